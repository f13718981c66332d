"""Vision -> text hand-off on the GPU: the vision actor's embeddings are written into the ``<image>`` slots of
the text embeddings, and the gradient of those slots is handed back.

Mirrors the text actor's side of the exchange in the reference, python/ray/text.py:
  * ``prepare_vision_embeddings``  text.py:860-872  (batch dimension, detached leaf that collects ``.grad``)
  * ``merge_vision_embeddings``    text.py:883-913  (placeholder mask, the three count / label guards with their
                                                     error messages, ``masked_scatter``)
  * ``extract_vision_grad``        text.py:1000-1019 (gradient of the leaf, batch dimension removed, detached copy)

One ranking kernel and one row-merge kernel replace the expanded boolean mask, three reductions with host
read-backs and ``masked_scatter``; the backward is one pass over the gradient.
"""

from __future__ import annotations

from typing import Optional

import torch

from . import _lib
from .ops import _p, _stream

IMAGE_TOKEN_ID = 151655  # text.py:884


def _int64_row(t: torch.Tensor) -> torch.Tensor:
    t = t.reshape(-1)
    return t if t.dtype == torch.int64 and t.is_contiguous() else t.to(torch.int64).contiguous()


class _Arrival:
    """Counts that a kernel on `stream` writes to pinned host memory, -1 until then.  They are seen there as soon as they arrive, some 10 us
    before an event behind the kernel would tell the host."""

    __slots__ = ("counts", "stream")

    def __init__(self, counts: torch.Tensor, stream: int):
        self.counts, self.stream = counts, stream

    def query(self) -> bool:
        return _lib.load().mvit_wait_host_values(self.counts.data_ptr(), self.counts.numel(), 0) == 0

    def _wait(self) -> None:
        # one call, which no signal handler ends early
        _lib.check(_lib.load().mvit_await_host_values(self.counts.data_ptr(), self.counts.numel(), self.stream), "mvit_await_host_values")

    def synchronize(self) -> None:
        """Returns or raises when the counts are there or the stream has nothing left that could write them."""
        try:
            self._wait()
        except BaseException:  # of a signal handler that ran before the call, too
            self._wait()
            raise


def _ranks(input_ids: torch.Tensor, labels: Optional[torch.Tensor], image_token_id: int):
    """(rank of every token, pinned counts, their arrival).  The pinned allocator does not know of the kernel that writes the
    counts: the caller holds them until they have arrived, on every way out."""
    ids = _int64_row(input_ids)
    lab = None
    if labels is not None:
        if labels.numel() != ids.numel():
            raise ValueError("labels and input_ids differ in size")
        lab = _int64_row(labels)
    n, stream = ids.numel(), _stream(ids)
    rank = torch.empty(n, dtype=torch.int32, device=ids.device)
    counts = torch.empty(2, dtype=torch.int64, pin_memory=True).fill_(-1)  # the kernel writes them where the host reads them
    try:
        rc = _lib.load().mvit_image_token_ranks(ids.data_ptr(), None if lab is None else lab.data_ptr(), n, image_token_id, -100,
                                                rank.data_ptr(), None, counts.data_ptr(), stream)
        _lib.check(rc, "mvit_image_token_ranks")
        return rank, counts, _Arrival(counts, stream)
    except BaseException:
        torch.cuda.synchronize(ids.device)
        raise


class _MergeRowsFn(torch.autograd.Function):
    """Row merge over the last dimension of embeds [..., O] and vision [..., O]; the gradients keep those shapes."""

    @staticmethod
    def forward(ctx, embeds, vision, rank):
        embeds, vision = embeds.contiguous(), vision.contiguous()
        hidden = embeds.shape[-1]
        n_vision = vision.numel() // hidden
        out = torch.empty_like(embeds)
        rc = _lib.load().mvit_merge_rows(embeds.data_ptr(), vision.data_ptr(), rank.data_ptr(), out.data_ptr(), rank.numel(), n_vision,
                                         hidden * embeds.element_size(), _stream(embeds))
        _lib.check(rc, "mvit_merge_rows")
        ctx.save_for_backward(rank)
        ctx.vision_shape = vision.shape
        return out

    @staticmethod
    def backward(ctx, grad):
        (rank,) = ctx.saved_tensors
        grad = grad.contiguous()
        hidden = grad.shape[-1]
        d_embeds = torch.empty_like(grad) if ctx.needs_input_grad[0] else None
        d_vision = torch.empty(ctx.vision_shape, dtype=grad.dtype, device=grad.device) if ctx.needs_input_grad[1] else None
        rc = _lib.load().mvit_split_rows(grad.data_ptr(), rank.data_ptr(), _p(d_embeds), _p(d_vision), rank.numel(),
                                         ctx.vision_shape.numel() // hidden, hidden * grad.element_size(), _stream(grad))
        _lib.check(rc, "mvit_split_rows")
        return d_embeds, d_vision, None


def prepare_vision_embeddings(vision_embeddings: torch.Tensor) -> torch.Tensor:
    """[M, O] or [B, M, O] from the vision actor -> a detached leaf [B, M, O] that collects ``.grad`` (text.py:860-872)."""
    if vision_embeddings.dim() == 2:
        vision_embeddings = vision_embeddings.unsqueeze(0)
    vision_embeddings = vision_embeddings.detach().clone().requires_grad_(True)
    vision_embeddings.retain_grad()
    return vision_embeddings


def merge_vision_embeddings(inputs_embeds: torch.Tensor, input_ids: torch.Tensor, vision_embeddings: torch.Tensor,
                            labels: Optional[torch.Tensor] = None, image_token_id: int = IMAGE_TOKEN_ID, rank: int = 0) -> torch.Tensor:
    """``inputs_embeds`` [B, T, O] with the rows at ``input_ids == image_token_id`` replaced, in order, by the rows of
    ``vision_embeddings`` ([*, O]); differentiable in both.  Raises the reference's RuntimeErrors when there is no
    placeholder, when the counts differ, or when a placeholder position carries a label other than -100."""
    if not inputs_embeds.is_cuda:
        raise RuntimeError("merge_vision_embeddings needs tensors on the GPU; there is no CPU path")
    if tuple(inputs_embeds.shape[:-1]) != tuple(input_ids.shape):
        raise ValueError(f"inputs_embeds {tuple(inputs_embeds.shape)} does not match input_ids {tuple(input_ids.shape)}")
    hidden = inputs_embeds.shape[-1]
    n_vision = vision_embeddings.numel() // hidden if hidden else 0
    if vision_embeddings.shape[-1] != hidden or vision_embeddings.dtype != inputs_embeds.dtype or vision_embeddings.device != inputs_embeds.device:
        raise ValueError("vision embeddings must share hidden size, dtype and device with inputs_embeds")
    ranks, counts, ready = _ranks(input_ids, labels, image_token_id)
    # the merge is queued before the host waits for the counts: it stays inside its arrays whatever they are, and its result
    # is dropped when one of the checks below refuses the call
    try:
        merged = _MergeRowsFn.apply(inputs_embeds, vision_embeddings, ranks)
    finally:  # also when the merge cannot be allocated: the counts must not go back to the allocator while the kernel may write them
        ready.synchronize()  # the one host wait (the reference has three)
    n_image, n_bad = counts.tolist()
    if n_image == 0:
        raise RuntimeError(
            f"[r{rank}] No <image> tokens (ID={image_token_id}) found in input_ids! "
            f"This likely means modality filter is wrong. input_ids shape: {input_ids.shape}")
    if n_vision != n_image:
        raise RuntimeError(
            f"[r{rank}] Mismatch: {n_vision} vision embeddings but "
            f"{n_image} <image> tokens in input_ids! "
            f"Vision and text trainers are out of sync.")
    if n_bad:
        raise RuntimeError(
            f"[r{rank}] Labels should be -100 at <image> positions, but found {n_bad} "
            f"positions with other values. This indicates incorrect label preprocessing.")
    return merged


def extract_vision_grad(vision_embeddings: Optional[torch.Tensor], rank: int = 0) -> torch.Tensor:
    """The gradient to send back to the vision actor (text.py:1000-1019): ``.grad`` of the leaf made by
    ``prepare_vision_embeddings``, without a batch dimension of one, as a detached copy."""
    if vision_embeddings is None or vision_embeddings.grad is None:
        raise RuntimeError(
            f"[r{rank}] vision_embeddings or its gradient is None! "
            f"This should not happen - check that vision_embeddings.requires_grad=True in forward.")
    grad = vision_embeddings.grad
    if grad.dim() == 3 and grad.shape[0] == 1:
        grad = grad.squeeze(0)
    return grad.detach().clone()
