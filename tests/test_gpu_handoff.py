"""Parity of the vision -> text hand-off kernels (through the C ABI) against the CPU oracle: index / copy work,
bit-exact; error behaviour as python/ray/text.py:883-910 and :1000-1007."""

import numpy as np
import pytest
import torch

from oracle import handoff_oracle as ho

pytestmark = pytest.mark.gpu
DEV = "cuda:0"
IMG = ho.IMAGE_TOKEN_ID


def _announce(msg):
    print(f"[case] {msg}", flush=True)


def _case(seed, B, T, frac, hidden, dtype):
    g = torch.Generator().manual_seed(seed)
    ids = torch.randint(0, 1000, (B, T), generator=g)
    ids[torch.rand(B, T, generator=g) < frac] = IMG
    if int((ids == IMG).sum()) == 0:
        ids[0, T // 2] = IMG
    n = int((ids == IMG).sum())
    mk = lambda *s: torch.randn(*s, generator=g).to(dtype)
    return ids, mk(B, T, hidden), mk(n, hidden), mk(B, T, hidden)


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("B,T,frac,hidden", [(1, 4096, 0.6, 3584), (3, 1000, 0.3, 256), (2, 77, 1.0, 40), (1, 5000, 0.001, 64),
                                             (1, 1, 1.0, 8), (2, 1500, 0.5, 6), (1, 333, 0.4, 7)])
def test_merge_and_backward_bit_exact(dtype, B, T, frac, hidden):
    from mi355_vit.handoff import extract_vision_grad, merge_vision_embeddings, prepare_vision_embeddings

    _announce(f"handoff {dtype} B={B} T={T} frac={frac} hidden={hidden}")
    ids, emb, vis, gout = _case(1, B, T, frac, hidden, dtype)
    labels = torch.randint(0, 1000, (B, T))
    labels[ids == IMG] = -100
    e = emb.to(DEV).requires_grad_(True)
    leaf = prepare_vision_embeddings(vis.to(DEV))
    assert leaf.shape == (1, vis.shape[0], hidden) and leaf.is_leaf and leaf.requires_grad
    out = merge_vision_embeddings(e, ids.to(DEV), leaf, labels.to(DEV))
    out.backward(gout.to(DEV))
    as_np = lambda t: t.detach().cpu().float().numpy()
    assert np.array_equal(as_np(out), ho.merge(as_np(emb), ids.numpy(), as_np(vis), labels.numpy()))
    d_e, d_v = ho.merge_backward(as_np(gout), ids.numpy())
    assert np.array_equal(as_np(e.grad), d_e)
    sent = extract_vision_grad(leaf)
    assert sent.shape == (vis.shape[0], hidden) and sent.dtype == dtype and np.array_equal(as_np(sent), d_v)
    # and against the reference's own call on the same device
    ref = emb.to(DEV).masked_scatter((ids.to(DEV) == IMG).unsqueeze(-1).expand(B, T, hidden), vis.to(DEV))
    assert torch.equal(out.detach(), ref)


@pytest.mark.parametrize("n", [0, 1, 63, 64, 511, 512, 513, 8191, 8192, 8193, 16384, 20001])
@pytest.mark.parametrize("with_labels", [True, False])
def test_ranks_over_the_edges_of_waves_and_spans(n, with_labels):
    """A wave takes 512 tokens, the work-group 8,192 at a time: ranks, positions and both counts are exact around those edges."""
    from mi355_vit import _lib

    _announce(f"image token ranks n={n} labels={with_labels}")
    g = torch.Generator().manual_seed(n)
    ids, labels = torch.randint(0, 3, (n,), generator=g), torch.where(torch.rand(n, generator=g) < 0.7, -100, 5)
    dev = [ids.to(DEV), labels.to(DEV)]
    rank = torch.full((n + 8,), -7, dtype=torch.int32, device=DEV)
    positions = torch.full((n + 8,), -7, dtype=torch.int64, device=DEV)
    counts = torch.full((2,), -7, dtype=torch.int64, device=DEV)
    rc = _lib.load().mvit_image_token_ranks(dev[0].data_ptr(), dev[1].data_ptr() if with_labels else None, n, 1, -100, rank.data_ptr(),
                                            positions.data_ptr(), counts.data_ptr(), torch.cuda.current_stream().cuda_stream)
    if n == 0 and rc != 0:  # nothing to rank is refused, or counts nothing
        return
    assert rc == 0
    img = ids == 1
    want = torch.where(img, torch.cumsum(img, 0) - 1, -1)
    assert torch.equal(rank[:n].cpu().long(), want) and bool((rank[n:] == -7).all())
    at = img.nonzero().flatten()
    assert torch.equal(positions[: at.numel()].cpu(), at) and bool((positions[at.numel():] == -7).all())
    assert counts.tolist() == [at.numel(), int((img & (labels != -100)).sum()) if with_labels else 0]


def test_guards_raise_like_the_reference():
    from mi355_vit.handoff import extract_vision_grad, merge_vision_embeddings

    ids = torch.tensor([[7, IMG, 3, IMG]], device=DEV)
    emb = torch.zeros(1, 4, 8, device=DEV)
    vis = torch.ones(2, 8, device=DEV)
    with pytest.raises(RuntimeError, match=r"\[r2\] No <image> tokens \(ID=151655\) found in input_ids!"):
        merge_vision_embeddings(emb, torch.tensor([[1, 2, 3, 4]], device=DEV), vis, rank=2)
    with pytest.raises(RuntimeError, match=r"Mismatch: 3 vision embeddings but 2 <image> tokens in input_ids!"):
        merge_vision_embeddings(emb, ids, torch.ones(3, 8, device=DEV))
    with pytest.raises(RuntimeError, match=r"Labels should be -100 at <image> positions, but found 1 positions"):
        merge_vision_embeddings(emb, ids, vis, labels=torch.tensor([[5, -100, 6, 9]], device=DEV))
    with pytest.raises(RuntimeError, match="vision_embeddings or its gradient is None"):
        extract_vision_grad(None)
    with pytest.raises(RuntimeError, match="no CPU path"):
        merge_vision_embeddings(emb.cpu(), ids.cpu(), vis.cpu())
    out = merge_vision_embeddings(emb, ids, vis, labels=torch.tensor([[5, -100, 6, -100]], device=DEV))
    assert out[0, :, 0].tolist() == [0.0, 1.0, 0.0, 1.0]


def test_a_merge_that_fails_still_waits_for_the_counts(monkeypatch):
    """The ranking kernel writes the counts in pinned host memory: they are not given back before it has run."""
    from mi355_vit import handoff

    taken = []
    ranks = handoff._ranks

    def spy(*args):
        out = ranks(*args)
        taken.append(out[2])
        return out

    class Fails:
        @staticmethod
        def apply(*args):
            torch.cuda._sleep(1 << 20)  # work behind the ranking kernel: the wait is for the counts, not for the stream
            raise torch.OutOfMemoryError("no room for the merged rows")

    monkeypatch.setattr(handoff, "_ranks", spy)
    monkeypatch.setattr(handoff, "_MergeRowsFn", Fails)
    ids = torch.randint(0, 1000, (1, 200000), device=DEV)
    emb = torch.zeros(1, ids.shape[1], 8, device=DEV)
    torch.cuda.synchronize()
    torch.cuda._sleep(1 << 26)  # some 30 ms in front of the ranking kernel
    with pytest.raises(torch.OutOfMemoryError):
        handoff.merge_vision_embeddings(emb, ids, torch.zeros(2, 8, device=DEV))
    assert len(taken) == 1 and taken[0].query()


def test_the_wait_behind_queued_work_is_one_call(monkeypatch):
    """The counts arrive long after the merge has been queued: the host waits for them without sleeping in between, and they are right."""
    import time

    from mi355_vit.handoff import merge_vision_embeddings

    _announce("hand-off behind queued work")

    def sleeps(seconds):
        raise AssertionError("the host slept while it waited")

    monkeypatch.setattr(time, "sleep", sleeps)
    ids = torch.full((1, 40), 11, device=DEV)
    ids[0, 3:8] = IMG
    emb, vis = torch.randn(1, 40, 64, device=DEV), torch.randn(5, 64, device=DEV)
    merge_vision_embeddings(emb, ids, vis)
    torch.cuda._sleep(1 << 25)  # some 15 ms in front of the ranking kernel
    got = merge_vision_embeddings(emb, ids, vis)
    assert torch.equal(got[0, 3:8], vis) and torch.equal(got[0, 8:], emb[0, 8:])
    torch.cuda._sleep(1 << 25)
    with pytest.raises(RuntimeError, match="4 vision embeddings but 5 <image> tokens"):
        merge_vision_embeddings(emb, ids, vis[:4])


def test_tower_output_feeds_the_handoff():
    """End of the path: the tower's [M, O] output goes into the placeholders and its gradient comes back unchanged
    in shape and order (the vision actor's backward_step accepts the 2-D gradient)."""
    from mi355_vit.config import Qwen2_5_VLVisionConfig
    from mi355_vit.handoff import extract_vision_grad, merge_vision_embeddings, prepare_vision_embeddings
    from mi355_vit.modeling import Qwen2_5_VisionTransformerPretrainedModel

    torch.manual_seed(0)
    kw = dict(depth=2, hidden_size=256, intermediate_size=300, num_heads=8, out_hidden_size=128, window_size=56, fullatt_block_indexes=[1])
    model = Qwen2_5_VisionTransformerPretrainedModel(Qwen2_5_VLVisionConfig(**kw)).to(torch.bfloat16).to(DEV).train()
    grid = torch.tensor([[1, 16, 16], [1, 8, 24]])
    S = int((grid[:, 0] * grid[:, 1] * grid[:, 2]).sum())
    emb = model(torch.randn(S, 1176, device=DEV, dtype=torch.bfloat16), grid.to(DEV))
    M = S // 4
    ids = torch.full((1, M + 20), 11, device=DEV)
    ids[0, 5 : 5 + M] = IMG
    leaf = prepare_vision_embeddings(emb)
    text = torch.randn(1, M + 20, 128, device=DEV, dtype=torch.bfloat16)
    merged = merge_vision_embeddings(text, ids, leaf)
    assert torch.equal(merged[0, 5 : 5 + M], emb.detach()) and torch.equal(merged[0, :5], text[0, :5])
    (merged.float() ** 2).sum().backward()
    g = extract_vision_grad(leaf)
    assert g.shape == emb.shape and torch.equal(g, (2 * emb.detach().float()).to(torch.bfloat16))
    emb.backward(g)
    assert all(p.grad is not None for p in model.parameters())
