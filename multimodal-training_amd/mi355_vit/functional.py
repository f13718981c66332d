"""Autograd functions of the vision tower.  Each one is a fixed sequence of C-ABI kernel launches with a
hand-written backward (no autograd graph inside), so a transformer block is one node of PyTorch's graph.

Reference spans (python/models/qwen2_5_vl/modeling_qwen2_5_vl.py):
  VisionBlockFn   Qwen2_5_VLVisionBlock.forward :776-792 with _forward_standard :385-472 and the MLP :203-204
  PatchEmbedFn    Qwen2_5_VisionPatchEmbed.forward :225-231
  PermuteRowsFn   window reorder :934-937 and its inverse :1067-1068
  MergerFn        Qwen2_5_VLPatchMerger.forward :260-262
"""

from __future__ import annotations

import ctypes
import math
import os
from dataclasses import dataclass
from typing import Dict, List, Optional, Tuple

import torch

from . import _lib, ops

E = _lib


def round_up(v: int, m: int) -> int:
    return (v + m - 1) // m * m


def padded_inner(inner: int) -> int:
    """Columns that a block's gate, up and hidden activations are laid out in: whole 128-byte cache lines of bf16 for MLPs wide
    enough that the padding is small, else the 8 columns that 16-byte accesses need.  Rows of 3,424 columns (3,420 rounded up
    to 8) begin in the middle of a line every other time, and a K tile of the down projection, 128 bytes of each row, then
    touches two (us at 4,096 / 16,384 / 65,536 rows: 53 / 162 / 479 with 3,424 columns, 43 / 138 / 460 with 3,456; SwiGLU
    backward 61 / 225 / 779 and 59 / 219 / 760; the products that grow with the padding, gate/up forward and input gradient,
    take 1 % more)."""
    return round_up(inner, 64 if inner >= 512 else 8)


@dataclass
class BlockWeights:
    """Compute-dtype operands of one block, laid out for the fused GEMMs.

    wqkv [3C, C] / bqkv [3C]         q, k, v stacked
    wgu  [2*Ipad, C] / bgu [2*Ipad]  gate rows [0, I), up rows [Ipad, Ipad+I); padding rows are zero
    wdown [C, Ipad] / bdown [C]      padding columns are zero
    """

    norm1: torch.Tensor
    norm2: torch.Tensor
    wqkv: torch.Tensor
    bqkv: torch.Tensor
    wproj: torch.Tensor
    bproj: torch.Tensor
    wgu: torch.Tensor
    bgu: torch.Tensor
    wdown: torch.Tensor
    bdown: torch.Tensor
    C: int
    I: int
    Ipad: int
    alias: bool = False  # norm1 / norm2 / wproj / bproj / bdown are the parameters themselves (same dtype), not copies
    args: Optional[tuple] = None  # (what the struct was filled from, the struct), see block_args

    def block_args(self) -> Optional["_lib.BlockArgs"]:
        """The weight operands as the C calls take them; None: not laid out for them.  Layouts, types and addresses are looked at on
        every call (3.2 us), as the call-by-call wrappers do; the struct that is kept saves filling another (1.2 us) and is taken
        only while the operands are what it was filled from.  Another thread may run the same model: `args` is set to a struct that
        is complete, and not written again."""
        w = (self.norm1, self.norm2, self.wqkv, self.bqkv, self.wproj, self.bproj, self.wgu, self.bgu, self.wdown, self.bdown)
        dtype = self.wqkv.dtype
        if dtype not in ops._DT:
            return None
        source = [dtype, self.C, self.I, self.Ipad]
        for t in w:
            if t.dtype is not dtype or not t.is_contiguous():
                return None
            source.append(t.data_ptr())
        kept = self.args
        if kept is not None and kept[0] == source:
            return kept[1]
        a = _lib.BlockArgs()
        a.dtype, a.C, a.I, a.Ipad = ops._DT[dtype], self.C, self.I, self.Ipad
        a.norm1, a.norm2, a.wqkv, a.bqkv, a.wproj, a.bproj, a.wgu, a.bgu, a.wdown, a.bdown = source[4:]
        self.args = (source, a)
        return a

    def __getstate__(self):  # addresses are not copied or saved with the operands
        return dict(self.__dict__, args=None)


# order of the parameter tensors handed to VisionBlockFn
LOG2E = 1.4426950408889634  # log2(e): the attention kernels work in base-2 exponentials

BLOCK_PARAM_ORDER = (
    "norm1.weight", "norm2.weight",
    "attn.q_proj.weight", "attn.q_proj.bias", "attn.k_proj.weight", "attn.k_proj.bias",
    "attn.v_proj.weight", "attn.v_proj.bias", "attn.proj.weight", "attn.proj.bias",
    "mlp.gate_proj.weight", "mlp.gate_proj.bias", "mlp.up_proj.weight", "mlp.up_proj.bias",
    "mlp.down_proj.weight", "mlp.down_proj.bias",
)


def pack_block_weights(params: List[torch.Tensor], dtype: torch.dtype, into: Optional[BlockWeights]) -> BlockWeights:
    """(Re)fill the packed operands from the 16 parameters (cast to `dtype` on the way).

    Operands that are a single parameter (norm weights, proj, the down bias) are the parameter itself when it
    already has the compute dtype; the fused ones (q|k|v, gate|up, the padded down weight) are copies.  Every copy is
    declared to the optimizer (``optim.attach_shadow``): ``FusedAdam.step`` writes updated values into it directly, so
    an optimizer step never forces a re-pack; any other in-place change of a parameter bumps its version counter and
    the owner of the pack calls this function again."""
    from .optim import attach_shadow

    (n1, n2, wq, bq, wk, bk, wv, bv, wp, bp, wg, bg, wu, bu, wd, bd) = params
    C = wq.shape[1]
    I = wg.shape[0]
    Ipad = padded_inner(I)
    dev = wq.device
    alias = all(p.dtype == dtype and p.is_contiguous() for p in (n1, n2, wp, bp, bd))
    if into is None or into.wqkv.dtype != dtype or into.wqkv.device != dev or into.alias != alias:
        z = lambda *s: torch.zeros(*s, dtype=dtype, device=dev)  # noqa: E731
        e = (lambda *s: None) if alias else z  # noqa: E731
        into = BlockWeights(e(1, C), e(1, C), z(3 * C, C), z(1, 3 * C), e(C, C), e(1, C), z(2 * Ipad, C), z(1, 2 * Ipad),
                            z(C, Ipad), e(1, C), C, I, Ipad, alias)
    cp = ops.cast2d
    v = lambda t: t.detach().view(1, -1)  # noqa: E731

    def fill(param: torch.Tensor, dst: torch.Tensor) -> None:
        cp(param.detach() if param.dim() == 2 else v(param), dst)
        attach_shadow(param, dst if param.dim() == 2 else dst.view(-1))

    if alias:
        into.norm1, into.norm2, into.wproj, into.bproj, into.bdown = v(n1), v(n2), wp.detach(), v(bp), v(bd)
        for param in (n1, n2, wp, bp, bd):
            param._mvit_shadow = None  # read in place: nothing to keep in step
    else:
        for param, dst in ((n1, into.norm1), (n2, into.norm2), (wp, into.wproj), (bp, into.bproj), (bd, into.bdown)):
            fill(param, dst)
    for j, (w, b) in enumerate(((wq, bq), (wk, bk), (wv, bv))):
        fill(w, into.wqkv[j * C : (j + 1) * C])
        fill(b, into.bqkv[:, j * C : (j + 1) * C])
    for j, (w, b) in enumerate(((wg, bg), (wu, bu))):
        fill(w, into.wgu[j * Ipad : j * Ipad + I])
        fill(b, into.bgu[:, j * Ipad : j * Ipad + I])
    fill(wd, into.wdown[:, :I])
    return into


@dataclass
class AttnGeometry:
    """Per-layer attention layout: device cu_seqlens, the longest segment, head counts, rotary tables."""

    cu: torch.Tensor
    max_seqlen: int
    nheads: int
    head_dim: int
    cos: torch.Tensor  # fp32 [S, head_dim]
    sin: torch.Tensor
    order: Optional[torch.Tensor] = None  # device int32 permutation of the segments, longest first (ops.segment_order)

    def block_call_ok(self, x: torch.Tensor) -> bool:
        """What the call-by-call wrappers check launch by launch of the geometry, once for the block."""
        S, hd = x.shape[0], self.head_dim
        return (self.cu.dtype == torch.int32 and self.cu.is_contiguous() and self.cu.device == x.device
                and all(t.dtype == torch.float32 and tuple(t.shape) == (S, hd) and t.is_contiguous() for t in (self.cos, self.sin))
                and (self.order is None or (self.order.dtype == torch.int32 and self.order.is_contiguous() and self.order.numel() == self.cu.numel() - 1)))


# One C call per block and direction (mvit_block_fwd / mvit_block_bwd) instead of one per kernel: the same steps on the
# same operands, issued from inside the library, where the weight gradients of a few rows are one launch.  MVIT_BLOCK_CALLS=0 keeps the call-by-call sequence below, which is
# also what runs while launches are being timed one by one (ops.set_trace) and for parameters of mixed gradient dtypes.
BLOCK_CALLS = os.environ.get("MVIT_BLOCK_CALLS", "1") != "0"
_join_events: dict = {}
_GRAD_DTYPES = (torch.bfloat16, torch.float32)  # one dtype for all of a block's gradients, as the C call writes them


def _block_args(x: torch.Tensor, W: BlockWeights, geo: AttnGeometry, eps: float) -> Optional["_lib.BlockArgs"]:
    """The arguments that a block's C calls share, or None where an operand is not laid out as their sequence assumes: what the
    call-by-call wrappers check launch by launch, once for the block."""
    weights = W.block_args()
    if (weights is None or not x.is_cuda or not x.is_contiguous() or x.shape[1] != W.C or geo.nheads * geo.head_dim != W.C
            or x.dtype != W.wqkv.dtype or not geo.block_call_ok(x)):
        return None
    a = _lib.BlockArgs.from_buffer_copy(weights)
    a.S, a.nheads, a.head_dim = x.shape[0], geo.nheads, geo.head_dim
    a.eps, a.q_lead_scale, a.attn_scale = eps, geo.head_dim**-0.5 * LOG2E, 1.0 / LOG2E
    a.n_seg, a.max_seqlen = geo.cu.shape[0] - 1, geo.max_seqlen
    a.cu, a.cos, a.sin = geo.cu.data_ptr(), geo.cos.data_ptr(), geo.sin.data_ptr()
    if geo.order is not None:
        a.seg_order = geo.order.data_ptr()
    a.x = x.data_ptr()
    return a


class _Buffers:
    """Pieces of one allocation, each at a 256-byte address: a block's saved activations, or the scratch of its backward.  At few
    rows an allocation per tensor costs the host more than the kernels cost the GPU."""

    __slots__ = ("buf", "at", "shapes", "dtypes")

    def __init__(self, device, shapes, dtypes):
        self.shapes, self.dtypes, self.at, end = shapes, dtypes, [], 0
        for shape, dtype in zip(shapes, dtypes):
            self.at.append(end)
            n = dtype.itemsize
            for d in shape:
                n *= d
            end += (n + 255) // 256 * 256
        self.buf = torch.empty(end, dtype=torch.uint8, device=device)

    def ptr(self, i: int) -> int:
        return self.buf.data_ptr() + self.at[i]

    def tensor(self, i: int) -> torch.Tensor:
        shape, dtype = self.shapes[i], self.dtypes[i]
        return self.buf[self.at[i] : self.at[i] + math.prod(shape) * dtype.itemsize].view(dtype).view(shape)


class _Saved:
    """What a one-call forward keeps for the backward, in the order (rstd1, n1, qkv, o, lse, x1, rstd2, n2, gu, h): addresses for the
    C call, tensors for whoever asks for one by position or for all of them."""

    __slots__ = ("buffers", "index", "attn")

    def __init__(self, buffers, index, attn):
        self.buffers, self.index, self.attn = buffers, index, attn  # index: position -> piece (None: not kept); attn: (o, lse) when they are tensors of their own

    def ptr(self, i: int):
        if self.attn is not None and i in (3, 4):
            return self.attn[i - 3].data_ptr()
        piece = self.index[i]
        return None if piece is None else self.buffers.ptr(piece)

    def __getitem__(self, i: int) -> Optional[torch.Tensor]:
        if self.attn is not None and i in (3, 4):
            return self.attn[i - 3]
        piece = self.index[i]
        return None if piece is None else self.buffers.tensor(piece)

    def __iter__(self):
        return (self[i] for i in range(10))


def _block_forward_one_call(a, x, W, geo, attn_out, for_backward, output):
    S, C = x.shape
    T, f32, Ipad = x.dtype, torch.float32, W.Ipad
    if attn_out is None and geo.max_seqlen > KEEP_ATTENTION_ABOVE:  # may outlive the rest
        attn_out, skip = (torch.empty_like(x), torch.empty(geo.nheads, S, dtype=f32, device=x.device)), 0
    else:
        skip = int(attn_out is not None)
    shapes, dtypes = [(S,), (S, C), (S, 3 * C), (S, C), (S,), (S, C), (S, Ipad)], [f32, T, T, T, f32, T, T]
    index = [0, 1, 2, None, None, 3, 4, 5, None, 6]
    if for_backward:
        index[8] = len(shapes)
        shapes.append((S, 2 * Ipad))
        dtypes.append(T)
    if attn_out is None:
        index[3], index[4] = len(shapes), len(shapes) + 1
        shapes += [(S, C), (geo.nheads, S)]
        dtypes += [T, f32]
    saved = _Saved(_Buffers(x.device, shapes, dtypes), index, attn_out)
    x2 = torch.empty_like(x) if output else None
    a.skip_attention = skip
    p = saved.ptr
    a.rstd1, a.n1, a.qkv, a.o, a.lse, a.x1, a.rstd2, a.n2, a.gu, a.h = p(0), p(1), p(2), p(3), p(4), p(5), p(6), p(7), p(8), p(9)
    if output:
        a.x2 = x2.data_ptr()
    _lib.check(_lib.load().mvit_block_fwd(ctypes.byref(a), ops._stream(x)), "mvit_block_fwd")
    return x2, saved


def _block_split_k(out_rows: int, out_cols: int, rows: int) -> int:
    """K slices of a block's weight gradient: those of a product beside the input-gradient chain, also where the second stream is
    switched off, so that the gradients are the same bits either way."""
    return ops.wgrad_split_k(out_rows, out_cols, rows, True)


def _block_backward_one_call(a, dx2, x, saved, W, G):
    S, Cc = x.shape
    I, Ipad = W.I, W.Ipad
    dev, T = x.device, x.dtype
    a.grad_dtype = ops._DT[G]
    if type(saved) is _Saved:
        p = saved.ptr
        a.rstd1, a.n1, a.qkv, a.o, a.lse, a.x1, a.rstd2, a.n2, a.gu, a.h = p(0), p(1), p(2), p(3), p(4), p(5), p(6), p(7), p(8), p(9)
    else:
        a.rstd1, a.n1, a.qkv, a.o, a.lse, a.x1, a.rstd2, a.n2, a.gu, a.h = (t.data_ptr() for t in saved)
    sk = _block_split_k
    a.split_k_down, a.split_k_gate_up, a.split_k_proj, a.split_k_qkv = sk(Cc, I, S), sk(2 * Ipad, Cc, S), sk(Cc, Cc, S), sk(3 * Cc, Cc, S)
    lib = _lib.load()
    nbytes = lib.mvit_block_bwd_workspace_bytes(ctypes.byref(a))
    scratch = _Buffers(dev, ((S, 2 * Ipad), (S, 3 * Cc), (S, Cc), (S, Cc), (nbytes,)), (T, T, T, T, torch.uint8))
    a.dgu, a.dqkv, a.dn, a.dx1, a.workspace = scratch.ptr(0), scratch.ptr(1), scratch.ptr(2), scratch.ptr(3), scratch.ptr(4)
    a.workspace_bytes = nbytes
    dx = torch.empty_like(x)
    a.dx2, a.dx = dx2.data_ptr(), dx.data_ptr()
    e = torch.empty
    g_n1, g_n2, g_bp, g_bd = e(Cc, dtype=G, device=dev), e(Cc, dtype=G, device=dev), e(Cc, dtype=G, device=dev), e(Cc, dtype=G, device=dev)
    g_wqkv, g_bqkv = e(3, Cc, Cc, dtype=G, device=dev), e(3, Cc, dtype=G, device=dev)
    g_wp, g_wgu, g_bgu, g_wd = e(Cc, Cc, dtype=G, device=dev), e(2, Ipad, Cc, dtype=G, device=dev), e(2, Ipad, dtype=G, device=dev), e(Cc, I, dtype=G, device=dev)
    a.g_norm1, a.g_norm2, a.g_wqkv, a.g_bqkv, a.g_wproj = g_n1.data_ptr(), g_n2.data_ptr(), g_wqkv.data_ptr(), g_bqkv.data_ptr(), g_wp.data_ptr()
    a.g_bproj, a.g_wgu, a.g_bgu, a.g_wdown, a.g_bdown = g_bp.data_ptr(), g_wgu.data_ptr(), g_bgu.data_ptr(), g_wd.data_ptr(), g_bd.data_ptr()
    side = ops.side_stream(dev)
    if side is not None:
        key = dev.index if dev.index is not None else torch.cuda.current_device()
        evs = _join_events.get(key)
        if evs is None:
            evs = [torch.cuda.Event() for _ in range(5)]
            for ev in evs:
                ev.record()  # an event object gets its handle with its first record
            _join_events[key] = evs
        a.side_stream = side.cuda_stream
        a.events[:] = [ev.cuda_event for ev in evs]
    _lib.check(lib.mvit_block_bwd(ctypes.byref(a), ops._stream(x)), "mvit_block_bwd")
    wq, wk, wv = g_wqkv.unbind(0)
    bq, bk, bv = g_bqkv.unbind(0)
    wg, wu = g_wgu[:, :I].unbind(0)
    bg, bu = g_bgu[:, :I].unbind(0)
    return dx, (g_n1, g_n2, wq, bq, wk, bk, wv, bv, g_wp, g_bp, wg, bg, wu, bu, g_wd, g_bd)


def _block_forward(x: torch.Tensor, W: BlockWeights, geo: AttnGeometry, eps: float,
                   attn_out: Optional[Tuple[torch.Tensor, torch.Tensor]] = None, *,
                   for_backward: bool = True, output: bool = True) -> Tuple[Optional[torch.Tensor], tuple]:
    """``attn_out`` = (o, lse) kept from an earlier run of the same block on the same input: the attention product is
    then not computed again (the recomputation of a checkpointed block).

    ``for_backward=False``: nothing but the block's output (and the attention output) will be used, so the gate / up
    pre-activations are not written (the first run of a checkpointed block).  ``output=False``: the block's output is
    not wanted, so the down projection is skipped (the re-run of a checkpointed block: the backward reads `h`, not
    `x2`)."""
    a = _block_args(x, W, geo, eps) if BLOCK_CALLS and ops._trace is None else None
    if a is not None:
        return _block_forward_one_call(a, x, W, geo, attn_out, for_backward, output)
    S, C = x.shape
    H, hd = geo.nheads, geo.head_dim
    n1, rstd1 = ops.rmsnorm_fwd(x, W.norm1.view(-1), eps)
    qkv = torch.empty(S, 3 * C, dtype=x.dtype, device=x.device)
    ops.gemm(n1, W.wqkv, qkv, epilogue=E.EPI_BIAS, bias=W.bqkv.view(-1))
    # q and k are the first 2*H heads of every row.  The queries leave the rotary pass multiplied by the softmax scale
    # in base-2 units (Q_SCALE), in the same fp32 -> storage rounding as the rotation; the attention kernels then get
    # scale = 1 / log2(e), for which their own pre-scaling of the queries is the identity.  Scores are computed from
    # operands rounded once, as in the reference (the kernels alone would round q * scale a second time).
    ops.rope_(qkv, geo.cos, geo.sin, 2 * H, hd, lead_heads=H, lead_scale=hd**-0.5 * LOG2E)
    if attn_out is None:
        o, lse = ops.attn_fwd(qkv[:, :C], qkv[:, C : 2 * C], qkv[:, 2 * C :], geo.cu, geo.max_seqlen, H, hd, 1.0 / LOG2E,
                              seg_order=geo.order)
    else:
        o, lse = attn_out
    x1 = torch.empty_like(x)
    ops.gemm(o, W.wproj, x1, epilogue=E.EPI_BIAS_RES, bias=W.bproj.view(-1), residual=x)
    n2, rstd2 = ops.rmsnorm_fwd(x1, W.norm2.view(-1), eps)
    gu = torch.empty(S, 2 * W.Ipad, dtype=x.dtype, device=x.device) if for_backward else None
    h = torch.empty(S, W.Ipad, dtype=x.dtype, device=x.device)
    bgu = W.bgu.view(-1)
    ops.gemm(n2, W.wgu[: W.Ipad], h, epilogue=E.EPI_SWIGLU, b2=W.wgu[W.Ipad :], bias=bgu[: W.Ipad], bias2=bgu[W.Ipad :],
             aux=gu, aux_off=W.Ipad)
    x2 = None
    if output:
        x2 = torch.empty_like(x)
        ops.gemm(h, W.wdown, x2, epilogue=E.EPI_BIAS_RES, bias=W.bdown.view(-1), residual=x1)
    return x2, (rstd1, n1, qkv, o, lse, x1, rstd2, n2, gu, h)


def _block_backward(dx2: torch.Tensor, x: torch.Tensor, saved: tuple, W: BlockWeights, geo: AttnGeometry, gdt):
    """Returns (dx, grads in BLOCK_PARAM_ORDER).  gdt: the gradients' dtype, or a map parameter name -> gradient dtype."""
    dx2 = dx2.contiguous()
    a = _block_args(x, W, geo, 0.0) if BLOCK_CALLS and ops._trace is None and gdt in _GRAD_DTYPES and dx2.dtype == x.dtype else None
    if a is not None:
        return _block_backward_one_call(a, dx2, x, saved, W, gdt)
    if not isinstance(gdt, dict):
        gdt = dict.fromkeys(BLOCK_PARAM_ORDER, gdt)
    rstd1, n1, qkv, o, lse, x1, rstd2, n2, gu, h = saved
    S, C = x.shape
    H, hd = geo.nheads, geo.head_dim
    I, Ipad = W.I, W.Ipad
    dev = x.device
    main = torch.cuda.current_stream(dev)
    side = ops.side_stream(dev)

    def off_chain(fn):
        # work that feeds nothing else in this block (weight and bias gradients) runs on the second stream, after
        # the point its inputs are complete on the main stream, and is joined before the gradients are handed back;
        # one event and one stream switch per point serve the bias and the weight gradient that start there
        if side is None:
            return fn()
        ev = torch.cuda.Event()
        ev.record(main)
        with torch.cuda.stream(side):
            side.wait_event(ev)
            return fn()

    beside = side is not None

    def weight_grad(dy, act, out, bias_dtype, n=None):
        return ops.weight_grad(dy, act, out, bias_dtype, n=n, split_k=_block_split_k(out.shape[0], out.shape[1], S), overlapped=beside)

    # ---- MLP: x2 = x1 + down(silu(g) * u)
    g_wd = torch.empty(C, I, dtype=gdt["mlp.down_proj.weight"], device=dev)
    g_bd = off_chain(lambda: weight_grad(dx2, h, g_wd, gdt["mlp.down_proj.bias"], n=I))
    dgu = torch.empty(S, 2 * Ipad, dtype=x.dtype, device=dev)
    # the bf16 epilogue also hands back per-tile column sums of dgu, of its fp32 values: the gate / up bias gradient
    fused = x.dtype == torch.bfloat16
    part = torch.empty(-(-S // ops.swiglu_bwd_colsum_rows(S, Ipad, C)), 2 * Ipad, dtype=torch.float32, device=dev) if fused else None
    ops.gemm(dx2, W.wdown, dgu, trans_b=True, epilogue=E.EPI_SWIGLU_BWD, residual=gu, aux_off=Ipad, colsum_partial=part, overlapped=beside)
    g_wgu = torch.empty(2 * Ipad, C, dtype=gdt["mlp.gate_proj.weight"], device=dev)
    b_gu = gdt["mlp.gate_proj.bias"]
    g_bgu = off_chain(lambda: (ops.reduce_partials(part, b_gu), weight_grad(dgu, n2, g_wgu, None))[0] if fused else weight_grad(dgu, n2, g_wgu, b_gu))
    dn2 = torch.empty_like(x)
    ops.gemm(dgu, W.wgu, dn2, trans_b=True, overlapped=beside)
    dx1, g_n2 = ops.rmsnorm_bwd(dn2, x1, W.norm2.view(-1), rstd2, dx_add=dx2, w_grad_dtype=gdt["norm2.weight"])

    # ---- attention: x1 = x + proj(attn(rope(qkv(norm1(x)))))
    g_wp = torch.empty(C, C, dtype=gdt["attn.proj.weight"], device=dev)
    g_bp = off_chain(lambda: weight_grad(dx1, o, g_wp, gdt["attn.proj.bias"]))
    d_o = dn2  # reuse the buffer
    ops.gemm(dx1, W.wproj, d_o, trans_b=True, overlapped=beside)
    dqkv = torch.empty_like(qkv)
    ops.attn_bwd(qkv[:, :C], qkv[:, C : 2 * C], qkv[:, 2 * C :], o, d_o, lse, geo.cu, geo.max_seqlen, H, hd, 1.0 / LOG2E,
                 dqkv[:, :C], dqkv[:, C : 2 * C], dqkv[:, 2 * C :], seg_order=geo.order)
    # dq arrives as the gradient with respect to the scaled, rotated queries: the same factor on the way back
    ops.rope_(dqkv, geo.cos, geo.sin, 2 * H, hd, backward=True, lead_heads=H, lead_scale=hd**-0.5 * LOG2E)
    g_wqkv = torch.empty(3 * C, C, dtype=gdt["attn.q_proj.weight"], device=dev)
    g_bqkv = off_chain(lambda: weight_grad(dqkv, n1, g_wqkv, gdt["attn.q_proj.bias"]))
    dn1 = d_o
    ops.gemm(dqkv, W.wqkv, dn1, trans_b=True, overlapped=beside)
    dx, g_n1 = ops.rmsnorm_bwd(dn1, x, W.norm1.view(-1), rstd1, dx_add=dx1, w_grad_dtype=gdt["norm1.weight"])
    if side is not None:
        main.wait_stream(side)

    grads = (
        g_n1, g_n2,
        g_wqkv[:C], g_bqkv[:C], g_wqkv[C : 2 * C], g_bqkv[C : 2 * C], g_wqkv[2 * C :], g_bqkv[2 * C :],
        g_wp, g_bp,
        g_wgu[:I], g_bgu[:I], g_wgu[Ipad : Ipad + I], g_bgu[Ipad : Ipad + I],
        g_wd, g_bd,
    )
    return dx, grads


KEEP_ATTENTION_ABOVE = 64  # segments longer than this (the full-attention layers) keep their attention output when checkpointed


class VisionBlockFn(torch.autograd.Function):
    """One transformer block.  With `checkpoint` only the block input is kept and the forward is re-run in
    the backward (the native counterpart of torch.utils.checkpoint around the block, [tf] modeling_layers.py:79).
    A full-attention layer also keeps its attention output and log-sum-exp ([S, C] + [H, S] fp32: 164 MiB at 65,536
    patches), so the re-run skips the one product whose cost grows with the square of the segment length; the values
    it would recompute are bit-identical, hence so are the gradients."""

    @staticmethod
    def forward(ctx, x, holder, geo: AttnGeometry, eps: float, checkpoint: bool, *params):
        W = holder.packed(x.dtype)
        x = x.contiguous()
        differentiated = any(ctx.needs_input_grad)  # False under torch.no_grad() and for frozen inputs and weights
        x2, saved = _block_forward(x, W, geo, eps, for_backward=differentiated and not checkpoint)
        if not differentiated:
            return x2
        ctx.holder, ctx.geo, ctx.eps, ctx.checkpoint = holder, geo, eps, checkpoint
        G = params[0].dtype
        ctx.gdt = G if all([p.dtype is G for p in params]) else {name: p.dtype for name, p in zip(BLOCK_PARAM_ORDER, params)}
        ctx.x = x
        ctx.saved = None if checkpoint else saved
        ctx.attn_out = (saved[3], saved[4]) if checkpoint and geo.max_seqlen > KEEP_ATTENTION_ABOVE else None
        return x2

    @staticmethod
    def backward(ctx, dx2):
        x, geo = ctx.x, ctx.geo
        W = ctx.holder.packed(x.dtype)
        saved = ctx.saved
        if saved is None:
            ops.recomputing = True
            try:
                _, saved = _block_forward(x, W, geo, ctx.eps, ctx.attn_out, output=False)
            finally:
                ops.recomputing = False
        dx, grads = _block_backward(dx2, x, saved, W, geo, ctx.gdt)
        ctx.saved = None
        ctx.x = None
        ctx.attn_out = None
        return (dx, None, None, None, None) + tuple(grads)


class PatchEmbedFn(torch.autograd.Function):
    """[S, 1176] pixels x Conv3d weight viewed as [C, 1176]: a GEMM without bias."""

    @staticmethod
    def forward(ctx, pixels, weight, compute_dtype):
        w2 = weight.detach().reshape(weight.shape[0], -1)
        K = w2.shape[1]
        px = pixels.detach().reshape(-1, K)
        if px.dtype != compute_dtype or not px.is_contiguous():
            px = ops.cast2d(px if px.stride(1) == 1 else px.contiguous(), torch.empty(px.shape, dtype=compute_dtype, device=px.device))
        if w2.dtype != compute_dtype:
            w2 = ops.cast2d(w2, torch.empty(w2.shape, dtype=compute_dtype, device=w2.device))
        out = torch.empty(px.shape[0], w2.shape[0], dtype=compute_dtype, device=px.device)
        ops.gemm(px, w2, out)
        ctx.px, ctx.wshape, ctx.wdtype = px, weight.shape, weight.dtype
        return out

    @staticmethod
    def backward(ctx, dout):
        px = ctx.px
        gw = torch.empty(dout.shape[1], px.shape[1], dtype=ctx.wdtype, device=px.device)
        ops.gemm(dout.contiguous(), px, gw, trans_a=True, trans_b=True, split_k=ops.wgrad_split_k(gw.shape[0], gw.shape[1], px.shape[0]))
        return None, gw.view(ctx.wshape), None


class PatchEmbedFramesFn(torch.autograd.Function):
    """The patch embedding straight from decoded uint8 frames (bf16 compute): the forward makes the rows of
    ``pixel_values`` inside the GEMM and never writes them; the weight gradient needs them as a matrix, so the backward
    writes them once (``patchify``) just before its GEMM and drops them again."""

    @staticmethod
    def forward(ctx, weight, out_dtype, *frames):
        from . import pixels

        out, _ = pixels.patch_embed_frames(frames, pixels.pack_patch_embed_weight(weight), dtype=out_dtype)
        ctx.frames, ctx.wshape, ctx.wdtype = frames, weight.shape, weight.dtype
        return out

    @staticmethod
    def backward(ctx, dout):
        from . import pixels

        px, _ = pixels.patchify(ctx.frames, dtype=torch.bfloat16)
        dy = dout.contiguous()
        if dy.dtype != torch.bfloat16:
            dy = ops.cast2d(dy, torch.empty(dy.shape, dtype=torch.bfloat16, device=dy.device))
        gw = torch.empty(dy.shape[1], px.shape[1], dtype=ctx.wdtype, device=px.device)
        ops.gemm(dy, px, gw, trans_a=True, trans_b=True, split_k=ops.wgrad_split_k(gw.shape[0], gw.shape[1], px.shape[0]))
        return (gw.view(ctx.wshape), None) + (None,) * len(ctx.frames)


class PermuteRowsFn(torch.autograd.Function):
    """out.view(n, unit*cols)[i] = x.view(n, unit*cols)[index[i]]; `inverse` is the inverse permutation."""

    @staticmethod
    def forward(ctx, x, index, inverse, unit):
        ctx.inverse, ctx.unit = inverse, unit
        return ops.gather_rows(x.contiguous(), index, unit)

    @staticmethod
    def backward(ctx, dout):
        return ops.gather_rows(dout.contiguous(), ctx.inverse, ctx.unit), None, None, None


def _as_dtype(t: torch.Tensor, dtype: torch.dtype) -> torch.Tensor:
    t = t.detach()
    if t.dtype == dtype and t.is_contiguous():
        return t
    t2 = t.reshape(1, -1) if t.dim() == 1 else t
    out = ops.cast2d(t2.contiguous() if t2.stride(-1) != 1 else t2, torch.empty(t2.shape, dtype=dtype, device=t.device))
    return out.view(t.shape)


class MergerFn(torch.autograd.Function):
    """RMSNorm(C) -> view [S/unit, unit*C] -> Linear + exact GELU -> Linear."""

    @staticmethod
    def forward(ctx, x, ln_w, w0, b0, w2, b2, unit, eps):
        T = x.dtype
        x = x.contiguous()
        lw, W0, B0, W2, B2 = (_as_dtype(t, T) for t in (ln_w, w0, b0, w2, b2))
        ln, rstd = ops.rmsnorm_fwd(x, lw, eps)
        M = x.shape[0] // unit
        ln2 = ln.view(M, -1)
        z = torch.empty(M, W0.shape[0], dtype=T, device=x.device)
        y1 = torch.empty_like(z)
        ops.gemm(ln2, W0, y1, epilogue=E.EPI_BIAS_GELU, bias=B0, aux=z)
        y2 = torch.empty(M, W2.shape[0], dtype=T, device=x.device)
        ops.gemm(y1, W2, y2, epilogue=E.EPI_BIAS, bias=B2)
        ctx.saved = (x, lw, rstd, ln2, z, y1, W0, W2)
        ctx.gdt = (ln_w.dtype, w0.dtype, b0.dtype, w2.dtype, b2.dtype)
        return y2

    @staticmethod
    def backward(ctx, dy):
        x, lw, rstd, ln2, z, y1, W0, W2 = ctx.saved
        ctx.saved = None
        dy = dy.contiguous()
        dev = x.device
        g_w2 = torch.empty(W2.shape, dtype=ctx.gdt[3], device=dev)
        g_b2 = ops.weight_grad(dy, y1, g_w2, ctx.gdt[4])
        dz = torch.empty_like(z)
        ops.gemm(dy, W2, dz, trans_b=True, epilogue=E.EPI_GELU_BWD, residual=z)
        g_w0 = torch.empty(W0.shape, dtype=ctx.gdt[1], device=dev)
        g_b0 = ops.weight_grad(dz, ln2, g_w0, ctx.gdt[2])
        dln = torch.empty_like(ln2)
        ops.gemm(dz, W0, dln, trans_b=True)
        dx, g_ln = ops.rmsnorm_bwd(dln.view(x.shape), x, lw, rstd, w_grad_dtype=ctx.gdt[0])
        return dx, g_ln, g_w0, g_b0, g_w2, g_b2, None, None
