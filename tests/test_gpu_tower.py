"""End-to-end parity of the vision tower (forward, every parameter gradient) against the CPU oracle, and the
VisionTrainer step API on the GPU."""

import copy

import pytest
import torch

from oracle import vit_oracle
from oracle.vit_oracle import OracleConfig, max_rel_err

pytestmark = pytest.mark.gpu
DEV = "cuda:0"


def _build(cfg_kwargs, seed, dtype):
    from mi355_vit.config import Qwen2_5_VLVisionConfig
    from mi355_vit.modeling import Qwen2_5_VisionTransformerPretrainedModel

    torch.manual_seed(seed)
    model = Qwen2_5_VisionTransformerPretrainedModel(Qwen2_5_VLVisionConfig(**cfg_kwargs))
    model.to(dtype)
    return model


def _oracle_cfg(kw):
    return OracleConfig(**{k: v for k, v in kw.items() if k in OracleConfig.__dataclass_fields__})


def _oracle_run(model_cpu, kw, pixels, grid, gout):
    """fp32 oracle forward/backward on the (possibly bf16-rounded) weights of `model_cpu`."""
    params = {k: v.detach().float().clone().requires_grad_(True) for k, v in model_cpu.state_dict().items()}
    inv_freq = model_cpu.rotary_pos_emb.inv_freq.detach().clone()  # keeps its dtype: bf16 towers build a bf16 table
    out = vit_oracle.tower_forward(pixels.float(), grid, params, _oracle_cfg(kw), inv_freq=inv_freq)
    out.backward(gout.float())
    return out.detach(), {k: p.grad for k, p in params.items()}


def _run_gpu(model, pixels, grid, gout):
    model.to(DEV).train()
    model.zero_grad(set_to_none=True)
    out = model(hidden_states=pixels.to(DEV), grid_thw=grid.to(DEV))
    out.backward(gout.to(device=DEV, dtype=out.dtype))
    return out.detach(), {n: p.grad.detach() for n, p in model.named_parameters()}


CFG1 = dict(depth=4, hidden_size=1280, intermediate_size=3420, num_heads=16, out_hidden_size=2048, fullatt_block_indexes=[3])


def test_config1_fp32_parity():
    """Benchmark configuration 1: reduced tower, fp32, 2 images of 224x224; outputs and all gradients within 1e-4."""
    print("[case] config-1 fp32 tower", flush=True)
    model = _build(CFG1, 0, torch.float32)
    g = torch.Generator().manual_seed(0)
    grid = torch.tensor([[1, 16, 16], [1, 16, 16]])
    pixels = torch.randn(512, 1176, generator=g)
    gout = torch.randn(128, 2048, generator=g)
    ref_out, ref_grads = _oracle_run(copy.deepcopy(model), CFG1, pixels, grid, gout)
    out, grads = _run_gpu(model, pixels, grid, gout)
    assert out.shape == (128, 2048) and out.dtype == torch.float32
    assert max_rel_err(out, ref_out) < 1e-4
    worst = max((max_rel_err(grads[k], ref_grads[k]), k) for k in ref_grads)
    assert worst[0] < 1e-4, worst
    assert set(grads) == set(ref_grads)


@pytest.mark.parametrize("checkpoint", [False, True])
def test_small_ragged_tower_bf16_parity(checkpoint):
    """Ragged images + a video, windows with edge remainders, bf16 kernels vs the fp32 oracle on the same bf16 weights."""
    print(f"[case] bf16 ragged tower checkpoint={checkpoint}", flush=True)
    kw = dict(depth=3, hidden_size=1280, intermediate_size=3420, num_heads=16, out_hidden_size=512, fullatt_block_indexes=[1])
    model = _build(kw, 1, torch.bfloat16)
    if checkpoint:
        model.gradient_checkpointing_enable()
    g = torch.Generator().manual_seed(1)
    grid = torch.tensor([[1, 18, 22], [2, 8, 12], [1, 34, 16]])
    S = int((grid[:, 0] * grid[:, 1] * grid[:, 2]).sum())
    pixels = torch.randn(S, 1176, generator=g).to(torch.bfloat16)
    gout = torch.randn(S // 4, 512, generator=g).to(torch.bfloat16)
    ref_out, ref_grads = _oracle_run(copy.deepcopy(model), kw, pixels, grid, gout)
    out, grads = _run_gpu(model, pixels, grid, gout)
    assert out.dtype == torch.bfloat16
    assert max_rel_err(out, ref_out) < 2e-2
    worst = max((max_rel_err(grads[k], ref_grads[k]), k) for k in ref_grads)
    assert worst[0] < 2e-2, worst


@pytest.mark.parametrize("dtype,tol", [(torch.float32, 1e-4), (torch.bfloat16, 2e-2)])
def test_smallest_images_parity(dtype, tol):
    """The smallest inputs the model takes: one 28 x 28 image (4 patches, one merged token: every GEMM has 4 rows, every
    attention segment 4 tokens) alone and beside a 2-frame video of the same size and a 28 x 56 image, against the oracle."""
    kw = dict(depth=2, hidden_size=256, intermediate_size=300, num_heads=8, out_hidden_size=128, fullatt_block_indexes=[1])
    for grid in (torch.tensor([[1, 2, 2]]), torch.tensor([[1, 2, 2], [2, 2, 2], [1, 2, 4]])):
        print(f"[case] smallest images {grid.tolist()} {dtype}", flush=True)
        model = _build(kw, 2, dtype)
        g = torch.Generator().manual_seed(4)
        S = int((grid[:, 0] * grid[:, 1] * grid[:, 2]).sum())
        pixels = torch.randn(S, 1176, generator=g).to(dtype)
        gout = torch.randn(S // 4, 128, generator=g).to(dtype)
        ref_out, ref_grads = _oracle_run(copy.deepcopy(model), kw, pixels, grid, gout)
        out, grads = _run_gpu(model, pixels, grid, gout)
        assert tuple(out.shape) == (S // 4, 128) and max_rel_err(out, ref_out) < tol
        worst = max((max_rel_err(grads[k], ref_grads[k]), k) for k in ref_grads)
        assert worst[0] < tol, worst


def test_checkpointing_gives_identical_gradients():
    kw = dict(depth=2, hidden_size=256, intermediate_size=300, num_heads=8, out_hidden_size=256, window_size=56, fullatt_block_indexes=[1])
    g = torch.Generator().manual_seed(3)
    grid = torch.tensor([[1, 16, 16], [1, 16, 32]])
    pixels = torch.randn(768, 1176, generator=g)
    gout = torch.randn(192, 256, generator=g)
    res = []
    for ck in (False, True):
        model = _build(kw, 5, torch.float32)
        if ck:
            model.gradient_checkpointing_enable()
        res.append(_run_gpu(model, pixels, grid, gout))
    assert torch.equal(res[0][0], res[1][0])
    for k in res[0][1]:
        assert torch.equal(res[0][1][k], res[1][1][k]), k


def test_second_stream_overlap_gives_identical_gradients():
    """Weight / bias gradients computed on the second stream (default) against the single-stream order: the
    kernels are deterministic, so every gradient must be bit-identical; bf16 at a size where a weight-gradient
    GEMM spans many work-groups and uses split-K, and two backward passes so that buffers are recycled."""
    from mi355_vit import ops

    kw = dict(depth=3, hidden_size=512, intermediate_size=1200, num_heads=8, out_hidden_size=256, window_size=56, fullatt_block_indexes=[1])
    g = torch.Generator().manual_seed(11)
    grid = torch.tensor([[1, 32, 48], [1, 40, 28], [2, 16, 16]])
    S = int((grid[:, 0] * grid[:, 1] * grid[:, 2]).sum())
    pixels = torch.randn(S, 1176, generator=g)
    gout = torch.randn(S // 4, 256, generator=g)
    res = []
    old = ops.OVERLAP_WGRAD
    try:
        for overlap in (True, False):
            ops.OVERLAP_WGRAD = overlap
            model = _build(kw, 7, torch.bfloat16)
            _run_gpu(model, pixels, grid, gout)
            for p_ in model.parameters():
                p_.grad = None
            res.append(_run_gpu(model, pixels, grid, gout))
    finally:
        ops.OVERLAP_WGRAD = old
    assert ops.side_stream(torch.device(DEV)) is not None or not old
    assert torch.equal(res[0][0], res[1][0])
    for k in res[0][1]:
        assert torch.equal(res[0][1][k], res[1][1][k]), k


def test_products_are_told_whether_a_second_stream_runs_beside_them(monkeypatch):
    """Backward products of a block are chosen as ones that share the GPU where its second stream runs, and only there: not the
    forward's, not the merger's and the patch embedding's, and none with the second stream switched off."""
    from mi355_vit import functional, ops

    kw = dict(depth=2, hidden_size=256, intermediate_size=300, num_heads=8, out_hidden_size=128, fullatt_block_indexes=[1])
    told, gemm = [], ops.gemm
    monkeypatch.setattr(ops, "gemm", lambda *a, **k: (told.append(bool(k.get("overlapped"))), gemm(*a, **k))[1])
    monkeypatch.setattr(functional, "BLOCK_CALLS", False)
    pixels, gout = torch.randn(256, 1176), torch.randn(64, 128)
    for overlap in (True, False):
        monkeypatch.setattr(ops, "OVERLAP_WGRAD", overlap)
        told.clear()
        _run_gpu(_build(kw, 3, torch.bfloat16), pixels, torch.tensor([[1, 16, 16]]), gout)
        merger, patch_embedding, block = 4, 1, 8
        assert told == [False] * (1 + 2 * 4 + 2 + merger) + [overlap] * (2 * block) + [False] * patch_embedding


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float32])
@pytest.mark.parametrize("checkpoint", [False, True])
def test_one_call_per_block_equals_the_call_by_call_sequence(dtype, checkpoint):
    """mvit_block_fwd / mvit_block_bwd issue a block's launches from inside the library; the sequence issued call by call
    (MVIT_BLOCK_CALLS=0, and what runs while launches are being timed) must give the same bits: output and every
    gradient, plain and checkpointed, with the weight gradients on the second stream and in line."""
    from mi355_vit import functional, ops

    kw = dict(depth=3, hidden_size=512, intermediate_size=1200, num_heads=8, out_hidden_size=256, window_size=56, fullatt_block_indexes=[1])
    g = torch.Generator().manual_seed(12)
    grid = torch.tensor([[1, 32, 48], [1, 40, 28], [2, 16, 16]])
    S = int((grid[:, 0] * grid[:, 1] * grid[:, 2]).sum())
    pixels = torch.randn(S, 1176, generator=g)
    gout = torch.randn(S // 4, 256, generator=g)
    res = {}
    old_calls, old_overlap = functional.BLOCK_CALLS, ops.OVERLAP_WGRAD
    try:
        for one_call in (True, False):
            for overlap in (True, False):
                functional.BLOCK_CALLS, ops.OVERLAP_WGRAD = one_call, overlap
                model = _build(kw, 7, dtype)
                if checkpoint:
                    model.gradient_checkpointing_enable()
                _run_gpu(model, pixels, grid, gout)
                for p_ in model.parameters():
                    p_.grad = None
                res[(one_call, overlap)] = _run_gpu(model, pixels, grid, gout)  # second pass: buffers are recycled
    finally:
        functional.BLOCK_CALLS, ops.OVERLAP_WGRAD = old_calls, old_overlap
    ref_out, ref_grads = res[(False, False)]
    assert torch.isfinite(ref_out).all()
    for key, (out, grads) in res.items():
        assert torch.equal(out, ref_out), key
        for k in ref_grads:
            assert torch.equal(grads[k], ref_grads[k]), (key, k)


@pytest.mark.parametrize("heads,rows,ragged,tables_alike", [(1, 1, False, True), (1, 64, False, False), (2, 77, True, True), (3, 500, True, False), (16, 256, False, True),
                                                            (16, 4033, True, False), (16, 22000, False, True), (16, 22001, True, False), (6, 60000, True, True), (5, 70000, False, False)])
def test_windows_with_the_rotation_inside_give_the_bits_of_two_passes(heads, rows, ragged, tables_alike):
    """A windowed block behind one call rotates q and k inside its attention, both ways: output, attention output and log-sum-exp, what a backward
    reads of q, k and v, and its gradients are those of the call-by-call sequence with its pass of its own; one, two and four heads to a work-group, windows of 1 to 64
    tokens, rotary tables whose halves differ, with gradients to come and without."""
    from mi355_vit import functional as F

    C, I, g = 80 * heads, 128, torch.Generator().manual_seed(rows + heads)
    lengths = []
    left = rows
    while left > 0:
        lengths.append(min(left, int(torch.randint(1, 65, (1,), generator=g)) if ragged else 64))
        left -= lengths[-1]
    cu = torch.tensor([0] + lengths).cumsum(0).to(torch.int32).to(DEV)
    angle = torch.randn(rows, 40, generator=g)
    angle = torch.cat([angle, angle if tables_alike else angle + 1], 1).to(DEV)
    geo = F.AttnGeometry(cu, max(lengths), heads, 80, angle.cos().contiguous(), angle.sin().contiguous())
    r = lambda *shape: (torch.randn(*shape, generator=g) * 0.05).to(torch.bfloat16).to(DEV)  # noqa: E731
    Ipad = F.padded_inner(I)
    W = F.BlockWeights(r(1, C) + 1, r(1, C) + 1, r(3 * C, C), r(1, 3 * C), r(C, C), r(1, C), r(2 * Ipad, C), r(1, 2 * Ipad), r(C, Ipad), r(1, C), C, I, Ipad)
    x, old = torch.randn(rows, C, generator=g).to(torch.bfloat16).to(DEV), F.BLOCK_CALLS
    try:
        for for_backward in (True, False):
            F.BLOCK_CALLS = True
            y, saved = F._block_forward(x, W, geo, 1e-6, for_backward=for_backward)
            F.BLOCK_CALLS = False
            want, want_saved = F._block_forward(x, W, geo, 1e-6, for_backward=for_backward)
            assert torch.isfinite(want).all() and torch.equal(y, want)
            for i in (2, 3, 4) if for_backward else (3, 4):
                assert torch.equal(saved[i], want_saved[i]), (for_backward, i)
            if for_backward:  # the backward turns dq and dk back inside
                kept, dy = tuple(want_saved), torch.randn(rows, C, generator=g).to(torch.bfloat16).to(DEV)
                dx, grads = F._block_backward(dy, x, kept, W, geo, torch.bfloat16)  # call by call
                F.BLOCK_CALLS = True
                dx1, grads1 = F._block_backward(dy, x, kept, W, geo, torch.bfloat16)
                assert torch.isfinite(dx).all() and torch.equal(dx1, dx) and all(torch.equal(a, b) for a, b in zip(grads1, grads))
    finally:
        F.BLOCK_CALLS = old


@pytest.mark.parametrize("rows", [4100, 12000, 12100])
def test_weight_gradients_of_many_rows_are_summed_in_the_slices_of_their_products(rows):
    """A block's weight and bias gradients are those of its products one by one with the K slices that ``wgrad_split_k`` names, bit for bit, behind one call
    and call by call, on the second stream and in line: with longer chains of fp32 additions more of them are rounded to the wrong side."""
    from mi355_vit import functional as F
    from mi355_vit import ops

    C, H, I, g = 1280, 16, 3420, torch.Generator().manual_seed(rows)
    cu = torch.tensor(list(range(0, rows, 64)) + [rows], dtype=torch.int32).to(DEV)
    angle = torch.randn(rows, 40, generator=g).repeat(1, 2).to(DEV)
    geo = F.AttnGeometry(cu, 64, H, 80, angle.cos().contiguous(), angle.sin().contiguous())
    r = lambda *shape: (torch.randn(*shape, generator=g) * 0.03).to(torch.bfloat16).to(DEV)  # noqa: E731
    Ipad = F.padded_inner(I)
    W = F.BlockWeights(r(1, C) + 1, r(1, C) + 1, r(3 * C, C), r(1, 3 * C), r(C, C), r(1, C), r(2 * Ipad, C), r(1, 2 * Ipad), r(C, Ipad), r(1, C), C, I, Ipad)
    x, dy = torch.randn(rows, C, generator=g).to(torch.bfloat16).to(DEV), torch.randn(rows, C, generator=g).to(torch.bfloat16).to(DEV)
    names = {n: i for i, n in enumerate(F.BLOCK_PARAM_ORDER)}
    old = F.BLOCK_CALLS, ops.OVERLAP_WGRAD
    try:
        for F.BLOCK_CALLS, ops.OVERLAP_WGRAD in ((True, True), (True, False), (False, True), (False, False)):
            _, saved = F._block_forward(x, W, geo, 1e-6)
            h = saved[9].clone()
            _, grads = F._block_backward(dy, x, saved, W, geo, torch.bfloat16)
            want = torch.empty(C, I, dtype=torch.bfloat16, device=DEV)
            bias = ops.weight_grad(dy, h, want, torch.bfloat16, n=I, split_k=ops.wgrad_split_k(C, I, rows, True), overlapped=True)
            assert torch.equal(grads[names["mlp.down_proj.weight"]], want) and torch.equal(grads[names["mlp.down_proj.bias"]], bias)
    finally:
        F.BLOCK_CALLS, ops.OVERLAP_WGRAD = old


@pytest.mark.parametrize("rows,window", [(1000, 4), (999, 9), (1000, 10), (1001, 11), (22000, 4), (22003, 16), (22016, 39), (22000, 40), (22008, 47), (22032, 48)])
def test_windows_give_the_bits_of_two_passes_on_both_sides_of_the_lines(rows, window):
    """Short windows are rotated by a pass of their own; many rows of long ones take several heads to a work-group."""
    from mi355_vit import functional as F

    H, C, I, g = 16, 1280, 64, torch.Generator().manual_seed(rows)
    cu = torch.tensor(list(range(0, rows, window)) + [rows], dtype=torch.int32).to(DEV)
    angle = torch.randn(rows, 40, generator=g).repeat(1, 2).to(DEV)
    geo = F.AttnGeometry(cu, window, H, 80, angle.cos().contiguous(), angle.sin().contiguous())
    r = lambda *shape: (torch.randn(*shape, generator=g) * 0.05).to(torch.bfloat16).to(DEV)  # noqa: E731
    Ipad = F.padded_inner(I)
    W = F.BlockWeights(r(1, C) + 1, r(1, C) + 1, r(3 * C, C), r(1, 3 * C), r(C, C), r(1, C), r(2 * Ipad, C), r(1, 2 * Ipad), r(C, Ipad), r(1, C), C, I, Ipad)
    x, dy, old, got = r(rows, C) * 20, r(rows, C) * 20, F.BLOCK_CALLS, {}
    try:
        for F.BLOCK_CALLS in (True, False):
            y0, saved0 = F._block_forward(x, W, geo, 1e-6, for_backward=False)
            y, saved = F._block_forward(x, W, geo, 1e-6)
            kept = [saved[i].clone() for i in (2, 3, 4)]
            dx, grads = F._block_backward(dy, x, tuple(saved), W, geo, torch.bfloat16)
            got[F.BLOCK_CALLS] = [y0, saved0[3], saved0[4], y, *kept, dx, *grads]
    finally:
        F.BLOCK_CALLS = old
    assert all(torch.equal(a, b) for a, b in zip(got[True], got[False]))


@pytest.mark.parametrize("kind", ["permuted", "named twice", "outside the list"])
def test_windows_that_rotate_are_taken_once_each_whatever_the_order_of_segments_says(kind):
    """q and k are rotated in place inside the windows' attention: an order that names a window twice must not have it rotated twice."""
    from mi355_vit import functional as F

    H, C, I, g = 16, 1280, 64, torch.Generator().manual_seed(5)
    lengths = torch.randint(1, 65, (97,), generator=g)
    cu = torch.cat([torch.zeros(1, dtype=torch.int64), lengths.cumsum(0)]).to(torch.int32).to(DEV)
    rows, n = int(lengths.sum()), lengths.numel()
    order = torch.randperm(n, generator=g) if kind == "permuted" else torch.randint(0, n, (n,), generator=g)
    if kind == "outside the list":
        order[::2] = n + order[::2]
    angle = torch.randn(rows, 40, generator=g).repeat(1, 2).to(DEV)
    tables = angle.cos().contiguous(), angle.sin().contiguous()
    r = lambda *shape: (torch.randn(*shape, generator=g) * 0.05).to(torch.bfloat16).to(DEV)  # noqa: E731
    Ipad = F.padded_inner(I)
    W = F.BlockWeights(r(1, C) + 1, r(1, C) + 1, r(3 * C, C), r(1, 3 * C), r(C, C), r(1, C), r(2 * Ipad, C), r(1, 2 * Ipad), r(C, Ipad), r(1, C), C, I, Ipad)
    x, dy = r(rows, C) * 20, r(rows, C) * 20

    def run(order):
        geo = F.AttnGeometry(cu, 64, H, 80, *tables, order)
        y, saved = F._block_forward(x, W, geo, 1e-6)
        kept = [saved[i].clone() for i in (2, 3, 4)]
        dx, grads = F._block_backward(dy, x, saved, W, geo, torch.bfloat16)
        return [y, *kept, F._block_forward(x, W, geo, 1e-6, for_backward=False)[0], dx, *grads]

    assert all(torch.equal(a, b) for a, b in zip(run(order.to(torch.int32).to(DEV)), run(None)))


@pytest.mark.parametrize("where", ["a token", "a channel of v", "a channel of q", "a gradient"])
@pytest.mark.parametrize("value", [float("inf"), float("-inf"), float("nan")])
def test_windows_with_the_rotation_inside_keep_infinities_and_nans_where_two_passes_do(value, where):
    """One token's row (NaN behind its norm), one channel of one head, one row of the incoming gradient; ragged windows."""
    from mi355_vit import functional as F

    H, C, I, g = 3, 240, 64, torch.Generator().manual_seed(9)
    lengths = torch.tensor([64, 17, 1, 50, 33, 64, 16])
    cu = torch.cat([torch.zeros(1, dtype=torch.int64), lengths.cumsum(0)]).to(torch.int32).to(DEV)
    rows = int(lengths.sum())
    angle = torch.randn(rows, 40, generator=g).repeat(1, 2).to(DEV)
    geo = F.AttnGeometry(cu, 64, H, 80, angle.cos().contiguous(), angle.sin().contiguous())
    r = lambda *shape: (torch.randn(*shape, generator=g) * 0.05).to(torch.bfloat16).to(DEV)  # noqa: E731
    Ipad = F.padded_inner(I)
    W = F.BlockWeights(r(1, C) + 1, r(1, C) + 1, r(3 * C, C), r(1, 3 * C), r(C, C), r(1, C), r(2 * Ipad, C), r(1, 2 * Ipad), r(C, Ipad), r(1, C), C, I, Ipad)
    x, dy = r(rows, C) * 20, r(rows, C) * 20
    if where == "a token":
        x[70, 11] = value  # in the second window
    elif where == "a gradient":
        dy[70, 11] = value
    else:
        W.bqkv[0, (2 * C if where == "a channel of v" else 0) + 80 + 7] = value  # of the second head
    old = F.BLOCK_CALLS
    same = lambda a, b: torch.equal(torch.isnan(a), torch.isnan(b)) and torch.equal(torch.nan_to_num(a), torch.nan_to_num(b))  # noqa: E731
    try:
        got = {}
        for one_call in (True, False):
            F.BLOCK_CALLS = one_call
            y0, saved0 = F._block_forward(x, W, geo, 1e-6, for_backward=False)
            y, saved = F._block_forward(x, W, geo, 1e-6)
            kept = [saved[i].clone() for i in (2, 3, 4)]
            dx, grads = F._block_backward(dy, x, tuple(saved), W, geo, torch.bfloat16)
            got[one_call] = [y0, saved0[3], saved0[4], y, *kept, dx, *grads]
    finally:
        F.BLOCK_CALLS = old
    assert all(same(a, b) for a, b in zip(got[True], got[False]))
    y, o = got[True][3], got[True][5]
    if where == "a token":  # its window and no other
        hit = torch.isnan(y).any(1).cpu()
        assert hit[64:81].any() and not hit[:64].any() and not hit[81:].any()
    elif where != "a gradient":  # its head and no other
        hit = (~torch.isfinite(o.view(rows, H, 80))).any(2).cpu()
        assert hit[:, 1].all() and not hit[:, 0].any() and not hit[:, 2].any()


def test_windowed_block_refuses_the_tensors_that_the_attention_calls_refuse():
    """A log-sum-exp that does not start at a 16-byte address, in both directions, as mvit_attn_fwd and mvit_attn_bwd answer it."""
    import ctypes

    from mi355_vit import _lib
    from mi355_vit import functional as F
    from mi355_vit import ops

    H, C, I, rows, g = 2, 160, 64, 100, torch.Generator().manual_seed(2)
    cu = torch.tensor([0, 64, 100], dtype=torch.int32, device=DEV)
    angle = torch.randn(rows, 40, generator=g).repeat(1, 2).to(DEV)
    geo = F.AttnGeometry(cu, 64, H, 80, angle.cos().contiguous(), angle.sin().contiguous())
    r = lambda *shape: (torch.randn(*shape, generator=g) * 0.05).to(torch.bfloat16).to(DEV)  # noqa: E731
    Ipad = F.padded_inner(I)
    W = F.BlockWeights(r(1, C) + 1, r(1, C) + 1, r(3 * C, C), r(1, 3 * C), r(C, C), r(1, C), r(2 * Ipad, C), r(1, 2 * Ipad), r(C, Ipad), r(1, C), C, I, Ipad)
    x, dy = r(rows, C) * 20, r(rows, C) * 20
    _, saved = F._block_forward(x, W, geo, 1e-6)
    kept = [t.clone() for t in saved]
    moved = torch.empty(H * rows + 1, dtype=torch.float32, device=DEV)[1:].view(H, rows)
    moved.copy_(kept[4])
    F._block_backward(dy, x, tuple(kept), W, geo, torch.bfloat16)
    with pytest.raises(RuntimeError, match="unaligned"):
        F._block_backward(dy, x, tuple(kept[:4] + [moved] + kept[5:]), W, geo, torch.bfloat16)
    a = F._block_args(x, W, geo, 1e-6)
    a.rstd1, a.n1, a.qkv, a.o, a.lse, a.x1, a.rstd2, a.n2, a.gu, a.h = (t.data_ptr() for t in kept)
    y = torch.empty_like(x)
    a.x2, a.lse = y.data_ptr(), moved.data_ptr()
    with pytest.raises(RuntimeError, match="unaligned"):
        _lib.check(_lib.load().mvit_block_fwd(ctypes.byref(a), ops._stream(x)), "mvit_block_fwd")


def test_windowed_block_takes_as_many_windows_and_heads_as_the_two_passes():
    """65,535 windows, all but one of them empty, of 205 heads: together more threads than one dimension of a grid holds.  Of so few tokens on
    average they go as two passes too; inside, windows and heads have a grid dimension each."""
    from mi355_vit import functional as F

    H, rows, I = 205, 64, 8
    C, g = 80 * H, torch.Generator(device=DEV).manual_seed(3)
    cu = torch.full((65536,), rows, dtype=torch.int32, device=DEV)
    cu[:40000] = 0
    angle = torch.randn(rows, 40, generator=g, device=DEV).repeat(1, 2)
    geo = F.AttnGeometry(cu, 64, H, 80, angle.cos().contiguous(), angle.sin().contiguous())
    r = lambda *shape: (torch.randn(*shape, generator=g, device=DEV) * 0.02).to(torch.bfloat16)  # noqa: E731
    Ipad = F.padded_inner(I)
    W = F.BlockWeights(r(1, C) + 1, r(1, C) + 1, r(3 * C, C), r(1, 3 * C), r(C, C), r(1, C), r(2 * Ipad, C), r(1, 2 * Ipad), r(C, Ipad), r(1, C), C, I, Ipad)
    x, old, got = r(rows, C) * 50, F.BLOCK_CALLS, {}
    try:
        for F.BLOCK_CALLS in (False, True):
            y, saved = F._block_forward(x, W, geo, 1e-6)
            got[F.BLOCK_CALLS] = [y] + [saved[i] for i in (2, 3, 4)]
    finally:
        F.BLOCK_CALLS = old
    assert torch.isfinite(got[True][0]).all() and all(torch.equal(a, b) for a, b in zip(got[True], got[False]))


_FEW_ROWS = ([[1, 2, 2]], [[1, 6, 10]], [[1, 16, 16], [1, 2, 6]], [[1, 32, 40]], [[1, 32, 40], [1, 2, 2]])


@pytest.mark.parametrize("hidden,inner,grid", [(h, i, g) for h, i in ((512, 1200), (64, 72)) for g in _FEW_ROWS] + [(1280, 3420, g) for g in _FEW_ROWS[1:4]])
def test_weight_gradients_of_few_rows_in_one_launch_equal_a_launch_each(grid, hidden, inner):
    """Up to 1,280 rows the backward of a block sends its weight gradients in one launch and its column sums in another (4, 60, 268 and
    1,280 rows; 1,284 go as longer ones do), on tiles of 64 x 128, 64 x 64 and, at the tower's own width, 128 x 128: output and gradients
    have the bits of the call-by-call sequence."""
    from mi355_vit import functional

    kw = dict(depth=2, hidden_size=hidden, intermediate_size=inner, num_heads=hidden // 32, out_hidden_size=256, window_size=56, fullatt_block_indexes=[1])
    g = torch.Generator().manual_seed(13)
    grid = torch.tensor(grid)
    S = int(grid.prod(1).sum())
    pixels, gout = torch.randn(S, 1176, generator=g), torch.randn(S // 4, 256, generator=g)
    res, old = [], functional.BLOCK_CALLS
    try:
        for functional.BLOCK_CALLS in (True, False):
            res.append(_run_gpu(_build(kw, 8, torch.bfloat16), pixels, grid, gout))
    finally:
        functional.BLOCK_CALLS = old
    assert torch.equal(res[0][0], res[1][0]) and torch.isfinite(res[0][0]).all()
    for k in res[1][1]:
        assert torch.equal(res[0][1][k], res[1][1][k]), k


def test_reference_smoke_shape():
    """The reference's own smoke case (tests/test_ragged_sp_smoke.py:27-98): output [192, 256]."""
    kw = dict(hidden_size=256, num_heads=8, depth=2, patch_size=14, in_channels=3, out_hidden_size=256, spatial_merge_size=2,
              window_size=28, fullatt_block_indexes=[1])
    model = _build(kw, 0, torch.float32).to(DEV).eval()
    grid = torch.tensor([[1, 16, 16], [1, 16, 32]], dtype=torch.int64)
    pixels = torch.randn(768, 1176)
    with torch.no_grad():
        out = model(pixels.to(DEV), grid.to(DEV))
    assert out.shape == (192, 256)
    params = {k: v.detach().float().cpu() for k, v in model.state_dict().items()}
    ref = vit_oracle.tower_forward(pixels, grid, params, _oracle_cfg(kw))
    assert ref.shape == (192, 256)
    assert max_rel_err(out, ref) < 1e-4
    flat = model(pixels.flatten().to(DEV), grid.to(DEV))  # the reference's GPU tests pass a flat tensor
    assert torch.equal(flat.detach(), out)


def _trainer_config(**over):
    cfg = dict(seed=0, model_name="unit-test", parallelism="none", dtype="bfloat16", attention_backend="flash_attention_2",
               activation_checkpointing=False, autocast=True, learning_rate=1e-2, weight_decay=0.01, warmup_ratio=0.0,
               warmup_steps=0, lr_scheduler_type="cosine", num_iterations=10, max_grad_norm=1.0, profile_time=True,
               vision_config=dict(depth=2, hidden_size=256, intermediate_size=300, num_heads=8, out_hidden_size=128, fullatt_block_indexes=[1]),
               synthetic_grids=[[1, 16, 16], [1, 8, 24]])
    cfg.update(over)
    return cfg


def test_trainer_steps_on_gpu():
    from mi355_vit.trainer import VisionTrainer

    tr = VisionTrainer(_trainer_config(), rank=0)
    tr.build_model()
    tr.initialize_trainer()
    tr.zero_grad()
    res = tr.forward_step(iteration=3)
    emb = res["vision_embeddings"]
    M = (16 * 16 + 8 * 24) // 4
    assert emb.shape == (1, M, 128) and emb.dtype == torch.bfloat16 and res["iteration"] == 3 and res["sample_index"] == 0
    assert res["forward_time_ms"] > 0
    before = {n: p.detach().clone() for n, p in tr.model.named_parameters()}
    back = tr.backward_step({"grad": torch.randn(M, 128, device=DEV, dtype=torch.bfloat16)})  # 2-D grad for a 3-D output
    assert back["backward_time_ms"] > 0
    contrib = tr.compute_grad_norm_contribution()
    assert contrib["type"] == "none" and contrib["norm_sq"] > 0
    coeff = tr.optimizer_step(global_grad_norm=contrib["norm_sq"] ** 0.5)
    assert coeff == pytest.approx(min(1.0, 1.0 / (contrib["norm_sq"] ** 0.5 + 1e-6)))
    changed = sum(int(not torch.equal(before[n], p.detach())) for n, p in tr.model.named_parameters())
    assert changed == len(before)
    # packed weights follow the optimizer step: a second forward differs from the first
    res2 = tr.forward_step(iteration=4)
    assert res2["sample_index"] == 1
    tr.backward_step(torch.zeros(1, M, 128, device=DEV, dtype=torch.bfloat16))
    with pytest.raises(RuntimeError, match="No pending vision outputs"):
        tr.backward_step(torch.zeros(1, M, 128, device=DEV))
    tr.forward_step()
    with pytest.raises(ValueError, match="No gradient provided"):
        tr.backward_step(None)
    stats = tr.get_memory_stats()
    assert stats["peak_mb"] >= stats["allocated_mb"] > 0


def test_trainer_batched_five_dimensional_pixel_values():
    """The collated [B, C, T, H, W] input of python/ray/vision.py:732-760: every sample is viewed as consecutive
    1176-value rows, one grid is broadcast to all samples, and the output comes back as [B, tokens per image, hidden];
    gradients of a 3-D output arrive in the same shape."""
    from mi355_vit.trainer import VisionTrainer

    torch.manual_seed(3)
    px = torch.randn(3, 3, 2, 56, 56)  # 16 rows of 1176 values per sample
    batches = [{"pixel_values": px, "image_grid_thw": torch.tensor([1, 4, 4]), "sample_index": torch.tensor([5, 6, 7])},
               {"pixel_values": px.reshape(-1, 1176), "image_grid_thw": torch.tensor([[1, 4, 4]] * 3), "sample_index": torch.tensor([0])}]
    outs = []
    for batch in batches:
        tr = VisionTrainer(_trainer_config(autocast=False), rank=0)
        tr.build_model()
        tr.set_data_iterator([batch])
        tr.initialize_trainer()
        res = tr.forward_step(0)
        outs.append(res["vision_embeddings"])
        if batch["pixel_values"].dim() == 5:
            assert res["sample_index"] == [5, 6, 7] and tuple(outs[0].shape) == (3, 4, 128)
            tr.backward_step(torch.ones(3, 4, 128, device=DEV, dtype=torch.bfloat16))
            assert all(p.grad is not None and torch.isfinite(p.grad).all() for p in tr.model.parameters())
            with pytest.raises(ValueError, match="doesn't match pixel_values batch dimension"):
                tr._model_forward({"pixel_values": px.to(DEV), "image_grid_thw": torch.tensor([[1, 4, 4]] * 2, device=DEV)})
    assert tuple(outs[1].shape) == (1, 12, 128) and torch.equal(outs[0].reshape(1, 12, 128), outs[1])


def test_trainer_fifo_and_checkpoint_roundtrip(tmp_path):
    from mi355_vit.trainer import VisionTrainer

    tr = VisionTrainer(_trainer_config(dtype="float32", activation_checkpointing=True, weight_decay=0.0), rank=0)
    tr.build_model()
    tr.initialize_trainer()
    o1 = tr.forward_step(0)["vision_embeddings"]
    o2 = tr.forward_step(1)["vision_embeddings"]
    assert len(tr._pending_outputs) == 2 and tr._pending_outputs[0] is o1
    tr.backward_step(torch.ones_like(o1))
    assert len(tr._pending_outputs) == 1 and tr._pending_outputs[0] is o2
    tr.backward_step(torch.ones_like(o2))
    path = tr.save_checkpoint(str(tmp_path), epoch=2)
    assert path.endswith("epoch_2/vision/rank_0.pt")
    sd = torch.load(path, weights_only=True, map_location="cpu")["model"]
    assert "blocks.0.attn.q_proj.weight" in sd and "merger.mlp.2.bias" in sd and "rotary_pos_emb.inv_freq" not in sd
    tr.optimizer_step()
    assert tr.load_checkpoint(str(tmp_path), epoch=2)
    for k, v in tr.model.state_dict().items():
        assert torch.equal(v.cpu(), sd[k]), k
    assert not tr.load_checkpoint(str(tmp_path), epoch=9)


@pytest.mark.parametrize("dtype,autocast", [(torch.bfloat16, False), (torch.float32, False), (torch.float32, True)])
def test_forward_after_a_fused_adam_step_uses_the_updated_weights(dtype, autocast):
    """The step writes parameters through raw pointers (no version counter moves): the packed operands the blocks
    read must follow anyway.  Same input before and after one step; the second output must match the oracle run on
    the updated parameters and differ from the first output."""
    from mi355_vit.optim import FusedAdam

    print(f"[case] forward after FusedAdam step {dtype} autocast={autocast}", flush=True)
    kw = dict(depth=2, hidden_size=256, intermediate_size=300, num_heads=8, out_hidden_size=128, fullatt_block_indexes=[1])
    model = _build(kw, 5, dtype).to(DEV).train()
    g = torch.Generator().manual_seed(5)
    grid = torch.tensor([[1, 16, 16], [1, 8, 24]])
    S = 16 * 16 + 8 * 24
    pixels = torch.randn(S, 1176, generator=g).to(DEV)
    gout = torch.randn(S // 4, 128, generator=g).to(DEV)
    # gradients for the block parameters only: a change of the output can then only come from the blocks
    block_params = [p for n, p in model.named_parameters() if n.startswith("blocks.")]
    opt = FusedAdam(block_params, lr=5e-3, weight_decay=0.01)

    def forward():
        with torch.autocast("cuda", dtype=torch.bfloat16, enabled=autocast):
            return model(hidden_states=pixels, grid_thw=grid.to(DEV))

    outs = []
    for step in range(3):
        out = forward()
        outs.append(out.detach().float().cpu())
        model.zero_grad(set_to_none=True)
        out.backward(gout.to(out.dtype))
        for n, p in model.named_parameters():
            if not n.startswith("blocks."):
                p.grad = None
        opt.step()
    final = forward().detach().float().cpu()
    torch.cuda.synchronize()
    assert max_rel_err(final, outs[0]) > 5e-2, "three optimizer steps left the output unchanged: stale operands"
    assert max_rel_err(outs[1], outs[0]) > 1e-2
    low = dtype == torch.bfloat16 or autocast
    cpu = copy.deepcopy(model).cpu()
    params = {k: (v.detach().to(torch.bfloat16).float() if low else v.detach().float()).clone() for k, v in cpu.state_dict().items()}
    inv_freq = cpu.rotary_pos_emb.inv_freq.detach().clone()
    with torch.no_grad():
        ref = vit_oracle.tower_forward(pixels.cpu().float(), grid, params, _oracle_cfg(kw), inv_freq=inv_freq)
    assert max_rel_err(final, ref) < (2e-2 if low else 1e-4)
    # a torch optimizer (in-place torch ops) on the same parameters is followed as well
    sgd = torch.optim.SGD(block_params, lr=0.5)
    out = forward()
    model.zero_grad(set_to_none=True)
    out.backward(gout.to(out.dtype))
    sgd.step()
    after_sgd = forward().detach().float().cpu()
    assert max_rel_err(after_sgd, final) > 1e-2


def test_windowed_block_on_each_sequence_parallel_share_equals_the_unsharded_block():
    """One rank's share of a windowed layer under Ulysses sequence parallelism (modeling:492-581): the pack is cut at
    window boundaries, so a block run on a rank's rows with the rank-local window boundaries and rotary rows needs no
    exchange.  For sp = 4 every rank's output (and input gradient) must equal the matching rows of the unsharded block
    bit for bit."""
    from mi355_vit import ops
    from mi355_vit import sequence_parallel_utils as spu
    from mi355_vit.config import Qwen2_5_VLVisionConfig
    from mi355_vit.modeling import Qwen2_5_VLVisionBlock

    print("[case] windowed block on sp=4 shares", flush=True)
    torch.manual_seed(7)
    cfg = Qwen2_5_VLVisionConfig(depth=1, hidden_size=1280, intermediate_size=3420, num_heads=16, out_hidden_size=256, fullatt_block_indexes=[])
    blk = Qwen2_5_VLVisionBlock(cfg, 0).to(torch.bfloat16).to(DEV)
    grid = torch.tensor([[1, 18, 22], [2, 8, 12], [1, 34, 16], [1, 4, 4]])
    _, cu_w = ops.window_index(grid, 2, 112, 14)
    cu_f = ops.cu_seqlens(grid)
    lengths = (cu_f[1:] - cu_f[:-1]).tolist()
    S = sum(lengths)
    g = torch.Generator().manual_seed(7)
    x = torch.randn(S, 1280, generator=g).to(torch.bfloat16).to(DEV)
    ang = torch.randn(S, 40, generator=g)
    emb = torch.cat((ang, ang), dim=-1)
    cos, sin = emb.cos().to(DEV), emb.sin().to(DEV)
    gy = torch.randn(S, 1280, generator=g).to(torch.bfloat16).to(DEV)

    xf = x.clone().requires_grad_(True)
    y_full = blk(xf, cu_seqlens=cu_w.to(DEV), position_embeddings=(cos, sin))
    y_full.backward(gy)
    outs, dxs, metas = [], [], []
    for r in range(4):
        xr, meta = spu.split_pack_by_sp(x, lengths, r, 4, cu_window_seqlens=cu_w)
        gr, _ = spu.split_pack_by_sp(gy, lengths, r, 4, cu_window_seqlens=cu_w)
        cu_local = spu.rebuild_local_cu_seqlens(meta, use_windows=True)
        cos_r, sin_r, _ = spu.build_local_rope(meta, cos, sin)
        assert int(cu_local[-1]) == xr.shape[0] == cos_r.shape[0]
        xr = xr.clone().requires_grad_(True)
        if xr.shape[0]:
            yr = blk(xr, cu_seqlens=cu_local.to(DEV), position_embeddings=(cos_r, sin_r))
            yr.backward(gr)
            outs.append(yr.detach())
            dxs.append(xr.grad)
        else:
            outs.append(xr.detach())
            dxs.append(torch.zeros_like(xr))
        metas.append(meta)
    lm = [m.local_lengths for m in metas]
    assert torch.equal(spu.gather_rank_packs(outs, lm), y_full.detach())
    assert torch.equal(spu.gather_rank_packs(dxs, lm), xf.grad)
    assert sum(o.shape[0] for o in outs) == S and min(o.shape[0] for o in outs) > 0


def test_windowed_block_of_4096_rows_equals_its_four_shares():
    """The same at 4,096 rows, where the whole block and its shares run on tiles of different sizes."""
    from mi355_vit import ops
    from mi355_vit.config import Qwen2_5_VLVisionConfig
    from mi355_vit.modeling import Qwen2_5_VLVisionBlock

    print("[case] windowed block, 4096 rows and four shares", flush=True)
    torch.manual_seed(8)
    cfg = Qwen2_5_VLVisionConfig(depth=1, hidden_size=1280, intermediate_size=3420, num_heads=16, out_hidden_size=256, fullatt_block_indexes=[])
    blk = Qwen2_5_VLVisionBlock(cfg, 0).to(torch.bfloat16).to(DEV)
    S, n = 4096, 1024
    _, cu = ops.window_index(torch.tensor([[1, 64, 64]]), 2, 112, 14)
    assert cu.tolist() == list(range(0, S + 1, 64))
    g = torch.Generator().manual_seed(8)
    x, gy = (torch.randn(S, 1280, generator=g).to(torch.bfloat16).to(DEV) for _ in range(2))
    ang = torch.randn(S, 40, generator=g)
    emb = torch.cat((ang, ang), dim=-1)
    cos, sin = emb.cos().to(DEV), emb.sin().to(DEV)

    def run(a, b):
        xr = x[a:b].clone().requires_grad_(True)
        y = blk(xr, cu_seqlens=cu[: (b - a) // 64 + 1].to(DEV), position_embeddings=(cos[a:b], sin[a:b]))
        y.backward(gy[a:b])
        return y.detach(), xr.grad

    y_full, dx_full = run(0, S)
    for a in range(0, S, n):
        y, dx = run(a, a + n)
        assert torch.equal(y, y_full[a : a + n]) and torch.equal(dx, dx_full[a : a + n]), a


@pytest.mark.parametrize("one_call", [True, False])
@pytest.mark.parametrize("S", [320, 4096, 5120])
def test_gate_and_up_bias_gradients_are_sums_of_fp32_values(S, one_call, monkeypatch):
    """The SwiGLU backward's results are summed before they are rounded to bf16, at any number of rows."""
    from mi355_vit import functional as MF
    from mi355_vit.config import Qwen2_5_VLVisionConfig
    from mi355_vit.modeling import Qwen2_5_VLVisionBlock

    print(f"[case] gate/up bias gradients, {S} rows, one call {one_call}", flush=True)
    monkeypatch.setattr(MF, "BLOCK_CALLS", one_call)
    torch.manual_seed(9)
    cfg = Qwen2_5_VLVisionConfig(depth=1, hidden_size=1280, intermediate_size=3420, num_heads=16, out_hidden_size=256, fullatt_block_indexes=[])
    blk = Qwen2_5_VLVisionBlock(cfg, 0).to(DEV)  # fp32 parameters: their gradients are not rounded
    g = torch.Generator().manual_seed(9)
    x, gy = (torch.randn(S, 1280, generator=g).to(torch.bfloat16).to(DEV) for _ in range(2))
    emb = torch.randn(S, 40, generator=g).repeat(1, 2)
    cu = torch.arange(0, S + 1, 64, dtype=torch.int32, device=DEV)
    kept = []
    backward = MF._block_backward
    monkeypatch.setattr(MF, "_block_backward", lambda dx2, x, saved, W, *rest: (kept.append((saved[8], W)), backward(dx2, x, saved, W, *rest))[1])
    xr = x.clone().requires_grad_(True)
    blk(xr, cu_seqlens=cu, position_embeddings=(emb.cos().to(DEV), emb.sin().to(DEV))).backward(gy)
    (gu, W), = kept
    gate, up = gu[:, : W.I].double(), gu[:, W.Ipad : W.Ipad + W.I].double()
    dh, s = gy.double() @ W.wdown.double()[:, : W.I], torch.sigmoid(gate)
    for param, exact in ((blk.mlp.gate_proj.bias, (dh * up * s * (1 + gate * (1 - s))).sum(0)), (blk.mlp.up_proj.bias, (dh * gate * s).sum(0))):
        err = float((param.grad.double() - exact).norm() / exact.norm())
        # fp32 sums of 1,280 products, each value then with a relative error near sqrt(1280) * 2^-24 = 2e-6 (and as much again
        # from the hardware exponential and reciprocal); summed after a rounding to bf16 it would be near 2^-9 / sqrt(3) = 1e-3
        assert param.grad.dtype == torch.float32 and err < 2e-5, err


def test_a_step_recorded_in_a_hip_graph_replays_bit_identically():
    """The library's launches allocate nothing, wait for nothing and use no stream but the caller's (the eager backward's
    second stream joins through events), so a whole forward and a whole backward can be recorded in HIP graphs.  Three
    replays with different inputs, eager steps and synchronisations between them, each equal to the eager step bit for
    bit (kernel order and arguments are the eager ones)."""
    print("[case] forward and backward recorded in HIP graphs", flush=True)
    kw = dict(depth=3, hidden_size=1280, intermediate_size=3420, num_heads=16, out_hidden_size=512, fullatt_block_indexes=[1])
    model = _build(kw, 5, torch.bfloat16).to(DEV).train()
    model.gradient_checkpointing_enable()
    grid = torch.tensor([[1, 18, 22], [2, 8, 12], [1, 34, 16]])  # a host tensor: planning needs no device read-back
    S = int(grid.prod(dim=1).sum())
    params = list(model.parameters())

    def inputs(seed):
        g = torch.Generator().manual_seed(seed)
        return torch.randn(S, 1176, generator=g).to(torch.bfloat16).to(DEV), torch.randn(S // 4, 512, generator=g).to(torch.bfloat16).to(DEV)

    def eager(px, gout):
        model.zero_grad(set_to_none=True)
        out = model(hidden_states=px, grid_thw=grid)
        out.backward(gout)
        torch.cuda.synchronize()
        return out.detach().clone(), [p.grad.detach().clone() for p in params]

    static_px, static_gout = inputs(0)
    side = torch.cuda.Stream()
    side.wait_stream(torch.cuda.current_stream())
    with torch.cuda.stream(side):  # plans, packed weights and library handles come into being before the recording
        for _ in range(2):
            torch.autograd.grad(model(hidden_states=static_px, grid_thw=grid), params, static_gout)
    torch.cuda.current_stream().wait_stream(side)
    pool = torch.cuda.graph_pool_handle()
    fwd, bwd = torch.cuda.CUDAGraph(), torch.cuda.CUDAGraph()
    with torch.cuda.graph(fwd, pool=pool):
        static_out = model(hidden_states=static_px, grid_thw=grid)
    with torch.cuda.graph(bwd, pool=pool):
        static_grads = torch.autograd.grad(static_out, params, static_gout)
    for seed in (1, 2, 1):
        px, gout = inputs(seed)
        out_e, grads_e = eager(px, gout)
        static_px.copy_(px)
        static_gout.copy_(gout)
        fwd.replay()
        bwd.replay()
        torch.cuda.synchronize()
        assert torch.equal(static_out.detach(), out_e), f"output, inputs {seed}"
        for i, (a, b) in enumerate(zip(static_grads, grads_e)):
            assert torch.equal(a, b), f"gradient {i}, inputs {seed}"
