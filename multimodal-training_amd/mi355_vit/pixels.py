"""Input side on the GPU: decoded RGB frames -> (resize ->) ``pixel_values`` and ``image_grid_thw``.

The reference produces these two tensors on CPU dataloader workers: ``python/data/preprocessing.py:134`` calls
``processor.apply_chat_template``, whose image processor (transformers 4.57.0, ``Qwen2VLImageProcessor``)
rescales, normalises and cuts every image into ``[grid_t * grid_h * grid_w, 1176]`` rows, and
``python/data/collator.py:134-156`` concatenates the samples.  ``patchify`` does the same for frames that are
already on the GPU as uint8 ``[frames, height, width, 3]`` (height and width multiples of 28, i.e. after the
processor's resize step, which stays where the frames are decoded), for the whole batch in one launch, with the
processor's arithmetic (float32 results are bit-identical to a numpy restatement of it) and, optionally, the cast
to the model dtype that the tower applies first.

``resize_frames`` is the step in front of it: ``PIL.Image.resize`` for 8-bit RGB frames (BILINEAR: the reference's own
fixed-size resize, ``python/data/preprocessing.py:126-131``; BICUBIC: the image processor's resize to the
``smart_resize`` target), bit for bit, as two resampling passes on the GPU; the coefficient tables are computed on the
host exactly as Pillow computes them.  ``preprocess`` chains smart_resize -> resize -> patchify for still images.

There is no CPU path: frames must live on the GPU and the HIP library must be built.
"""

from __future__ import annotations

import ctypes as C
import functools
import itertools
import math
import struct
from typing import Optional, Sequence, Tuple

import numpy as np
import torch

from . import _lib
from .ops import _stream

OPENAI_CLIP_MEAN = (0.48145466, 0.4578275, 0.40821073)
OPENAI_CLIP_STD = (0.26862954, 0.26130258, 0.27577711)
PATCH_SIZE, TEMPORAL_PATCH_SIZE, MERGE_SIZE = 14, 2, 2

_IMAGE_FORMAT = "Q4iq"  # pixels, frames, height, width, reserved, first_row
assert struct.calcsize("<" + _IMAGE_FORMAT) == C.sizeof(_lib.Image) == 32
_HOST_TABLE_IMAGES = 64  # image tables up to this length travel with the launch


def grid_thw_of(frames: Sequence[torch.Tensor]) -> torch.Tensor:
    """``image_grid_thw`` ([n, 3] int64, CPU) of resized frame stacks, as the processor reports it."""
    rows = []
    for i, f in enumerate(frames):
        if f.dim() != 4 or f.shape[3] != 3 or f.dtype != torch.uint8:
            raise ValueError(f"image {i}: expected uint8 [frames, height, width, 3], got {f.dtype} {tuple(f.shape)}")
        n, h, w, _ = f.shape
        unit = PATCH_SIZE * MERGE_SIZE
        if n < 1 or h < unit or w < unit or h % unit or w % unit:
            raise ValueError(f"image {i}: {n} frames of {h}x{w}; height and width must be multiples of {unit} "
                             "(run the processor's resize first)")
        rows.append(((n + TEMPORAL_PATCH_SIZE - 1) // TEMPORAL_PATCH_SIZE, h // PATCH_SIZE, w // PATCH_SIZE))
    return torch.tensor(rows, dtype=torch.int64).reshape(-1, 3)


def _packed(form: str, rows: Sequence[tuple]) -> bytes:
    return struct.pack("<" + form * len(rows), *itertools.chain.from_iterable(rows))


def _image_table(frames: Sequence[torch.Tensor], what: str):
    """Checks the frame stacks and builds the table of ``mvit_image`` entries (32 bytes per image).  Returns (frames as a
    list, image_grid_thw, table on the host, total rows)."""
    frames = list(frames)
    if not frames:
        raise ValueError(f"{what}: no images")
    grid = grid_thw_of(frames)
    device = frames[0].device
    for i, f in enumerate(frames):
        if not f.is_cuda or f.device != device:
            raise RuntimeError(f"image {i} on {f.device}: frames must be on one GPU (there is no CPU path)")
        if not f.is_contiguous():
            raise RuntimeError(f"image {i}: frames must be contiguous")
    rows, total = [], 0
    for f, (t, gh, gw) in zip(frames, grid.tolist()):
        rows.append((f.data_ptr(), f.shape[0], f.shape[1], f.shape[2], 0, total))
        total += t * gh * gw
    rows.append((0, 0, 0, 0, 0, total))
    return frames, grid, _packed(_IMAGE_FORMAT, rows), total


def _on_device(table: bytes, device: torch.device) -> torch.Tensor:
    """A table of a few tens of bytes per image on the GPU.  It goes through pinned memory, which the allocator keeps until the copy
    is done, so the host need not wait for the GPU; a stream that is being captured could not replay that."""
    host = torch.frombuffer(bytearray(table), dtype=torch.uint8)
    if torch.cuda.is_current_stream_capturing():
        return host.to(device)
    return torch.empty(len(table), dtype=torch.uint8, pin_memory=True).copy_(host).to(device, non_blocking=True)


def _dtype_code(dtype: torch.dtype) -> int:
    if dtype == torch.float32:
        return _lib.F32
    if dtype == torch.bfloat16:
        return _lib.BF16
    raise TypeError(f"unsupported dtype {dtype} (float32 and bfloat16 only)")


def _norm(image_mean, image_std, rescale_factor) -> tuple:
    return (float(rescale_factor), *(float(np.float32(v)) for v in image_mean), *(float(np.float32(v)) for v in image_std))


def _patchify_table(table: bytes, n: int, total: int, out: torch.Tensor, code: int, norm: tuple) -> None:
    """The launch, on the current device."""
    lib, stream = _lib.load(), _stream(out)
    if n <= _HOST_TABLE_IMAGES:
        rc = lib.mvit_patchify_host_table(table, n, total, out.data_ptr(), *norm, code, stream)
    else:
        dev_table = _on_device(table, out.device)
        rc = lib.mvit_patchify(dev_table.data_ptr(), n, total, out.data_ptr(), *norm, code, stream)
    _lib.check(rc, "mvit_patchify")


def patchify(frames: Sequence[torch.Tensor], dtype: torch.dtype = torch.float32,
             image_mean: Sequence[float] = OPENAI_CLIP_MEAN, image_std: Sequence[float] = OPENAI_CLIP_STD,
             rescale_factor: float = 1.0 / 255.0, out: Optional[torch.Tensor] = None) -> Tuple[torch.Tensor, torch.Tensor]:
    """Frames of a batch of images / videos -> (``pixel_values`` [rows, 1176] on the GPU, ``image_grid_thw`` [n, 3]).

    ``frames``: one contiguous uint8 GPU tensor ``[frames, height, width, 3]`` per image (one frame) or video.
    ``dtype``: float32 (what the processor returns) or bfloat16 (what the tower casts it to).
    """
    code = _dtype_code(dtype)
    frames, grid, table, total = _image_table(frames, "patchify")
    n, device = len(frames), frames[0].device
    if out is None:
        out = torch.empty((total, _lib.PIXEL_ROW), dtype=dtype, device=device)
    elif out.shape != (total, _lib.PIXEL_ROW) or out.dtype != dtype or out.device != device or not out.is_contiguous():
        raise RuntimeError(f"patchify: out must be a contiguous {dtype} [{total}, {_lib.PIXEL_ROW}] tensor on {device}")
    with torch.cuda.device(device):
        _patchify_table(table, n, total, out, code, _norm(image_mean, image_std, rescale_factor))
    return out, grid


PACKED_PATCH_K = 1344  # 28 pixel lines of a patch (frame of the pair, y), each 14 x 3 bytes padded to 48


def frames_fit_fused_patch_embed(frames: Sequence[torch.Tensor]) -> bool:
    """Whether ``patch_embed_frames`` can read these frame stacks: 4-byte aligned buffers below 2 GiB each."""
    return all(f.data_ptr() % 4 == 0 and f.numel() < 2**31 for f in frames)


def pack_patch_embed_weight(weight: torch.Tensor) -> torch.Tensor:
    """The patch-embedding weight ([embed_dim, 1176] or the Conv3d's [embed_dim, 3, 2, 14, 14], float32 or bfloat16)
    in the contraction order of ``patch_embed_frames``: bfloat16 ``[embed_dim, 1344]``."""
    w = weight.detach().reshape(weight.shape[0], -1)
    if w.shape[1] != _lib.PIXEL_ROW or w.dtype not in (torch.float32, torch.bfloat16) or not w.is_cuda:
        raise ValueError(f"pack_patch_embed_weight: expected a float32 / bfloat16 GPU weight with {_lib.PIXEL_ROW} inputs, got {w.dtype} {tuple(w.shape)} on {w.device}")
    if w.stride(1) != 1:
        w = w.contiguous()
    packed = torch.empty((w.shape[0], PACKED_PATCH_K), dtype=torch.bfloat16, device=w.device)
    lib = _lib.load()
    with torch.cuda.device(w.device):
        rc = lib.mvit_patch_embed_pack_weight(w.data_ptr(), _lib.BF16 if w.dtype == torch.bfloat16 else _lib.F32, w.stride(0),
                                              w.shape[0], packed.data_ptr(), torch.cuda.current_stream(w.device).cuda_stream)
    _lib.check(rc, "mvit_patch_embed_pack_weight")
    return packed


def patch_embed_frames(frames: Sequence[torch.Tensor], packed_weight: torch.Tensor, dtype: torch.dtype = torch.bfloat16,
                       image_mean: Sequence[float] = OPENAI_CLIP_MEAN, image_std: Sequence[float] = OPENAI_CLIP_STD,
                       rescale_factor: float = 1.0 / 255.0) -> Tuple[torch.Tensor, torch.Tensor]:
    """Frames -> (patch embeddings ``[rows, embed_dim]``, ``image_grid_thw``): ``patchify(frames, bfloat16)`` times the
    weight, in one kernel that makes the rows on the fly and never writes them.  ``packed_weight`` comes from
    ``pack_patch_embed_weight``.  Raises ``_lib.Unsupported`` when the normalisation constants cannot be folded into
    one multiply-add per byte without changing a bfloat16 value (the caller then uses ``patchify`` and a GEMM)."""
    if dtype not in (torch.float32, torch.bfloat16):
        raise TypeError(f"unsupported dtype {dtype} (float32 and bfloat16 only)")
    frames, grid, table, total = _image_table(frames, "patch_embed_frames")
    device = frames[0].device
    if not frames_fit_fused_patch_embed(frames):
        raise RuntimeError("patch_embed_frames: frame buffers must be 4-byte aligned and smaller than 2 GiB")
    if (packed_weight.dim() != 2 or packed_weight.shape[1] != PACKED_PATCH_K or packed_weight.dtype != torch.bfloat16
            or packed_weight.device != device or not packed_weight.is_contiguous()):
        raise ValueError("patch_embed_frames: packed_weight must be the contiguous bfloat16 [embed_dim, 1344] result of pack_patch_embed_weight on the frames' GPU")
    out = torch.empty((total, packed_weight.shape[0]), dtype=dtype, device=device)
    dev_table = _on_device(table, device)
    mean = [float(np.float32(m)) for m in image_mean]
    std = [float(np.float32(s)) for s in image_std]
    lib = _lib.load()
    with torch.cuda.device(device):
        rc = lib.mvit_patch_embed_frames(dev_table.data_ptr(), len(frames), total, packed_weight.data_ptr(), packed_weight.shape[0],
                                         out.data_ptr(), out.stride(0), _lib.BF16 if dtype == torch.bfloat16 else _lib.F32,
                                         float(rescale_factor), *mean, *std, torch.cuda.current_stream(device).cuda_stream)
    _lib.check(rc, "mvit_patch_embed_frames")
    return out, grid


# ------------------------------------------------------------------------------------------------ resize

BILINEAR, BICUBIC = "bilinear", "bicubic"
_FILTER_SUPPORT = {BILINEAR: 1.0, BICUBIC: 2.0}
_PRECISION_BITS = 22  # Pillow: 32 - 8 bits of pixel - 2 bits of head-room


def smart_resize(height: int, width: int, factor: int = PATCH_SIZE * MERGE_SIZE, min_pixels: int = 56 * 56,
                 max_pixels: int = 14 * 14 * 4 * 1280) -> Tuple[int, int]:
    """The (height, width) the image processor resizes to (transformers 4.57.0 ``smart_resize``): multiples of
    ``factor``, pixel count within [min_pixels, max_pixels], aspect ratio kept as closely as that allows."""
    if height <= 0 or width <= 0:
        raise ValueError(f"smart_resize: {height}x{width}")
    if max(height, width) / min(height, width) > 200:
        raise ValueError(f"absolute aspect ratio must be smaller than 200, got {max(height, width) / min(height, width)}")
    h_bar = round(height / factor) * factor
    w_bar = round(width / factor) * factor
    if h_bar * w_bar > max_pixels:
        beta = math.sqrt((height * width) / max_pixels)
        h_bar = max(factor, math.floor(height / beta / factor) * factor)
        w_bar = max(factor, math.floor(width / beta / factor) * factor)
    elif h_bar * w_bar < min_pixels:
        beta = math.sqrt(min_pixels / (height * width))
        h_bar = math.ceil(height * beta / factor) * factor
        w_bar = math.ceil(width * beta / factor) * factor
    return h_bar, w_bar


def resample_coefficients(in_size: int, out_size: int, resample: str = BICUBIC) -> Tuple[np.ndarray, np.ndarray]:
    """Window bounds ([out_size, 2] int32: first input index, tap count) and 22-bit fixed-point weights ([out_size, ksize]
    int32) of one axis, as Pillow's Resample.c computes them (precompute_coeffs + normalize_coeffs_8bpc): the filter's
    support is widened by the scale factor when shrinking; weights are evaluated and normalised in double precision, the
    sum taken tap by tap in index order.  Every step is one IEEE double operation, in the order of the C source, so the
    tables are Pillow's bit for bit."""
    if resample not in _FILTER_SUPPORT:
        raise ValueError(f"resample must be '{BILINEAR}' or '{BICUBIC}', got {resample!r}")
    if in_size < 1 or out_size < 1:
        raise ValueError(f"resample_coefficients: sizes {in_size} -> {out_size}")
    scale = in_size / out_size
    filterscale = scale if scale >= 1.0 else 1.0
    support = _FILTER_SUPPORT[resample] * filterscale
    ksize = int(math.ceil(support)) * 2 + 1
    ss = 1.0 / filterscale
    center = (np.arange(out_size, dtype=np.float64) + 0.5) * scale
    xmin = np.maximum((center - support + 0.5).astype(np.int64), 0)  # (int) truncates; the operand is > -1 here
    xmax = np.minimum((center + support + 0.5).astype(np.int64), in_size) - xmin
    taps = np.arange(ksize, dtype=np.int64)[None, :]
    active = taps < xmax[:, None]
    x = np.abs(((taps + xmin[:, None]).astype(np.float64) - center[:, None] + 0.5) * ss)
    if resample == BILINEAR:
        w = np.where(x < 1.0, 1.0 - x, 0.0)
    else:
        a = -0.5
        w = np.where(x < 1.0, ((a + 2.0) * x - (a + 3.0)) * x * x + 1, np.where(x < 2.0, (((x - 5) * x + 8) * x - 4) * a, 0.0))
    w = np.where(active, w, 0.0)
    ww = np.cumsum(w, axis=1)[:, -1:]  # left-to-right sum, like the C loop (numpy's sum() adds pairwise)
    w = np.where(ww != 0.0, w / np.where(ww != 0.0, ww, 1.0), w)
    fixed = np.where(w < 0, -0.5 + w * (1 << _PRECISION_BITS), 0.5 + w * (1 << _PRECISION_BITS)).astype(np.int64)  # truncation
    kk = np.where(active, fixed, 0).astype(np.int32)
    bounds = np.stack([xmin, xmax], axis=1).astype(np.int32)
    return bounds, kk


@functools.lru_cache(maxsize=64)
def _device_coefficients(in_size: int, out_size: int, resample: str, device_index: int):
    bounds, kk = resample_coefficients(in_size, out_size, resample)
    dev = torch.device("cuda", device_index)
    return torch.from_numpy(bounds).to(dev), torch.from_numpy(kk).to(dev), kk.shape[1]


def _check_resizable(frames: torch.Tensor) -> None:
    if frames.dim() != 4 or frames.dtype != torch.uint8 or frames.shape[0] < 1:
        raise ValueError(f"resize_frames: expected uint8 [frames, height, width, channels], got {frames.dtype} {tuple(frames.shape)}")
    if not frames.is_cuda:
        raise RuntimeError("resize_frames: frames must be on the GPU (there is no CPU path)")
    if not frames.is_contiguous():
        raise RuntimeError("resize_frames: frames must be contiguous")


_RESIZED_FORMAT = "3Q4iq"  # mvit_resized_image: src, bounds, kk, src_height, height, width, ksize, first_row
_JOB_FORMAT = "8q2i"  # mvit_resample_job: src, dst, bounds, kk, outer, in_len, out_len, inner, ksize, reserved


def _resample_passes(jobs: list, stream: int) -> None:
    if jobs:
        _lib.check(_lib.load().mvit_resample_u8_batch(_packed(_JOB_FORMAT, jobs), len(jobs), stream), "mvit_resample_u8_batch")


def _across_job(src: int, dst: int, n: int, h: int, w: int, ow: int, ch: int, resample: str, index: int, held: list) -> tuple:
    bounds, kk, ksize = _device_coefficients(w, ow, resample, index)
    held.append((bounds, kk))  # tables may leave the cache before the launch is queued
    return (src, dst, bounds.data_ptr(), kk.data_ptr(), n * h, w, ow, ch, ksize, 0)


def _down_job(src: int, dst: int, n: int, h: int, oh: int, ow: int, ch: int, resample: str, index: int, held: list) -> tuple:
    bounds, kk, ksize = _device_coefficients(h, oh, resample, index)
    held.append((bounds, kk))
    return (src, dst, bounds.data_ptr(), kk.data_ptr(), n, h, oh, ow * ch, ksize, 0)


def resize_frames(frames: torch.Tensor, out_height: int, out_width: int, resample: str = BICUBIC) -> torch.Tensor:
    """``PIL.Image.resize((out_width, out_height), resample)`` applied to every frame of a contiguous uint8 GPU tensor
    ``[frames, height, width, 3]``, bit for bit: a horizontal pass into an 8-bit intermediate image, then a vertical
    pass (a pass whose size does not change is skipped, as Pillow does)."""
    _check_resizable(frames)
    if out_height < 1 or out_width < 1:
        raise ValueError(f"resize_frames: target {out_height}x{out_width}")
    device = frames.device
    index, (n, h, w, ch) = device.index or 0, frames.shape
    cur, across, down, held = frames, [], [], []
    if w != out_width:
        cur = torch.empty((n, h, out_width, ch), dtype=torch.uint8, device=device)
        across.append(_across_job(frames.data_ptr(), cur.data_ptr(), n, h, w, out_width, ch, resample, index, held))
    between = cur  # the intermediate image lives until both launches are queued
    if h != out_height:
        cur = torch.empty((n, out_height, out_width, ch), dtype=torch.uint8, device=device)
        down.append(_down_job(between.data_ptr(), cur.data_ptr(), n, h, out_height, out_width, ch, resample, index, held))
    with torch.cuda.device(device):
        stream = _stream(frames)
        _resample_passes(across, stream)
        _resample_passes(down, stream)
    return frames.clone() if cur is frames else cur


def preprocess(images: Sequence[torch.Tensor], dtype: torch.dtype = torch.float32, min_pixels: int = 56 * 56,
               max_pixels: int = 14 * 14 * 4 * 1280, resample: str = BICUBIC) -> Tuple[torch.Tensor, torch.Tensor]:
    """Decoded still images (uint8 GPU tensors ``[1, height, width, 3]`` of any size) -> (``pixel_values``,
    ``image_grid_thw``): the image processor's smart_resize + resize + rescale + normalise + patchify, on the GPU.

    The horizontal passes of all images are one launch, the vertical ones and patchify another, and the images in between share one
    allocation: the host would take longer than the GPU with a tensor for each (four photographs 69 us of host time, now 40)."""
    images, plans = list(images), []  # per image: height, width, resized height and width
    for i, f in enumerate(images):
        if f.dim() != 4 or f.shape[0] != 1 or f.shape[3] != 3:
            raise ValueError(f"image {i}: expected uint8 [1, height, width, 3], got {tuple(f.shape)}")
        _, h, w, _ = f.shape
        plans.append((h, w) + smart_resize(h, w, min_pixels=min_pixels, max_pixels=max_pixels))
        _check_resizable(f)
        if f.device != images[0].device:
            raise RuntimeError(f"image {i} on {f.device}: frames must be on one GPU (there is no CPU path)")
    if not images:
        raise ValueError("patchify: no images")
    code, device = _dtype_code(dtype), images[0].device
    index, ch, size, places = device.index or 0, 3, 0, []
    for h, w, oh, ow in plans:  # places of the images as wide as they have to be
        places.append(size)
        size += -(-h * ow * ch // 256) * 256 if w != ow else 0
    between = torch.empty(size, dtype=torch.uint8, device=device)  # lives until the last launch is queued
    base, across, held, rows, grid, total = between.data_ptr(), [], [], [], [], 0
    for f, (h, w, oh, ow), place in zip(images, plans, places):
        at = f.data_ptr()
        if w != ow:
            across.append(_across_job(at, base + place, 1, h, w, ow, ch, resample, index, held))
            at = base + place
        bounds, kk, ksize = 0, 0, 0
        if h != oh:
            job = _down_job(at, 0, 1, h, oh, ow, ch, resample, index, held)
            bounds, kk, ksize = job[2], job[3], job[8]
        rows.append((at, bounds, kk, h, oh, ow, ksize, total))
        grid.append((1, oh // PATCH_SIZE, ow // PATCH_SIZE))
        total += (oh // PATCH_SIZE) * (ow // PATCH_SIZE)
    rows.append((0, 0, 0, 0, 0, 0, 0, total))
    out = torch.empty((total, _lib.PIXEL_ROW), dtype=dtype, device=device)
    norm = _norm(OPENAI_CLIP_MEAN, OPENAI_CLIP_STD, 1.0 / 255.0)
    with torch.cuda.device(device):
        stream = _stream(out)
        _resample_passes(across, stream)
        try:
            _lib.check(_lib.load().mvit_resize_patchify(_packed(_RESIZED_FORMAT, rows), len(images), total, out.data_ptr(), *norm, code, stream),
                       "mvit_resize_patchify")
        except _lib.Unsupported:  # many images, or one made a quarter as high and less
            _resize_down_and_patchify(rows, out, code, norm, stream, device)
    return out, torch.tensor(grid, dtype=torch.int64)


def _resize_down_and_patchify(rows: list, out: torch.Tensor, code: int, norm: tuple, stream: int, device: torch.device) -> None:
    """The vertical passes in one launch and patchify in another, for the table of ``mvit_resize_patchify``."""
    ch, size, places = 3, 0, []
    for _, bounds, _, _, oh, ow, _, _ in rows[:-1]:
        places.append(size)
        size += -(-oh * ow * ch // 256) * 256 if bounds else 0
    resized = torch.empty(size, dtype=torch.uint8, device=device)
    down, images = [], []
    for (at, bounds, kk, h, oh, ow, ksize, first), place in zip(rows, places):
        if bounds:
            down.append((at, resized.data_ptr() + place, bounds, kk, 1, h, oh, ow * ch, ksize, 0))
            at = resized.data_ptr() + place
        images.append((at, 1, oh, ow, 0, first))
    images.append((0, 0, 0, 0, 0, rows[-1][-1]))
    _resample_passes(down, stream)
    _patchify_table(_packed(_IMAGE_FORMAT, images), len(images) - 1, rows[-1][-1], out, code, norm)
