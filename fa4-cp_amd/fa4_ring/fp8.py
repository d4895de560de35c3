"""FP8 producer: OCP e4m3 shards and their descales for the e4m3 ring sweep.

The reference leaves this step to its caller (README.md:63-70: pass e4m3 q/k/v shards and
per-tensor descales, the k/v ones all-gathered and indexed by source rank; Descales at
ring_attention.py:43-52).  The recipe is the one its FP8 inputs assume:
``scale = amax / 448``, ``x8 = clamp(x / scale, -448, 448).to(float8_e4m3fn)``,
descale = scale.  Here it is one library call per tensor (``fa4cp_quantize_e4m3``: an amax
pass and a quantise pass over HBM) instead of the four torch passes.
"""

from __future__ import annotations

import ctypes
from typing import List, Optional, Sequence, Tuple

import torch

from . import _lib
from .ring_attention import Descales


def quantize_e4m3(x: torch.Tensor, *, heads_per_scale: int = 0,
                  out: Optional[torch.Tensor] = None) -> Tuple[torch.Tensor, torch.Tensor]:
    """x [rows, h, d] (bf16 / fp16 / fp32, on the device, unit stride in d) ->
    (x8 [rows, h, d] float8_e4m3fn contiguous, descale float32).

    ``heads_per_scale`` 0 gives one scale (a 0-dim descale); g > 0 one scale per g
    consecutive heads (a [h / g] descale): 1 for K/V per kv head, ``H_q / H_kv`` for Q in
    the (1, H_kv) layout of the sweep's q descale.  An all-zero group gets scale 1."""
    lib = _lib.load()
    assert x.is_cuda and x.dim() == 3 and x.stride(2) == 1, "x must be a [rows, h, d] device tensor, unit stride in d"
    rows, h, d = x.shape
    g = int(heads_per_scale)
    assert g == 0 or (g > 0 and h % g == 0), f"heads_per_scale {g} must be 0 or divide h = {h}"
    nscale = 1 if g == 0 else h // g
    if out is None:
        out = torch.empty((rows, h, d), dtype=torch.float8_e4m3fn, device=x.device)
    assert out.shape == (rows, h, d) and out.dtype == torch.float8_e4m3fn and out.is_contiguous() \
        and out.device == x.device, f"out must be a contiguous [{rows}, {h}, {d}] float8_e4m3fn tensor on {x.device}"
    amax = torch.empty(nscale, dtype=torch.float32, device=x.device)
    descale = torch.empty(nscale, dtype=torch.float32, device=x.device)
    a = _lib.QuantArgs()
    a.x, a.rows, a.h, a.d = x.data_ptr(), rows, h, d
    a.row_stride, a.head_stride = x.stride(0), x.stride(1)
    a.dtype = _lib.dtype_code(x.dtype)
    a.heads_per_scale = g
    a.amax, a.descale, a.y = amax.data_ptr(), descale.data_ptr(), out.data_ptr()
    _lib.check(lib.fa4cp_quantize_e4m3(ctypes.byref(a), _lib.stream_handle(x.device)), "fa4cp_quantize_e4m3")
    return out, (descale.reshape(()) if g == 0 else descale)


QUANT_MAX_TENSORS = 33  # FA4CP_QUANT_MAX_TENSORS
# Input bytes of one call's tensors.  The second pass starts on what the first one left in the 256 MB last-level cache;
# beyond that a call with fewer tensors reads more of its input from there (five of 1510 MB in all: together
# 756 us, in calls of up to 384 MB 688; 768 MB in five 359 and 357; smaller calls lose: 320 MB in 17 tensors 168,
# in two calls 188).
QUANT_MAX_BYTES = 384 << 20


def _quant_calls(xs: Sequence[torch.Tensor]) -> List[range]:
    """The tensors of each fa4cp_quantize_e4m3_many call: at most QUANT_MAX_TENSORS, and QUANT_MAX_BYTES
    where they are several."""
    calls, first, held = [], 0, 0
    for i, x in enumerate(xs):
        size = x.numel() * x.element_size()
        if i > first and (i - first == QUANT_MAX_TENSORS or held + size > QUANT_MAX_BYTES):
            calls.append(range(first, i))
            first, held = i, 0
        held += size
    return calls + [range(first, len(xs))]


def quantize_e4m3_many(xs: Sequence[torch.Tensor], *, heads_per_scale: Sequence[int]
                       ) -> List[Tuple[torch.Tensor, torch.Tensor]]:
    """quantize_e4m3 of every xs[i] with heads_per_scale[i], three launches for up to 33 tensors and 384
    MB (fa4cp_quantize_e4m3_many).  The tensors share a device and dtype; the descales are views of
    one small tensor."""
    lib = _lib.load()
    dev, nscale = xs[0].device, []
    for x, g in zip(xs, heads_per_scale):
        assert x.is_cuda and x.dim() == 3 and x.stride(2) == 1, \
            "x must be a [rows, h, d] device tensor, unit stride in d"
        assert x.device == dev and x.dtype == xs[0].dtype, "the tensors must share a device and dtype"
        assert g == 0 or (g > 0 and x.shape[1] % g == 0), f"heads_per_scale {g} must be 0 or divide h = {x.shape[1]}"
        nscale.append(1 if g == 0 else x.shape[1] // g)
    words = torch.empty(2 * sum(nscale), dtype=torch.float32, device=dev)  # amax words, then descales
    amax, descales = words.data_ptr(), words[sum(nscale):].split(nscale)
    code, stream, out = _lib.dtype_code(xs[0].dtype), _lib.stream_handle(dev), []
    for part in _quant_calls(xs):
        args = (_lib.QuantArgs * len(part))()
        for a, i in zip(args, part):
            x = xs[i]
            rows, a.h, a.d = x.shape
            y = torch.empty((rows, a.h, a.d), dtype=torch.float8_e4m3fn, device=dev)
            a.x, a.rows, a.dtype, a.heads_per_scale = x.data_ptr(), rows, code, heads_per_scale[i]
            a.row_stride, a.head_stride, _ = x.stride()
            a.amax, a.descale, a.y = amax, descales[i].data_ptr(), y.data_ptr()
            amax += 4 * nscale[i]
            out.append((y, descales[i] if heads_per_scale[i] else descales[i].reshape(())))
        _lib.check(lib.fa4cp_quantize_e4m3_many(args, len(part), stream), "fa4cp_quantize_e4m3_many")
    return out


QUANT_MAX_SCALES = 1024  # FA4CP_QUANT_MAX_SCALES


def quantize_e4m3_into(x: torch.Tensor, out: torch.Tensor, descale: torch.Tensor, *,
                       heads_per_scale: int = 0) -> None:
    """quantize_e4m3 into caller-provided ``out`` ([rows, h, d] float8_e4m3fn, contiguous) and
    ``descale`` (float32, one element per scale, contiguous), allocating nothing on the
    device: the amax workspace is the library's static per-GPU array
    (fa4cp_quantize_e4m3_noalloc), so this can run where allocation is not allowed.  At most
    QUANT_MAX_SCALES scales.  Calls that overlap on one GPU (on different streams) share that
    workspace and race."""
    lib = _lib.load()
    assert x.is_cuda and x.dim() == 3 and x.stride(2) == 1, "x must be a [rows, h, d] device tensor, unit stride in d"
    rows, h, d = x.shape
    g = int(heads_per_scale)
    assert g == 0 or (g > 0 and h % g == 0), f"heads_per_scale {g} must be 0 or divide h = {h}"
    nscale = 1 if g == 0 else h // g
    assert nscale <= QUANT_MAX_SCALES, f"{nscale} scales exceed the static workspace ({QUANT_MAX_SCALES})"
    assert out.shape == (rows, h, d) and out.dtype == torch.float8_e4m3fn and out.is_contiguous() \
        and out.device == x.device, f"out must be a contiguous [{rows}, {h}, {d}] float8_e4m3fn tensor on {x.device}"
    assert descale.numel() == nscale and descale.dtype == torch.float32 and descale.is_contiguous() \
        and descale.device == x.device, f"descale must be {nscale} contiguous float32 values on {x.device}"
    a = _lib.QuantArgs()
    a.x, a.rows, a.h, a.d = x.data_ptr(), rows, h, d
    a.row_stride, a.head_stride = x.stride(0), x.stride(1)
    a.dtype = _lib.dtype_code(x.dtype)
    a.heads_per_scale = g
    a.amax, a.descale, a.y = None, descale.data_ptr(), out.data_ptr()
    with torch.cuda.device(x.device):  # the library looks up the current device's workspace
        rc = lib.fa4cp_quantize_e4m3_noalloc(ctypes.byref(a), _lib.stream_handle(x.device))
    _lib.check(rc, "fa4cp_quantize_e4m3_noalloc")


def quantize_ring(local_q: torch.Tensor, k_shards: Sequence[torch.Tensor], v_shards: Sequence[torch.Tensor],
                  *, per_head: bool = False
                  ) -> Tuple[torch.Tensor, List[torch.Tensor], List[torch.Tensor], Descales]:
    """The e4m3 inputs of one rank's sweep: its local q and every source rank's k / v shard
    quantised, with the Descales ring_flash_attn takes (k / v indexed by source rank).
    ``per_head`` scales q per kv-head group and k / v per kv head; otherwise per tensor."""
    h_q, h_kv = local_q.shape[1], k_shards[0].shape[1]
    assert h_q % h_kv == 0
    g = 1 if per_head else 0
    n = len(k_shards)
    xs = [local_q, *k_shards, *v_shards]
    groups = [(h_q // h_kv) if per_head else 0] + [g] * (n + len(v_shards))
    if all(x.dtype == local_q.dtype and x.device == local_q.device for x in xs):
        (q8, qd), *kv = quantize_e4m3_many(xs, heads_per_scale=groups)
    else:
        (q8, qd), *kv = [quantize_e4m3(x, heads_per_scale=hs) for x, hs in zip(xs, groups)]
    k8, kd = zip(*kv[:n])
    v8, vd = zip(*kv[n:])
    return q8, list(k8), list(v8), Descales(q=qd, k=list(kd), v=list(vd))
