"""The backward where several workgroups share a tile, and its gradients in the inputs' type
(fa4cp_ring_sweep_bwd_shared).

The shared sums are the unshared ones' float32 terms in another order: every partial sum of n terms is
off by at most n 2^-24 of the sum of their magnitudes, far below the 1e-5 of the largest gradient
allowed here.  The gradients in 16 bits are the float32 ones rounded once, so they equal them
bit for bit after that rounding."""

import ctypes

import pytest
import torch

import plans
from fa4_ring import LocalKVRing, RingConfig, _lib, ring_flash_attn, ring_flash_attn_backward, ring_flash_attn_func
from fa4_ring.backward import _backward
from gpu_helpers import DEV, say

pytestmark = pytest.mark.gpu

CASES = [  # (local lens, H, H_kv, D, cp, rank, dtype, what is shared: dq's and dk / dv's tiles)
    ([512], 8, 2, 128, 4, 1, torch.bfloat16, "dq kv"),
    ([386], 4, 4, 64, 8, 2, torch.float16, "dq"),         # one query head per kv head, partial blocks
    ([1024], 8, 2, 128, 2, 0, torch.bfloat16, "dq kv"),   # no earlier source
    ([640], 16, 2, 128, 8, 7, torch.float16, "dq kv"),    # no later source
    ([1024, 66, 0, 514], 4, 1, 128, 8, 3, torch.bfloat16, "dq"),  # packed
    ([2048], 16, 4, 64, 4, 1, torch.bfloat16, "dq"),
    ([512], 8, 2, 256, 4, 1, torch.bfloat16, "dq kv"),    # head dim 256: the shares summed by kernels of their own
    ([386], 8, 1, 256, 8, 5, torch.float16, "dq kv"),     # a partial key tile, tiles no row attends
    ([300, 0, 70, 2], 4, 1, 256, 4, 3, torch.bfloat16, "dq kv"),  # packed
    ([256], 8, 1, 256, 4, 0, torch.bfloat16, "dq kv"),    # the shorter row tiles whole beside shared ones
    ([4096], 16, 2, 256, 4, 1, torch.bfloat16, "kv"),
    ([2048], 16, 16, 256, 2, 0, torch.bfloat16, ""),      # more tiles than are shared
    ([2], 4, 2, 128, 4, 2, torch.bfloat16, ""),
]


@pytest.mark.parametrize("lens,h,h_kv,d,cp,rank,dtype,shared", CASES)
def test_shared_backward(lens, h, h_kv, d, cp, rank, dtype, shared, monkeypatch):
    say(f"shared backward lens={lens} h={h}/{h_kv} d={d} cp={cp} rank={rank} {dtype}")
    g = torch.Generator(device="cuda").manual_seed(23)
    total, packed = sum(lens), len(lens) > 1
    cu = torch.tensor([0] + torch.tensor(lens).cumsum(0).tolist(), dtype=torch.int32, device=DEV) if packed else None
    kw = dict(cu_seqlens=cu, max_seqlen=max(lens) if packed else None)
    mk = lambda hh: torch.randn(total, hh, d, generator=g, device=DEV).to(dtype)  # noqa: E731
    q, dout = mk(h), mk(h)
    ring = LocalKVRing([mk(h_kv) for _ in range(cp)], [mk(h_kv) for _ in range(cp)])
    cfg = RingConfig(cp_size=cp, cp_rank=rank)
    lk, lv = ring.kv(rank)
    out, lse = ring_flash_attn(q, lk, lv, cfg, group=ring, return_lse=True, **kw)

    lib = _lib.load()
    need = lib.fa4cp_ring_sweep_bwd_share_bytes(ctypes.byref(plans.backward_args(lens, h, h_kv, d, cp, rank)))
    assert (need > 0) == bool(shared)

    def grads(dt=torch.float32):
        r = _backward(dout, q, lk, lv, out, lse, cfg, ring, cu, kw["max_seqlen"], None, None, None, False, dt)
        return [r[0], *r[1], *r[2]]

    got = grads()
    for _ in range(6):  # the same bits every time, whichever workgroup sums
        assert all(torch.equal(x, y) for x, y in zip(grads(), got))
    for x, y in zip(grads(dtype), got):
        assert x.dtype == dtype and torch.equal(x, y.to(dtype))
    # unshared: the entry point without the second workspace
    monkeypatch.setattr(lib, "fa4cp_ring_sweep_bwd_share_bytes", lambda _: 0)  # (an attribute of the loaded library)
    for x, y in zip(grads(), got):
        assert (x - y).abs().max() <= 1e-5 * max(1e-3, float(x.abs().max()))
    monkeypatch.undo()
    # adding to what is there
    base = [torch.randn(x.shape, generator=g, device=DEV) for x in got]
    acc = [b.clone() for b in base]
    ring_flash_attn_backward(dout, q, lk, lv, out, lse, cfg, group=ring, dq=acc[0], dk=acc[1:1 + cp], dv=acc[1 + cp:],
                             accumulate=True, **kw)
    for x, b, y in zip(acc, base, got):
        assert torch.equal(x, b + y)
    with pytest.raises(RuntimeError, match="grad_dtype"):
        _backward(dout, q, lk, lv, out, lse, cfg, ring, cu, kw["max_seqlen"], None, None, None, True, dtype)


def test_autograd_gradients_are_the_rounded_ones():
    say("autograd gradients in the inputs' type")
    g = torch.Generator(device="cuda").manual_seed(4)
    mk = lambda hh: torch.randn(512, hh, 128, generator=g, device=DEV).to(torch.bfloat16).requires_grad_()  # noqa: E731
    q, ks, vs = mk(8), [mk(2) for _ in range(4)], [mk(2) for _ in range(4)]
    ring, cfg = LocalKVRing(ks, vs), RingConfig(cp_size=4, cp_rank=2)
    out = ring_flash_attn_func(q, ring, cfg)
    dout = torch.randn(out.shape, generator=g, device=DEV).to(torch.bfloat16)
    got = torch.autograd.grad(out, [q, *ks, *vs], dout)
    with torch.no_grad():
        o, lse = ring_flash_attn(q, ks[2], vs[2], cfg, group=ring, return_lse=True)
        dq, dk, dv = ring_flash_attn_backward(dout, q, ks[2], vs[2], o, lse, cfg, group=ring)
    assert all(torch.equal(x, y.to(torch.bfloat16)) for x, y in zip(got, [dq, *dk, *dv]))


@pytest.mark.parametrize("n,rows,h,h_kv,d,cp,rank", [
    (126, 126, 32, 32, 64, 16, 3),   # one key tile: no pair
    (130, 130, 32, 16, 128, 16, 5),  # one pair
    (386, 386, 16, 16, 128, 8, 0),   # no earlier source, the last tile partial
    (640, 640, 16, 8, 64, 8, 7),     # no later source, a tile without a partner
    (386, 900, 16, 16, 64, 8, 4),    # a shorter sequence than the tensors hold: the second tiles past its end,
    (130, 900, 16, 16, 128, 8, 4),   # and both
])
def test_paired_key_tiles(n, rows, h, h_kv, d, cp, rank):
    """One sequence (its own key tiles taken in pairs) against the same one packed with an empty one (never
    in pairs): each tile sums the same terms in the same order, so the bits are equal."""
    say(f"paired key tiles n={n} rows={rows} h={h}/{h_kv} d={d} cp={cp} rank={rank}")
    assert cp * h_kv * -(-rows // 128) > 256  # (else no tile is paired)
    g = torch.Generator(device="cuda").manual_seed(41)
    mk = lambda hh: torch.randn(rows, hh, d, generator=g, device=DEV).to(torch.bfloat16)  # noqa: E731
    q, dout = mk(h), mk(h)
    ring = LocalKVRing([mk(h_kv) for _ in range(cp)], [mk(h_kv) for _ in range(cp)])
    cfg = RingConfig(cp_size=cp, cp_rank=rank)
    lk, lv = ring.kv(rank)
    out, lse = torch.zeros_like(q), torch.zeros(rows, h, device=DEV)
    part = LocalKVRing([k[:n] for k in ring.k], [v[:n] for v in ring.v])
    out[:n], lse[:n] = ring_flash_attn(q[:n], *part.kv(rank), cfg, group=part, return_lse=True)
    one = dict(cu_seqlens=torch.tensor([0, n], dtype=torch.int32, device=DEV), max_seqlen=rows) if rows > n else {}
    two = dict(cu_seqlens=torch.tensor([0, n, n], dtype=torch.int32, device=DEV), max_seqlen=n)
    got = ring_flash_attn_backward(dout, q, lk, lv, out, lse, cfg, group=ring, **one)
    ref = ring_flash_attn_backward(dout, q, lk, lv, out, lse, cfg, group=ring, **two)
    for x, y in zip([*got[1], *got[2]], [*ref[1], *ref[2]]):
        assert torch.equal(x[:n], y[:n])
