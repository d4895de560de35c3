"""The split form of the fused sweep (fa4cp_ring_sweep_fwd_ws): several workgroups share a row
tile's keys and the last of them merges the shares.

Every case is run split and, over the same inputs, unsplit; the split result is checked against the
oracle's ring and against the unsplit one.  Those two differ by the rounding of their
probabilities (a share's are relative to its own maximum) and of the output: each is off by at
most u relative, the unit roundoff of its type, in either form, so the outputs differ by at most
about 4 u in the 2-norm.  The LSEs are fp32 sums in another order."""

import ctypes

import pytest
import torch

from fa4_ring import Descales, LocalKVRing, PagedKVRing, RingConfig, _lib, ring_flash_attn
from fa4_ring import ring_attention as RA
from gpu_helpers import DEV, TOL_BF16_OUT, TOL_FP8_OUT, TOL_LSE, say
from oracle import ring_oracle as O

pytestmark = pytest.mark.gpu

E4 = torch.float8_e4m3fn
CASES = [  # (local lens, H, H_kv, D, cp, rank, dtype, page size): row tiles of 256 / (heads per workgroup) rows
    ([512], 8, 2, 128, 4, 1, torch.bfloat16, 0),
    ([512], 8, 2, 128, 4, 3, torch.bfloat16, 256),     # no later source; shares start inside a page
    ([386], 8, 2, 128, 8, 0, torch.bfloat16, 128),     # no earlier source; a partial row tile and key tile
    ([386], 4, 4, 64, 8, 2, torch.float16, 0),         # one query head per kv head: row tiles of 256 and 130 rows
    ([62], 16, 1, 128, 16, 9, torch.float16, 0),       # the largest ring, one row tile, a half of 31 keys
    ([300], 6, 3, 64, 8, 5, torch.bfloat16, 0),        # two heads per workgroup, three head groups in turns
    ([258], 12, 12, 128, 4, 1, torch.bfloat16, 0),     # twelve head groups: neither a divisor nor a multiple of 8
    ([640], 16, 2, 256, 8, 3, torch.bfloat16, 384),    # 32-key tiles, twelve per page
    ([2], 4, 1, 128, 8, 3, torch.bfloat16, 0),         # two rows: one tile per step
    ([640, 2, 0, 322, 126], 4, 1, 128, 8, 2, torch.bfloat16, 0),    # packed: empty and short sequences
    ([640, 2, 0, 322, 126], 4, 1, 128, 8, 2, torch.bfloat16, 256),
    ([512], 8, 2, 128, 8, 0, E4, 0),                   # rank 0: the front rows take the causal precision rules
    ([768], 8, 2, 128, 4, 2, E4, 128),                 # one 128-key tile per page
    ([450], 8, 1, 256, 8, 5, E4, 0),
    ([400, 50, 262], 4, 2, 128, 8, 1, E4, 128),
]


def _unsplit(monkeypatch):
    launch = RA.launch_sweep
    monkeypatch.setattr(RA, "launch_sweep", lambda a, dev, kp=None, ws=None, n=0: launch(a, dev, kp))


def _shares(lens, h, h_kv, d, cp, rank, dtype):
    a = _lib.SweepArgs()
    a.total, a.h_q, a.h_kv, a.d, a.dtype = sum(lens), h, h_kv, d, _lib.dtype_code(dtype)
    a.cp_rank, a.cp_size = rank, cp
    if len(lens) > 1:
        a.cu, a.nseq, a.max_seqlen = 1 << 20, len(lens), max(lens)
    return _lib.load().fa4cp_ring_sweep_workspace_bytes(ctypes.byref(a), None)


@pytest.mark.parametrize("lens,h,h_kv,d,cp,rank,dtype,page", CASES)
def test_split_sweep(lens, h, h_kv, d, cp, rank, dtype, page, monkeypatch):
    say(f"split sweep lens={lens} h={h}/{h_kv} d={d} cp={cp} rank={rank} {dtype} page={page}")
    g = torch.Generator().manual_seed(17)
    total = sum(lens)
    cu = [0]
    for n in lens:
        cu.append(cu[-1] + n)

    def rand(*shape):
        return torch.randn(*shape, generator=g).to(torch.bfloat16 if dtype == E4 else dtype).to(dtype)

    q = rand(total, h, d)
    ks, vs = [rand(total, h_kv, d) for _ in range(cp)], [rand(total, h_kv, d) for _ in range(cp)]
    desc = None
    qs_, ks_, vs_ = 1.0, [1.0] * cp, [1.0] * cp
    if dtype == E4:
        qs_, ks_, vs_ = 0.8, [0.4 + 0.1 * r for r in range(cp)], [1.3 - 0.1 * r for r in range(cp)]
        desc = Descales(q=torch.tensor(qs_, device=DEV), k=[torch.tensor(x, device=DEV) for x in ks_],
                        v=[torch.tensor(x, device=DEV) for x in vs_])
    packed = len(lens) > 1
    kw = dict(descales=desc)
    if packed:
        kw.update(cu_seqlens=torch.tensor(cu, dtype=torch.int32, device=DEV), max_seqlen=max(lens))
    ring = LocalKVRing([x.to(DEV) for x in ks], [x.to(DEV) for x in vs])
    qd, lk, lv = q.to(DEV), ring.k[rank], ring.v[rank]
    cfg = RingConfig(cp_size=cp, cp_rank=rank)

    def sweep(group=ring):
        return ring_flash_attn(qd, lk, lv, cfg, group=group, return_lse=True, **kw)

    if max(lens) > 2:
        assert _shares(lens, h, h_kv, d, cp, rank, dtype) > 0, "the case is meant to be split"
    out, lse = sweep()
    ref, ref_lse = O.ring_rank(q.float() * qs_, [k.float() * s for k, s in zip(ks, ks_)],
                               [v.float() * s for v, s in zip(vs, vs_)], rank, cp, d ** -0.5, cu=cu if packed else None)
    assert (out.float().cpu() - ref).abs().max() <= (TOL_FP8_OUT if dtype == E4 else TOL_BF16_OUT)
    assert (lse.cpu() - ref_lse).abs().max() <= TOL_LSE
    # the same bits every time, whichever workgroup merges; and over a paged cache
    for _ in range(8):
        o, l = sweep()
        assert torch.equal(o, out) and torch.equal(l, lse)
    if page:
        paged = PagedKVRing.from_shards(ring.k, ring.v, page, cu if packed else None, spare_pages=2,
                                        generator=torch.Generator().manual_seed(5), fill=0.0)
        o, l = sweep(paged)
        assert torch.equal(o, out) and torch.equal(l, lse)
    _unsplit(monkeypatch)
    o, l = sweep()
    u = 2.0 ** -4 if dtype == E4 else 2.0 ** -11 if dtype == torch.float16 else 2.0 ** -8  # (e4m3 rounds P)
    assert (o.float() - out.float()).norm() <= 4 * u * o.float().norm()
    assert (l - lse).abs().max() <= 1e-5 * max(1.0, float(l.abs().max()))


def test_split_sweep_graph_replays():
    """A captured split sweep (the V^T launch that clears its counters, then the sweep) replayed five
    times with eager sweeps between: the eager result every time."""
    say("split sweep graph replays")
    g = torch.Generator(device="cuda").manual_seed(3)
    cp, rank = 4, 1
    mk = lambda hh: torch.randn(512, hh, 128, generator=g, device=DEV).to(torch.bfloat16)  # noqa: E731
    ring = LocalKVRing([mk(2) for _ in range(cp)], [mk(2) for _ in range(cp)])
    q, cfg = mk(8), RingConfig(cp_size=cp, cp_rank=rank)

    def sweep():
        return ring_flash_attn(q, ring.k[rank], ring.v[rank], cfg, group=ring, return_lse=True)

    out, lse = sweep()
    side = torch.cuda.Stream()
    with torch.cuda.stream(side):
        sweep()
    torch.cuda.synchronize()
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph, stream=side):
        go, gl = sweep()
    for _ in range(5):
        go.zero_()
        graph.replay()
        torch.cuda.synchronize()
        assert torch.equal(go, out) and torch.equal(gl, lse)
        o, l = sweep()
        torch.cuda.synchronize()
        assert torch.equal(o, out) and torch.equal(l, lse)


def test_transpose_v_ring_reads_the_front_halves():
    """fa4cp_transpose_v_ring: of the first n_front tensors the front half of every sequence,
    rounded up to 128 positions, as transpose_v_many writes it; the rest whole; and the words to
    clear zero, the next one untouched."""
    from fa4_ring.fa4_backend import transpose_v_many

    say("transpose_v_ring")
    lens = [700, 2, 0, 258]
    cu = torch.tensor([0, 700, 702, 702, 960], dtype=torch.int32, device=DEV)
    for dtype, d in ((torch.bfloat16, 128), (torch.float16, 64), (E4, 256)):
        vs = [torch.randn(960, 2, d, device=DEV).to(dtype) for _ in range(4)]
        words = torch.full((70,), 7, dtype=torch.int32, device=DEV)
        whole, stride = transpose_v_many(vs, cu_seqlens_k=cu, max_seqlen_k=700)
        ring, _ = transpose_v_many(vs, cu_seqlens_k=cu, max_seqlen_k=700, n_front=2, clear=(words, 69))
        for i, (a, b) in enumerate(zip(whole, ring)):
            a, b = (x.view(torch.uint8).view(2 * d, stride, -1) for x in (a, b))
            at = 0
            for n in lens:
                w = (n // 2 if i < 2 else n) + 127
                assert torch.equal(a[:, at:at + w // 128 * 128], b[:, at:at + w // 128 * 128]), (dtype, i, n)
                at += (n + 127) // 128 * 128
        assert not words[:69].any() and int(words[69]) == 7
