"""Head dim 64 launches of many workgroups (more than the chip has CUs, or two for each) run two on a CU, in
kernels built for half the registers.

Every case has enough heads for them; a slice of its heads alone has not, and goes to the kernels that
the other tests hold against the oracle.  Both forms round the same probabilities and outputs, each off by
at most u relative, the unit roundoff of the type, so the outputs differ by at most about 4 u in the
2-norm.  The LSEs are fp32 sums, whose order may differ."""

import pytest
import torch

from fa4_ring import LocalKVRing, PagedKVRing, RingConfig, ring_flash_attn
from gpu_helpers import DEV, say

pytestmark = pytest.mark.gpu

CASES = [  # (local lens, H, H_kv, cp, rank, dtype, page, heads alone): row tiles of 256 / (heads per workgroup) rows
    ([386], 144, 144, 2, 0, torch.bfloat16, 0, 8),             # 2 x 144: a partial row tile
    ([258], 130, 130, 3, 2, torch.float16, 128, 26),           # 260
    ([1026], 96, 48, 2, 1, torch.bfloat16, 0, 16),             # two heads per workgroup: 9 x 48, one per CU
    ([1026], 128, 64, 2, 1, torch.bfloat16, 0, 16),            # 9 x 64
    ([2048], 32, 8, 8, 3, torch.bfloat16, 0, 4),               # four; 256 row tiles whose keys are shared
    ([2048], 32, 8, 8, 3, torch.float16, 256, 4),
    ([640, 2, 0, 322, 126, 514], 128, 32, 4, 1, torch.bfloat16, 0, 16),  # packed: empty and short sequences
    ([640, 2, 0, 322, 126, 514], 128, 32, 4, 3, torch.float16, 128, 16),
]


@pytest.mark.parametrize("fused", [True, False])
@pytest.mark.parametrize("lens,h,h_kv,cp,rank,dtype,page,alone", CASES)
def test_two_per_cu(lens, h, h_kv, cp, rank, dtype, page, alone, fused):
    say(f"two per CU lens={lens} h={h}/{h_kv} cp={cp} rank={rank} {dtype} page={page} fused={fused}")
    g = torch.Generator(device="cuda").manual_seed(3)
    total, packed = sum(lens), len(lens) > 1
    cu = torch.tensor([0] + torch.tensor(lens).cumsum(0).tolist(), dtype=torch.int32)
    kw = dict(cu_seqlens=cu.to(DEV), max_seqlen=max(lens)) if packed else {}
    mk = lambda hh: torch.randn(total, hh, 64, generator=g, device=DEV).to(dtype)  # noqa: E731
    q, ks, vs = mk(h), [mk(h_kv) for _ in range(cp)], [mk(h_kv) for _ in range(cp)]
    cfg = RingConfig(cp_size=cp, cp_rank=rank)

    def attend(q, ks, vs):
        group = LocalKVRing(ks, vs)
        if page and fused:
            group = PagedKVRing.from_shards(ks, vs, page, cu if packed else None, spare_pages=2,
                                            generator=torch.Generator().manual_seed(5), fill=0.0)
        return ring_flash_attn(q, ks[rank], vs[rank], cfg, group=group, fused=fused, return_lse=True, **kw)

    out, lse = attend(q, ks, vs)
    u = 2.0 ** -11 if dtype == torch.float16 else 2.0 ** -8
    kv = alone * h_kv // h
    for i in (0, h // alone // 2, h // alone - 1):
        s, t = slice(i * alone, (i + 1) * alone), slice(i * kv, (i + 1) * kv)
        o, l = attend(q[:, s].contiguous(), [k[:, t].contiguous() for k in ks], [v[:, t].contiguous() for v in vs])
        assert (o.float() - out[:, s].float()).norm() <= 4 * u * o.float().norm()
        assert (l - lse[:, s]).abs().max() <= 1e-5 * max(1.0, float(l.abs().max()))
