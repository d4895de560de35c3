"""How the attention launches are laid out (csrc/attn_plan.h), without a GPU."""

import pytest

import plans
from test_gpu_split_backward import CASES as BACKWARD


@pytest.mark.parametrize("lens,h,h_kv,d,cp,rank,dtype,shared", BACKWARD)
def test_backward_cases_share_what_they_say(lens, h, h_kv, d, cp, rank, dtype, shared):
    dq, kv = plans.backward_plan(lens, h, h_kv, d, cp, rank)
    assert (dq.k > 1) == ("dq" in shared) and (kv.k > 1) == ("kv" in shared), (dq, kv)


def test_backward_cases_reach_every_form():
    """Up to head dim 128 (merged by the last workgroup) and at 256 (by sum kernels): tiles of both
    classes shared, and the second class whole beside a shared first."""
    for wide in (False, True):
        dq, kv = zip(*(plans.backward_plan(*c[:6]) for c in BACKWARD if (c[3] == 256) == wide))
        for shares in (dq, kv):
            assert any(s.k > 1 and s.k2 > 1 for s in shares), (wide, shares)
        assert any(s.k > 1 and s.top2 and s.k2 == 1 for s in dq + kv), (wide, dq, kv)
