"""How the attention launches are laid out (csrc/attn_plan.h), without a GPU."""

import pytest
import torch

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


BF16, FP16, E4M3 = torch.bfloat16, torch.float16, torch.float8_e4m3fn
NINE = [260, 216, 144, 112, 96, 64, 46, 32, 16]


@pytest.mark.parametrize("lens,h,h_kv,cp,rank,dtype,least,most", [
    # (the times beside split_plan: within 2 % of the fastest share count are least..most)
    ([512], 8, 2, 2, 1, FP16, 1, 1),
    ([2000], 32, 8, 4, 3, BF16, 1, 1),
    ([4386], 32, 8, 2, 1, E4M3, 1, 1),
    ([290], 8, 2, 8, 7, E4M3, 1, 1),
    ([182], 16, 2, 8, 3, FP16, 1, 3),
    ([296], 8, 2, 8, 5, BF16, 2, 3),
    ([2048], 16, 2, 8, 3, BF16, 3, 3),   # still shared where that is 1.7 times as fast
    (NINE, 16, 2, 8, 6, BF16, 1, 3),
])
def test_wide_sweeps_are_not_split_at_a_loss(lens, h, h_kv, cp, rank, dtype, least, most):
    """Head dim 256: the merge and the slots' traffic are charged."""
    assert least <= plans.split_plan(lens, h, h_kv, 256, cp, rank, dtype).back <= most


@pytest.mark.parametrize("lens,h,h_kv,d,least,most", [
    ([4416], 32, 8, 128, 1, 1),   # 340 us, in halves 387
    ([10440], 8, 2, 128, 1, 1),   # 425, 470
    ([8824], 16, 2, 64, 1, 1),    # 383, 420
    ([5360], 16, 16, 256, 1, 1),  # 453, 545
    ([2054], 8, 2, 128, 2, 6),    # 77, in three 51
])
def test_sweeps_of_uneven_row_tiles_are_not_split_at_a_loss(lens, h, h_kv, d, least, most):
    """Rank 1 of 2: one class of row tiles, the longest of three times the shortest's keys."""
    assert least <= plans.split_plan(lens, h, h_kv, d, 2, 1, FP16).back <= most


@pytest.mark.parametrize("lens,h,h_kv,cp,rank,dtype,least,most", [
    # (as above; unsplit, and in the shares that an average sequence's two classes of row tiles gave, us)
    ([216, 78, 252, 314, 82, 340, 166, 102, 924], 32, 8, 2, 0, BF16, 1, 1),  # 64, 80
    ([1024, 4608, 662], 16, 16, 4, 2, E4M3, 1, 1),                           # 252, 304
    ([360, 2034, 334], 32, 8, 2, 0, E4M3, 1, 1),                             # 84, 102
    ([344, 414], 32, 8, 4, 2, BF16, 2, 3),                                   # 50, 60 (4; now 44)
    ([308, 56, 40, 60, 24, 76, 82, 230, 104], 24, 8, 4, 3, FP16, 1, 1),      # 44, 55
    ([8410, 4742, 2496], 8, 2, 8, 6, BF16, 1, 1),                            # 1425, 1540 (4)
    ([706, 730], 16, 2, 2, 0, BF16, 1, 3),                                   # 48, 54 (4)
    ([968, 598, 574], 8, 1, 8, 4, FP16, 3, 6),                               # 140, 75
])
def test_packed_sweeps_are_not_split_at_a_loss(lens, h, h_kv, cp, rank, dtype, least, most):
    """Head dim 128: packed sequences' tiles of many lengths fill the chip unsplit, and slots cost bandwidth."""
    assert least <= plans.split_plan(lens, h, h_kv, 128, cp, rank, dtype).back <= most


@pytest.mark.parametrize("lens,h,h_kv", [
    ([350, 150, 124, 100, 100, 80, 60, 40, 20], 32, 8),  # 432 workgroups with the longest one's tiles for each
    ([2048] + [64] * 31, 8, 2),
    ([256] * 8, 32, 8),                                  # whole tiles: 256 workgroups, none to spare
    ([322] * 8, 32, 8),
    ([1024] * 8, 32, 8),
    ([4098], 32, 8),
    ([4096], 32, 8),                                     # 512
    ([2050], 32, 8),
    ([27782], 8, 1),                                     # two head groups: 870, a sweep needs four for each CU
    ([34000], 8, 1),
    ([1300] * 12, 16, 16),
    ([600] * 9, 6, 3),
    ([386], 144, 144),                                   # short row tiles: from 256 on
    ([250], 144, 144),
])
@pytest.mark.parametrize("q_sel", [0, 1])
def test_two_per_cu_counts_the_workgroups_with_rows(lens, h, h_kv, q_sel):
    """Two workgroups per CU (head dim 64) only where more than two for each have rows (four in a sweep of few
    head groups), or one where all row tiles are short (then, per step, those of the grid); half a tile per sequence off at
    most, as the host doesn't know the lengths."""
    hp = plans.heads_per_wg(h // h_kv)
    tiles = lambda n: -(-n * hp // 256)  # noqa: E731
    for step, two, ns in ((True, plans.attn_two_per_cu(lens, h, h_kv, 64, q_sel), [n if q_sel == 0 else n // 2 for n in lens]),
                          (False, plans.sweep_two_per_cu(lens, h, h_kv, 64), lens)):
        few = max(ns) <= 512 and tiles(max(ns)) <= 4
        n = h // hp * (len(ns) * tiles(max(ns)) if step and few else sum(map(tiles, ns)))
        slack = h // hp * len(lens) // 2 if len(lens) > 1 and not (step and few) else 0
        most = 256 if few else 512 if step or h // hp >= 4 else 1024
        assert two == (n > most) or abs(n - most) <= slack, (two, n)
    assert not plans.attn_two_per_cu(lens, h, h_kv, 128, q_sel)


def test_two_per_cu_where_measured():
    step, sweep = plans.attn_two_per_cu, plans.sweep_two_per_cu
    nine, short = [350, 150, 124, 100, 100, 80, 60, 40, 20], [222] + [70] * 8
    assert not step(nine, 32, 8, 64) and not sweep(nine, 32, 8, 64)
    assert not step([256] * 8, 32, 8, 64) and not sweep([256] * 8, 32, 8, 64)
    assert step(short, 32, 8, 64) and not sweep(short, 32, 8, 64)  # the grid, empty workgroups and all
    assert sweep([296], 144, 144, 64) and step([296], 144, 144, 64)
    # all at once on two per CU the longest tiles share CUs while others fall idle (800 us, 1170; 730, 930)
    for lens, h, h_kv in (([4504], 24, 8), ([16208], 8, 2), ([7096], 16, 2)):
        assert not sweep(lens, h, h_kv, 64) and not step(lens, h, h_kv, 64)
    assert not sweep([27782], 8, 1, 64) and step([27782], 8, 1, 64)
    assert sweep([16384], 32, 8, 64) and step([16384], 32, 8, 64)


@pytest.mark.parametrize("h,h_kv,d,cp,rank", [(16, 2, 256, 4, 1), (8, 1, 256, 4, 0), (16, 2, 256, 4, 3), (8, 2, 256, 8, 5),
                                              (8, 2, 128, 4, 1), (8, 1, 64, 8, 3), (2, 1, 128, 2, 0)])
def test_key_tiles_take_their_classes_shares(h, h_kv, d, cp, rank):
    """dk / dv: a tile walks the 32-row blocks that hold a row of its own, of every query head.  A
    later source's tiles (the back-half rows, from the middle of a block on where half the length
    is no multiple of 32) are the second class's longest, an earlier source's of the first."""
    group, seen = h // h_kv, 0
    for length in list(range(2, 900, 2)) + [1022, 1024, 1534, 2046, 2048, 3070, 3072, 4094, 4096]:
        kv = plans.backward_plan([length], h, h_kv, d, cp, rank)[1]
        if kv.k == 1:
            continue

        def blocks(first):
            return group * len({row // 32 for row in range(first, length)})

        late, early = blocks(length // 2), blocks(0)
        own = [blocks(first) for first in range(0, length, 128)]
        assert kv.top2 == (late if late < early and (rank < cp - 1 or min(own) <= late) else 0), length
        if kv.top2:
            seen += 1
            assert plans.shares_of(kv, late) == min(kv.k, -(-kv.top2 // kv.chunk2)) <= kv.k2, length
            assert plans.shares_of(kv, early) == min(kv.k, -(-early // kv.chunk)), length
    assert seen


def test_turned_shares():
    """Packed sequences: every tile's workgroups take its shares once each, and over the tiles share 0 comes
    to each XCD and, within it, to each shader engine (workgroups in turn) about as often."""
    for ns in range(2, 9):
        for k in (1, 2, 4, 8):  # XCDs that a head group's workgroups go to in turn
            seen = [0] * (4 * k)
            for tile in range(128):
                shares = [plans.turned_share(i, tile, ns) for i in range(ns)]
                assert sorted(shares) == list(range(ns))
                seen[(tile * ns + shares.index(0)) % (4 * k)] += 1
            assert max(seen) <= 1.6 * 128 / (4 * k), (ns, k, seen)
