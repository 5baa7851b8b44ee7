"""The batched linear kernel's host-side rules (csrc/linear_tile.h), compiled for the host."""
from __future__ import annotations

import linear_plan as lp
import pytest


@pytest.mark.parametrize("ntb", [1, 2, 3, 4])
@pytest.mark.parametrize("nb", [1, 2, 5, 7, 16, 97, 65535, 65537, 92683, 113512, 131072, 131073, 200001, 0x8000000])
def test_every_token_block_once(nb, ntb):
    """Token tiles take consecutive, non-empty runs of at most ntb blocks, from 0 to nb, also where
    tile x block count passes 32 bits (from 2.1 million tokens of one-block tiles on)."""
    plan = lp.lib()
    tiles = -(-nb // ntb)
    pick = range(tiles) if tiles < 70000 else [*range(100), *range(tiles // 2, tiles // 2 + 100), *range(tiles - 100, tiles)]
    for tt in pick:
        lo, hi = plan.plan_share0(tt, nb, tiles), plan.plan_share0(tt + 1, nb, tiles)
        assert 0 < hi - lo <= ntb and lo <= nb and hi <= nb, (tt, lo, hi)
    assert plan.plan_share0(0, nb, tiles) == 0 and plan.plan_share0(tiles, nb, tiles) == nb


@pytest.mark.parametrize("t", lp.TYPES)
def test_splits_are_whole_units(t):
    """Every chosen split gets at least one unit of n_in (64 elements, 256 of Q6_K, per k group), so
    that as many splits run as are reported, and a request is met while n_in has 256 elements a split."""
    unit, plan = 256 if t == "Q6_K" else 64, lp.lib()
    for n_in in (256, 512, 1024, 2048, 3072, 5120, 8192, 14336):
        for n_out in (96, 1024, 3072, 4096, 8192, 14336):
            for n_tok in (2, 13, 40, 100, 157, 300, 512, 700):
                for requested in (0, 1, 2, 3, 5, 8):
                    ntb, kg, splits = lp.linear(t, n_in, n_out, n_tok, requested)
                    units = -(-n_in // (unit * kg))
                    assert 1 <= splits <= units and 1 <= ntb <= 4 and kg in (1, 2, 4)
                    shares = [plan.plan_share0(i + 1, units, splits) - plan.plan_share0(i, units, splits) for i in range(splits)]
                    assert sum(shares) == units and min(shares) >= 1
                    if requested > 1 and -(-n_out // 128) * -(-n_tok // 96) <= 256:  # (counters for 256 tiles)
                        assert splits == min(requested, max(1, n_in // 256)), (n_in, n_out, n_tok, requested, kg)


@pytest.mark.parametrize("t", lp.TYPES)
def test_every_kernel_is_reached(t):
    """Every kernel that is built (token blocks, k groups; split, not split, gate/up) is the choice for
    some call of test_gpu_linear_shapes, and no other shape is ever chosen."""
    one, two = lp.smallest(t)
    want = set(lp.kernels(t))
    assert {k[:2] for k in one if not k[2]} == want and {k[:2] for k in one if k[2]} == want and set(two) == want
