"""The batched linear kernel's host-side rules (csrc/linear_tile.h), compiled for the host."""
from __future__ import annotations

import ctypes
import os
import subprocess

import pytest

from conftest import ROOT


@pytest.fixture(scope="module")
def plan(tmp_path_factory):
    so = str(tmp_path_factory.mktemp("plan") / "plan.so")
    subprocess.run(["g++", "-std=c++17", "-O1", "-shared", "-fPIC", "-D__HIP_PLATFORM_AMD__", "-I/opt/rocm/include",
                    os.path.join(ROOT, "tests", "cpp", "linear_plan.cpp"), "-o", so], check=True)
    return ctypes.CDLL(so)


@pytest.mark.parametrize("ntb", [1, 2, 3, 4])
@pytest.mark.parametrize("nb", [1, 2, 5, 7, 16, 97, 65535, 65537, 92683, 113512, 131072, 131073, 200001, 0x8000000])
def test_every_token_block_once(plan, nb, ntb):
    """Token tiles take consecutive, non-empty runs of at most ntb blocks, from 0 to nb, also where
    tile x block count passes 32 bits (from 2.1 million tokens of one-block tiles on)."""
    tiles = -(-nb // ntb)
    pick = range(tiles) if tiles < 70000 else [*range(100), *range(tiles // 2, tiles // 2 + 100), *range(tiles - 100, tiles)]
    for tt in pick:
        lo, hi = plan.plan_block0(tt, nb, tiles), plan.plan_block0(tt + 1, nb, tiles)
        assert 0 < hi - lo <= ntb and lo <= nb and hi <= nb, (tt, lo, hi)
    assert plan.plan_block0(0, nb, tiles) == 0 and plan.plan_block0(tiles, nb, tiles) == nb
