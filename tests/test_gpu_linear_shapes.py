"""Every kernel of the batched linear layer (token blocks, k groups; split, not split, gate/up) on the
smallest ragged call that its shape rule gives it, and the production shapes of long rows, against the
CPU oracle with both operands rounded to f16. The weights repeat 97 rows, so that every output is
checked and a row taken from another wave or tile shows. The bar is the one of test_gpu_linear: only
the order of the f32 sums differs (rel-L2 <= 1e-5, max|d| <= 1e-5 * max|ref| + 1e-6)."""
from __future__ import annotations

import linear_plan as lp
import numpy as np
import pytest

from conftest import ensure_built

import gguf_blocks as gb

pytestmark = pytest.mark.gpu
ROWS = 97


@pytest.fixture(scope="module")
def dev():
    import torch

    if not torch.cuda.is_available():
        pytest.fail("GPU test run without a GPU")
    ensure_built("lib")
    import ingot_attn

    ingot_attn.load_library()
    return torch.device("cuda:0")


def _matrix(dev, t, n_in, n_out, seed):
    """Raw bytes of n_out rows on the device, row r a copy of row r % 97, and those 97."""
    import torch

    few = gb.random_weights(t, ROWS, n_in, seed=seed).reshape(ROWS, -1).view(np.uint8)
    return torch.from_numpy(few).to(dev)[torch.arange(n_out, device=dev) % ROWS].reshape(-1), few


def _close(got, want, what):
    want = np.take(want, np.arange(got.shape[1]) % ROWS, axis=1)
    d = np.abs(got - want)
    assert np.all(np.isfinite(got)), what
    assert d.max() <= 1e-5 * np.abs(want).max() + 1e-6 and np.linalg.norm(d) <= 1e-5 * np.linalg.norm(want), what


def _linear(dev, oracle_mod, t, n_in, n_out, n_tok, n_splits, what):
    import torch
    import ingot_attn as ia

    w, few = _matrix(dev, t, n_in, n_out, n_tok)
    x = np.random.default_rng(n_in).standard_normal((n_tok, n_in)).astype(np.float32)
    out = torch.full((n_tok * n_out + 64,), float("nan"), device=dev)
    ia.linear(w, torch.from_numpy(x).to(dev), out, ia.linear_desc(t, n_in, n_out, n_tok, n_splits=n_splits), workspace=ia.Workspace(dev))
    assert bool(torch.isnan(out[n_tok * n_out:]).all()), "wrote past its rows"
    _close(out[: n_tok * n_out].view(n_tok, n_out).cpu().numpy(),
           oracle_mod.linear(t, few.reshape(-1), x, n_in, ROWS, f16_path=True), what)


@pytest.mark.parametrize("t", lp.TYPES)
def test_every_kernel(dev, oracle_mod, t):
    for key, case in lp.smallest(t)[0].items():
        _linear(dev, oracle_mod, t, *case, (key, case))


@pytest.mark.parametrize("t", lp.TYPES)
def test_walks_spread_over_the_rows(dev, oracle_mod, t):
    """Token tiles that start their walks of n_in at different stages and wrap: two and more of them,
    split and not, every tile height."""
    assert len(lp.spread(t)) >= 4 and len({k[0] for k in lp.spread(t)}) >= 2
    for key, case in lp.spread(t).items():
        _linear(dev, oracle_mod, t, *case, (key, case))


@pytest.mark.parametrize("t", lp.TYPES)
def test_every_pair_kernel(dev, oracle_mod, t):
    """silu(gate) * up of each tile: equal bit for bit to the two products (n_splits = 1) and
    ingot_silu_mul, and near the oracle's sums (silu' <= 1.1: the bar on the sums, times |up| and |gate|)."""
    import torch
    import ingot_attn as ia

    for key, (n_in, n_out, n_tok) in lp.smallest(t)[1].items():
        ws = [_matrix(dev, t, n_in, n_out, seed) for seed in (5, 6)]
        x = np.random.default_rng(n_in).standard_normal((n_tok, n_in)).astype(np.float32)
        xd = torch.from_numpy(x).to(dev)
        out = torch.full((n_tok * n_out + 64,), float("nan"), device=dev)
        ia.proj([w for w, _ in ws], xd, [out], ia.proj_desc(t, n_in, [n_out, n_out], epilogue=ia.PROJ_SILU_GATE, n_tok=n_tok))
        g, u = (torch.empty(n_tok * n_out + 4, device=dev) for _ in range(2))
        for (w, _), o in zip(ws, (g, u)):
            ia.linear(w, xd, o, ia.linear_desc(t, n_in, n_out, n_tok, n_splits=1), use_workspace=False)
        sums = [o[: n_tok * n_out].view(n_tok, n_out).cpu().numpy() for o in (g, u)]
        ia.silu_mul(g, u, (n_tok * n_out + 3) // 4 * 4)
        assert torch.equal(out[: n_tok * n_out], g[: n_tok * n_out]), (key, n_in, n_out, n_tok)
        assert bool(torch.isnan(out[n_tok * n_out:]).all()), "wrote past its rows"
        for got, (_, few) in zip(sums, ws):
            _close(got, oracle_mod.linear(t, few.reshape(-1), x, n_in, ROWS, f16_path=True), key)


@pytest.mark.parametrize("t", ["Q4_0", "Q8_0", "F16", "Q6_K"])
@pytest.mark.parametrize("n_tok,n_in,n_out", [(300, 8192, 3072), (512, 8192, 3072), (1024, 8192, 3072), (600, 2048, 2048)])
def test_long_rows_and_many_tokens(dev, oracle_mod, t, n_tok, n_in, n_out):
    """The down projection of a prompt chunk, split over n_in, and a square product of many tokens."""
    _linear(dev, oracle_mod, t, n_in, n_out, n_tok, 0, "")
