"""The batched linear kernel at the edges of its tiles: token blocks of 32 (and where the number of
k groups changes), tiles of 64 / 128 / 256 rows, k shares that end inside a step of 64 elements,
against the CPU oracle with both operands rounded to f16. The bar is the one of test_gpu_linear:
only the order of the f32 sums differs (rel-L2 <= 1e-5, max|d| <= 1e-5 * max|ref| + 1e-6)."""
from __future__ import annotations

import numpy as np
import pytest

from conftest import ensure_built

import gguf_blocks as gb

pytestmark = pytest.mark.gpu

TYPES = ["F32", "F16", "BF16", "Q8_0", "Q4_0", "Q4_1", "Q6_K"]


@pytest.fixture(scope="module")
def dev():
    import torch

    if not torch.cuda.is_available():
        pytest.fail("GPU test run without a GPU")
    ensure_built("lib")
    import ingot_attn

    ingot_attn.load_library()
    return torch.device("cuda:0")


def _run(dev, t, raw, x, n_in, n_out, n_splits):
    import torch
    import ingot_attn as ia

    out = torch.full((x.shape[0] * n_out + 64,), float("nan"), device=dev)
    ia.linear(torch.from_numpy(raw.reshape(-1)).to(dev), torch.from_numpy(x).to(dev), out,
              ia.linear_desc(t, n_in, n_out, x.shape[0], n_splits=n_splits), workspace=ia.Workspace(dev))
    torch.cuda.synchronize()
    got = out.cpu().numpy()
    assert np.all(np.isnan(got[x.shape[0] * n_out:])), "wrote past its rows"
    return got[: x.shape[0] * n_out].reshape(x.shape[0], n_out)


@pytest.mark.parametrize("t", TYPES)
@pytest.mark.parametrize("n_tok,n_in,n_out,n_splits", [
    (2, 32, 1, 0), (31, 96, 33, 0), (33, 160, 65, 1), (64, 288, 63, 0), (96, 352, 129, 1), (97, 1056, 130, 0),
    (129, 2336, 127, 3), (288, 544, 257, 1), (289, 1312, 255, 1), (300, 800, 31, 2)])
def test_tile_edges(dev, oracle_mod, t, n_tok, n_in, n_out, n_splits):
    n_in = n_in if t != "Q6_K" else -(-n_in // 256) * 256
    raw = gb.random_weights(t, n_out, n_in, seed=n_tok + n_in)
    x = np.random.default_rng(n_out).standard_normal((n_tok, n_in)).astype(np.float32)
    got = _run(dev, t, raw, x, n_in, n_out, n_splits)
    want = oracle_mod.linear(t, raw, x, n_in, n_out, f16_path=True)
    d = np.abs(got - want)
    assert np.all(np.isfinite(got))
    assert d.max() <= 1e-5 * np.abs(want).max() + 1e-6 and np.linalg.norm(d) <= 1e-5 * np.linalg.norm(want)


@pytest.mark.parametrize("t", ["F16", "Q8_0"])
def test_ragged_end_reads_no_neighbour(dev, t):
    """A row whose share of n_in ends inside a step: the elements past its end are the next row's
    and must not reach the sum, not even where that row is infinite."""
    n_in, n_out, n_tok = 96, 6, 5
    raw = gb.random_weights(t, n_out, n_in, seed=3).copy()
    raw.view(np.uint8).reshape(n_out, -1)[4, 0:2] = (0x00, 0x7C)  # an infinite value or scale
    x = np.random.default_rng(4).standard_normal((n_tok, n_in)).astype(np.float32)
    got = _run(dev, t, raw, x, n_in, n_out, 0)
    assert np.all(np.isfinite(np.delete(got, 4, axis=1))) and not np.any(np.isfinite(got[:, 4]))


@pytest.mark.parametrize("t", ["Q4_0", "F16"])
@pytest.mark.parametrize("n_tok", [40, 130, 300])
def test_chunk_of_narrow_and_wide_matrices(dev, oracle_mod, t, n_tok):
    """Matrices narrower and wider than n_in, which take different numbers of k groups, in one
    ingot_proj call: each output equals ingot_linear (n_splits = 1) on its matrix bit for bit, and the
    oracle within the bar."""
    import torch
    import ingot_attn as ia

    n_in, n_outs = 512, (4100, 96, 4096)
    g = torch.Generator(device=dev)
    g.manual_seed(n_tok)
    x = torch.randn(n_tok, n_in, generator=g, device=dev)
    raw = [gb.random_weights(t, n, n_in, seed=n) for n in n_outs]
    ws = [torch.from_numpy(w.reshape(-1)).to(dev) for w in raw]
    outs = [torch.zeros(n_tok, n, device=dev) for n in n_outs]
    refs = [torch.zeros(n_tok, n, device=dev) for n in n_outs]
    ia.proj(ws, x, outs, ia.proj_desc(t, n_in, list(n_outs), n_tok=n_tok))
    for w, r, n in zip(ws, refs, n_outs):
        ia.linear(w, x, r, ia.linear_desc(t, n_in, n, n_tok, n_splits=1), use_workspace=False)
    torch.cuda.synchronize()
    for o, r, w, n in zip(outs, refs, raw, n_outs):
        assert torch.equal(o, r) and bool(torch.isfinite(o).all())
        want = oracle_mod.linear(t, w, x.cpu().numpy(), n_in, n, f16_path=True)
        d = np.abs(o.cpu().numpy() - want)
        assert d.max() <= 1e-5 * np.abs(want).max() + 1e-6 and np.linalg.norm(d) <= 1e-5 * np.linalg.norm(want)


@pytest.mark.parametrize("t", ["Q4_0", "Q4_1", "Q8_0", "Q6_K"])
@pytest.mark.parametrize("n_out", [16384, 66000])
def test_one_token_many_rows(dev, oracle_mod, t, n_out):
    """One token over more row blocks than the grid holds (each workgroup loops over several, the
    last ones ragged), against the f32 oracle (bar of test_gpu_linear), plain and with the norm."""
    import torch
    import ingot_attn as ia

    n_in = 256
    n_out += 5
    raw = gb.random_weights(t, n_out, n_in, seed=n_out)
    rng = np.random.default_rng(7)
    x, nw = rng.standard_normal((1, n_in)).astype(np.float32), np.ones(n_in, np.float32)
    w, xd = torch.from_numpy(raw.reshape(-1)).to(dev), torch.from_numpy(x).to(dev)
    for norm in (False, True):
        out = torch.full((n_out + 16,), float("nan"), device=dev)
        d = ia.proj_desc(t, n_in, [n_out], prologue=ia.PROJ_RMSNORM if norm else ia.PROJ_X, eps=1e-5)
        ia.proj([w], xd, [out], d, norm_w=torch.from_numpy(nw).to(dev))
        torch.cuda.synchronize()
        xr = (x / np.sqrt((x.astype(np.float64) ** 2).mean() + 1e-5)).astype(np.float32) if norm else x
        want = oracle_mod.linear(t, raw, xr, n_in, n_out)[0]
        got = out.cpu().numpy()
        dd = np.abs(got[:n_out] - want)
        assert np.all(np.isnan(got[n_out:])) and np.all(np.isfinite(dd))
        assert dd.max() <= 1e-5 * np.abs(want).max() + 1e-6 and np.linalg.norm(dd) <= 1e-5 * np.linalg.norm(want)


def test_millions_of_tokens(dev):
    """Above 4.2 million tokens a product of token tile and token block count passes 32 bits: every
    row of out is written, and accumulated into, once (checked against torch in f32, both operands
    rounded to f16: only the order of 32 f32 products differs)."""
    import torch
    import ingot_attn as ia

    n_tok, n_in, n_out = 4_194_304 + 33, 32, 32
    g = torch.Generator(device=dev)
    g.manual_seed(5)
    x = torch.randn(n_tok, n_in, generator=g, device=dev)
    w = (torch.randn(n_out, n_in, generator=g, device=dev) / n_in ** 0.5).half()
    want = x.half().float() @ w.float().t()
    out = torch.full((n_tok, n_out), float("nan"), device=dev)
    for acc in (False, True):
        ia.linear(w.view(torch.uint8).reshape(-1), x, out, ia.linear_desc("F16", n_in, n_out, n_tok, accumulate=acc))
        d = (out - want * (2 if acc else 1)).abs().max()
        assert bool(torch.isfinite(out).all()) and float(d) <= 1e-5 * float(want.abs().max()) * 2


@pytest.mark.parametrize("t,n_in,n_out,n_tok", [("F16", 18_000_000, 2, 64), ("Q8_0", 72_000_000, 34, 15), ("F32", 18_000_000, 70, 3)])
@pytest.mark.parametrize("pair", [False, True])
def test_rows_beyond_2gib(dev, t, n_in, n_out, n_tok, pair):
    """Rows so long that a tile's tokens, or a wave's 32 weight rows, span more than 2 GiB. x is zero
    but for 256 columns (the last among them), so that the sums hold few terms: rel-L2 <= 1e-5 against
    the same columns in 64 bits, both operands rounded to f16."""
    import torch
    import ingot_attn as ia

    g = torch.Generator(device=dev)
    g.manual_seed(n_out)
    cols = torch.cat([torch.randint(0, n_in, (255,), generator=g, device=dev), torch.tensor([n_in - 1], device=dev)]).unique()
    x = torch.zeros(n_tok, n_in, device=dev)
    x[:, cols] = torch.randn(n_tok, len(cols), generator=g, device=dev)

    def matrix():
        if t == "Q8_0":
            raw = torch.randint(0, 256, (n_out, n_in // 32, 34), generator=g, device=dev, dtype=torch.uint8)
            raw[..., :2] = torch.tensor([0x00, 0x24], dtype=torch.uint8, device=dev)  # d = 2^-6
            q = raw.view(torch.int8)[:, cols // 32, 2 + cols % 32].double() / 64
            return raw.reshape(-1), q
        w = torch.randn(n_out, n_in, generator=g, device=dev)
        w = w if t == "F32" else w.half()
        return w.view(torch.uint8).reshape(-1), w[:, cols].half().double()

    xs = x[:, cols].half().double()
    mats = [matrix() for _ in range(2 if pair else 1)]
    sums = [xs @ q.t() for _, q in mats]
    if pair:
        want = torch.nn.functional.silu(sums[0]) * sums[1]
        out = torch.empty(n_tok, n_out, device=dev)
        ia.proj([m for m, _ in mats], x, [out], ia.proj_desc(t, n_in, [n_out, n_out], epilogue=ia.PROJ_SILU_GATE, n_tok=n_tok))
    else:
        want = sums[0] * 2
        out = torch.zeros(n_tok, n_out, device=dev)
        for _ in range(2):
            ia.linear(mats[0][0], x, out, ia.linear_desc(t, n_in, n_out, n_tok, accumulate=True), workspace=ia.Workspace(dev))
    assert float((out - want).norm()) <= 1e-5 * float(want.norm())
