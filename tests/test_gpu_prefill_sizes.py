"""Prefill at head sizes that share the MFMA kernel with zero-filled dims (multiples of 8 below 256
other than 64 and 128): against a float64 reference on the CPU. q and the probabilities enter as
two f16 parts (a relative 2^-22 each, the probabilities down to 2^-24), sums are f32: with scores of magnitude s the result is off by
about (s + 4) * 2^-22, so rel-L2 <= 2e-6 at s ~ 4 and <= 2e-5 at s ~ 100 (the first maximum of a
key group may then lie far below zero)."""
from __future__ import annotations

import numpy as np
import pytest

from conftest import ensure_built

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def dev():
    import torch

    if not torch.cuda.is_available():
        pytest.fail("GPU test run without a GPU")
    ensure_built("lib")
    import ingot_attn

    ingot_attn.load_library()
    return torch.device("cuda:0")


@pytest.mark.parametrize("hd,nh,nkv,pos,n,pad", [
    (8, 2, 1, 0, 2, 0), (56, 4, 2, 31, 33, 0), (72, 3, 1, 63, 65, 3), (96, 6, 2, 127, 64, 0),
    (120, 2, 2, 190, 129, 1), (136, 4, 1, 5, 70, 0), (248, 2, 1, 33, 31, 2),
    # (calls of one key chunk and few workgroups run the fallback kernel: the same sizes with more keys)
    (24, 2, 2, 255, 2, 0), (56, 4, 2, 261, 33, 0), (72, 3, 1, 263, 65, 3), (96, 6, 2, 327, 64, 0), (136, 4, 1, 205, 70, 0),
    (248, 2, 1, 233, 31, 2), (200, 2, 1, 1000, 5, 4),
    # and both sides of that line
    (96, 8, 8, 0, 128, 0), (96, 8, 8, 1, 128, 0), (96, 8, 8, 192, 64, 0), (96, 8, 8, 193, 64, 0), (40, 8, 2, 100, 64, 0),
    (40, 8, 2, 100, 65, 0), (96, 17, 17, 0, 64, 0)])
@pytest.mark.parametrize("gain,bar", [(1.0, 2e-6), (100.0, 2e-5)])
def test_zero_filled_dims(dev, hd, nh, nkv, pos, n, pad, gain, bar):
    import torch
    import ingot_attn as ia

    rng = np.random.default_rng(hd + n)
    L, kvd, stride = pos + n, nkv * hd, nh * hd + pad
    q = (rng.standard_normal((n, stride)) * gain).astype(np.float32)
    # a layer behind a slice of NaNs: nothing outside the visible rows may be read into a sum
    k = np.full((2 * L, kvd), np.nan, np.float16)
    v = np.full((2 * L, kvd), np.nan, np.float16)
    k[L:] = rng.standard_normal((L, kvd)).astype(np.float16)
    v[L:] = rng.standard_normal((L, kvd)).astype(np.float16)
    t = lambda a: torch.from_numpy(a).to(dev)  # noqa: E731
    out = torch.full((n, stride), float("nan"), device=dev)
    ia.attn_prefill(t(q), t(k), t(v), out, ia.prefill_desc(nh, nkv, hd, pos, n, kv_offset=L * kvd, q_stride=stride))
    torch.cuda.synchronize()
    got = out.cpu().numpy()
    assert np.all(np.isnan(got[:, nh * hd:])), "wrote past the heads"
    for h in range(nh):
        c = slice((h // (nh // nkv)) * hd, (h // (nh // nkv) + 1) * hd)
        s = q[:, h * hd:(h + 1) * hd].astype(np.float64) @ k[L:, c].astype(np.float64).T / np.sqrt(hd)
        s[np.arange(L)[None, :] > pos + np.arange(n)[:, None]] = -np.inf
        p = np.exp(s - s.max(1, keepdims=True))
        want = p / p.sum(1, keepdims=True) @ v[L:, c].astype(np.float64)
        d = got[:, h * hd:(h + 1) * hd] - want
        assert np.all(np.isfinite(d)) and np.linalg.norm(d) <= bar * np.linalg.norm(want), f"head {h}"


def test_rows_beyond_2gib(dev):
    """Rows of q and out so far apart that a block of 64 tokens spans more than 2 (and 4) GiB: the
    same values as from dense rows, up to f32 rounding (such calls run the fallback kernel)."""
    import torch
    import ingot_attn as ia

    hd, nh, nkv, pos, n = 96, 3, 1, 400, 64
    g = torch.Generator(device=dev)
    g.manual_seed(1)
    q = torch.randn(n, nh * hd, generator=g, device=dev)
    k = torch.randn(pos + n, nkv * hd, generator=g, device=dev).half()
    v = torch.randn(pos + n, nkv * hd, generator=g, device=dev).half()
    want = torch.empty_like(q)
    ia.attn_prefill(q, k, v, want, ia.prefill_desc(nh, nkv, hd, pos, n))
    for stride in (8_388_607, 8_388_608, 9_000_003, 18_000_000):
        far, out = (torch.zeros(n, stride, device=dev) for _ in range(2))
        far[:, : nh * hd] = q
        ia.attn_prefill(far, k, v, out, ia.prefill_desc(nh, nkv, hd, pos, n, q_stride=stride))
        assert float((out[:, : nh * hd] - want).norm() / want.norm()) <= 2e-6, stride
        assert not bool(out[:, nh * hd:].any()), "wrote past the heads"
        del far, out


@pytest.mark.parametrize("hd", [40, 96, 136])
@pytest.mark.parametrize("where", ["first", "last"])
@pytest.mark.parametrize("gap,bar", [(8.0, 2e-6), (12.0, 2e-6), (16.0, 2e-6), (20.0, 4e-6), (24.0, 2e-4)])
def test_small_probabilities(dev, hd, where, gap, bar):
    """An attention sink: one key `gap` nats above the others' mean score, with a zero V row, so that
    the output is made of probabilities around e^-gap alone. They are held to a relative 2^-22 down to
    2^-24 and the scores (up to 1.44 gap in the exponent of 2) rounded to f32, about 1.44 * 24 *
    2^-25 * ln 2 = 7e-7: rel-L2 <= 2e-6, the bar of ordinary scores. Below 2^-24 (gap 16.6) the
    probabilities keep an absolute 2^-47 of the largest: at e^-20 2^-18 (4e-6), at e^-24 2^-12 (2e-4)."""
    import torch
    import ingot_attn as ia

    nh, nkv, pos, n = 2, 1, 2000, 48
    L, kvd = pos + n, nkv * hd
    rng = np.random.default_rng(int(gap) + hd)
    at = 0 if where == "first" else pos  # (visible to every query)
    q = rng.standard_normal((n, nh * hd)).astype(np.float32)
    k = rng.standard_normal((L, kvd)).astype(np.float16)
    v = rng.standard_normal((L, kvd)).astype(np.float16)
    # dimension 0 carries the sink's score: q = 8 there, the sink's k such that 8 k / sqrt(hd) = gap
    q[:, ::hd] = 8.0
    k[:, 0], k[at] = 0, 0
    k[at, 0] = gap * np.sqrt(hd) / 8.0
    v[at] = 0
    t = lambda a: torch.from_numpy(a).to(dev)  # noqa: E731
    out = torch.empty(n, nh * hd, device=dev)
    ia.attn_prefill(t(q), t(k), t(v), out, ia.prefill_desc(nh, nkv, hd, pos, n))
    got = out.cpu().numpy()
    for h in range(nh):
        c = slice(h * hd, (h + 1) * hd)
        s = q[:, c].astype(np.float64) @ k.astype(np.float64).T * np.float64(np.float32(1.0 / np.sqrt(hd)))
        s[np.arange(L)[None, :] > pos + np.arange(n)[:, None]] = -np.inf
        p = np.exp(s - s.max(1, keepdims=True))
        want = p / p.sum(1, keepdims=True) @ v.astype(np.float64)
        rel = np.linalg.norm(got[:, c] - want) / np.linalg.norm(want)
        assert rel <= bar


@pytest.mark.parametrize("hd", [8, 96, 200])
@pytest.mark.parametrize("size", [1e-38, 1e-30, 1e30, 3e32, 1e35])
def test_any_finite_query(dev, hd, size):
    """Queries of any finite size: the softmax of the tiny ones is uniform, of the huge ones all on
    one key (test and reference agree on which: the best score leads by far more than f32 rounding)."""
    import torch
    import ingot_attn as ia

    n, pos = 40, 300
    rng = np.random.default_rng(hd)
    k = rng.standard_normal((pos + n, hd)).astype(np.float16)
    v = rng.standard_normal((pos + n, hd)).astype(np.float16)
    q = (rng.standard_normal((n, hd)) * size).astype(np.float32)
    t = lambda a: torch.from_numpy(a).to(dev)  # noqa: E731
    out = torch.empty(n, hd, device=dev)
    ia.attn_prefill(t(q), t(k), t(v), out, ia.prefill_desc(1, 1, hd, pos, n))
    s = q.astype(np.float64) @ k.astype(np.float64).T / np.sqrt(hd)
    s[np.arange(pos + n)[None, :] > pos + np.arange(n)[:, None]] = -np.inf
    p = np.exp(s - s.max(1, keepdims=True))
    want = p / p.sum(1, keepdims=True) @ v.astype(np.float64)
    got = out.cpu().numpy()
    assert np.all(np.isfinite(got)) and np.linalg.norm(got - want) <= 2e-6 * np.linalg.norm(want)


@pytest.mark.parametrize("hd", [8, 40, 96, 136, 200])
@pytest.mark.parametrize("where", ["v", "k", "q"])
def test_infinities(dev, hd, where):
    """A value that became infinite (the f16 cache has no more above 65504) reaches what it is a part
    of and nothing else: an infinite V element its dimension of the queries that see its key, a key
    whose score is -inf no output, a query with a NaN itself. Every other element keeps the bar of
    ordinary scores, also of queries before the key and of the same query's other dimensions."""
    import torch
    import ingot_attn as ia

    nh, nkv, pos, n = 4, 2, 300, 150
    L, kvd = pos + n, nkv * hd
    rng = np.random.default_rng(hd)
    q = rng.standard_normal((n, nh * hd)).astype(np.float32)
    k = rng.standard_normal((L, kvd)).astype(np.float16)
    v = rng.standard_normal((L, kvd)).astype(np.float16)
    if where == "v":  # (KV head 0; of one sign in dimensions 0 and hd - 1, of both from key 400 on in 5)
        v[pos + 40, 0], v[pos + 77, hd - 1], v[pos + 20, 5], v[pos + 100, 5] = np.inf, -np.inf, np.inf, -np.inf
    elif where == "k":
        q[:, :2 * hd:hd] = 1 + np.abs(q[:, :2 * hd:hd])  # (the heads of KV head 0)
        k[33, 0], k[pos + 55, 0] = -np.inf, -np.inf
    else:
        q[70, hd + 3] = np.nan
    t = lambda a: torch.from_numpy(a).to(dev)  # noqa: E731
    out = torch.zeros(n, nh * hd, device=dev)
    ia.attn_prefill(t(q), t(k), t(v), out, ia.prefill_desc(nh, nkv, hd, pos, n))
    got = out.cpu().numpy()
    for h in range(nh):
        c, kc = slice(h * hd, (h + 1) * hd), slice(h // 2 * hd, (h // 2 + 1) * hd)
        with np.errstate(invalid="ignore"):
            s = q[:, c].astype(np.float64) @ k[:, kc].astype(np.float64).T / np.sqrt(hd)
            s[np.arange(L)[None, :] > pos + np.arange(n)[:, None]] = -np.inf
            p = np.exp(s - s.max(1, keepdims=True))
            vis = np.arange(L)[None, :, None] <= (pos + np.arange(n))[:, None, None]
            want = np.where(vis, p[:, :, None] * v[None, :, kc].astype(np.float64), 0).sum(1) / p.sum(1, keepdims=True)
        fin, g = np.isfinite(want), got[:, c]
        assert np.array_equal(fin, np.isfinite(g)) and np.array_equal(want[~fin], g[~fin], equal_nan=True), h
        assert np.linalg.norm(g[fin] - want[fin]) <= 2e-6 * np.linalg.norm(want[fin]), h
        assert fin.mean() > 0.7 and fin.all() == (where == "k" or h > 1 or (where == "q" and h == 0)), h
