"""The batched linear kernel's shape rule (csrc/linear_shape.h), compiled for the host, and the smallest
calls that reach each of its shapes."""
from __future__ import annotations

import ctypes
import functools
import os
import subprocess
import tempfile

from conftest import ROOT

TYPES = {"F32": 0, "F16": 1, "Q4_0": 2, "Q4_1": 3, "Q8_0": 8, "Q6_K": 14, "BF16": 30}


@functools.lru_cache(maxsize=1)
def lib():
    so = os.path.join(tempfile.mkdtemp(prefix="linear_plan"), "plan.so")
    subprocess.run(["g++", "-std=c++17", "-O2", "-shared", "-fPIC", "-D__HIP_PLATFORM_AMD__", "-I/opt/rocm/include",
                    os.path.join(ROOT, "tests", "cpp", "linear_plan.cpp"), "-o", so], check=True)
    return ctypes.CDLL(so)


def linear(t, n_in, n_out, n_tok, requested=0, ws=1 << 40):
    """(token blocks, k groups, splits) of ingot_linear."""
    out = (ctypes.c_uint32 * 3)()
    lib().plan_shape(TYPES[t], n_in, n_out, n_tok, requested, ctypes.c_uint64(ws), out)
    return tuple(out)


def pair(t, n_in, n_out, n_tok):
    out = (ctypes.c_uint32 * 3)()
    lib().plan_pair(TYPES[t], n_in, n_out, n_tok, out)
    return tuple(out)


def kernels(t):
    """(token blocks, k groups) of the type's kernels."""
    all_ = [(b, 4) for b in (1, 2, 3)] + [(b, kg) for kg in (2, 1) for b in (2, 3, 4)]
    return [k for k in all_ if t != "F32" or k not in ((3, 4), (4, 2), (4, 1))]


def _sizes(t):
    # (most rows end inside a step of 64 or a stage of 128; Q6_K: whole blocks of 256)
    for n_in in ((512, 768, 1280, 2304, 4352, 8448) if t == "Q6_K" else (96, 160, 512, 544, 800, 2080, 3104, 4128, 8224, 14368)):
        for n_out in (33, 130, 257, 1025, 2050, 3073, 4100, 8201, 14337):
            for n_tok in (2, 33, 65, 97, 129, 161, 200, 257, 290, 321, 390, 450, 513, 600, 700):
                yield n_in, n_out, n_tok


@functools.lru_cache(maxsize=None)
def smallest(t):
    """{(token blocks, k groups, split?): (n_in, n_out, n_tok, n_splits)} and the same for pairs with
    {(token blocks, k groups): (n_in, n_out, n_tok)}: the call of least work that runs each kernel."""
    one, two = {}, {}
    for n_in, n_out, n_tok in sorted(_sizes(t), key=lambda s: s[0] * s[1] * s[2]):
        for req in (0, 1, 2, 3, 8):
            b, kg, splits = linear(t, n_in, n_out, n_tok, req)
            one.setdefault((b, kg, splits > 1), (n_in, n_out, n_tok, req))
        two.setdefault(pair(t, n_in, n_out, n_tok)[:2], (n_in, n_out, n_tok))
    return one, two


@functools.lru_cache(maxsize=None)
def spread(t):
    """{(token blocks, split?, more than two token tiles?): (n_in, n_out, n_tok, n_splits)}: the call of
    least work whose token tiles start apart (whole stages of weights: 256 elements of every k group)."""
    per = {"F32": 4, "F16": 2, "BF16": 2, "Q8_0": 34 / 32, "Q4_0": 18 / 32, "Q4_1": 20 / 32, "Q6_K": 210 / 256}[t]
    out = {}
    sizes = [(i, o, n) for i in (1024, 1536, 2560, 3072, 4096) for o in (130, 257, 514, 1025, 2050, 3073)
             for n in (65, 97, 129, 161, 200, 257, 321, 390, 450, 513, 600, 700)]
    for n_in, n_out, n_tok in sorted(sizes, key=lambda s: s[0] * s[1] * s[2]):
        for req in (0, 2, 3, 4):
            b, kg, splits = linear(t, n_in, n_out, n_tok, req)
            tiles = -(-(-(-n_tok // 32)) // b)
            if tiles > 1 and n_in % (512 * splits) == 0 and lib().plan_spread(kg, ctypes.c_uint64(int(n_in * n_out * per)), ctypes.c_uint64(4 * n_in * n_tok)):
                out.setdefault((b, splits > 1, tiles > 2), (n_in, n_out, n_tok, req))
    return out
