"""What the framework's speed is judged by: the calls that a Llama-style engine makes, at the
sizes this repository configures, tests and benchmarks.

Four kinds of case ("op"):
  decode    attention of one new token over the f16 cache, for every layer of a model
  prefill   causal attention of a chunk over the f16 cache, for a few layers
  linears   embedding rows, then the projections of a few layers (norm, q/k/v, wo, gate/up, down)
            around a given attention output: for one token with the fused decode entry points, for
            a chunk with the batched ones, chosen as the forward pass chooses them
  linear    one linear layer (the logits projection with its norm, or a plain product)
  model     a whole forward pass, returning logits
One-token work is captured once and replayed as a graph, as a decode loop runs it; chunks are
launched call by call.
"""
import math
import os
import sys

import numpy as np
import torch

sys.path.insert(0, os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "inference-agent_amd"))

import ingot_attn as ia  # noqa: E402
import ingot_forward as fwd  # noqa: E402

DEV = "cuda:0"
F32 = dict(dtype=torch.float32, device=DEV)
EPS = 1e-5
THETA = 500000.0
# elements and bytes of a block of each GGUF weight type
BLOCK = {"F32": (1, 4), "F16": (1, 2), "BF16": (1, 2), "Q8_0": (32, 34), "Q4_0": (32, 18), "Q4_1": (32, 20), "Q6_K": (256, 210)}
# Llama-3.2-3B: the shapes this repository is benchmarked on
LLAMA = dict(n_embd=3072, n_head=24, n_head_kv=8, head_dim=128, n_ff=8192)


def listed():
    return [
        # Token generation early in a chat: one token's attention through the 28 layers, short
        # cache. The smallest launches the engine makes.
        dict(name="decode-512", op="decode", n_head=24, n_head_kv=8, head_dim=128, n_keys=512, layers=28),
        # The same with the server's whole default context (8192) filled.
        dict(name="decode-8192", op="decode", n_head=24, n_head_kv=8, head_dim=128, n_keys=8192, layers=28),
        # A long prompt arrives in 512-token chunks: the chunk that ends at 4096.
        dict(name="prefill-512@3584", op="prefill", n_head=24, n_head_kv=8, head_dim=128, pos=3584, n_tok=512, layers=4),
        # The largest attention call benchmarked: a 2048-token chunk that ends at 8192.
        dict(name="prefill-2048@6144", op="prefill", n_head=24, n_head_kv=8, head_dim=128, pos=6144, n_tok=2048, layers=1),
        # A model whose head size is none of the common three (96), a ragged follow-up chunk.
        dict(name="prefill-hd96-301@211", op="prefill", n_head=24, n_head_kv=8, head_dim=96, pos=211, n_tok=301, layers=2),
        # The projections of one generated token, Q4_0 weights (the usual download).
        dict(name="linears-q4_0-1", op="linears", type="Q4_0", n_tok=1, pos=700, layers=8, **LLAMA),
        # A short follow-up message, 8-bit weights.
        dict(name="linears-q8_0-13", op="linears", type="Q8_0", n_tok=13, pos=0, layers=4, **LLAMA),
        # A full prompt chunk, Q4_0 weights.
        dict(name="linears-q4_0-512", op="linears", type="Q4_0", n_tok=512, pos=0, layers=4, **LLAMA),
        # The ragged last chunk of a prompt, unquantized f16 weights.
        dict(name="linears-f16-389", op="linears", type="F16", n_tok=389, pos=0, layers=2, **LLAMA),
        # Next-token logits over the full vocabulary, from a Q6_K output matrix.
        dict(name="logits-q6_k", op="linear", type="Q6_K", n_in=3072, n_out=128256, n_tok=1, norm=True),
        # One whole generated token (eight layers, Q4_0).
        dict(name="model-decode", op="model", type="Q4_0", n_layer=8, n_vocab=32064, pos=600, n_tok=1, **LLAMA),
        # A whole prompt of ordinary length (eight layers, Q4_0).
        dict(name="model-prefill-157", op="model", type="Q4_0", n_layer=8, n_vocab=32064, pos=0, n_tok=157, **LLAMA),
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    op = rng.choice(["decode", "prefill", "linears", "linear", "prefill", "linears", "linear"])
    if op in ("decode", "prefill"):
        # head sizes: mostly the three with tuned kernels, and others of the same range
        hd = rng.choice([64, 128, 128, 128, 256, 80, 96, 112])
        n_head_kv = rng.choice([2, 4, 8])
        n_head = n_head_kv * rng.choice([1, 2, 3, 3, 4, 7, 8])
        if op == "decode":
            n_keys = _log(rng, 16, 8192)
            return dict(op=op, n_head=n_head, n_head_kv=n_head_kv, head_dim=hd, n_keys=n_keys,
                        layers=max(2, min(28, 60_000_000 // (n_keys * n_head_kv * hd))))
        n_tok = _log(rng, 2, 1024)
        pos = rng.choice([0, _log(rng, 1, 4096)])
        return dict(op=op, n_head=n_head, n_head_kv=n_head_kv, head_dim=hd, pos=pos, n_tok=n_tok, layers=1)
    t = rng.choice(["Q4_0", "Q4_0", "Q8_0", "F16", "Q6_K", "Q4_1", "BF16", "F32"])
    if op == "linear":
        n_in = 256 * _log(rng, 1, 32)
        n_out = _log(rng, 48, 16384)
        return dict(op=op, type=t, n_in=n_in, n_out=n_out, n_tok=rng.choice([1, _log(rng, 2, 64), _log(rng, 64, 1024)]), norm=False)
    # a whole layer's projections, of the benchmarked model's width or half of it
    half = rng.choice([False, True])
    shape = dict(n_embd=2048, n_head=32, n_head_kv=8, head_dim=64, n_ff=8192) if half else dict(LLAMA)
    n_tok = rng.choice([1, _log(rng, 2, 64), _log(rng, 64, 700)])
    return dict(op=op, type=t, n_tok=n_tok, pos=rng.randrange(0, 2048) if n_tok == 1 else 0, layers=2, **shape)


# ---------------------------------------------------------------- inputs

def _gen(seed):
    g = torch.Generator(device=DEV)
    g.manual_seed(int(seed))
    return g


def _f16_bytes(x):
    return x.to(torch.float16).contiguous().view(torch.uint8)


def weights(t, n_out, n_in, g, gain=1.0):
    """Rows of GGUF type t whose values are about N(0, gain / sqrt(n_in)), as raw bytes."""
    sd = gain / math.sqrt(n_in)
    if BLOCK[t][0] == 1:
        w = torch.randn(n_out, n_in, generator=g, **F32) * sd
        w = {"F32": w, "F16": w.half(), "BF16": w.bfloat16()}[t]
        return w.contiguous().view(torch.uint8).reshape(-1)
    be, bb = BLOCK[t]
    nb = n_in // be
    out = torch.empty(n_out, nb, bb, dtype=torch.uint8, device=DEV)
    spread = 0.7 + 0.6 * torch.rand(n_out, nb, 1, generator=g, **F32)
    z = torch.randn(n_out, nb, be, generator=g, **F32)
    if t == "Q8_0":
        out[..., 2:] = (z * 40).round().clamp(-127, 127).to(torch.int8).view(torch.uint8)
        out[..., :2] = _f16_bytes(spread * sd / 40)
    elif t in ("Q4_0", "Q4_1"):
        q = ((z * 2.7).round() + 8).clamp(0, 15).to(torch.uint8)
        d = spread * sd / 2.7
        out[..., bb - 16:] = q[..., :16] | (q[..., 16:] << 4)
        out[..., :2] = _f16_bytes(d)
        if t == "Q4_1":
            out[..., 2:4] = _f16_bytes(-8 * d)
    else:  # Q6_K: halves of 128: ql[64], qh[32]; then 16 scales and d
        q = ((z * 10).round() + 32).clamp(0, 63).to(torch.uint8).view(n_out, nb, 2, 4, 32)
        lo, hi = q & 15, q >> 4
        out[..., :128] = (lo[..., :2, :] | (lo[..., 2:, :] << 4)).reshape(n_out, nb, 128)
        out[..., 128:192] = (hi[..., 0, :] | (hi[..., 1, :] << 2) | (hi[..., 2, :] << 4) | (hi[..., 3, :] << 6)).reshape(n_out, nb, 64)
        out[..., 192:208] = torch.randint(40, 90, (n_out, nb, 16), generator=g, device=DEV, dtype=torch.int8).view(torch.uint8)
        out[..., 208:] = _f16_bytes(spread * sd / 640)
    return out.reshape(-1)


def dequant(t, raw, n_out, n_in):
    """The rows of `weights` (or of any such bytes) in 64 bits."""
    if t == "F32":
        return raw.view(torch.float32).view(n_out, n_in).double()
    if t == "F16":
        return raw.view(torch.float16).view(n_out, n_in).double()
    if t == "BF16":
        return raw.view(torch.bfloat16).view(n_out, n_in).double()
    be, bb = BLOCK[t]
    b = raw.view(n_out, n_in // be, bb)

    def half(lo):
        return b[..., lo:lo + 2].contiguous().view(torch.float16).double()

    if t == "Q8_0":
        w = half(0) * b[..., 2:].contiguous().view(torch.int8).double()
    elif t in ("Q4_0", "Q4_1"):
        qs = b[..., bb - 16:]
        q = torch.cat([qs & 15, qs >> 4], -1).double()
        w = half(0) * (q - 8) if t == "Q4_0" else half(0) * q + half(2)
    else:
        ql = b[..., :128].reshape(*b.shape[:2], 2, 2, 32)
        qh = b[..., 128:192].reshape(*b.shape[:2], 2, 1, 32)
        lo = torch.cat([ql & 15, ql >> 4], -2)
        hi = torch.cat([(qh >> s) & 3 for s in (0, 2, 4, 6)], -2)
        q = (lo | (hi << 4)).double() - 32
        sc = b[..., 192:208].contiguous().view(torch.int8).double().view(*b.shape[:2], 2, 4, 2, 1)
        w = (half(208).view(*b.shape[:2], 1, 1, 1, 1) * sc * q.view(*b.shape[:2], 2, 4, 2, 16))
    return w.reshape(n_out, n_in)


def _inv_freq(hd):
    """Rotary frequencies theta^(-2i/hd), formed in f32 by repeated products."""
    step, f, out = np.float32(THETA ** (-2.0 / hd)), np.float32(1), []
    for _ in range(hd // 2):
        out.append(f)
        f = np.float32(f * step)
    return np.array(out, dtype=np.float32)


def _norm_w(n, g):
    return 1.0 + 0.1 * torch.randn(n, generator=g, **F32)


def _acts(n_tok, n, g):
    """Activations: normal, some channels larger than others."""
    return torch.randn(n_tok, n, generator=g, **F32) * torch.exp(0.4 * torch.randn(n, generator=g, **F32))


def _attn_inputs(case, seed):
    g = _gen(seed)
    n_keys = case["n_keys"] if case["op"] == "decode" else case["pos"] + case["n_tok"]
    kvd, n_tok = case["n_head_kv"] * case["head_dim"], case.get("n_tok", 1)
    rows = case["layers"] * n_keys
    k = torch.randn(rows, kvd, generator=g, **F32).half()
    v = torch.randn(rows, kvd, generator=g, **F32).half()
    q = torch.randn(case["layers"], n_tok, case["n_head"] * case["head_dim"], generator=g, **F32)
    return k, v, q, n_keys, kvd


def _linears_inputs(case, seed):
    g = _gen(seed)
    t, ne, nf = case["type"], case["n_embd"], case["n_ff"]
    qd, kvd = case["n_head"] * case["head_dim"], case["n_head_kv"] * case["head_dim"]
    layers = []
    for _ in range(case["layers"]):
        layers.append(dict(
            norm1=_norm_w(ne, g), norm2=_norm_w(ne, g),
            wq=weights(t, qd, ne, g), wk=weights(t, kvd, ne, g), wv=weights(t, kvd, ne, g),
            wo=weights(t, ne, qd, g, 0.5), gate=weights(t, nf, ne, g), up=weights(t, nf, ne, g),
            down=weights(t, ne, nf, g, 0.5), attn=_acts(case["n_tok"], qd, g)))
    table = weights("F16", 1024, ne, g, math.sqrt(ne))
    tokens = torch.randint(0, 1024, (case["n_tok"],), generator=g, device=DEV, dtype=torch.int32)
    return layers, table, tokens, qd, kvd


def _linear_inputs(case, seed):
    g = _gen(seed)
    w = weights(case["type"], case["n_out"], case["n_in"], g)
    return w, _acts(case["n_tok"], case["n_in"], g), _norm_w(case["n_in"], g)


def _model_inputs(case, seed):
    """A model dict as HipForward takes it (two different layers, used in turn), a filled cache
    below pos, and the tokens."""
    g = _gen(seed)
    t, ne, nf = case["type"], case["n_embd"], case["n_ff"]
    qd, kvd = case["n_head"] * case["head_dim"], case["n_head_kv"] * case["head_dim"]
    up = lambda n_out, n_in, gain=1.0: (t, weights(t, n_out, n_in, g, gain).cpu().numpy())  # noqa: E731
    kinds = [dict(attn_norm=_norm_w(ne, g).cpu().numpy(), ffn_norm=_norm_w(ne, g).cpu().numpy(),
                  wq=up(qd, ne), wk=up(kvd, ne), wv=up(kvd, ne), wo=up(ne, qd, 0.5),
                  w_gate=up(nf, ne), w_up=up(nf, ne), w_down=up(ne, nf, 0.5)) for _ in range(2)]
    embd = up(case["n_vocab"], ne, math.sqrt(ne))
    m = dict(cfg=dict(n_layer=case["n_layer"], n_embd=ne, n_head=case["n_head"], n_head_kv=case["n_head_kv"],
                      head_dim=case["head_dim"], n_ff=nf, n_vocab=case["n_vocab"], rope_theta=THETA, rms_eps=EPS),
             rope_inv_freq=_inv_freq(case["head_dim"]), layers=[kinds[i % 2] for i in range(case["n_layer"])],
             tok_embd=embd, output=embd, output_norm=_norm_w(ne, g).cpu().numpy())
    rows = case["n_layer"] * (case["pos"] + case["n_tok"])
    k = torch.randn(rows, kvd, generator=g, **F32).half()
    v = torch.randn(rows, kvd, generator=g, **F32).half()
    tokens = torch.randint(0, case["n_vocab"], (case["n_tok"],), generator=g, device=DEV, dtype=torch.int32)
    return m, k, v, tokens


# ---------------------------------------------------------------- a pass

def prepare(case, seed):
    s = {"ws": ia.Workspace(DEV), "lws": ia.Workspace(DEV)}
    if case["op"] in ("decode", "prefill"):
        k, v, q, n_keys, kvd = _attn_inputs(case, seed)
        heads = (case["n_head"], case["n_head_kv"], case["head_dim"])
        out = torch.empty_like(q)
        if case["op"] == "decode":
            d = [ia.decode_desc(*heads, n_keys, kv_offset=i * n_keys * kvd) for i in range(case["layers"])]
            s["pass"] = lambda: [ia.attn_decode(q[i], k, v, out[i], x, workspace=s["ws"]) for i, x in enumerate(d)]
        else:
            d = [ia.prefill_desc(*heads, case["pos"], case["n_tok"], kv_offset=i * n_keys * kvd) for i in range(case["layers"])]
            s["pass"] = lambda: [ia.attn_prefill(q[i], k, v, out[i], x, workspace=s["ws"]) for i, x in enumerate(d)]
        s["out"] = out
    elif case["op"] == "linears":
        _prepare_linears(case, seed, s)
    elif case["op"] == "linear":
        w, x, nw = _linear_inputs(case, seed)
        out = torch.empty(case["n_tok"], case["n_out"], **F32)
        if case["norm"]:
            d = ia.proj_desc(case["type"], case["n_in"], [case["n_out"]], prologue=ia.PROJ_RMSNORM, eps=EPS)
            s["pass"] = lambda: ia.proj([w], x, [out], d, norm_w=nw)
        else:
            d = ia.linear_desc(case["type"], case["n_in"], case["n_out"], case["n_tok"])
            s["pass"] = lambda: ia.linear(w, x, out, d, workspace=s["lws"])
        s["out"] = out
    else:
        m, k, v, tokens = _model_inputs(case, seed)
        f = fwd.HipForward(m, n_ctx=case["pos"] + case["n_tok"], n_batch=case["n_tok"], device=DEV)
        f.k_cache.copy_(k)
        f.v_cache.copy_(v)
        ids = tokens.cpu().tolist()
        s["pass"] = lambda: f.forward_batch(ids, case["pos"], tokens_on_device=tokens)
        s["out"] = {"logits": f.logits, "k": f.k_cache, "v": f.v_cache}
    one_token = case["op"] == "decode" or (case["op"] in ("linears", "model") and case["n_tok"] == 1)
    if one_token:  # a decode loop replays its token step as a graph
        s["pass"]()
        torch.cuda.synchronize()
        s["graph"] = torch.cuda.CUDAGraph()
        with torch.cuda.graph(s["graph"]):
            s["pass"]()
    return s


def _prepare_linears(case, seed, s):
    layers, table, tokens, qd, kvd = _linears_inputs(case, seed)
    t, ne, nf, n, lws = case["type"], case["n_embd"], case["n_ff"], case["n_tok"], s["lws"]
    x, h = torch.empty(n, ne, **F32), torch.empty(n, ne, **F32)
    # the q/k/v of the first layer and the feed-forward activations of the last come back
    q, k, v = (torch.empty(n, c, **F32) for c in (qd, kvd, kvd))
    gate, up = torch.empty(n, nf, **F32), torch.empty(n, nf, **F32)
    wo, down = ia.linear_desc(t, qd, ne, n, accumulate=True), ia.linear_desc(t, nf, ne, n, accumulate=True)

    def ffn_tail(L):
        ia.linear(L["down"], gate, x, down, workspace=lws)

    if n == 1:
        kc = torch.zeros(case["layers"] * (case["pos"] + 1), kvd, dtype=torch.float16, device=DEV)
        vc = torch.zeros_like(kc)
        inv = torch.from_numpy(_inv_freq(case["head_dim"])).to(DEV)
        qkv = ia.proj_desc(t, ne, [qd, kvd, kvd], prologue=ia.PROJ_RMSNORM, eps=EPS)
        ffn = ia.proj_desc(t, ne, [nf, nf], prologue=ia.PROJ_RMSNORM, epilogue=ia.PROJ_SILU_GATE, eps=EPS)
        ropes = [ia.rope_kv_desc(case["n_head"], case["n_head_kv"], case["head_dim"], case["pos"], 1,
                                 dst_offset=(i * (case["pos"] + 1) + case["pos"]) * kvd) for i in range(case["layers"])]

        def one_pass():
            ia.get_rows("F16", table, ne, 1024, tokens, 1, x)
            for L, r in zip(layers, ropes):
                ia.proj_rope_kv([L["wq"], L["wk"], L["wv"]], x, q, k, v, kc, vc, inv, qkv, r, norm_w=L["norm1"])
                ia.linear(L["wo"], L["attn"], x, wo, workspace=lws)
                ia.proj([L["gate"], L["up"]], x, [gate], ffn, norm_w=L["norm2"])
                ffn_tail(L)

        s["pass"], s["out"] = one_pass, {"q": q, "k": kc, "v": vc, "ffn": gate, "x": x}
        return
    qkv = ia.proj_desc(t, ne, [qd, kvd, kvd], n_tok=n)
    ffn = ia.proj_desc(t, ne, [nf, nf], epilogue=ia.PROJ_SILU_GATE, n_tok=n)
    dq, dkv, dff = (ia.linear_desc(t, ne, c, n) for c in (qd, kvd, nf))

    def chunk_pass():
        ia.get_rows("F16", table, ne, 1024, tokens, n, x)
        for L in layers:
            ia.rmsnorm(x, L["norm1"], h, ne, n, EPS)
            if fwd.qkv_one_launch(n, qd, kvd):
                ia.proj([L["wq"], L["wk"], L["wv"]], h, [q, k, v], qkv)
            else:
                for w, o, d in ((L["wq"], q, dq), (L["wk"], k, dkv), (L["wv"], v, dkv)):
                    ia.linear(w, h, o, d, workspace=lws)
            ia.linear(L["wo"], L["attn"], x, wo, workspace=lws)
            ia.rmsnorm(x, L["norm2"], h, ne, n, EPS)
            if fwd.ffn_one_launch(n, nf):
                ia.proj([L["gate"], L["up"]], h, [gate], ffn)
            else:
                ia.linear(L["gate"], h, gate, dff, workspace=lws)
                ia.linear(L["up"], h, up, dff, workspace=lws)
                ia.silu_mul(gate, up, n * nf)
            ffn_tail(L)

    s["pass"], s["out"] = chunk_pass, {"q": q, "k": k, "v": v, "ffn": gate, "x": x}


def run(state):
    if "graph" in state:
        state["graph"].replay()
    else:
        state["pass"]()
    return state["out"]


# ---------------------------------------------------------------- what it cannot do without

def _wbytes(t, n_out, n_in):
    return n_out * (n_in // BLOCK[t][0]) * BLOCK[t][1]


def _layer_work(t, n, ne, nf, qd, kvd):
    w = sum(_wbytes(t, o, i) for o, i in ((qd, ne), (kvd, ne), (kvd, ne), (ne, qd), (nf, ne), (nf, ne), (ne, nf)))
    flops = 2 * n * (ne * (qd + 2 * kvd) + qd * ne + 3 * ne * nf)
    return w, flops


def _attn_work(nh, nkv, hd, pos, n):
    keys = n * pos + n * (n + 1) // 2  # visible (query, key) pairs of a head
    return 2 * (pos + n) * nkv * hd * 2 + 2 * n * nh * hd * 4, 4 * hd * nh * keys


def work(case):
    op = case["op"]
    if op in ("decode", "prefill"):
        pos, n = (case["n_keys"] - 1, 1) if op == "decode" else (case["pos"], case["n_tok"])
        b, f = _attn_work(case["n_head"], case["n_head_kv"], case["head_dim"], pos, n)
        return {"bytes": case["layers"] * b, "flops": case["layers"] * f}
    n = case["n_tok"]
    if op == "linear":
        return {"bytes": _wbytes(case["type"], case["n_out"], case["n_in"]) + 4 * n * (case["n_in"] + case["n_out"]),
                "flops": 2 * n * case["n_in"] * case["n_out"]}
    ne, nf, qd, kvd = case["n_embd"], case["n_ff"], case["n_head"] * case["head_dim"], case["n_head_kv"] * case["head_dim"]
    w, f = _layer_work(case["type"], n, ne, nf, qd, kvd)
    if op == "linears":  # weights, the embedding rows and attention output in, the outputs out
        return {"bytes": case["layers"] * (w + 4 * n * qd) + n * (2 * ne + 4 * (ne + nf + qd + 2 * kvd)),
                "flops": case["layers"] * f}
    b, fa = _attn_work(case["n_head"], case["n_head_kv"], case["head_dim"], case["pos"], n)
    return {"bytes": case["n_layer"] * (w + b) + _wbytes(case["type"], case["n_vocab"], ne) + 4 * case["n_vocab"],
            "flops": case["n_layer"] * (f + fa) + 2 * ne * case["n_vocab"]}


def tolerance(case):
    op, n = case["op"], case.get("n_tok", 1)
    # About four times the distance measured between this path and 64 bits.
    if op == "decode":
        return {"rel": 2e-6, "max": 3e-5}
    if op == "prefill":  # q and the probabilities in f16 at the tuned head sizes, f32 at the others
        return {"rel": 1.5e-3, "max": 2e-2} if case["head_dim"] in (64, 128, 256) else {"rel": 2e-6, "max": 3e-5}
    if op == "linear":  # a chunk's inputs and weights are rounded to f16
        return {"rel": 4e-6, "max": 4e-5} if n == 1 else {"rel": 1.5e-3, "max": 1e-2}
    # chains of layers: a cache value may round to the other f16 neighbour; a chunk's inputs are
    # rounded to f16 in every product
    return {"rel": 3e-5, "max": 3e-3} if n == 1 else {"rel": 2.5e-3, "max": 5e-2}


# ---------------------------------------------------------------- the same in 64 bits

def _attn64(q, k, v, nh, nkv, hd, pos):
    """q [n][nh*hd] at positions pos.., k and v [pos + n][nkv*hd], all f64."""
    n, L = q.shape[0], k.shape[0]
    out = torch.empty_like(q)
    hide = torch.arange(L, device=q.device)[None, :] > pos + torch.arange(n, device=q.device)[:, None]
    for h in range(nh):
        c = slice((h // (nh // nkv)) * hd, (h // (nh // nkv) + 1) * hd)
        s = q[:, h * hd:(h + 1) * hd] @ k[:, c].t().contiguous() / math.sqrt(hd)
        out[:, h * hd:(h + 1) * hd] = torch.softmax(s.masked_fill(hide, -math.inf), -1) @ v[:, c].contiguous()
    return out


def _rms64(x, w):
    return x / torch.sqrt((x * x).mean(-1, keepdim=True) + EPS) * w.double()


def _rope64(x, pos, hd):
    n = x.shape[0]
    p = torch.arange(pos, pos + n, dtype=torch.float32, device=x.device)
    a = (p[:, None] * torch.from_numpy(_inv_freq(hd)).to(x.device)[None, :]).double()[:, None, :]
    y = x.view(n, -1, hd // 2, 2)
    c, s = torch.cos(a), torch.sin(a)
    return torch.stack([y[..., 0] * c - y[..., 1] * s, y[..., 0] * s + y[..., 1] * c], -1).view(n, -1)


def _mul64(x, t, raw, n_out, n_in):
    """x times the rows' transpose, some rows at a time."""
    per = max(1, (1 << 27) // n_in)
    rb = raw.numel() // n_out
    return torch.cat([x @ dequant(t, raw[r * rb:min(n_out, r + per) * rb], min(n_out, r + per) - r, n_in).t()
                      for r in range(0, n_out, per)], -1)


def exact(case, seed):
    op = case["op"]
    if op in ("decode", "prefill"):
        k, v, q, n_keys, kvd = _attn_inputs(case, seed)
        pos = n_keys - q.shape[1]
        return torch.stack([_attn64(q[i].double(), k[i * n_keys:(i + 1) * n_keys].double(), v[i * n_keys:(i + 1) * n_keys].double(),
                                    case["n_head"], case["n_head_kv"], case["head_dim"], pos) for i in range(case["layers"])])
    t = case["type"]
    if op == "linear":
        w, x, nw = _linear_inputs(case, seed)
        x = _rms64(x.double(), nw) if case["norm"] else x.double()
        return _mul64(x, t, w, case["n_out"], case["n_in"])
    n, ne, nf, hd, pos = case["n_tok"], case["n_embd"], case["n_ff"], case["head_dim"], case["pos"]
    if op == "linears":
        layers, table, tokens, qd, kvd = _linears_inputs(case, seed)
        x = dequant("F16", table, 1024, ne)[tokens.long()]
        kc = torch.zeros(case["layers"] * (pos + 1), kvd, dtype=torch.float64, device=DEV)
        vc = torch.zeros_like(kc)
        for i, L in enumerate(layers):
            h = _rms64(x, L["norm1"])
            q, k, v = (_mul64(h, t, L[w], o, ne) for w, o in (("wq", qd), ("wk", kvd), ("wv", kvd)))
            if n == 1:
                q, k = _rope64(q, pos, hd), _rope64(k, pos, hd)
                kc[i * (pos + 1) + pos], vc[i * (pos + 1) + pos] = k[0].half(), v[0].half()  # the cache holds f16
            x = x + _mul64(L["attn"].double(), t, L["wo"], ne, qd)
            h = _rms64(x, L["norm2"])
            ffn = torch.nn.functional.silu(_mul64(h, t, L["gate"], nf, ne)) * _mul64(h, t, L["up"], nf, ne)
            x = x + _mul64(ffn, t, L["down"], ne, nf)
        return {"q": q, "k": kc if n == 1 else k, "v": vc if n == 1 else v, "ffn": ffn, "x": x}
    m, k0, v0, tokens = _model_inputs(case, seed)
    qd, kvd, rows = case["n_head"] * hd, case["n_head_kv"] * hd, pos + n
    kc, vc = k0.double(), v0.double()
    dev = lambda a: torch.from_numpy(np.ascontiguousarray(a)).reshape(-1).to(DEV)  # noqa: E731
    table = dev(m["tok_embd"][1])
    x = dequant(t, table, case["n_vocab"], ne)[tokens.long()]
    for i, L in enumerate(m["layers"]):
        mul = lambda a, w, o, j: _mul64(a, t, dev(L[w][1]), o, j)  # noqa: E731
        h = _rms64(x, dev(L["attn_norm"]))
        at = slice(i * rows + pos, (i + 1) * rows)
        kc[at] = _rope64(mul(h, "wk", kvd, ne), pos, hd).half().double()  # the cache holds f16
        vc[at] = mul(h, "wv", kvd, ne).half().double()
        all_ = slice(i * rows, (i + 1) * rows)
        a = _attn64(_rope64(mul(h, "wq", qd, ne), pos, hd), kc[all_], vc[all_], case["n_head"], case["n_head_kv"], hd, pos)
        x = x + mul(a, "wo", ne, qd)
        h = _rms64(x, dev(L["ffn_norm"]))
        x = x + mul(torch.nn.functional.silu(mul(h, "w_gate", nf, ne)) * mul(h, "w_up", nf, ne), "w_down", ne, nf)
    logits = _mul64(_rms64(x[-1:], dev(m["output_norm"])), t, table, case["n_vocab"], ne)[0]
    return {"logits": logits, "k": kc, "v": vc}
