"""What is measured: the work a user of the framework has it do, call by call.

Every case goes through the public entry points (`myelith_amd.backend`,
`myelith_amd.model`, `myelith_amd.moe`).  The sizes are those of the two
architectures the repository knows (the Qwen2.5-0.5B and -7B layouts) and of
its MoE layer, with odd row counts among them.  Every output is an integer
that the numeric contract defines bit for bit, so every tolerance is "exact".

Kinds of case:
  linear   W8A16 projections of consecutive layers, M activation rows each
           (1: a decode step; 2-32: a decode batch; more: prefill chunks)
  head     the LM head over M rows, int16 or int8 weights
  score    teacher-forced scoring of logit rows: the integer log-softmax at
           the target token and the argmax of every row
  sample   choosing the next tokens of a decode batch: the seeded integer
           CDF draw and the argmax of every row
  moe      the integer MoE layer over T tokens
  decode   greedy decode of one sequence, the last step's logits returned
  batch    lock-step greedy decode of B sequences with contexts of different
           lengths, the last step's logits returned
  prefill  a prompt (or its next chunk) into the KV cache, the last row's
           logits returned
"""
from __future__ import annotations

import math

import numpy as np
import torch

from myelith_amd.backend import RocmBackend
from myelith_amd.luts import LutSet, exp_lut
from myelith_amd.model import QWEN25_05B, QWEN25_7B, IntegerModel, make_spec
from myelith_amd.moe import MoeLayer, moe_spec

# The 7B layout is cut to four layers (the widths, the rows and the positions
# choose the kernels, the depth does not), so that several states fit and are
# built quickly; the 0.5B layout keeps its 24.
ARCHS = {"7b": dict(QWEN25_7B, layers=4), "0.5b": dict(QWEN25_05B)}
V7, V05 = QWEN25_7B["vocab"], QWEN25_05B["vocab"]

# (N, K) of the projections of both layouts: q/k/v, o_proj, gate (or up), down.
PROJECTIONS = [(1152, 896), (896, 896), (4864, 896), (896, 4864),
               (4608, 3584), (3584, 3584), (18944, 3584), (3584, 18944)]

_BACKEND = None


def backend() -> RocmBackend:
    """One context per process, as a serving program keeps it."""
    global _BACKEND
    if _BACKEND is None:
        _BACKEND = RocmBackend(0)
    return _BACKEND


def listed():
    return [
        # the smallest projection, one row, through the 24 layers of the 0.5B layout: launches and latency count
        dict(name="linear_m1_small", kind="linear", M=1, N=896, K=896, layers=24, requant="channel"),
        # a decode batch of 13 sequences through the down projection: the weights' stream counts
        dict(name="linear_m13_down", kind="linear", M=13, N=3584, K=18944, layers=4, requant="channel"),
        # a prompt chunk of 200 tokens through q/k/v: too few tiles for the chip, too many rows for a stream
        dict(name="linear_m200_qkv", kind="linear", M=200, N=4608, K=3584, layers=4, requant="shift"),
        # a full prefill through one gate projection with multiplier requant: the matrix cores count
        dict(name="linear_m4001_gate", kind="linear", M=4001, N=18944, K=3584, layers=1, requant="mult"),
        # the int16 head over five rows (a small batch, or the drafts of one step)
        dict(name="head16_m5", kind="head", M=5, N=V7, K=3584, bits=16),
        # perplexity over a chunk of text: 600 logit rows
        dict(name="score_600", kind="score", M=600, V=V7),
        # one step's token choice for 24 sequences
        dict(name="sample_24", kind="sample", M=24, V=V7),
        # the MoE layer in a decode batch of 16 and over a prompt of 3001 tokens
        dict(name="moe_t16", kind="moe", T=16),
        dict(name="moe_t3001", kind="moe", T=3001),
        # one user's chat turn: 16 tokens at a 2000-token context
        dict(name="decode_7b", kind="decode", arch="7b", ctx=2000, steps=16),
        # a serving batch: 24 sequences of mixed lengths, four tokens each
        dict(name="batch_7b_b24", kind="batch", arch="7b", B=24, ctx=1900, steps=4),
        # a long prompt into an empty cache
        dict(name="prefill_7b_1500", kind="prefill", arch="7b", n=1500, pos0=0),
    ]


def _log(rng, lo, hi):
    return max(lo, min(hi, int(round(math.exp(rng.uniform(math.log(lo), math.log(hi + 0.5)))))))


def draw(rng):
    kind = rng.choice(["linear", "linear", "linear", "head", "score", "sample", "moe", "moe", "decode", "batch",
                       "prefill"])
    if kind == "linear":
        N, K = rng.choice(PROJECTIONS)
        if rng.random() < 0.3:
            N -= rng.randrange(1, 64)  # a shard or a pruned projection: any row count
        M = _log(rng, 1, 4000)
        layers = 4 if M <= 64 else 2 if M <= 512 else 1
        return dict(kind=kind, M=M, N=N, K=K, layers=layers, requant=rng.choice(["shift", "channel", "mult"]))
    if kind == "head":
        N, K, bits = rng.choice([(V7, 3584, 16), (V7, 3584, 8), (V05, 896, 8)])
        return dict(kind=kind, M=_log(rng, 1, 64), N=N, K=K, bits=bits)
    if kind == "score":
        return dict(kind=kind, M=_log(rng, 16, 2000), V=rng.choice([V7, V05, 32001]))
    if kind == "sample":
        return dict(kind=kind, M=_log(rng, 1, 64), V=rng.choice([V7, V05, 32001]))
    if kind == "moe":
        return dict(kind=kind, T=_log(rng, 1, 4000))
    arch = rng.choice(["7b", "0.5b"])
    if kind == "decode":
        return dict(kind=kind, arch=arch, ctx=_log(rng, 16, 2040), steps=rng.randrange(8, 17))
    if kind == "batch":
        return dict(kind=kind, arch=arch, B=_log(rng, 2, 32), ctx=_log(rng, 32, 2000), steps=4)
    return dict(kind=kind, arch=arch, n=_log(rng, 16, 1500), pos0=rng.choice([0, 0, rng.randrange(1, 500)]))


def _gen(seed):
    g = torch.Generator(device="cuda")
    g.manual_seed(seed)
    return g


def _gauss16(shape, g, sigma=2000.0):
    return torch.clamp(torch.round(torch.randn(shape, device="cuda", generator=g) * sigma), -32767, 32767).to(torch.int16)


def _linear_inputs(case, seed):
    """Per layer: activations (Gaussian, sd 2000), uniform int8 weights and the
    scales that bring the sums back to int16 activations of the same size."""
    g, layers = _gen(seed), []
    M, N, K = case["M"], case["N"], case["K"]
    growth = int(math.log2(73.0 * math.sqrt(K)))  # log2 of the sums' sd over the inputs'
    for _ in range(case["layers"]):
        x = _gauss16((M, K), g)
        W = torch.randint(-127, 128, (N, K), dtype=torch.int8, device="cuda", generator=g)
        if case["requant"] == "mult":
            a = torch.randint(1 << 29, (1 << 30) + 1, (N,), dtype=torch.int32, device="cuda", generator=g)
            b = torch.randint(growth + 29, growth + 32, (N,), dtype=torch.uint8, device="cuda", generator=g)
        else:
            a = torch.randint(growth, growth + 2, (N,), dtype=torch.uint8, device="cuda", generator=g)
            b = torch.randint(8, 12, (N,), dtype=torch.uint8, device="cuda", generator=g)
        layers.append((x, W, a, b))
    return layers


def _head_inputs(case, seed):
    g = _gen(seed)
    M, N, K, bits = case["M"], case["N"], case["K"], case["bits"]
    x = _gauss16((M, K), g)
    lim = 127 if bits == 8 else 32767
    W = torch.randint(-lim, lim + 1, (N, K), dtype=torch.int8 if bits == 8 else torch.int16, device="cuda", generator=g)
    lo = 8 if bits == 8 else 17
    return x, W, torch.randint(lo, lo + 3, (N,), dtype=torch.uint8, device="cuda", generator=g)


def _logit_rows(case, seed):
    """Q6 logits: Gaussian of sd 2.5 with a few likely tokens per row."""
    g = _gen(seed)
    M, V = case["M"], case["V"]
    z = torch.round(torch.randn((M, V), device="cuda", generator=g) * 160).to(torch.int32)
    top = torch.randint(0, V, (M, 8), device="cuda", generator=g)
    z.scatter_(1, top, torch.randint(500, 1200, (M, 8), dtype=torch.int32, device="cuda", generator=g))
    return z, top[:, 0].contiguous(), g


def _model(case, seed, max_pos):
    return IntegerModel(backend(), make_spec(ARCHS[case["arch"]], seed=seed, max_pos=max_pos))


def _contexts(case, rng):
    """Context lengths of a serving batch: one at the full length, the others down to an eighth of it."""
    ctx = rng.integers(max(1, case["ctx"] // 8), case["ctx"] + 1, case["B"])
    ctx[rng.integers(case["B"])] = case["ctx"]
    return ctx.astype(np.uint32)


def prepare(case, seed):
    be, kind = backend(), case["kind"]
    s = dict(case, be=be)
    rng = np.random.default_rng(seed)
    if kind == "linear":
        s["in"] = _linear_inputs(case, seed)
        s["out"] = [torch.empty((case["M"], case["N"]), dtype=torch.int16, device="cuda") for _ in s["in"]]
    elif kind == "head":
        s["in"] = _head_inputs(case, seed)
        s["out"] = torch.empty((case["M"], case["N"]), dtype=torch.int32, device="cuda")
    elif kind == "score":
        s["z"], s["targets"], _ = _logit_rows(case, seed)
        s["lut"] = torch.from_numpy(exp_lut()).cuda()
    elif kind == "sample":
        s["z"], _, g = _logit_rows(case, seed)
        s["states"] = torch.randint(-2**63, 2**63 - 1, (case["M"],), dtype=torch.int64, device="cuda", generator=g)
    elif kind == "moe":
        s["layer"] = MoeLayer(be, moe_spec(seed))
        s["x"] = _gauss16((case["T"], s["layer"].spec["hidden"]), _gen(seed))
        s["out"] = torch.empty_like(s["x"])
    elif kind == "decode":
        m = s["model"] = _model(case, seed, case["ctx"] + case["steps"] + 8)
        prompt = rng.integers(0, m.vocab_size, case["ctx"]).astype(np.uint32)
        m.prefill(prompt, 0, want_logits=False)
        s["token"] = int(rng.integers(m.vocab_size))
    elif kind == "batch":
        m = s["model"] = _model(case, seed, case["ctx"] + case["steps"] + 8)
        B, ctx = case["B"], _contexts(case, rng)
        m.batch_begin(B)
        rows = [(b, p) for b in range(B) for p in range(ctx[b])]
        for r0 in range(0, len(rows), 4096):
            seq, pos = np.array(rows[r0:r0 + 4096], np.uint32).T
            m.forward_batch(seq, pos, rng.integers(0, m.vocab_size, seq.size), want_logits=False)
        s.update(seq=np.arange(B, dtype=np.uint32), pos=ctx, tokens=rng.integers(0, m.vocab_size, B).astype(np.uint32))
    else:
        n, pos0 = case["n"], case["pos0"]
        m = s["model"] = _model(case, seed, n + pos0 + 8)
        toks = rng.integers(0, m.vocab_size, pos0 + n).astype(np.uint32)
        if pos0:
            m.prefill(toks[:pos0], 0, want_logits=False)
        s["tokens"] = toks[pos0:]
    torch.cuda.synchronize()
    return s


def run(s):
    be, kind = s["be"], s["kind"]
    if kind == "linear":
        for (x, W, a, b), out in zip(s["in"], s["out"]):
            if s["requant"] == "mult":
                be.linear_w8a16_mult_dev(x, W, a, b, out=out)
            elif s["requant"] == "channel":
                be.linear_w8a16_dev(x, W, a, 10, out_frac_pc=b, out=out)
            else:
                be.linear_w8a16_dev(x, W, a, 10, 10, out=out)
        return s["out"]
    if kind == "head":
        x, W, shifts = s["in"]
        return be.logits_dev(x, W, shifts, 10, 6, out=s["out"])
    if kind == "score":
        return be.logsoftmax_dev(s["z"], s["lut"], s["targets"]), be.argmax_dev(s["z"])
    if kind == "sample":
        return be.sample_dev(s["z"], s["states"]) + (be.argmax_dev(s["z"]),)
    if kind == "moe":
        return s["layer"].forward(s["x"], out=s["out"])
    m = s["model"]
    if kind == "decode":
        toks, _ = m.decode_greedy(s["token"], s["ctx"], s["steps"] - 1)
        return toks, m.forward_token(int(toks[-1]), s["ctx"] + s["steps"] - 1)
    if kind == "batch":
        toks = m.batch_decode_greedy(s["seq"], s["pos"], s["tokens"], s["steps"])
        # the view is the model's own memory until its next batched call: a caller who keeps the logits copies them
        return toks, m.batch_logits_dev(s["B"]).clone()
    return m.prefill(s["tokens"], s["pos0"])


def _layer_weights(a):
    nq, nkv = a["heads"] * a["head_dim"], a["kv_heads"] * a["head_dim"]
    return a["hidden"] * (2 * nq + 2 * nkv) + 3 * a["hidden"] * a["inter"]


def work(case):
    kind = case["kind"]
    if kind == "linear":
        M, N, K, n = case["M"], case["N"], case["K"], case["layers"]
        scales = {"shift": 1, "channel": 2, "mult": 5}[case["requant"]]
        return {"bytes": n * (N * K + 2 * M * K + 2 * M * N + scales * N), "flops": 2 * n * M * N * K}
    if kind == "head":
        M, N, K = case["M"], case["N"], case["K"]
        return {"bytes": N * K * case["bits"] // 8 + 2 * M * K + 4 * M * N + N, "flops": 2 * M * N * K}
    if kind in ("score", "sample"):
        M, V = case["M"], case["V"]
        return {"bytes": 4 * M * V + 32 * M, "flops": 2 * M * V}
    if kind == "moe":
        p = moe_spec(0)
        T, H, E, I, k, S = case["T"], p["hidden"], p["n_experts"], p["inter"], p["top_k"], p["shared_inter"]
        load = 1.0 / np.arange(1, E + 1)
        load = np.minimum(1.0, k * load / load.sum())  # expected share of the tokens per expert
        used = float((1.0 - (1.0 - load) ** T).sum())
        return {"bytes": int(used * 3 * H * I + 3 * H * S + E * H + 4 * T * H), "flops": 2 * T * (E * H + 3 * H * (k * I + S))}
    a = ARCHS[case["arch"]]
    H, V = a["hidden"], a["vocab"]
    layer, head_w = a["layers"] * _layer_weights(a), (2 if a["lm_head_int16"] else 1) * V * H
    kv_row = 4 * a["layers"] * a["kv_heads"] * a["head_dim"]      # K and V bytes of one position
    attn = 4 * a["layers"] * a["heads"] * a["head_dim"]           # operations per (query, position)
    if kind == "decode":
        n, pos = case["steps"], case["ctx"] + case["steps"] / 2
        return {"bytes": int(n * (layer + head_w + kv_row * pos + 4 * V)), "flops": int(n * (2 * (layer + V * H) + attn * pos))}
    if kind == "batch":
        n, B, pos = case["steps"], case["B"], case["ctx"] * 9 / 16  # contexts between an eighth and the whole
        return {"bytes": int(n * (layer + head_w + B * (kv_row * pos + 4 * V))),
                "flops": int(n * B * (2 * (layer + V * H) + attn * pos))}
    n, pos0 = case["n"], case["pos0"]
    return {"bytes": int(layer + head_w + kv_row * (pos0 + n) + 2 * n * H + 4 * V),
            "flops": int(2 * n * layer + 2 * V * H + attn * n * (pos0 + n / 2))}


def tolerance(case):
    return "exact"


def _rne(v, shift):
    """v / 2^shift of int64 tensors, rounded half to even."""
    q = v >> shift
    r, half = v - (q << shift), torch.ones_like(shift) << (shift - 1)
    return q + ((r > half) | ((r == half) & ((q & 1) == 1))).to(torch.int64)


def exact(case, seed):
    """The products and their requantization in 64 bits: the sums are whole
    numbers below 2^53, so a float64 product holds them exactly.  The other
    kinds' outputs are whole numbers chosen by tables and comparisons (tokens,
    table logarithms, whole models), which have no value in real arithmetic to
    be near to."""
    if case["kind"] == "linear":
        outs = []
        for x, W, a, b in _linear_inputs(case, seed):
            acc = (x.double() @ W.double().T).to(torch.int64)
            a, b = a.to(torch.int64), b.to(torch.int64)
            if case["requant"] == "mult":
                y = _rne(acc * a, b)
            else:
                y = _rne(acc, a + 10 - (b if case["requant"] == "channel" else 10))
            outs.append(torch.clamp(y, -32768, 32767).to(torch.int16))
        return outs
    if case["kind"] == "head":
        x, W, shifts = _head_inputs(case, seed)
        out = torch.empty((case["M"], case["N"]), dtype=torch.int32, device="cuda")
        for n0 in range(0, case["N"], 16384):
            acc = (x.double() @ W[n0:n0 + 16384].double().T).to(torch.int64)
            y = _rne(acc, shifts[n0:n0 + 16384].to(torch.int64) + 10 - 6)
            out[:, n0:n0 + 16384] = torch.clamp(y, -2**31, 2**31 - 1).to(torch.int32)
        return out
    return None
