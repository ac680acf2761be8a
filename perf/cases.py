"""The workloads whose time counts: what a user of this library has it do, through its
public entry points (the C API of include/gehtp_kernels.h and the runlist engine), from a
one-token call to a 2048-token prompt.

    listed()             the named cases
    draw(rng)            one more case of the same ranges
    prepare(case, seed)  inputs, weights, workspaces and parsed blobs, on the GPU
    run(state)           one pass; returns its outputs
    work(case)           bytes and floating-point operations of one pass
    tolerance(case)      how far two correct implementations may differ
    exact(case, seed)    the same outputs in 64 bits, in plain torch / numpy

Kinds of case:
  mlp          the decoder MLP block on M tokens: RMSNorm, gate/up linear with SwiGLU,
               down linear with residual (W4A16 group 64). M <= 4 takes the RMSNorm inside
               the gate/up call, as the decode step does; longer inputs normalize first.
  proj         one W4A16 linear: the attention projections, and generic (odd) widths.
  attn_prefill causal (or full) GQA attention over a prompt, head dim 128.
  attn_decode  one token's attention over a KV ring, head dim 128.
  f16          OP_MATMUL_F16, the reference runlist's plain fp16 linear, weights stored
               [K, N] (as its front-end writes them) or [N, K].
  attn_ops     attention as the reference runlist's separate ops (batched MATMUL_F16,
               SOFTMAX, MATMUL_F16) for head dims the fused kernels do not take.
  w4a16        opcode 1: u16 crouton surfaces times int4 weights, divided by 7.
  request      a whole small model through the engine: prompt, then decode steps, logits
               of each (this build's fused opcodes).
  chain        the same model's prompt in the reference front-end's own op chain.
"""
from __future__ import annotations

import functools
import math
from dataclasses import replace

import numpy as np
import torch

from gehtp_amd import Engine, lib_path, load_library
from gehtp_amd.qwen3 import CONFIG_08B_LAYER, CONFIG_4B, Weights, emit_decode, emit_prefill
from gehtp_amd.qwen3_chain import emit_prefill_chain

HD = 128
GEMV_TOKENS = 4          # up to this many tokens the linears take the RMSNorm themselves
MODELS = {"0.8b": CONFIG_08B_LAYER, "4b": CONFIG_4B}
# The whole-model cases: four layers of the 0.8B-class model with its vocabulary.
ENGINE_CFG = replace(CONFIG_08B_LAYER, layers=4)
MAX_POS = 1024
ENGINE_SEED = 0          # one model per process; only the prompts change


# ---------------------------------------------------------------------------- the cases
def listed():
    return [
        # a decode step's MLP in the small model: latency and launches
        {"name": "mlp_decode_small", "kind": "mlp", "model": "0.8b", "M": 1},
        # a few tokens at once: short prompts, speculative verification, small batches
        {"name": "mlp_tokens_8", "kind": "mlp", "model": "4b", "M": 8},
        # the benchmark model's prompt
        {"name": "mlp_prompt_2048", "kind": "mlp", "model": "4b", "M": 2048},
        # RMSNorm + linear of a 512-token prompt (benchmark configuration 2)
        {"name": "proj_prompt_512", "kind": "proj", "M": 512, "N": 3072, "K": 1024, "norm": True},
        # causal GQA attention over 1024 tokens, and one token over 4096 cached ones
        # (benchmark configuration 3)
        {"name": "attn_prompt_1024", "kind": "attn_prefill", "S": 1024, "H": 16, "KVH": 8, "causal": True},
        {"name": "attn_decode_4096", "kind": "attn_decode", "n_kv": 4096, "H": 16, "KVH": 8},
        # the reference runlist's fp16 linear over a prompt, and for one decoded token
        {"name": "f16_prompt_512", "kind": "f16", "M": 512, "N": 3072, "K": 1024, "t1": False},
        {"name": "f16_decode", "kind": "f16", "M": 1, "N": 3072, "K": 1024, "t1": False},
        # attention op by op at head dim 64, 256 tokens
        {"name": "attn_ops_256", "kind": "attn_ops", "S": 256, "T": 256, "H": 16, "hd": 64},
        # opcode 1 at the reference's own golden shape
        {"name": "w4a16_256", "kind": "w4a16", "M": 256, "N": 2560, "K": 2560},
        # a request through the engine: a 200-token prompt and 8 decode steps
        {"name": "request_200_8", "kind": "request", "S": 200, "steps": 8},
        # a 128-token prompt through the reference front-end's op chain
        {"name": "chain_prompt_128", "kind": "chain", "S": 128},
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["mlp", "mlp", "proj", "proj", "attn_prefill", "attn_decode", "f16", "f16", "attn_ops", "w4a16",
                       "request", "chain"])
    if kind == "mlp":
        return {"kind": kind, "model": rng.choice(sorted(MODELS)), "M": _log(rng, 1, 2048)}
    if kind == "proj":
        c = MODELS[rng.choice(sorted(MODELS))]
        n, k = rng.choice([(c.q_dim + 2 * c.kv_dim, c.hidden), (c.hidden, c.q_dim),
                           (_log(rng, 256, 8192), 64 * rng.randint(4, 64))])
        return {"kind": kind, "M": _log(rng, 1, 2048), "N": n, "K": k, "norm": rng.random() < 0.5}
    if kind == "attn_prefill":
        H, KVH = rng.choice([(16, 8), (32, 8), (8, 8)])
        return {"kind": kind, "S": _log(rng, 16, 2048), "H": H, "KVH": KVH, "causal": rng.random() < 0.75}
    if kind == "attn_decode":
        H, KVH = rng.choice([(16, 8), (32, 8), (8, 8)])
        return {"kind": kind, "n_kv": _log(rng, 64, 16384), "H": H, "KVH": KVH}
    if kind == "f16":
        return {"kind": kind, "M": _log(rng, 1, 1024), "N": _log(rng, 256, 4096) | rng.randint(0, 1),
                "K": rng.choice([512, 1024, 2560, 3072, _log(rng, 256, 4096)]), "t1": rng.random() < 0.4}
    if kind == "attn_ops":
        T = _log(rng, 32, 512)
        return {"kind": kind, "S": rng.choice([1, T]), "T": T, "H": rng.choice([4, 8, 16]), "hd": rng.choice([32, 64, 80])}
    if kind == "w4a16":
        return {"kind": kind, "M": 32 * _log(rng, 1, 32), "N": 32 * _log(rng, 8, 128), "K": 32 * _log(rng, 8, 128)}
    if kind == "request":
        return {"kind": kind, "S": _log(rng, 8, 512), "steps": rng.randint(1, 8)}
    return {"kind": kind, "S": _log(rng, 8, 256)}


# ---------------------------------------------------------------------------- inputs
def _gen(seed):
    g = torch.Generator(device="cuda")
    g.manual_seed(int(seed))
    return g


def _normal(g, *shape):
    return torch.randn(shape, device="cuda", generator=g).half()


def _uniform(g, lo, hi, *shape):
    return (torch.rand(shape, device="cuda", generator=g) * (hi - lo) + lo).half()


def _w4g(g, N, K):
    """int4 weights uniform on [-8, 7] (packed, stored q + 8), fp16 scales U[0.005, 0.02]."""
    return (torch.randint(0, 256, (N, K // 2), device="cuda", generator=g, dtype=torch.uint8),
            _uniform(g, 0.005, 0.02, N, K // 64))


def _inputs(case, seed):
    """The case's input tensors, from the seed alone."""
    g, kind = _gen(seed), case["kind"]
    if kind == "mlp":
        c, M = MODELS[case["model"]], case["M"]
        gu, gus = _w4g(g, 2 * c.ffn, c.hidden)   # gate and up rows interleaved
        d, ds = _w4g(g, c.hidden, c.ffn)
        return {"x": _normal(g, M, c.hidden), "gamma": _uniform(g, 0.8, 1.2, c.hidden), "gu": gu, "gus": gus, "d": d,
                "ds": ds}
    if kind == "proj":
        w, s = _w4g(g, case["N"], case["K"])
        t = {"x": _normal(g, case["M"], case["K"]), "w": w, "s": s}
        if case["norm"]:
            t["gamma"] = _uniform(g, 0.8, 1.2, case["K"])
        return t
    if kind == "attn_prefill":
        S, H, KVH = case["S"], case["H"], case["KVH"]
        return {"q": _normal(g, S, H, HD), "k": _normal(g, S, KVH, HD), "v": _normal(g, S, KVH, HD)}
    if kind == "attn_decode":   # a ring slot is one token's [K | V]
        return {"q": _normal(g, case["H"], HD), "ring": _normal(g, case["n_kv"], 2, case["KVH"], HD)}
    if kind == "f16":
        shape = (case["N"], case["K"]) if case["t1"] else (case["K"], case["N"])
        w = torch.randn(shape, device="cuda", generator=g) / math.sqrt(case["K"])
        return {"a": _normal(g, case["M"], case["K"]), "w": w.half()}
    if kind == "attn_ops":   # q already scaled, as the pre-scaled lowering hands it over
        S, T, H, hd = case["S"], case["T"], case["H"], case["hd"]
        return {"q": _normal(g, H, S, hd) * (hd ** -0.5), "k": _normal(g, H, T, hd), "v": _normal(g, H, T, hd)}
    if kind == "w4a16":
        M, N, K = case["M"], case["N"], case["K"]
        act = torch.randn((M, K), device="cuda", generator=g) * 900.0
        lin = (act.round().clamp(-32768, 32767) + 32768).to(torch.int32)
        return {"act": lin, "w": torch.randint(0, 256, (N, K // 2), device="cuda", generator=g, dtype=torch.uint8)}
    rng = np.random.default_rng(int(seed))
    t = {"ids": rng.integers(0, ENGINE_CFG.vocab, case["S"]).astype(np.int32)}
    if kind == "request":
        t["next"] = rng.integers(0, ENGINE_CFG.vocab, case["steps"]).astype(np.int32)
    return t


def _crouton(lin):
    """[rows, cols] u16 values (int32) -> the crouton16_row4 surface, as int16 bits."""
    R, Cc = lin.shape
    # row = g*32 + phase*4 + rp*2 + b, col = kt*32 + ci -> [phase][kt][g][rp][ci][b]
    v = lin.view(R // 32, 8, 2, 2, Cc // 32, 32).permute(1, 4, 0, 2, 5, 3)
    return v.contiguous().to(torch.int16).view(-1)


# ---------------------------------------------------------------------------- the engine's model
@functools.lru_cache(maxsize=1)
def _model():
    return Engine(), Weights(ENGINE_CFG, seed=ENGINE_SEED)


@functools.lru_cache(maxsize=32)
def _blobs(kind, S):
    """The parsed blobs a program keeps for prompts of S tokens."""
    eng, w = _model()
    if kind == "chain":
        blob, t = emit_prefill_chain(ENGINE_CFG, w, S, lowering="ref_pre", recycle=True)
        return (eng.parse(blob), t["logits"]), None
    pre, tp = emit_prefill(ENGINE_CFG, w, S, MAX_POS)
    dec, td = emit_decode(ENGINE_CFG, w, MAX_POS)
    return (eng.parse(pre), tp["logits"]), (eng.parse(dec), td["logits"])


# ---------------------------------------------------------------------------- prepare
def prepare(case, seed):
    t, kind = _inputs(case, seed), case["kind"]
    if kind in ("request", "chain"):
        eng, w = _model()
        pre, dec = _blobs(kind, case["S"])
        st = {"kind": kind, "eng": eng, "image": w.image.ctypes.data, "pre": pre, "dec": dec}
        if kind == "chain":
            st["prompt"] = t["ids"].tobytes()
        else:
            st["prompt"] = np.ascontiguousarray(w.embed()[t["ids"]]).tobytes()
            st["steps"] = [w.embed()[i].tobytes() for i in t["next"]]
        return st
    lib, sp = load_library(lib_path), torch.cuda.current_stream().cuda_stream
    st = {"kind": kind, "lib": lib, "t": t}

    def out(*shape):
        o = torch.empty(shape, dtype=torch.float16, device="cuda")
        st.setdefault("out", []).append(o)
        return o

    def linear(x, wq, ws, y, gamma=None, res=None, mode=0):
        """Calls of one W4A16 linear: [RMSNorm,] linear, with the workspace it asks for."""
        M, K, N = x.shape[0], x.shape[1], wq.shape[0]
        calls = []
        if gamma is not None and M > GEMV_TOKENS:
            h = torch.empty_like(x)
            st.setdefault("keep", []).append(h)
            calls.append((lib.gehtp_rmsnorm2, (x.data_ptr(), gamma.data_ptr(), None, h.data_ptr(), M, K, sp)))
            x, gamma = h, None
        nb = lib.gehtp_w4g_split_bytes(M, N, K)
        work = torch.empty(max(nb, 16), dtype=torch.uint8, device="cuda")
        st.setdefault("keep", []).append(work)
        calls.append((lib.gehtp_w4g_fused_ws,
                      (x.data_ptr(), K, wq.data_ptr(), ws.data_ptr(), y.data_ptr(), y.shape[1], M, N, K,
                       gamma.data_ptr() if gamma is not None else None, res.data_ptr() if res is not None else None,
                       res.shape[1] if res is not None else 0, mode, work.data_ptr(), nb, sp)))
        return calls

    if kind == "mlp":
        c, M = MODELS[case["model"]], case["M"]
        m, y = out(M, c.ffn), out(M, c.hidden)
        st["calls"] = (linear(t["x"], t["gu"], t["gus"], m, gamma=t["gamma"], mode=1)
                       + linear(m, t["d"], t["ds"], y, res=t["x"]))
    elif kind == "proj":
        st["calls"] = linear(t["x"], t["w"], t["s"], out(case["M"], case["N"]), gamma=t.get("gamma"))
    elif kind == "attn_prefill":
        S, H, KVH = case["S"], case["H"], case["KVH"]
        o = out(S, H, HD)
        st["calls"] = [(lib.gehtp_attn_prefill, (t["q"].data_ptr(), t["k"].data_ptr(), t["v"].data_ptr(), o.data_ptr(),
                                                 S, H, KVH, HD, HD ** -0.5, int(case["causal"]), sp))]
    elif kind == "attn_decode":
        H, KVH, n = case["H"], case["KVH"], case["n_kv"]
        wf = lib.gehtp_attn_decode_work_floats(n, H, HD)
        work, o = torch.empty(wf, dtype=torch.float32, device="cuda"), out(H, HD)
        st["keep"] = [work]
        st["calls"] = [(lib.gehtp_attn_decode, (t["q"].data_ptr(), t["ring"].data_ptr(), t["ring"].numel() * 2,
                                                o.data_ptr(), n, H, KVH, HD, HD ** -0.5, work.data_ptr(), wf, sp))]
    elif kind == "f16":
        M, N, K = case["M"], case["N"], case["K"]
        o = out(M, N)
        st["calls"] = [(lib.gehtp_matmul_f16, (t["a"].data_ptr(), t["w"].data_ptr(), o.data_ptr(), M, K, N, 0, N,
                                               2 if case["t1"] else 0, sp))]
    elif kind == "attn_ops":
        S, T, H, hd = case["S"], case["T"], case["H"], case["hd"]
        s, p, o = out(H, S, T), out(H, S, T), out(H, S, hd)
        st["calls"] = [
            (lib.gehtp_matmul_f16, (t["q"].data_ptr(), t["k"].data_ptr(), s.data_ptr(), S, hd, T, 0, T, 6 | (H << 16), sp)),
            (lib.gehtp_softmax, (s.data_ptr(), p.data_ptr(), H * S, T, sp)),
            (lib.gehtp_matmul_f16, (p.data_ptr(), t["v"].data_ptr(), o.data_ptr(), S, T, hd, 0, hd, 4 | (H << 16), sp))]
    elif kind == "w4a16":
        M, N, K = case["M"], case["N"], case["K"]
        surf = _crouton(t.pop("act"))
        o = torch.empty(M * N, dtype=torch.int16, device="cuda")
        st["out"], st["keep"] = [o], [surf]
        st["calls"] = [(lib.gehtp_matmul_w4a16, (surf.data_ptr(), t["w"].data_ptr(), o.data_ptr(), M, K, N, sp))]
    else:
        raise ValueError(kind)
    return st


# ---------------------------------------------------------------------------- run
def run(state):
    if "calls" in state:
        for fn, args in state["calls"]:
            rc = fn(*args)
            if rc:
                raise RuntimeError(f"{fn.__name__}: {rc}")
        return state["out"]
    eng = state["eng"]
    eng.set_ext_weights(state["image"])
    pb, logits = state["pre"]
    if state["kind"] == "chain":
        return [np.frombuffer(eng.run_io(pb, state["prompt"], logits)[0], np.float16)]
    eng.state_reset()   # a new request
    rows = [np.frombuffer(eng.run_io(pb, state["prompt"], logits)[0], np.float16)]
    pb, logits = state["dec"]
    for x in state["steps"]:
        rows.append(np.frombuffer(eng.run_io(pb, x, logits)[0], np.float16))
    return rows


# ---------------------------------------------------------------------------- work
def _linear_work(M, N, K, n_out, res=False, norm=False):
    b = N * K / 2 + N * (K // 64) * 2 + M * K * 2 + M * n_out * 2 + (M * n_out * 2 if res else 0) + (K * 2 if norm else 0)
    return b, 2.0 * M * N * K


def work(case):
    kind = case["kind"]
    if kind == "mlp":
        c, M = MODELS[case["model"]], case["M"]
        b1, f1 = _linear_work(M, 2 * c.ffn, c.hidden, c.ffn, norm=True)
        b2, f2 = _linear_work(M, c.hidden, c.ffn, c.hidden, res=True)
        return {"bytes": b1 + b2, "flops": f1 + f2}
    if kind == "proj":
        b, f = _linear_work(case["M"], case["N"], case["K"], case["N"], norm=case["norm"])
        return {"bytes": b, "flops": f}
    if kind == "attn_prefill":
        S, H, KVH = case["S"], case["H"], case["KVH"]
        return {"bytes": 4.0 * S * (H + KVH) * HD, "flops": 4.0 * H * HD * (S * (S + 1) / 2 if case["causal"] else S * S)}
    if kind == "attn_decode":
        return {"bytes": 4.0 * HD * (case["n_kv"] * case["KVH"] + case["H"]), "flops": 4.0 * case["H"] * HD * case["n_kv"]}
    if kind == "f16":
        M, N, K = case["M"], case["N"], case["K"]
        return {"bytes": 2.0 * (M * K + K * N + M * N), "flops": 2.0 * M * N * K}
    if kind == "attn_ops":
        S, T, H, hd = case["S"], case["T"], case["H"], case["hd"]
        return {"bytes": 2.0 * H * (2 * S * hd + 2 * T * hd + 4 * S * T), "flops": 4.0 * H * S * T * hd}
    if kind == "w4a16":
        M, N, K = case["M"], case["N"], case["K"]
        return {"bytes": 2.0 * M * K + N * K / 2 + 2.0 * M * N, "flops": 2.0 * M * N * K}
    c, S, steps = ENGINE_CFG, case["S"], case.get("steps", 0)
    per_token = 2.0 * (sum(n * k for _, n, k in c.linears()) * c.layers + c.vocab * c.hidden)
    attn = 4.0 * c.layers * c.heads * HD * sum(S + i + 1 for i in range(steps))
    return {"bytes": float(c.decode_weight_bytes() * (1 + steps)), "flops": c.prefill_flops(S) + steps * per_token + attn}


# ---------------------------------------------------------------------------- tolerance
def tolerance(case):
    """About four times the error against exact() that the kinds show over their ranges
    (fp16 outputs, fp32 sums; intermediates rounded to fp16 where the ops define it)."""
    kind = case["kind"]
    if kind == "w4a16":
        return "exact"
    return {"rel": {"mlp": 2.5e-3, "proj": 1.2e-3, "attn_prefill": 1.2e-3, "attn_decode": 1.2e-3, "f16": 9e-4,
                    "attn_ops": 2.6e-3, "request": 6.5e-3, "chain": 6.5e-3}[kind]}


# ---------------------------------------------------------------------------- 64 bits
def _deq64(wq, ws):
    """dequant(W) = fp16(q * s), the weight format's definition, as float64 [N, K]."""
    q = torch.stack([(wq & 15).to(torch.float32), (wq >> 4).to(torch.float32)], dim=2).flatten(1) - 8.0
    return (q * ws.float().repeat_interleave(64, dim=1)).half().double()


def _norm64(x, gamma):
    return x / torch.sqrt((x * x).mean(-1, keepdim=True) + 1e-6) * gamma


def _attn64(q, k, v, scale, causal):
    """q [S, H, hd], k / v [T, KVH, hd], the last S of T positions -> [S, H, hd]."""
    S, H, T = q.shape[0], q.shape[1], k.shape[0]
    rep, out = H // k.shape[1], torch.empty_like(q)
    future = torch.ones(S, T, dtype=torch.bool, device=q.device).triu(T - S + 1) if causal else None
    for h in range(H):
        s = (q[:, h] @ k[:, h // rep].t().contiguous()) * scale
        if causal:
            s.masked_fill_(future, -math.inf)
        out[:, h] = torch.softmax(s, -1) @ v[:, h // rep].contiguous()
    return out


def _silu64(x):
    return x / (1.0 + torch.exp(-x))


def _model64(ids):
    """Logits [len(ids), vocab] of the engine's model at every position, in float64."""
    c, (_, w) = ENGINE_CFG, _model()
    dev = lambda a: torch.from_numpy(np.array(a)).cuda()  # noqa: E731
    f64 = lambda name: dev(w.f16(name).view(np.int16)).view(torch.float16).double()  # noqa: E731

    def lin(l, nm, rows, k):
        s = dev(w.get(f"{l}.{nm}.s").view(np.int16)).view(torch.float16).view(rows, k // 64)
        return _deq64(dev(w.get(f"{l}.{nm}.q")).view(rows, k // 2), s)

    shapes = {nm: (n, k) for nm, n, k in c.fused_linears()}
    E = f64("embed").view(c.vocab, c.hidden)
    n = len(ids)
    x = E[torch.from_numpy(ids.astype(np.int64)).cuda()]
    ang = torch.arange(n, device="cuda", dtype=torch.float64)[:, None] / (
        c.theta ** (torch.arange(0, HD, 2, device="cuda", dtype=torch.float64) / HD))
    cos, sin = torch.cos(ang)[:, None, :], torch.sin(ang)[:, None, :]

    def rope(y):
        a, b = y[..., :HD // 2], y[..., HD // 2:]
        return torch.cat([a * cos - b * sin, b * cos + a * sin], -1)

    for l in range(c.layers):
        qkv = _norm64(x, f64(f"{l}.g_attn")) @ lin(l, "wqkv", *shapes["wqkv"]).t()
        q, k, v = qkv.split([c.q_dim, c.kv_dim, c.kv_dim], 1)
        q = rope(_norm64(q.reshape(n, c.heads, HD), f64(f"{l}.q_norm")))
        k = rope(_norm64(k.reshape(n, c.kv_heads, HD), f64(f"{l}.k_norm")))
        a = _attn64(q, k, v.reshape(n, c.kv_heads, HD), c.scale, True).reshape(n, c.q_dim)
        x = x + a @ lin(l, "wo", *shapes["wo"]).t()
        gu = _norm64(x, f64(f"{l}.g_ffn")) @ lin(l, "wgu", *shapes["wgu"]).t()
        x = x + (_silu64(gu[:, 0::2]) * gu[:, 1::2]) @ lin(l, "wd", *shapes["wd"]).t()
    return _norm64(x, f64("g_final")), E


def exact(case, seed):
    t, kind = _inputs(case, seed), case["kind"]
    if kind == "mlp":
        x = t["x"].double()
        gu = _norm64(x, t["gamma"].double()) @ _deq64(t["gu"], t["gus"]).t()
        m = _silu64(gu[:, 0::2]) * gu[:, 1::2]
        return [m, x + m @ _deq64(t["d"], t["ds"]).t()]
    if kind == "proj":
        x = t["x"].double()
        if case["norm"]:
            x = _norm64(x, t["gamma"].double())
        return [x @ _deq64(t["w"], t["s"]).t()]
    if kind == "attn_prefill":
        return [_attn64(t["q"].double(), t["k"].double(), t["v"].double(), HD ** -0.5, case["causal"])]
    if kind == "attn_decode":
        ring = t["ring"].double()
        return [_attn64(t["q"].double()[None], ring[:, 0], ring[:, 1], HD ** -0.5, False)[0]]
    if kind == "f16":
        w = t["w"].double()
        return [t["a"].double() @ (w.t() if case["t1"] else w)]
    if kind == "attn_ops":
        q, k, v = (t[n].double() for n in ("q", "k", "v"))
        s = torch.stack([q[h] @ k[h].t() for h in range(case["H"])])
        p = torch.softmax(s, -1)
        return [s, p, torch.stack([p[h] @ v[h] for h in range(case["H"])])]
    if kind == "w4a16":
        w = torch.stack([t["w"] & 15, t["w"] >> 4], dim=2).flatten(1).double() - 8.0
        s = (t["act"].double() - 32768.0) @ w.t()                      # whole numbers, exact
        y = torch.sign(s) * torch.floor((s.abs() + 3.0) / 7.0) + 32768.0   # nearest of s / 7 (no ties)
        return [_crouton(y.clamp(0, 65535).to(torch.int32))]
    ids = t["ids"] if kind == "chain" else np.concatenate([t["ids"], t["next"]])
    h, E = _model64(ids)
    h = h[case["S"] - 1:]
    return [row.cpu().numpy() for row in h @ E.t()]
