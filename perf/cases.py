"""The work that a user of the warm-tier cache has it do, as measurable cases.

Every case goes through a public entry point of the ``akv`` package: the fused decode
(an eager prepared call, a captured multi-layer step, the plain function), the chunked
prefill, the demotion (selection, gather, quantize and pack), the drop-in cache's
``update``, the production cache's attention, the KIVI tier and the importance scorer.
Sizes are those of the workloads in ``akv/workloads.py``, of the caches' defaults and of
the tests, with odd and ragged ones beside them.
"""
import math
import os
import sys

import torch

_PKG = os.path.join(os.getcwd(), "adaptive-kv-memory_amd")
if _PKG not in sys.path:
    sys.path.insert(0, _PKG)

import akv  # noqa: E402
from akv.warm_tier import DecodeCall  # noqa: E402

DEV = "cuda"
DTYPES = {"fp16": torch.float16, "bf16": torch.bfloat16, "fp32": torch.float32}


def listed():
    return [
        # one token of a short context on one GQA layer: the smallest call a serving loop
        # makes, prepared once and launched eagerly; launch latency counts
        dict(name="decode_4k_eager", kind="decode", how="call", layers=1, B=1, Hq=12, Hkv=2, D=128, M=1,
             n_hot=512, n_warm=3584, bits_k=4, bits_v=4, block_t=32, group_v=32, outliers=0.0, hot_first=False,
             weights=False, scores=False),
        # one decode step of a batch of eight 32k sequences over four layers (their tiers
        # exceed the last-level cache), the importance scores updated, replayed as a graph
        dict(name="decode_32k_step", kind="decode", how="graph", layers=4, B=8, Hq=12, Hkv=2, D=128, M=1,
             n_hot=1024, n_warm=31744, bits_k=3, bits_v=3, block_t=32, group_v=32, outliers=0.0, hot_first=False,
             weights=False, scores=True),
        # multi-head attention, 4-bit keys, 2-bit values, one protected channel per block
        dict(name="decode_16k_outliers", kind="decode", how="eager", layers=1, B=4, Hq=32, Hkv=32, D=128, M=1,
             n_hot=512, n_warm=15872, bits_k=4, bits_v=2, block_t=32, group_v=32, outliers=0.01, hot_first=False,
             weights=False, scores=False),
        # a few draft tokens at once, ragged tiers, the attention weights returned and the
        # scores updated, hot tokens first (the order of the mixed-precision ops)
        dict(name="decode_ragged_weights", kind="decode", how="eager", layers=1, B=3, Hq=28, Hkv=4, D=128, M=3,
             n_hot=333, n_warm=9001, bits_k=2, bits_v=2, block_t=32, group_v=64, outliers=0.0, hot_first=True,
             weights=True, scores=True),
        # one prompt chunk after 128k cached tokens: the largest contraction
        dict(name="prefill_128k", kind="prefill", B=1, Hq=64, Hkv=8, M=512, n_hot=4096, n_warm=126976, bits_k=2,
             bits_v=2, group_v=32, dtype="bf16", causal=False),
        # an odd prompt chunk with its own causal part after a ragged cache
        dict(name="prefill_ragged_causal", kind="prefill", B=2, Hq=12, Hkv=2, M=333, n_hot=1000, n_warm=10007,
             bits_k=3, bits_v=3, group_v=32, dtype="fp16", causal=True),
        # a batch of sixteen 64k sequences demoted at once: select, gather, quantize, pack
        dict(name="demote_64k", kind="demote", B=16, H=8, D=128, S=65536, keep=1024, bits_k=3, bits_v=3, group_v=32,
             outliers=0.0, dtype="fp16"),
        # the drop-in cache takes a long prompt: everything past the hot budget is demoted in
        # one event, and the model gets the layer's chronological keys and values
        dict(name="cache_prompt_16k", kind="cache", B=1, H=8, D=128, prompt=16383, steps=0, preset="balanced",
             outliers=0.0, dtype="fp16"),
        # a bfloat16 model's batch of two: prompt, then generated tokens one by one, keys
        # and values at different widths with protected channels
        dict(name="cache_generate_bf16", kind="cache", B=2, H=2, D=128, prompt=2049, steps=12, preset="k4v2",
             outliers=0.02, dtype="bf16"),
        # one decode step of eight layers of the production cache at its default sizes
        dict(name="production_step", kind="production", layers=8, B=1, H=32, D=128, M=1, n_hot=1024, n_warm=4096,
             bits=4, group=64),
        # the KIVI tier takes a prompt: quantized rows, their dequantized view, residual
        dict(name="kivi_prompt_4k", kind="kivi", B=1, H=32, D=128, prompt=4097, bits=2, group=128, residual=128,
             dtype="fp16"),
        # a prefill's attention weights folded into the running importance
        dict(name="importance_prefill", kind="importance", B=1, H=32, M=256, N=8191, strategy="importance",
             dtype="bf16"),
    ]


def _log(rng, lo, hi):
    """An integer spread over the logarithm of [lo, hi]; half of them odd."""
    x = int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))
    if rng.random() < 0.5:
        x |= 1
    return max(lo, min(hi, x))


def draw(rng):
    kind = rng.choice(["decode", "decode", "decode", "prefill", "prefill", "demote", "demote", "cache", "cache",
                       "production", "kivi", "importance"])
    if kind == "decode":
        Hkv = rng.choice([1, 2, 4, 8, 32])
        g = 1 if Hkv == 32 else rng.choice([1, 4, 6, 7, 8])
        B = rng.choice([1, 2, 3, 4, 8])
        n_warm = _log(rng, 512, max(1024, min(32768, 524288 * 4 // (B * Hkv))))
        D = rng.choice([128, 128, 128, 128, 64])
        out = rng.choice([0.0, 0.0, 0.0, 0.01, 0.02])
        M = rng.choice([1, 1, 1, 2, 4])
        big = B * Hkv * g * M * n_warm > 64 * 1024 * 1024
        return dict(kind="decode", how=rng.choice(["call", "eager", "graph"]), layers=rng.choice([1, 2]), B=B,
                    Hq=g * Hkv, Hkv=Hkv, D=D, M=M, n_hot=_log(rng, 16, 2048), n_warm=n_warm,
                    bits_k=rng.choice([2, 3, 4]), bits_v=rng.choice([2, 3, 4]), block_t=rng.choice([32, 32, 64]),
                    group_v=32 if out else rng.choice([32, 64]), outliers=out, hot_first=rng.random() < 0.3,
                    weights=(not big) and rng.random() < 0.25, scores=rng.random() < 0.4)
    if kind == "prefill":
        Hkv = rng.choice([2, 4, 8])
        g = rng.choice([1, 4, 6, 8])
        M = _log(rng, 17, 1024)
        cap = 64 * 512 * 131072 // (Hkv * g * M)
        return dict(kind="prefill", B=1, Hq=g * Hkv, Hkv=Hkv, M=M, n_hot=_log(rng, 16, 4096),
                    n_warm=_log(rng, 1024, max(2048, min(65536, cap // 2))), bits_k=rng.choice([2, 3, 4]),
                    bits_v=rng.choice([2, 3, 4]), group_v=rng.choice([32, 64, 128]),
                    dtype=rng.choice(["fp16", "bf16"]), causal=rng.random() < 0.6)
    if kind == "demote":
        B = rng.choice([1, 2, 4, 8])
        out = rng.choice([0.0, 0.0, 0.01])
        return dict(kind="demote", B=B, H=rng.choice([2, 4, 8]), D=rng.choice([128, 128, 128, 64]),
                    S=_log(rng, 1500, 65536 * 2 // B), keep=rng.choice([64, 128, 1024]), bits_k=rng.choice([2, 3, 4]),
                    bits_v=rng.choice([2, 3, 4]), group_v=rng.choice([32, 64]), outliers=out,
                    dtype=rng.choice(["fp16", "fp16", "bf16"]))
    if kind == "cache":
        steps = rng.choice([0, 0, 4])
        return dict(kind="cache", B=rng.choice([1, 2]), H=rng.choice([2, 4, 8]), D=rng.choice([128, 128, 64]),
                    prompt=_log(rng, 300, 4096 if steps else 8192),
                    steps=steps, preset=rng.choice(["quality", "balanced", "compact", "k4v2", "k4v3"]),
                    outliers=rng.choice([0.0, 0.0, 0.02]), dtype=rng.choice(["fp16", "bf16"]))
    if kind == "production":
        return dict(kind="production", layers=rng.choice([1, 2, 4]), B=rng.choice([1, 1, 2]),
                    H=rng.choice([8, 16, 32]), D=128, M=rng.choice([1, 1, 2]), n_hot=_log(rng, 64, 1024),
                    n_warm=_log(rng, 512, 4096), bits=rng.choice([2, 4, 8]), group=rng.choice([32, 64, 128]))
    if kind == "kivi":
        return dict(kind="kivi", B=rng.choice([1, 2]), H=rng.choice([8, 16, 32]), D=rng.choice([64, 128]),
                    prompt=_log(rng, 200, 4096), bits=rng.choice([2, 4, 8]), group=rng.choice([32, 64, 128]),
                    residual=rng.choice([32, 128]), dtype=rng.choice(["fp16", "bf16"]))
    return dict(kind="importance", B=rng.choice([1, 2]), H=rng.choice([8, 12, 32]), M=_log(rng, 1, 256),
                N=_log(rng, 700, 8192), strategy=rng.choice(["importance", "observation_window"]),
                dtype=rng.choice(["fp16", "bf16", "fp32"]))


# ------------------------------------------------------------------ inputs


def _gen(seed, role):
    g = torch.Generator(device=DEV)
    g.manual_seed(1000003 * int(seed) + role)
    return g


def _kv(shape, seed, role, dtype):
    """Keys with two large channels per head (the structure of real key caches), plain values."""
    B, H, N, D = shape
    k = torch.randn(shape, generator=_gen(seed, role), device=DEV)
    ch = torch.randint(0, D, (H, 2), generator=_gen(seed, role + 1), device=DEV)
    gain = torch.ones(1, H, 1, D, device=DEV)
    gain.scatter_(3, ch.view(1, H, 1, 2), 6.0)
    k = (k * gain).to(dtype)
    v = torch.randn(shape, generator=_gen(seed, role + 2), device=DEV).to(dtype)
    return k, v


def _decode_inputs(c, seed):
    out = []
    for i in range(c["layers"]):
        r = 100 * i
        kw, vw = _kv((c["B"], c["Hkv"], c["n_warm"], c["D"]), seed, r, torch.float16)
        kh, vh = _kv((c["B"], c["Hkv"], c["n_hot"], c["D"]), seed, r + 10, torch.float16)
        q = torch.randn(c["B"], c["Hq"], c["M"], c["D"], generator=_gen(seed, r + 20), device=DEV).half()
        s = torch.rand(c["n_hot"] + c["n_warm"], generator=_gen(seed, r + 21), device=DEV) if c["scores"] else None
        out.append((q, kw, vw, kh, vh, s))
    return out


def _prefill_inputs(c, seed):
    dt = DTYPES[c["dtype"]]
    kw, vw = _kv((c["B"], c["Hkv"], c["n_warm"], 128), seed, 0, torch.float16)
    kh, vh = _kv((c["B"], c["Hkv"], c["n_hot"], 128), seed, 10, torch.float16)
    q = torch.randn(c["B"], c["Hq"], c["M"], 128, generator=_gen(seed, 20), device=DEV).to(dt)
    kc = vc = None
    if c["causal"]:
        kc, vc = _kv((c["B"], c["Hkv"], c["M"], 128), seed, 30, dt)
    return q, kw, vw, kh, vh, kc, vc


def _attn_weights(c, seed, M, role):
    x = torch.randn(c["B"], c["H"], M, c["N"], generator=_gen(seed, role), device=DEV) * 2.0
    return torch.softmax(x, dim=-1).to(DTYPES[c["dtype"]])


def _strategy(c):
    return akv.ImportanceConfig(strategy=akv.ScoringStrategy(c["strategy"]))


def _cache(c):
    return akv.AKVCache(preset=c["preset"], outlier_fraction=c["outliers"])


def _production_inputs(c, seed):
    out = []
    for i in range(c["layers"]):
        r = 100 * i
        kw, vw = _kv((1, c["H"], c["n_warm"], c["D"]), seed, r, torch.float16)
        kh, vh = _kv((1, c["H"], c["n_hot"], c["D"]), seed, r + 10, torch.float16)
        out.append((kw[0], vw[0], kh[0], vh[0]))
    q = torch.randn(c["B"], c["H"], c["M"], c["D"], generator=_gen(seed, 20), device=DEV).half()
    return q, out


def _capture(calls):
    """A serving loop's captured step: one eager run, then the graph and its outputs."""
    side = torch.cuda.Stream()
    side.wait_stream(torch.cuda.current_stream())
    with torch.cuda.stream(side):
        calls()
    torch.cuda.current_stream().wait_stream(side)
    torch.cuda.synchronize()
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        outs = calls()
    return graph, outs


def prepare(case, seed):
    c, kind = case, case["kind"]
    st = {"case": c}
    if kind == "decode":
        st["layers"] = []
        for q, kw, vw, kh, vh, s in _decode_inputs(c, seed):
            warm = akv.quantize_kv(kw, vw, c["bits_k"], c["bits_v"], c["block_t"], c["group_v"], c["outliers"])
            st["layers"].append(dict(q=q, kh=kh, vh=vh, warm=warm, scores=s))
        if c["how"] != "eager":
            st["calls"] = []
            N = c["n_hot"] + c["n_warm"]
            for lay in st["layers"]:
                w = None
                if c["weights"]:
                    w = torch.empty(c["B"], c["Hq"], c["M"], N, dtype=torch.float32, device=DEV)
                st["calls"].append(DecodeCall(lay["q"], lay["kh"], lay["vh"], lay["warm"], hot_first=c["hot_first"],
                                              scores=lay["scores"], decay=0.9, attn_weights=w))
        if c["how"] == "graph":
            before = [None if lay["scores"] is None else lay["scores"].clone() for lay in st["layers"]]
            st["graph"], _ = _capture(lambda: [call() for call in st["calls"]])
            for lay, b in zip(st["layers"], before):  # the scores as they were before the eager run
                if b is not None:
                    lay["scores"].copy_(b)
    elif kind == "prefill":
        q, kw, vw, kh, vh, kc, vc = _prefill_inputs(c, seed)
        st.update(q=q, kh=kh, vh=vh, kc=kc, vc=vc,
                  warm=akv.quantize_kv(kw, vw, c["bits_k"], c["bits_v"], 32, c["group_v"]))
    elif kind == "demote":
        k, v = _kv((c["B"], c["H"], c["S"], c["D"]), seed, 0, DTYPES[c["dtype"]])
        st.update(k=k, v=v, imp=torch.rand(c["B"], c["S"], generator=_gen(seed, 4), device=DEV))
    elif kind == "cache":
        dt = DTYPES[c["dtype"]]
        st["prompt"] = _kv((c["B"], c["H"], c["prompt"], c["D"]), seed, 0, dt)
        st["tokens"] = [_kv((c["B"], c["H"], 1, c["D"]), seed, 100 + 10 * i, dt) for i in range(c["steps"])]
    elif kind == "production":
        q, layers = _production_inputs(c, seed)
        cfg = akv.ProductionCacheConfig(
            num_layers=c["layers"], num_heads=c["H"], head_dim=c["D"], hot_budget=c["n_hot"],
            warm_budget=c["n_warm"], warm_bits=c["bits"], group_size=c["group"], warm_quantizer="minmax",
            max_hot_pages=(c["n_hot"] + 15) // 16, device=DEV)
        cache = akv.ProductionCache(cfg)
        for lay, (kw, vw, kh, vh) in zip(cache._layers, layers):
            lay._warm_k.quantize_and_append(kw)
            lay._warm_v.quantize_and_append(vw)
            lay.append_hot(kh, vh)
        st.update(q=q, cache=cache)
        st["graph"], st["outs"] = _capture(lambda: [cache.fused_attention(q, i) for i in range(c["layers"])])
    elif kind == "kivi":
        st["kv"] = _kv((c["B"], c["H"], c["prompt"], c["D"]), seed, 0, DTYPES[c["dtype"]])
    else:
        st["scorer"] = akv.ImportanceScorer(_strategy(c))
        st["scorer"].update(_attn_weights(c, seed, 1, 1), 0)  # an earlier step's scores
        st["attn"] = _attn_weights(c, seed, c["M"], 0)
    return st


# --------------------------------------------------------------------- run


def run(state):
    c = state["case"]
    kind = c["kind"]
    if kind == "decode":
        if c["how"] == "graph":
            state["graph"].replay()
            outs = [call.out for call in state["calls"]]
        elif c["how"] == "call":
            outs = [call() for call in state["calls"]]
        else:
            outs, ws = [], []
            for lay in state["layers"]:
                r = akv.decode_attention(lay["q"], lay["kh"], lay["vh"], lay["warm"], hot_first=c["hot_first"],
                                         scores=lay["scores"], decay=0.9, return_weights=c["weights"])
                outs.append(r[0] if c["weights"] else r)
                if c["weights"]:
                    ws.append(r[1])
        if c["weights"]:
            outs = outs + (ws if c["how"] == "eager" else [call.attn_weights for call in state["calls"]])
        if c["scores"]:
            outs = outs + [lay["scores"] for lay in state["layers"]]
        return outs
    if kind == "prefill":
        return akv.prefill_attention(state["q"], state["kh"], state["vh"], state["warm"], k_chunk=state["kc"],
                                     v_chunk=state["vc"])
    if kind == "demote":
        idx = akv.select_demote_indices(state["imp"], c["S"] - c["keep"], c["S"], 64)
        w = akv.quantize_kv(state["k"], state["v"], c["bits_k"], c["bits_v"], 32, c["group_v"], c["outliers"], sel=idx)
        outs = [idx, w.k_codes, w.k_scale, w.k_zero, w.v_codes, w.v_scale, w.v_zero]
        return outs + ([w.k_oidx, w.k_odata, w.v_oidx, w.v_odata] if w.n_out else [])
    if kind == "cache":
        cache = _cache(c)
        k, v = cache.update(*state["prompt"], 0)
        outs = [k, v]
        for tk, tv in state["tokens"]:
            outs = list(cache.update(tk, tv, 0))
        return outs
    if kind == "production":
        state["graph"].replay()
        return state["outs"]
    if kind == "kivi":
        cache = akv.create_baseline("kivi_fused", key_bits=c["bits"], value_bits=c["bits"], group_size=c["group"],
                                    residual_length=c["residual"])
        return list(cache.update(*state["kv"], 0))
    state["scorer"].update(state["attn"], 0)
    return state["scorer"].get_scores(0)


# -------------------------------------------------------------------- work


def _row(D, bits):
    return D * bits // 8


def work(case):
    c, kind = case, case["kind"]
    size = {"fp16": 2, "bf16": 2, "fp32": 4}.get(c.get("dtype", "fp16"))
    if kind == "decode":
        B, Hkv, Hq, D, M, nw, nh = (c[k] for k in ("B", "Hkv", "Hq", "D", "M", "n_warm", "n_hot"))
        nblk, N = -(-nw // c["block_t"]), nw + nh
        n_out = max(1, int(D * c["outliers"])) if c["outliers"] > 0 else 0
        tok = _row(D, c["bits_k"]) + _row(D, c["bits_v"]) + 4 * (D // c["group_v"]) + 4 * n_out
        by = B * Hkv * (nw * tok + nblk * 4 * D + nh * 4 * D) + B * nblk * 16 * n_out + 4 * B * Hq * M * D
        by += 4 * B * Hq * M * N if c["weights"] else 0
        by += 8 * N if c["scores"] else 0
        return {"bytes": by * c["layers"], "flops": 4 * B * Hq * M * N * D * c["layers"]}
    if kind == "prefill":
        B, Hkv, Hq, M, nw, nh = (c[k] for k in ("B", "Hkv", "Hq", "M", "n_warm", "n_hot"))
        tok = _row(128, c["bits_k"]) + _row(128, c["bits_v"]) + 4 * (128 // c["group_v"])
        by = B * Hkv * (nw * tok + -(-nw // 32) * 512 + nh * 512) + 4 * B * Hq * M * 128
        fl = 4 * B * Hq * M * (nw + nh) * 128
        if c["causal"]:
            by += 4 * B * Hkv * M * 128
            fl += 2 * B * Hq * M * (M + 1) * 128
        return {"bytes": by, "flops": fl}
    if kind == "demote":
        B, H, D, n = c["B"], c["H"], c["D"], c["S"] - c["keep"]
        tok = 2 * D * size + _row(D, c["bits_k"]) + _row(D, c["bits_v"]) + 4 * (D // c["group_v"])
        return {"bytes": B * H * (n * tok + -(-n // 32) * 4 * D) + B * (4 * c["S"] + 8 * n), "flops": 0}
    if kind == "cache":
        # each step's views are written whole; the tokens are read once
        B, H, D, P = c["B"], c["H"], c["D"], c["prompt"]
        out = 2 if c["dtype"] == "fp16" else 4
        views = sum(P + i for i in range(c["steps"] + 1))
        return {"bytes": 2 * B * H * D * (size * (P + c["steps"]) + out * views), "flops": 0}
    if kind == "production":
        B, H, D, M, nw, nh = (c[k] for k in ("B", "H", "D", "M", "n_warm", "n_hot"))
        by = H * (nw * 2 * (_row(D, c["bits"]) + 4 * (D // c["group"])) + nh * 4 * D) + 4 * B * H * M * D
        return {"bytes": by * c["layers"], "flops": 4 * B * H * M * (nw + nh) * D * c["layers"]}
    if kind == "kivi":
        B, H, D, P = c["B"], c["H"], c["D"], c["prompt"]
        nq, pd = max(0, P - c["residual"]), -(-D // c["group"]) * c["group"]
        kept = nq * (_row(pd, c["bits"]) + 12 * (pd // c["group"])) + (P - nq) * D * size
        return {"bytes": 2 * B * H * (P * D * (size + size) + kept), "flops": 0}
    M = min(c["M"], 32) if c["strategy"] == "observation_window" else c["M"]
    return {"bytes": c["B"] * c["H"] * M * c["N"] * size + 8 * c["N"], "flops": 0}


# --------------------------------------------------------------- tolerance


def tolerance(case):
    kind = case["kind"]
    if kind in ("demote", "cache", "kivi"):
        return "exact"
    if kind == "importance":
        return {"rel": 1e-6}  # 2.3e-7 against float64
    if kind == "prefill" and case["dtype"] == "bf16":
        return {"rel": 7e-3}  # 1.7e-3 against float64: the output's own rounding
    return {"rel": 1.5e-3}  # 2.5e-4 to 4e-4 between two runs and against float64


# ------------------------------------------------------------------- exact


def _affine(x, dim, bits):
    """Codes, scale and zero of x reduced over ``dim``, one rounding to x.dtype per operation."""
    mn, mx = x.amin(dim, keepdim=True), x.amax(dim, keepdim=True)
    maxv = (1 << bits) - 1
    scale = (mx - mn) / torch.full_like(mx, maxv)  # a true division, not a product with 1 / maxv
    if x.dtype != torch.float16:  # 1e-8 is 0 in float16
        scale = torch.maximum(scale, torch.tensor(1e-8, dtype=x.dtype, device=x.device))
    codes = torch.nan_to_num(torch.round((x - mn) / scale), nan=0.0, posinf=float(maxv)).clamp(0, maxv)
    return codes, scale, mn


def _dequant16(codes, scale, zero):
    return codes.half() * scale.half() + zero.half()


def _protect(x, f):
    """(x with its largest channels zeroed, their mask) for one call over x (H, n, D)."""
    n = max(1, int(x.shape[-1] * f))
    idx = x.double().norm(dim=1).mean(dim=0).topk(n).indices
    mask = torch.zeros(x.shape[-1], dtype=torch.bool, device=x.device)
    mask[idx] = True
    return x.masked_fill(mask, 0), mask


def _warm64(kw, vw, c):
    """The warm tier's float16 values (K per block and channel, V per token and group) in float64."""
    B, H, N, D = kw.shape
    T, G, f = c.get("block_t", 32), c["group_v"], c.get("outliers", 0.0)
    k64 = torch.empty(B, H, N, D, dtype=torch.float64, device=DEV)
    v64 = torch.empty_like(k64)
    for b in range(B):
        full = N // T * T
        if not f:
            for a, n, t in ((0, full, T), (full, N - full, N - full)):
                if n:
                    x = kw[b, :, a:a + n].reshape(H, n // t, t, D)
                    k64[b, :, a:a + n] = _dequant16(*_affine(x, 2, c["bits_k"])).reshape(H, n, D).double()
            x = vw[b].reshape(H, N, D // G, G)
            v64[b] = _dequant16(*_affine(x, 3, c["bits_v"])).reshape(H, N, D).double()
            continue
        for a in range(0, N, T):
            e = min(a + T, N)
            x, m = _protect(kw[b, :, a:e], f)
            d = _dequant16(*_affine(x, 1, c["bits_k"]))
            k64[b, :, a:e] = torch.where(m, kw[b, :, a:e].half(), d).double()
            x, m = _protect(vw[b, :, a:e], f)
            d = _dequant16(*_affine(x.reshape(H, e - a, D // G, G), 3, c["bits_v"])).reshape(H, e - a, D)
            v64[b, :, a:e] = torch.where(m, vw[b, :, a:e].half(), d).double()
    return k64, v64


def _attend64(q, k, v, mask_from=None, weights=False):
    """softmax(q k^T / sqrt(D)) v in float64, head by head; with ``mask_from`` query m sees
    key mask_from + j only for j <= m."""
    B, Hq, M, D = q.shape
    g = Hq // k.shape[1]
    out = torch.empty(B, Hq, M, D, dtype=torch.float64, device=DEV)
    p_all = torch.empty(B, Hq, M, k.shape[2], dtype=torch.float64, device=DEV) if weights else None
    for b in range(B):
        for h in range(Hq):
            s = (q[b, h].double() @ k[b, h // g].t().contiguous()) / math.sqrt(D)
            if mask_from is not None:
                j = torch.arange(k.shape[2], device=DEV) - mask_from
                s.masked_fill_(j[None, :] > torch.arange(M, device=DEV)[:, None], float("-inf"))
            p = torch.softmax(s, dim=-1)
            out[b, h] = p @ v[b, h // g]
            if weights:
                p_all[b, h] = p
    return out, p_all


def _exact_decode(c, seed):
    outs, ws, scs = [], [], []
    for q, kw, vw, kh, vh, s in _decode_inputs(c, seed):
        k64, v64 = _warm64(kw, vw, c)
        order = (lambda w, h: [h, w]) if c["hot_first"] else (lambda w, h: [w, h])
        k = torch.cat(order(k64, kh.double()), dim=2)
        v = torch.cat(order(v64, vh.double()), dim=2)
        need = c["weights"] or c["scores"]
        out, p = _attend64(q, k, v, weights=need)
        outs.append(out)
        if c["weights"]:
            ws.append(p)
        if c["scores"]:
            scs.append(s.double() * 0.9 + p.mean(dim=(0, 1)).sum(dim=0))
    return outs + ws + scs


def _exact_demote(c, seed):
    if c["outliers"]:
        return None
    k, v = _kv((c["B"], c["H"], c["S"], c["D"]), seed, 0, DTYPES[c["dtype"]])
    imp = torch.rand(c["B"], c["S"], generator=_gen(seed, 4), device=DEV)
    B, H, S, D = k.shape
    n, G = S - c["keep"], c["group_v"]
    nblk = -(-n // 32)
    key = imp.clone()
    key[:, :4] = float("inf")
    key[:, S - 16:] = float("inf")
    idx = torch.sort(torch.sort(key, dim=1, stable=True).indices[:, :n], dim=1).values
    ks = torch.empty(B, H, nblk, D, dtype=torch.float64, device=DEV)
    kz, vs = torch.empty_like(ks), torch.empty(B, H, n, D // G, dtype=torch.float64, device=DEV)
    vz = torch.empty_like(vs)
    floor = 0.0 if c["dtype"] == "fp16" else 1e-8
    for b in range(B):
        x, full = k[b].index_select(1, idx[b]), n // 32 * 32
        for a, m, t, o in ((0, full, 32, 0), (full, n - full, n - full, full // 32)):
            if m:
                y = x[:, a:a + m].reshape(H, m // t, t, D)
                mn, mx = y.amin(2).double(), y.amax(2).double()
                ks[b, :, o:o + m // t] = ((mx - mn) / ((1 << c["bits_k"]) - 1)).clamp(min=floor)
                kz[b, :, o:o + m // t] = mn
        y = v[b].index_select(1, idx[b]).reshape(H, n, D // G, G)
        mn, mx = y.amin(3).double(), y.amax(3).double()
        vs[b] = ((mx - mn) / ((1 << c["bits_v"]) - 1)).clamp(min=floor)
        vz[b] = mn
    return [None, None, ks, kz, None, vs, vz]


def _exact_cache(c, seed):
    if c["steps"]:
        return None  # promotions follow reductions whose order is the implementation's
    k, v = _kv((c["B"], c["H"], c["prompt"], c["D"]), seed, 0, DTYPES[c["dtype"]])
    cache = {"quality": (4, 4, 256), "balanced": (3, 3, 128), "compact": (2, 2, 64), "k4v2": (4, 2, 128),
             "k4v3": (4, 3, 128)}[c["preset"]]
    n = c["prompt"] - cache[2]
    outs = []
    for x, bits, dim in ((k, cache[0], 1), (v, cache[1], 2)):
        y = x.double()
        if n > 0:
            for b in range(c["B"]):
                ev = x[b, :, 4:4 + n]  # equal scores: the oldest past the four protected ones
                z, m = _protect(ev, c["outliers"]) if c["outliers"] else (ev, None)
                d = _dequant16(*_affine(z, dim, bits))
                y[b, :, 4:4 + n] = (d if m is None else torch.where(m, ev.half(), d)).double()
        outs.append(y)
    return outs


def _exact_production(c, seed):
    q, layers = _production_inputs(c, seed)
    G, outs = c["group"], []
    for kw, vw, kh, vh in layers:
        kv = []
        for w, h in ((kw, kh), (vw, vh)):
            x = w.reshape(c["H"], c["n_warm"], c["D"] // G, G)
            codes, s, z = _affine(x, 3, c["bits"])
            d = (codes.float() * s.float() + z.float()).half().reshape(w.shape)
            kv.append(torch.cat([d, h], dim=1).double().unsqueeze(0).expand(c["B"], -1, -1, -1))
        outs.append(_attend64(q, kv[0], kv[1])[0])
    return outs


def _exact_kivi(c, seed):
    k, v = _kv((c["B"], c["H"], c["prompt"], c["D"]), seed, 0, DTYPES[c["dtype"]])
    n, G, D = c["prompt"] - c["residual"], c["group"], c["D"]
    outs = []
    for x in (k, v):
        y = x.double()
        if n > 0:
            z = x[:, :, :n].float()
            pad = (-D) % G
            z = torch.nn.functional.pad(z, (0, pad)).reshape(c["B"], c["H"], n, (D + pad) // G, G)
            mn, mx = z.amin(-1, keepdim=True), z.amax(-1, keepdim=True)
            s = ((mx - mn) / torch.full_like(mx, (1 << c["bits"]) - 1)).clamp(min=1e-10)
            codes = torch.round((z - mn) / s).clamp(0, (1 << c["bits"]) - 1)
            d = (codes * s + mn).reshape(c["B"], c["H"], n, D + pad)[..., :D]
            y[:, :, :n] = d.half().double()
        outs.append(y)
    return outs


def exact(case, seed):
    c, kind = case, case["kind"]
    if kind == "decode":
        return _exact_decode(c, seed)
    if kind == "prefill":
        q, kw, vw, kh, vh, kc, vc = _prefill_inputs(c, seed)
        k64, v64 = _warm64(kw, vw, c)
        ks, vs = [kh.double(), k64], [vh.double(), v64]
        if c["causal"]:
            ks.append(kc.double())
            vs.append(vc.double())
        n = c["n_hot"] + c["n_warm"]
        return _attend64(q, torch.cat(ks, dim=2), torch.cat(vs, dim=2), n if c["causal"] else None)[0]
    if kind == "demote":
        return _exact_demote(c, seed)
    if kind == "cache":
        return _exact_cache(c, seed)
    if kind == "production":
        return _exact_production(c, seed)
    if kind == "kivi":
        return _exact_kivi(c, seed)
    prev, attn = _attn_weights(c, seed, 1, 1), _attn_weights(c, seed, c["M"], 0)
    window, kernel = (32, 7) if c["strategy"] == "observation_window" else (0, 1)
    s = torch.zeros(c["N"], dtype=torch.float64, device=DEV)
    for a in (prev, attn):
        a = a[:, :, -window:] if window else a
        imp = sum(a[b, h].double().sum(dim=0) for b in range(c["B"]) for h in range(c["H"])) / (c["B"] * c["H"])
        if kernel > 1 and c["N"] > kernel:
            imp = torch.nn.functional.avg_pool1d(imp.view(1, 1, -1), kernel, 1, kernel // 2).view(-1)
        s = s * 0.95 + imp
    return s
