"""The work whose time this repository looks after: what a language-model program asks of the quantized-matmul path, through
machx_inference_engine_amd.ops.  One pass is a whole piece of such a program: a projection of one token, a feed-forward block
over a few tokens (decode) or over a prompt (prefill), a mixture-of-experts block with its routing.

  kind "proj"         quantize one token's row and multiply it with one matrix: attention projections, the language-model head
  kind "ffn"          feed-forward block of T <= 16 tokens over q8 rows: gate, up, SwiGLU, down
  kind "prefill"      the same block for a prompt of T tokens: fp16 rows on the matrix cores
  kind "moe_decode"   router, then the experts of every token slot by device-side id, then their weighted sum
  kind "moe_grouped"  router, packing by expert, the grouped expert products, the weighted sum; rows "f16" (gathered while they
                      are loaded) or "q8" (the signatures that take quantized rows)

Formats: "q4_K", "q6_K", "q8_0" (planes), "mxfp4" (planes), and "q4_K_M", the usual mix of a Q4_K file: gate and up in Q4_K, down
in Q6_K.  Weights are N(0, 0.02) tensors encoded in HBM.  Activation rows are N(0, 1) with a common component, and the router's
rows respond to it, so that experts differ in popularity (by rank^-0.5: a trained, roughly balanced router).  "graph": the pass is replayed from a
captured graph, as a serving loop does with its decode step; otherwise every call is made from Python.
"""
import math

import torch

import machx_inference_engine_amd as mx
from machx_inference_engine_amd import synth

ops = mx.ops
DEV = "cuda:0"
PARTS = {"q4_K_M": ("q4_K", "q6_K")}
KQ = {"q4_K": "q4k", "q6_K": "q6k"}
BITS = {fmt: 8.0 * b / e for fmt, (e, b) in synth.BLOCK.items()}


def listed():
    return [
        # an attention projection of one token, the smallest call: launches and host work count
        {"name": "proj_q4_K_T1", "kind": "proj", "fmt": "q4_K", "K": 4096, "N": 4096},
        # the language-model head of one token: the largest single matrix of a decode step
        {"name": "lm_head_q6_K_T1", "kind": "proj", "fmt": "q6_K", "K": 4096, "N": 151936},
        # the feed-forward block of a Llama-3-8B layer, one token
        {"name": "ffn_q8_0_T1", "kind": "ffn", "fmt": "q8_0", "H": 4096, "F": 14336, "T": 1, "graph": False},
        # the same block for a few sequences decoded together: a ragged batch, and the largest one of the path
        {"name": "ffn_q4_K_M_T5", "kind": "ffn", "fmt": "q4_K_M", "H": 4096, "F": 14336, "T": 5, "graph": False},
        {"name": "ffn_q6_K_T16", "kind": "ffn", "fmt": "q6_K", "H": 4096, "F": 14336, "T": 16, "graph": True},
        # prompts: a short ragged one, an ordinary one, a long one
        {"name": "prefill_q4_K_M_T77", "kind": "prefill", "fmt": "q4_K_M", "H": 4096, "F": 14336, "T": 77},
        {"name": "prefill_q8_0_T512", "kind": "prefill", "fmt": "q8_0", "H": 4096, "F": 14336, "T": 512},
        {"name": "prefill_q4_K_M_T4096", "kind": "prefill", "fmt": "q4_K_M", "H": 4096, "F": 14336, "T": 4096},
        # a gpt-oss layer: one token, and a batch of 32
        {"name": "moe_mxfp4_T1", "kind": "moe_decode", "fmt": "mxfp4", "H": 2880, "F": 2880, "E": 32, "k": 4, "T": 1, "graph": True},
        {"name": "moe_mxfp4_T32", "kind": "moe_grouped", "fmt": "mxfp4", "rows": "q8", "H": 2880, "F": 2880, "E": 32, "k": 4, "T": 32},
        # a Qwen3-30B-A3B layer: a prompt over fp16 rows, and a ragged one through the quantized-row signatures
        {"name": "moe_q8_0_T2048", "kind": "moe_grouped", "fmt": "q8_0", "rows": "f16", "H": 2048, "F": 768, "E": 128, "k": 8, "T": 2048},
        {"name": "moe_q4_K_M_T333_q8", "kind": "moe_grouped", "fmt": "q4_K_M", "rows": "q8", "H": 2048, "F": 768, "E": 128, "k": 8, "T": 333},
    ]


def _log(rng, lo, hi, step=1):
    """A multiple of `step` in [lo, hi], uniform in the logarithm."""
    return min(hi, max(lo, int(round(math.exp(rng.uniform(math.log(lo), math.log(hi))) / step)) * step))


def draw(rng):
    kind = rng.choice(["proj", "ffn", "prefill", "prefill", "moe_decode", "moe_grouped", "moe_grouped"])
    if kind == "proj":
        K = _log(rng, 1024, 8192, 256)
        return {"kind": kind, "fmt": rng.choice(["q4_K", "q6_K", "q8_0", "mxfp4"]), "K": K, "N": min(_log(rng, 1000, 151936), 151936 * 4096 // K)}
    if kind in ("ffn", "prefill"):
        H = _log(rng, 1024, 6144, 256)
        F = min(_log(rng, 2048, 20480, 256), 4096 * 14336 // H // 256 * 256)
        fmt = rng.choice(["q4_K_M", "q4_K", "q6_K", "q8_0"])
        if kind == "prefill":
            return {"kind": kind, "fmt": fmt, "H": H, "F": F, "T": _log(rng, 17, 4096)}
        return {"kind": kind, "fmt": fmt, "H": H, "F": F, "T": rng.choice([1, rng.randint(2, 16)]), "graph": rng.random() < 0.5}
    fmt = rng.choice(["mxfp4", "q8_0", "q4_K_M"])
    step = 256 if fmt == "q4_K_M" else 128
    H, F = _log(rng, 1024, 4096, step), _log(rng, 512, 3072, step)
    E, k = rng.choice([8, 16, 32, 60, 64, 128]), rng.choice([2, 4, 6, 8])
    while E * H * F > 32 * 2880 * 2880:
        E //= 2
    k = min(k, E // 2)
    if kind == "moe_decode":
        return {"kind": kind, "fmt": fmt, "H": H, "F": F, "E": E, "k": k, "T": rng.choice([1, 1, 2, 4]), "graph": rng.random() < 0.5}
    T = _log(rng, 8, 2048)
    return {"kind": kind, "fmt": fmt, "rows": rng.choice(["f16", "q8"]) if T >= 48 else "q8", "H": H, "F": F, "E": E, "k": k, "T": T}


# ---------------------------------------------------------------- what a program has in hand
def _matrix(fmt, N, K, seed):
    """The tensors an entry point takes for one [N, K] matrix: GGUF blocks, or the two planes of Q8_0 and MXFP4."""
    w = synth.normal_weights(fmt, N, K, seed, device=DEV)
    return synth.split_q8_0(w) if fmt == "q8_0" else synth.split_mxfp4(w) if fmt == "mxfp4" else (w.reshape(-1),)


def _fmts(fmt):
    return PARTS.get(fmt, (fmt, fmt))


def prepare(case, seed):
    st = dict(case)
    g = torch.Generator(device=DEV)
    g.manual_seed(seed * 1000003 + 17)
    rnd = lambda *shape: torch.randn(shape, device=DEV, generator=g)  # noqa: E731
    ws = seed * 16 + 1
    if case["kind"] == "proj":
        st["x"] = rnd(1, case["K"]).half()
        st["W"] = _matrix(case["fmt"], case["N"], case["K"], ws)
        return st
    H, F, T = case["H"], case["F"], case["T"]
    fa, fd = _fmts(case["fmt"])
    E = case.get("E", 1)
    st["gate"], st["up"], st["down"] = _matrix(fa, E * F, H, ws), _matrix(fa, E * F, H, ws + 1), _matrix(fd, E * H, F, ws + 2)
    x = rnd(T, H)
    if "E" in case:
        popular = -0.5 * torch.log(torch.arange(1, E + 1, device=DEV, dtype=torch.float32))[torch.randperm(E, device=DEV, generator=g)]
        x = x + 0.25                                                    # the common component: 0.25 sqrt(H) along the unit diagonal
        st["W_gate"] = rnd(E, H) / math.sqrt(H) + popular[:, None] / (0.25 * H)
        if case["fmt"] == "mxfp4":
            st["gate_b"], st["up_b"], st["down_b"] = (0.1 * rnd(E, n) for n in (F, F, H))
            st["slots"] = torch.arange(T * case["k"], device=DEV, dtype=torch.int32)   # packed row of slot i when rows stay in slot order
    st["x"] = x.half().contiguous()
    if case.get("graph"):
        ops.init()
        side = torch.cuda.Stream()
        side.wait_stream(torch.cuda.current_stream())
        with torch.cuda.stream(side):
            _pass(st)
        torch.cuda.current_stream().wait_stream(side)
        st["captured"] = torch.cuda.CUDAGraph()
        with torch.cuda.graph(st["captured"]):
            st["out"] = _pass(st)
    return st


# ---------------------------------------------------------------- one pass
def run(state):
    if "captured" in state:
        state["captured"].replay()
        return state["out"]
    return _pass(state)


def _pass(st):
    return {"proj": _proj, "ffn": _ffn, "prefill": _prefill, "moe_decode": _moe_decode, "moe_grouped": _moe_grouped}[st["kind"]](st)


GEMV = {"q4_K": ops.gemv_q4_K_q8, "q6_K": ops.gemv_q6_K_q8, "q8_0": ops.gemv_q8_0_soa_q8, "mxfp4": ops.gemv_mxfp4_soa_q8}
BATCHED = {"q4_K": ops.gemv_q4_K_q8_batched, "q6_K": ops.gemv_q6_K_q8_batched, "q8_0": ops.gemv_q8_0_soa_q8_batched}
GEMM = {"q4_K": ops.gemm_q4_K, "q6_K": ops.gemm_q6_K, "q8_0": ops.gemm_q8_0_soa}


def _proj(st):
    return GEMV[st["fmt"]](ops.quantize_q8_1(st["x"]), *st["W"], st["K"], st["N"])


def _ffn(st):
    H, F, T = st["H"], st["F"], st["T"]
    fa, fd = _fmts(st["fmt"])
    if T == 1:
        one = lambda fmt, W: ("q8_0_soa", W) if fmt == "q8_0" else (fmt, W[0])  # noqa: E731
        kind, gate = one(fa, st["gate"])
        h = ops.gemv_x2_silu(kind, st["x"], gate, one(fa, st["up"])[1], H, F)
        kind, down = one(fd, st["down"])
        return ops.gemv_f16q8(kind, h, down, F, H)
    xq = ops.quantize_q8_1(st["x"])
    gate = BATCHED[fa](xq, *st["gate"], H, F, T)
    up = BATCHED[fa](xq, *st["up"], H, F, T)
    _, hq = ops.swiglu_q8(gate, up, want_y=False)
    return BATCHED[fd](hq, *st["down"], F, H, T)


def _prefill(st):
    H, F, T = st["H"], st["F"], st["T"]
    fa, fd = _fmts(st["fmt"])
    gate = GEMM[fa](st["x"], *st["gate"], T, H, F)
    up = GEMM[fa](st["x"], *st["up"], T, H, F)
    h, _ = ops.swiglu_q8(gate, up)
    return GEMM[fd](h, *st["down"], T, F, H)


def _strides(st):
    """(elements per expert of the quant planes in bytes, of the scale planes) or bytes per expert of the block banks."""
    n = st["H"] * st["F"]
    if st["fmt"] == "q8_0":
        return n, n // 32
    if st["fmt"] == "mxfp4":
        return n // 2, n // 32
    return tuple(n // 256 * synth.BLOCK[f][1] for f in _fmts(st["fmt"]))


def _moe_decode(st):
    H, F, E, k, T = st["H"], st["F"], st["E"], st["k"], st["T"]
    s0, s1 = _strides(st)
    ids, w = ops.moe_router(st["x"], st["W_gate"], E, k)
    if st["fmt"] == "q4_K_M":
        h = ops.moe_decode_gate_up_silu_q4k(st["x"], st["gate"][0], st["up"][0], ids, H, F, k, s0, T)
        return ops.moe_decode_down_kquant("q6k", h, st["down"][0], ids, w, H, F, k, s1, T), ids
    xq = ops.quantize_q8_1(st["x"])
    if st["fmt"] == "q8_0":
        h = ops.moe_gate_up_silu_q8(xq, *st["gate"], *st["up"], s0, s1, ids, T, k, H, F, n_experts=E)
        o = ops.moe_down_q8_f16(h, *st["down"], s0, s1, ids, w, T, k, F, H, n_experts=E)
        return ops.moe_reduce_q8(o, T, k, H), ids
    h = ops.moe_gate_up_oai_mxfp4(xq, *st["gate"], *st["up"], s0, s1, st["gate_b"], st["up_b"], ids, T, k, H, F, E)
    o = ops.moe_down_mxfp4_f16(h, *st["down"], s0, s1, st["down_b"], ids, T, k, F, H, E)
    return ops.moe_prefill_reduce(o, st["slots"], w, torch.zeros((T, H), dtype=torch.float16, device=DEV), T, k, H), ids


def _moe_grouped(st):
    H, F, E, k, T = st["H"], st["F"], st["E"], st["k"], st["T"]
    s0, s1 = _strides(st)
    fmt, TK, x = st["fmt"], T * k, st["x"]
    ids, w = ops.moe_router(x, st["W_gate"], E, k)
    off, src, wp, where = ops.moe_build_packing_device(ids, w, E)
    weighted = fmt != "mxfp4"             # the down product applies the routing weights itself
    if st["rows"] == "f16":
        if fmt == "q8_0":
            h = ops.moe_gemm_gate_up_silu_q8(x, *st["gate"], *st["up"], s0, s1, off, TK, E, H, F, sorted_idx=src)
            o = ops.moe_gemm_down_q8(h, *st["down"], s0, s1, off, wp, TK, E, H, F)
        elif fmt == "mxfp4":
            h = ops.moe_gemm_gate_up_oai_mxfp4(x, *st["gate"], *st["up"], s0, s1, st["gate_b"], st["up_b"], off, TK, E, H, F, sorted_idx=src)
            o = ops.moe_gemm_down_mxfp4(h, *st["down"], s0, s1, st["down_b"], off, TK, E, H, F)
        else:
            h = ops.moe_gemm_gate_up_silu_q4k(x, st["gate"][0], st["up"][0], off, TK, E, H, F, s0, sorted_idx=src)
            o = ops.moe_gemm_down_kquant("q6k", h, st["down"][0], off, wp, TK, E, H, F, s1)
    else:
        xp = ops.moe_gather_rows(x, src, TK, H)
        if fmt == "q8_0":
            h = ops.moe_prefill_gate_up_silu_q8(ops.quantize_q8_1(xp), *st["gate"], *st["up"], s0, s1, off, TK, E, H, F)
            o = ops.moe_prefill_down_q8(ops.quantize_q8_1(h), *st["down"], s0, s1, off, wp, TK, E, H, F)
        elif fmt == "mxfp4":
            h = ops.moe_grouped_gate_up_oai_mxfp4(ops.quantize_q8_1(xp), *st["gate"], *st["up"], s0, s1, st["gate_b"], st["up_b"], off, TK, E, H, F)
            o = ops.moe_grouped_down_mxfp4(ops.quantize_q8_1(h), *st["down"], s0, s1, st["down_b"], off, TK, E, H, F)
        else:
            h = ops.moe_prefill_gate_up_silu_kquant_q8("q4k", ops.quantize_q8_1s(xp), st["gate"][0], st["up"][0], off, TK, E, H, F, s0)
            o = ops.moe_prefill_down_packed_kquant_q8("q6k", ops.quantize_q8_1s(h), st["down"][0], off, TK, E, H, F, s1)
            weighted = False
    if weighted:
        return ops.moe_prefill_reduce_sum(o, where, T, k, H), ids
    return ops.moe_prefill_reduce(o, where, wp, torch.zeros((T, H), dtype=torch.float16, device=DEV), T, k, H), ids


# ---------------------------------------------------------------- what a pass cannot do without
def work(case):
    """Weights (of the experts that routing is expected to reach), input rows and output rows once; two operations per product."""
    fa, fd = _fmts(case["fmt"])
    if case["kind"] == "proj":
        n = case["K"] * case["N"]
        return {"bytes": n * BITS[fa] / 8 + 2 * (case["K"] + case["N"]), "flops": 2.0 * n}
    H, F, T, k, E = case["H"], case["F"], case["T"], case.get("k", 1), case.get("E", 1)
    shares = [r ** -0.5 for r in range(1, E + 1)]
    reached = sum(1.0 - (1.0 - min(1.0, k * s / sum(shares))) ** T for s in shares)
    weights = reached * H * F * (2 * BITS[fa] + BITS[fd]) / 8
    router = E * H if E > 1 else 0
    return {"bytes": weights + 4 * router + 4.0 * T * H, "flops": 6.0 * T * k * H * F + 2.0 * T * router}


def tolerance(case):
    """About four times the distance from the same chain in 64 bits with the same roundings (fp16 rows between the products, q8
    codes where the path quantizes): 1.4e-5 / 7e-4 (rel / max) for one product, 1.3e-4 / 1.6e-3 for a feed-forward block, where a
    last-bit change of an intermediate moves a q8 code, 3.5e-4 / 2.7e-3 for an expert block, whose summands are fp16 rows."""
    if case["kind"] == "proj":
        return {"rel": 1e-4, "max": 3e-3}
    if case["kind"] in ("ffn", "prefill"):
        return {"rel": 5e-4, "max": 6e-3}
    return {"rel": 1.4e-3, "max": 1.1e-2, "differ": 1e-3}
