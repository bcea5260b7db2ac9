"""The work that users of this package have it do, as cases that can be timed and checked.

A case is one pass through the public entry points:

* op "gemm": `calls` consecutive `w4a16_opt.w4a16_gemm` calls of one projection shape with the weights
  of `calls` layers, as a model's forward pass makes them (each layer has its own weights, so a call
  finds little of its weights in the caches; one call alone is the smallest request);
* op "quantize": `w4a16_opt.quantize_pack` of one fp16 or fp32 weight matrix (weight loading);
* op "gemv": `calls` consecutive `w4a16_ext.w4a16_gemv` calls (the baseline extension's format).

Shapes are the Llama-3 projections, the ragged shape of the tests and bench.py's; `draw` spreads sizes
over the same ranges.  Inputs are made on the GPU from the seed alone.  `exact` restates each op in
plain torch in 64 bits.
"""
import os
import sys

import torch

sys.path.insert(0, os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "w4a16-gemm_amd"))

import w4a16_ext  # noqa: E402
import w4a16_opt  # noqa: E402

MAX_MNK = 2048 * 28672 * 8192          # the largest listed product
MAX_QUANT = 14336 * 8192               # values of the largest weight matrix quantised


def listed():
    def gemm(name, M, N, K, G, calls, dist="normal"):
        return {"name": name, "op": "gemm", "M": M, "N": N, "K": K, "G": G, "calls": calls, "dist": dist}

    return [
        # one request, one projection: what a single call costs (launch and latency)
        gemm("decode-single-m1", 1, 8192, 4096, 128, 1),
        # token generation: the gate/up projection for 4 sequences, the down projection for 16, and the
        # widest projection for one
        gemm("decode-gate-m4", 4, 14336, 4096, 128, 5),
        gemm("decode-down-m16", 16, 4096, 14336, 128, 5),
        gemm("decode-wide-m1", 1, 28672, 8192, 128, 2),
        # batched generation and short prompts: more rows than the decode route takes, few enough that
        # the weights are most of the traffic
        gemm("batch-o-m24", 24, 4096, 4096, 128, 16),
        gemm("batch-down-m48", 48, 4096, 14336, 128, 5),
        # a short prompt at group size 64 (bench.py's moderate leg)
        gemm("prompt-gate-m128-g64", 128, 14336, 4096, 64, 5),
        # ragged sizes with activation outliers: N not a multiple of 64, an odd number of 64-wide chunks
        gemm("ragged-m37-g64", 37, 4112, 4160, 64, 15, "outliers"),
        # prompts: a ragged one, and the largest (bench.py's prefill leg)
        gemm("prompt-qkv-m513", 513, 6144, 4096, 128, 4),
        gemm("prompt-wide-m2048", 2048, 28672, 8192, 128, 1),
        # loading a checkpoint: quantise and pack one fp16 projection
        {"name": "quantize-gate-fp16", "op": "quantize", "N": 14336, "K": 4096, "G": 128, "dtype": "fp16"},
        # the baseline extension's matrix-vector product
        {"name": "gemv-gate", "op": "gemv", "N": 14336, "K": 4096, "calls": 5},
    ]


def _log(rng, lo, hi):
    return lo * (hi / lo) ** rng.random()


def draw(rng):
    kind = rng.random()
    if kind < 0.12:
        G = rng.choice([64, 128])
        N = 16 * int(_log(rng, 64, 1792))
        K = G * int(_log(rng, 1024 // G, max(1024 // G + 1, min(14336, MAX_QUANT // N) // G)))
        return {"op": "quantize", "N": N, "K": K, "G": G, "dtype": rng.choice(["fp16", "fp32"])}
    if kind < 0.25:
        N = int(_log(rng, 500, 28672))
        K = 8 * int(_log(rng, 64, 2048))
        return {"op": "gemv", "N": N, "K": K, "calls": _calls(N * K // 2, 1)}
    lo, hi = rng.choice([(1, 16), (17, 256), (257, 2048)])
    M = min(hi, int(_log(rng, lo, hi + 1)))
    G = rng.choice([64, 128])
    # multiples of 512 as most models have them, and any size the format takes
    N = 512 * int(_log(rng, 2, 57)) if rng.random() < 0.5 else 16 * int(_log(rng, 64, 1793))
    top = min(28672, MAX_MNK // (M * N))
    K = 512 * int(_log(rng, 2, max(2.1, top / 512 + 1))) if rng.random() < 0.5 else G * int(_log(rng, 1024 // G, top / G + 1))
    K = max(1024, min(K, top // 128 * 128))
    return {"op": "gemm", "M": M, "N": N, "K": K, "G": G, "calls": _calls(N * K // 2, M),
            "dist": rng.choice(["normal", "normal", "outliers"])}


def _calls(weight_bytes, M):
    """Layers per pass: about 130 MB of weights while the calls are short, one call for long ones."""
    if M > 1024:
        return 1
    return max(1, min(16, 130_000_000 // weight_bytes, 2_000_000_000_000 // (4 * M * weight_bytes)))


# ------------------------------------------------------------------------------------------ inputs


def _gen(seed):
    return torch.Generator(device="cuda").manual_seed(int(seed))


def _words(g, n):
    return torch.randint(-2**31, 2**31, (n,), dtype=torch.int32, device="cuda", generator=g)


def _gemm_inputs(c, seed):
    g = _gen(seed)
    M, N, K, G = c["M"], c["N"], c["K"], c["G"]
    wild = c["dist"] == "outliers"
    lo, hi = (1e-4, 0.05) if wild else (0.002, 0.02)
    layers = []
    for _ in range(c["calls"]):
        x = torch.randn(M, K, device="cuda", generator=g)
        if wild:                          # N(0, 4) with 1% of the entries at +-60
            x *= 2
            pick = torch.rand(M, K, device="cuda", generator=g)
            x[pick < 0.005] = 60.0
            x[pick > 0.995] = -60.0
        s = torch.rand(K // G, N, device="cuda", generator=g) * (hi - lo) + lo
        layers.append((_words(g, N * K // 8), x.half(), s.half()))
    return layers


def _gemv_inputs(c, seed):
    g = _gen(seed)
    N, K = c["N"], c["K"]
    layers = []
    for _ in range(c["calls"]):
        W = _words(g, N * (K // 8)).view(N, K // 8)
        A = torch.randn(K, device="cuda", generator=g).half()
        sW = (torch.rand(N, device="cuda", generator=g) * 0.018 + 0.002).half()
        zW = torch.randn(N, device="cuda", generator=g).half()
        layers.append((W, A, sW, zW))
    return layers


def _weight(c, seed):
    W = torch.randn(c["N"], c["K"], device="cuda", generator=_gen(seed)) * 0.02
    return W.half() if c["dtype"] == "fp16" else W


def prepare(case, seed):
    if case["op"] == "gemm":
        return case, _gemm_inputs(case, seed)
    if case["op"] == "gemv":
        return case, _gemv_inputs(case, seed)
    return case, _weight(case, seed)


def run(state):
    case, data = state
    if case["op"] == "gemm":
        return [w4a16_opt.w4a16_gemm(Wp, x, s) for Wp, x, s in data]
    if case["op"] == "gemv":
        return [w4a16_ext.w4a16_gemv(W, A, sW, zW) for W, A, sW, zW in data]
    return w4a16_opt.quantize_pack(data, case["G"])


# ------------------------------------------------------------------------------- what it has to be


def work(case):
    N, K = case["N"], case["K"]
    if case["op"] == "gemm":
        M, G, n = case["M"], case["G"], case["calls"]
        return {"bytes": n * (N * K // 2 + (K // G) * N * 2 + M * K * 2 + M * N * 2), "flops": n * 2 * M * N * K}
    if case["op"] == "gemv":
        return {"bytes": case["calls"] * (N * K // 2 + 2 * K + 6 * N), "flops": case["calls"] * 2 * N * K}
    size = 2 if case["dtype"] == "fp16" else 4
    return {"bytes": N * K * size + N * K // 2 + (K // case["G"]) * N * 2, "flops": 2 * N * K}


def tolerance(case):
    """fp16 results of fp32 sums (gemm, gemv: 2.1e-4 off `exact` as measured, the rounding to fp16);
    packed words and scales bit for bit (quantize)."""
    return "exact" if case["op"] == "quantize" else {"rel": 8e-4, "max": 4e-3}


def _unpack(Wp, N, K):
    """Packed words [N/16][K/64][lane][4] -> codes [N, K] (0..15): nibble i = p + 4h of word s of lane
    4g + t is the code of n = g + 8 (p & 1), k = 16 s + 2 t + 8 (p >> 1) + h of its 16 x 64 block."""
    w = Wp.view(N // 16, K // 64, 8, 4, 4)                                  # nb, kc, g, t, s
    q = torch.empty(N // 16, 2, 8, K // 64, 4, 2, 4, 2, dtype=torch.int8, device=Wp.device)   # nb,a,g,kc,s,b,t,h
    for a in range(2):
        for b in range(2):
            for h in range(2):
                nib = (w >> (4 * (a + 2 * b + 4 * h))) & 15
                q[:, a, :, :, :, b, :, h] = nib.permute(0, 2, 1, 4, 3).to(torch.int8)
    return q.view(N, K)


def _exact_gemm(c, Wp, x, s):
    N, K, G = c["N"], c["K"], c["G"]
    out = torch.empty(c["M"], N, dtype=torch.float64, device="cuda")
    q = _unpack(Wp, N, K)
    xd = x.double()
    for n0 in range(0, N, 4096):                                            # fp16 weights (q - 8) * s, 64-bit sums
        n1 = min(N, n0 + 4096)
        w = (q[n0:n1].half() - 8).view(n1 - n0, K // G, G) * s[:, n0:n1].t().contiguous().unsqueeze(-1)
        out[:, n0:n1] = xd @ w.view(n1 - n0, K).double().t().contiguous()
    return out


def _exact_gemv(W, A, sW, zW):
    out = []
    for w in W.split(2048):
        q = torch.stack([(w >> (4 * j)) & 15 for j in range(8)], dim=-1).reshape(w.shape[0], -1)
        q = torch.where(q >= 8, q - 16, q)
        out.append((q.double() * A.double()).sum(1))
    return (torch.cat(out) - zW.double()) * sW.double()


def exact(case, seed):
    if case["op"] == "gemm":
        return [_exact_gemm(case, *layer) for layer in _gemm_inputs(case, seed)]
    if case["op"] == "gemv":
        return [_exact_gemv(*layer) for layer in _gemv_inputs(case, seed)]
    W = _weight(case, seed).double()
    amax = W.abs().view(case["N"], case["K"] // case["G"], case["G"]).amax(-1)
    return None, (amax / 7).clamp_min(1e-4).t().contiguous()
