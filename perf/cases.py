"""The work that programs built on this framework have it do, as a list of timed cases.

A batch is a number of segments of different sizes (graphs, sequences, pairs of the two) stored back to back, times a
number of heads.  Every case is one pass over one batch through the public entry points:

    call             capi.gemm_softmax_static: metadata in, probabilities out, no allocation (serving loops)
    fused            blockGEMMSoftmax: softmax(scale * A_g B_g^T)
    pair             blockGEMM then blockSoftmax, the reference's own two operators
    pair_train       the same, and the gradients of both operands from a gradient of the probabilities
    chain            blockGEMM, blockSoftmax, blockGEMM with transpose2: attention whose probabilities are kept
    attention        blockFusedAttention: softmax(scale * Q_g K_g^T) V_g in one pass
    attention_train  the same, and the gradients of queries, keys and values from a gradient of the output

listed() is the fixed list, draw() gives further cases of the same ranges.  The segment sizes belong to the case (its
`sizes` number seeds them); the values come from the seed given to prepare().
"""
import math

import numpy as np
import torch

import blockedAttention
from blockedattention_amd import capi

DTYPES = {"f16": torch.float16, "bf16": torch.bfloat16, "f32": torch.float32}
BYTES = {"f16": 2, "bf16": 2, "f32": 4}


def _case(op, dtype, segments, heads, spread, lo, hi, k_lo, k_hi, k_step=8, square=True, sizes=0):
    return {"op": op, "dtype": dtype, "segments": segments, "heads": heads, "spread": spread, "lo": lo, "hi": hi,
            "k_lo": k_lo, "k_hi": k_hi, "k_step": k_step, "square": square, "sizes": sizes}


def listed():
    cases = {
        # A batch of small molecules in a serving loop: one call, latency is all of it.
        "molecule_call": _case("call", "f16", 64, 1, "uniform", 8, 32, 64, 64),
        # The same molecules in a training step of an attention layer: launches and host work.
        "molecule_attention_train": _case("attention_train", "f16", 64, 8, "uniform", 8, 32, 64, 64),
        # Ordinary batch (medium graphs or sentences): attention weights for inference.
        "medium_fused": _case("fused", "f16", 256, 8, "uniform", 32, 128, 64, 64),
        # Ordinary batch, training through the reference's two operators.
        "medium_train": _case("pair_train", "f16", 256, 8, "uniform", 32, 128, 64, 64),
        # Ordinary batch in single precision (evaluation runs, models that do not tolerate 16 bits).
        "medium_f32": _case("pair", "f32", 256, 8, "uniform", 32, 128, 64, 64),
        # Graphs with power-law sizes: a few of 500 nodes among many of 30; attention weights.
        "powerlaw_fused": _case("fused", "bf16", 1024, 4, "lognormal", 2, 512, 128, 128),
        # The same graphs in a training step of an attention layer.
        "powerlaw_attention_train": _case("attention_train", "bf16", 1024, 4, "lognormal", 2, 512, 128, 128),
        # Cross attention, queries and keys of different lengths, one head's worth of work.
        "cross_attention": _case("attention", "f16", 512, 1, "uniform", 16, 256, 32, 128, square=False),
        # Odd lengths and head dimensions that are no multiple of eight, probabilities kept (inspection, dropout).
        "ragged_chain": _case("chain", "bf16", 300, 4, "uniform", 5, 200, 20, 100, k_step=1, square=False),
        # Few long sequences or whole graphs: attention weights, the largest output.
        "large_fused": _case("fused", "bf16", 16, 16, "uniform", 1024, 4096, 128, 128),
        # The same, attention forward: prefill of long sequences.
        "large_attention": _case("attention", "bf16", 16, 16, "uniform", 1024, 4096, 128, 128),
        # The same in a training step.
        "large_attention_train": _case("attention_train", "bf16", 16, 16, "uniform", 1024, 4096, 128, 128),
    }
    return [dict(c, name=name) for name, c in cases.items()]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    op = rng.choice(["call", "fused", "pair", "pair_train", "chain", "attention", "attention_train"])
    dtype = rng.choice(["f32", "f32", "f16", "bf16"] if op == "pair" else ["f16", "bf16"])
    spread = rng.choice(["uniform", "uniform", "lognormal"])
    square = rng.random() < 0.6
    if spread == "lognormal":
        lo, hi = 2, _log_int(rng, 200, 512)
        segments = _log_int(rng, 64, 1024)
    else:
        hi = _log_int(rng, 24, 256 if op in ("call", "pair", "pair_train", "chain") else 4096)
        lo = max(1, int(hi * rng.uniform(0.06, 0.4)))
        segments = _log_int(rng, 16, max(17, min(1024, 65536 // hi)))
    heads = _log_int(rng, 1, 16)
    if op == "call":
        segments = min(segments, 512)
        heads = max(1, min(heads, 1024 // segments))
    # (the fused pair takes odd reduction lengths element by element: long segments of those go through the pair)
    k_step = 1 if rng.random() < 0.25 and not (op == "fused" and hi > 256) else 8
    k_hi = rng.randint(20, 128) if k_step == 1 else 8 * rng.randint(4, 16)
    k_lo = k_hi if rng.random() < 0.7 else max(8, (k_hi // 2) // k_step * k_step)
    case = _case(op, dtype, segments, heads, spread, lo, hi, k_lo, k_hi, k_step, square, rng.randrange(1 << 30))
    # no dearer than the largest listed ones
    limit = [work(c) for c in listed()]
    most = {key: max(w[key] for w in limit) for key in ("bytes", "flops")}
    while any(work(case)[key] > most[key] for key in most):
        if case["heads"] > 1:
            case["heads"] -= 1
        else:
            case["segments"] = max(1, case["segments"] // 2)
    return case


def _sizes(case):
    rng = np.random.default_rng(case["sizes"])
    def lengths():
        if case["spread"] == "lognormal":
            v = np.clip(np.rint(rng.lognormal(3.5, 1.0, case["segments"])), case["lo"], case["hi"])
        else:
            v = rng.integers(case["lo"], case["hi"] + 1, case["segments"])
        return v.astype(np.int64)
    M = lengths()
    N = M.copy() if case["square"] else lengths()
    K = rng.choice(np.arange(case["k_lo"], case["k_hi"] + 1, case["k_step"]), case["segments"]).astype(np.int64)
    return M, N, K


def prepare(case, seed):
    """Operands of unit variance on the GPU, scaled as in attention, with the batch's size lists."""
    dev = torch.device("cuda")
    dtype, heads = DTYPES[case["dtype"]], case["heads"]
    M, N, K = _sizes(case)
    gen = torch.Generator(device=dev).manual_seed(seed)
    def values(n, train=False):
        t = torch.randn((heads, int(n)), generator=gen, device=dev, dtype=torch.float32).to(dtype)
        return t.requires_grad_(train)
    train = case["op"].endswith("_train")
    a, b, out = (M * K).sum(), (N * K).sum(), (M * N).sum()
    state = {"op": case["op"], "scale": float(np.mean(K)) ** -0.5,
             "M": torch.from_numpy(M).to(dev), "N": torch.from_numpy(N).to(dev), "K": torch.from_numpy(K).to(dev),
             "q": values(a, train), "k": values(b, train)}
    if case["op"] in ("chain", "attention", "attention_train"):
        state["v"] = values(b, train)
    if case["op"] == "pair_train":
        state["grad"] = values(out)
    if case["op"] == "attention_train":
        state["grad"] = values(a)
    if case["op"] == "call":
        state["dims"] = (heads, int(a), int(b), int(out))
        state["out"] = torch.empty((heads, int(out)), dtype=dtype, device=dev)
        state["accum"] = [torch.empty(case["segments"] + 1, dtype=torch.int64, device=dev) for _ in range(3)]
    return state


def run(state):
    op, M, N, K = state["op"], state["M"], state["N"], state["K"]
    q, k, scale = state["q"], state["k"], state["scale"]
    if op == "call":
        capi.gemm_softmax_static(M, N, K, q, k, state["out"], *state["dims"], scale, *state["accum"])
        return [state["out"], *state["accum"]]
    if op == "fused":
        return blockedAttention.blockGEMMSoftmax(q, k, MList=M, NList=N, KList=K, scale=scale)
    if op in ("attention", "attention_train"):
        out = blockedAttention.blockFusedAttention(q, k, state["v"], M, N, K, scale=scale)
        if op == "attention":
            return out
        return [out.detach(), *torch.autograd.grad(out, (q, k, state["v"]), state["grad"])]
    probs = blockedAttention.blockSoftmax(blockedAttention.blockGEMM(q, k, None, None, None, M, N, K), M, N, scale=scale)
    if op == "pair_train":
        return [probs.detach(), *torch.autograd.grad(probs, (q, k), state["grad"])]
    if op == "chain":
        out = blockedAttention.blockGEMM(probs, state["v"], None, None, None, M, K, N, False, True)
        return [probs, out]
    return probs


def work(case):
    """Inputs read once and outputs written once; the products the results need, without recomputed ones."""
    M, N, K = (x.astype(object) for x in _sizes(case))
    mk, nk, mn = int((M * K).sum()), int((N * K).sum()), int((M * N).sum())
    product = 2 * int((M * N * K).sum())
    elements, products = {
        "call": (mk + nk + mn, 1),
        "fused": (mk + nk + mn, 1),
        "pair": (mk + nk + mn, 1),
        "pair_train": (2 * (mk + nk) + 2 * mn, 3),                 # operands and their gradients; P and its gradient
        "chain": (mk + 2 * nk + mn + mk, 2),
        "attention": (2 * mk + 2 * nk, 2),
        "attention_train": (4 * mk + 4 * nk, 6),                   # Q, K, V, dO in; O, dQ, dK, dV out
    }[case["op"]]
    return {"bytes": BYTES[case["dtype"]] * case["heads"] * elements, "flops": case["heads"] * products * product}


def tolerance(case):
    """About four times the distance from the same path in 64 bits, over all listed shapes (2-norm; largest difference).

    One rounding at the store (call, fused): f16 2.1e-4 / 4.9e-4, bf16 1.7e-3 / 3.9e-3.  With 16-bit intermediate
    results (scores, probabilities, their gradients): forward f16 4.7e-4 / 7.1e-3, bf16 3.8e-3 / 5.4e-2; gradients f16
    6.3e-4 / 1.0e-2, bf16 5.0e-3 / 6.2e-2.  Single precision: 2.5e-7 / 1.7e-6 at K = 64, growing with its root.
    """
    if case["dtype"] == "f32":
        return {"rel": 1.5e-6, "max": 1e-5}
    if case["op"] in ("call", "fused"):
        return {"f16": {"rel": 8e-4, "max": 2e-3}, "bf16": {"rel": 7e-3, "max": 1.6e-2}}[case["dtype"]]
    if case["op"] in ("pair", "chain", "attention"):
        return {"f16": {"rel": 1.8e-3, "max": 3e-2}, "bf16": {"rel": 1.5e-2, "max": 0.2}}[case["dtype"]]
    return {"f16": {"rel": 2.5e-3, "max": 4e-2}, "bf16": {"rel": 2e-2, "max": 0.25}}[case["dtype"]]
