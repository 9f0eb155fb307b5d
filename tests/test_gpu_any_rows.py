"""Fused GEMM + softmax of segments at any operand alignment, against the per-segment fp32 oracle: edges of the row
strips, column panels and k chunks, both sweeps, tiny segments, scales of either sign, every way into the kernel (with
and without the plan summary, the one-launch entry), aligned segments and packs in the same batch."""
import numpy as np
import pytest
import torch

import oracle
from _util import assert_probs_close, dev_i64, make_plan, random_operands
from blockedattention_amd import capi

pytestmark = pytest.mark.gpu

ROWS = [1, 15, 16, 17, 63, 64, 65, 130]
K_ODD = [1, 3, 7, 9, 31, 33, 63, 65, 101, 127, 129, 200]


def batch(seed, cols, ks, n=40):
    rng = np.random.default_rng(seed)
    pick = lambda v: rng.choice(np.asarray(v), n).astype(np.int64)
    return pick(ROWS), pick(cols), pick(ks)


def fused(dev, A, B, M, N, K, scale, out_dtype, summary=True):
    H = A.shape[0]
    plan = make_plan(dev, M, N, K, read=summary)
    dims = (H, A.shape[1], B.shape[1], int((M * N).sum()))
    out = torch.full((H, dims[3]), float("nan"), dtype=out_dtype, device=dev)
    capi.gemm_softmax(plan, A.to(dev), B.to(dev), out, *dims, scale)
    torch.cuda.synchronize()
    return out


@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16])
@pytest.mark.parametrize("cols,heads,scale", [([1, 15, 16, 17, 100, 127, 128], 3, 0.2), ([2, 129, 240, 255, 256], 2, -0.15),
                                              ([1, 257, 272, 511, 513, 700], 1, 0.1), ([40, 300], 2, 0.0)])
def test_against_oracle(dev, dtype, cols, heads, scale):
    M, N, K = batch(len(cols), cols, K_ODD)
    A, B = random_operands(M, N, K, heads, dtype, 3)
    ref = oracle.per_segment_torch(A, B, M, N, K, scale)
    for summary in (True, False):
        assert_probs_close(fused(dev, A, B, M, N, K, scale, dtype, summary), ref, f"summary {summary}")


def test_fp32_results_are_fp32_accurate(dev):
    """A score's error is at most K 2^-24 sum |a b| (fp32 sums in any order), a probability's relative one twice
    scale times that, and a few roundings of the exponential and the division; the oracle's own sums count once more."""
    M, N, K = batch(8, [5, 60, 128, 200, 300], K_ODD)
    A, B = random_operands(M, N, K, 2, torch.bfloat16, 5)
    scale = 0.12
    got = fused(dev, A, B, M, N, K, scale, torch.float32).double().cpu()
    ref = oracle.per_segment_torch(A, B, M, N, K, scale).double()
    mags = oracle.per_segment_torch(A.abs(), B.abs(), M, N, K, want="scores").double()
    rel = 4 * scale * np.repeat(K, M * N) * 2.0 ** -24 * float(mags.max()) + 64 * 2.0 ** -24
    assert ((got - ref).abs() <= torch.as_tensor(rel) * ref + 1e-30).all()


@pytest.mark.parametrize("summary", [True, False])
def test_among_aligned_segments_and_packs(dev, summary):
    rng = np.random.default_rng(12)
    M = rng.integers(1, 80, 64).astype(np.int64); N = rng.integers(1, 200, 64).astype(np.int64)
    M[::3] = 5; N[::3] = 6
    K = np.full(64, 64, np.int64)
    K[40:42] = (61, 13)                     # everything behind them starts at odd offsets
    K[42] = 6                               # sums are multiples of eight again further on for some
    A, B = random_operands(M, N, K, 2, torch.float16, 9)
    assert_probs_close(fused(dev, A, B, M, N, K, 0.2, torch.float16, summary), oracle.per_segment_torch(A, B, M, N, K, 0.2), "mixed")


@pytest.mark.parametrize("cols", [[1, 17, 128], [200, 256, 300]])
def test_one_launch_entry(dev, cols):
    M, N, K = batch(21, cols, K_ODD)
    A, B = random_operands(M, N, K, 2, torch.bfloat16, 6)
    dims = (2, A.shape[1], B.shape[1], int((M * N).sum()))
    out = torch.full((2, dims[3]), float("nan"), dtype=torch.bfloat16, device=dev)
    capi.gemm_softmax_static(dev_i64(M, dev), dev_i64(N, dev), dev_i64(K, dev), A.to(dev), B.to(dev), out, *dims, 0.2)
    torch.cuda.synchronize()
    assert_probs_close(out, oracle.per_segment_torch(A, B, M, N, K, 0.2), "one launch")


def test_summary_of_another_plan_is_reported(dev):
    # equal segment count and totals; the summary counts two packs of tiny segments and no unaligned one, the plan has two of those
    M = N = np.full(4, 2)
    plan, other = make_plan(dev, M, N, np.array([9, 7, 16, 16])), make_plan(dev, M, N, np.array([8, 8, 16, 16]))
    assert plan.info.slow_items == 2 and other.info.slow_items == 0 and other.info.list_rest == other.info.pack_items == 2
    A = torch.ones((2, 96), dtype=torch.float16, device=dev)
    out = torch.full((2, 16), 7.0, dtype=torch.float16, device=dev)
    plan.info = other.info
    capi.gemm_softmax(plan, A, A, out, 2, 96, 96, 16, 0.05)
    assert plan.read(raise_on_bad=False).run_errors == 2
    assert bool((out[:, :8] == 7.0).all())
