"""Backward of the one-pass attention (ba_varlen_attention_train / ba_varlen_attention_backward) against autograd on the
per-segment fp32 oracle.

Bound, from what the kernels round: P and dS are rounded once to the 16-bit type before the product that reduces over
them (u = 2^-11 or 2^-9 each), delta uses the stored output, whose elements carry one rounding, and every gradient is
rounded once at the store.  With A = |dO| |V|^T + |delta| the per-element size of what enters dS, the gradients may
move by u times P^T |dO| (dV) and 3 u times scale (P o A) |K|, scale (P o A)^T |Q| (dQ, dK: P, dS, and the output's
rounding in delta); with a factor of two of room, plus 1e-3 of the gradient's rms for the fp32 sums and exponentials."""
import numpy as np
import pytest
import torch

import oracle
from blockedattention_amd import capi
from _util import make_plan
from test_gpu_attention import operands

pytestmark = pytest.mark.gpu


def reference(Q, Km, V, G, M, N, K, scale):
    """fp32 gradients and the sizes of the sums behind them, per segment and head."""
    H = Q.shape[0]
    res = [torch.zeros_like(t, dtype=torch.float32) for t in (Q, Km, V)]
    mag = [torch.zeros_like(t, dtype=torch.float32) for t in (Q, Km, V)]
    o1 = np.concatenate([[0], np.cumsum(M * K)]); o2 = np.concatenate([[0], np.cumsum(N * K)])
    for g in range(len(M)):
        a, b = slice(o1[g], o1[g + 1]), slice(o2[g], o2[g + 1])
        m, n, k = int(M[g]), int(N[g]), int(K[g])
        if m == 0 or n == 0 or k == 0:
            continue
        for h in range(H):
            q, kk, v, go = (t[h, s].float().reshape(r, k) for t, s, r in ((Q, a, m), (Km, b, n), (V, b, n), (G, a, m)))
            p = torch.softmax(scale * (q @ kk.t()), -1)
            dp = go @ v.t()
            delta = (p * dp).sum(-1, keepdim=True)
            ds = scale * p * (dp - delta)
            A = abs(scale) * p * (go.abs() @ v.abs().t() + (go.abs() * (p @ v).abs()).sum(-1, keepdim=True))
            for out, x in ((res[0], ds @ kk), (mag[0], 3 * A @ kk.abs())):
                out[h, a] = x.reshape(-1)
            for i, x, y in ((1, ds.t() @ q, 3 * A.t() @ q.abs()), (2, p.t() @ go, p.t() @ go.abs())):
                res[i][h, b] = x.reshape(-1); mag[i][h, b] = y.reshape(-1)
    return res, mag


def run(dev, M, N, K, H, dtype, scale, seed=0, sigma=1.0):
    M, N, K = (np.asarray(x, np.int64) for x in (M, N, K))
    Q, Km, V = operands(M, N, K, H, dtype, seed, sigma)
    G = torch.randn(Q.shape, generator=torch.Generator("cpu").manual_seed(seed + 1)).to(dtype)
    plan = make_plan(dev, M, N, K)
    d1, d2, do = int((M * K).sum()), int((N * K).sum()), int((M * N).sum())
    q, k, v, go = (t.to(dev) for t in (Q, Km, V, G))
    print(f"attention backward case M={M[:6]} N={N[:6]} K={K[:6]} H={H} {dtype} scale={scale}", flush=True)
    out = torch.full((H, d1), float("nan"), dtype=dtype, device=dev)
    rows = capi.attention_rows(plan, d1)
    lse = torch.full((H, rows), float("nan"), device=dev); delta = torch.full_like(lse, float("nan"))
    capi.varlen_attention_train(plan, q, k, v, out, lse, H, d1, d2, do, scale)
    grads = [torch.full_like(t, float("nan")) for t in (q, k, v)]
    capi.varlen_attention_backward(plan, q, k, v, out, go, lse, delta, *grads, H, d1, d2, do, scale)
    plain = capi.varlen_attention(plan, q, k, v, torch.empty_like(out), H, d1, d2, do, scale)
    assert torch.equal(out, plain)
    u = 2.0 ** -11 if dtype == torch.float16 else 2.0 ** -9
    for name, got, ref, mag in zip(("dq", "dk", "dv"), grads, *reference(Q, Km, V, G, M, N, K, scale)):
        got = got.float().cpu()
        assert not torch.isnan(got).any(), name
        rms = float(ref.pow(2).mean().sqrt()) if ref.numel() else 0.0
        excess = (got - ref).abs() - (2 * u * (mag + ref.abs()) + 1e-3 * rms)
        assert excess.numel() == 0 or excess.max().item() <= 0, f"{name}: off by {float((got - ref).abs().max())} (rms {rms})"
    again = [torch.full_like(t, float("nan")) for t in (q, k, v)]
    capi.varlen_attention_backward(plan, q, k, v, out, go, lse, delta, *again, H, d1, d2, do, scale)
    assert all(torch.equal(x, y) for x, y in zip(grads, again)), "two runs differ"
    assert plan.read().run_errors == 0


@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16])
def test_tile_edges_of_short_segments(dev, dtype):
    # one strip per wavefront, 64 keys a workgroup: around 1, 16, 32, 64 and 128 rows and columns
    M = [1, 15, 16, 17, 64, 65, 130, 5, 200, 33]; N = [1, 16, 17, 31, 33, 64, 65, 300, 31, 129]
    run(dev, M, N, [64] * 10, 3, dtype, 0.125)


@pytest.mark.parametrize("K", [8, 32, 40, 64, 96, 104, 128, 1, 7, 33, 100, 127])
def test_head_dimensions(dev, K):
    # every build (32, 64, 96, 128), multiples of eight and odd ones; N * K below eight elements in the last segment
    run(dev, [33, 70, 3], [50, 129, 1], [K, K, K], 2, torch.bfloat16 if K % 3 else torch.float16, K ** -0.5, seed=K)


def test_mixed_head_dimensions_and_odd_offsets(dev):
    run(dev, [3, 11, 40, 7, 65, 20], [5, 66, 13, 130, 64, 9], [5, 33, 100, 1, 127, 64], 3, torch.float16, 0.3)


@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16])
@pytest.mark.parametrize("K", [64, 96, 128, 113])
def test_tall_segments(dev, K, dtype):
    # two strips per wavefront, 128 keys a workgroup, with ragged last blocks on both sides
    run(dev, [300, 520, 257], [130, 77, 1025], [K] * 3, 2, dtype, K ** -0.5, seed=7)


@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16])
@pytest.mark.parametrize("K", [24, 64, 96, 128])
def test_two_strips_beside_workgroups_of_64_keys(dev, K, dtype):
    # the same heights, more workgroups of 128 keys than compute units: 64 keys a workgroup
    run(dev, [300, 520, 257], [130, 77, 1025], [K] * 3, 24, dtype, K ** -0.5, seed=8)


@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16])
@pytest.mark.parametrize("K", [32, 64, 96, 128, 101])
def test_scales_and_missing_queries_in_tall_segments(dev, K, dtype):
    # above every line of heights: 128 keys a workgroup; scores of either sign and none; without queries dK and dV are zeros
    for scale in (K ** -0.5, -0.3, 0.0):
        run(dev, [2100, 0, 1500, 700], [130, 300, 77, 1025], [K] * 4, 1, dtype, scale, seed=K)


@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16])
@pytest.mark.parametrize("K", [61, 90, 127])
def test_two_strips_at_any_alignment(dev, K, dtype):
    # dQ in one stage (fewer than 256 keys a query) and in two
    run(dev, [300, 520, 257], [130, 77, 33], [K] * 3, 2, dtype, K ** -0.5, seed=9)
    run(dev, [300, 520, 257], [330, 577, 1], [K] * 3, 2, dtype, K ** -0.5, seed=9)


@pytest.mark.parametrize("K", [24, 64, 96, 128, 101])
def test_block_counts_beside_a_tall_segment(dev, K):
    # 128 keys a workgroup, three stages of 64 queries: one, two, three and more blocks, full and ragged, and key blocks
    # of which one to all four pairs of wavefronts have keys
    # (dQ: 64 keys a block in two halves of which the last may have none, wavefronts without rows, no keys at all)
    M = [1, 63, 64, 65, 128, 129, 193, 6400, 260]; N = [200, 31, 33, 127, 1, 128, 129, 96, 0]
    run(dev, M, N, [K] * 9, 2, torch.bfloat16, K ** -0.5, seed=K)


@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16])
@pytest.mark.parametrize("K", [8, 32, 29])
def test_small_head_dimensions_many_workgroups(dev, K, dtype):
    # head dimensions up to 32, tall segments, more workgroups of 128 keys than compute units: two stages of 64 queries; one
    # block and more, full and ragged, key blocks of which one to all four pairs of wavefronts have keys
    M = [1, 63, 64, 65, 129, 193, 2500, 3200]; N = [200, 31, 33, 127, 1, 128, 129, 300]
    run(dev, M, N, [K] * 8, 20, dtype, K ** -0.5, seed=K)


def test_empty_segments(dev):
    # no queries: dk and dv are zeros; no keys: dq is zeros
    run(dev, [4, 0, 9, 30, 0], [6, 5, 0, 70, 300], [16, 8, 24, 64, 64], 2, torch.float16, 0.5)


def all_scores_far_below_zero(dev, M, N):
    K, rows, keys = np.full_like(M, 64), int(M.sum()), int(N.sum())
    q, k = torch.full((1, rows * 64), -2.0), torch.full((1, keys * 64), 2.0)      # every score is -256
    v = torch.randn((1, keys * 64), generator=torch.Generator("cpu").manual_seed(1))
    plan = make_plan(dev, M, N, K)
    q, k, v = (t.to(torch.bfloat16).to(dev) for t in (q, k, v))
    out = torch.empty_like(q); lse = torch.empty((1, capi.attention_rows(plan, q.shape[1])), device=dev)
    dims = (1, q.shape[1], k.shape[1], int((M * N).sum()), 2.0)
    capi.varlen_attention_train(plan, q, k, v, out, lse, *dims)
    grads = [torch.empty_like(t) for t in (q, k, v)]
    capi.varlen_attention_backward(plan, q, k, v, out, torch.ones_like(q), lse, torch.empty_like(lse), *grads, *dims)
    assert all(bool(torch.isfinite(g).all()) for g in grads)
    assert torch.allclose(grads[2][0, : N[0] * 64].float(), torch.full((int(N[0]) * 64,), M[0] / N[0], device=dev), rtol=2 ** -8)


def test_negative_zero_and_large_scale(dev):
    # large scores of both signs: probabilities close to 0 and 1, sums far below 2^-128 for a padding key of score zero
    for scale in (-0.3, 0.0):
        run(dev, [9, 70], [100, 17], [16, 64], 2, torch.float16, scale)
        run(dev, [300, 520], [130, 77], [128, 64], 1, torch.bfloat16, scale)
    all_scores_far_below_zero(dev, np.array([40, 300]), np.array([50, 270]))


def test_scores_far_below_zero_in_tall_segments(dev):
    # two strips a wavefront and 128 keys a workgroup, the last of them ragged
    all_scores_far_below_zero(dev, np.array([1000, 900, 1100]), np.array([50, 270, 1025]))


@pytest.mark.parametrize("seed", [21, 22, 23, 24])
def test_random_batches(dev, seed):
    rng = np.random.default_rng(seed)
    nseg = int(rng.integers(1, 40))
    M = rng.integers(0, 700 if seed % 2 else 150, nseg); N = rng.integers(0, 400, nseg)
    kmax = int(rng.choice([16, 32, 64, 96, 128]))
    K = rng.integers(1, kmax // 8 + 1, nseg) * 8 if seed % 3 else rng.integers(1, kmax + 1, nseg)
    run(dev, M, N, K, int(rng.integers(1, 4)), torch.float16 if seed % 2 else torch.bfloat16, float(rng.uniform(0.05, 0.3)), seed=seed)


def test_given_prefix_sums_with_gaps_and_partial_gradients(dev):
    # segments with unused elements between them, several leading dimensions, only the values differentiable
    import blockedAttention
    M = np.array([20, 70]); N = np.array([40, 30]); K = np.array([16, 32])
    a1 = np.array([0, 20 * 16 + 8, 20 * 16 + 8 + 70 * 32]); a2 = np.array([0, 40 * 16 + 16, 40 * 16 + 16 + 30 * 32])
    ao = np.array([0, 800, 800 + 2100])
    g = torch.Generator("cpu").manual_seed(3)
    q, k, v, go = (torch.randn((2, 2, int(a[-1])), generator=g).half() for a in (a1, a2, a2, a1))
    meta = [torch.from_numpy(x).to(dev) for x in (M, N, K, a1, a2, ao)]
    vd = v.to(dev).requires_grad_()
    out = blockedAttention.blockFusedAttention(q.to(dev), k.to(dev), vd, *meta, scale=0.2)
    out.backward(go.reshape(out.shape).to(dev))
    for s in range(2):
        b, a = slice(a2[s], a2[s] + N[s] * K[s]), slice(a1[s], a1[s] + M[s] * K[s])
        for h in range(4):
            qq, kk, gg = (t.reshape(4, -1)[h, i].float().reshape(-1, int(K[s])) for t, i in ((q, a), (k, b), (go, a)))
            ref = torch.softmax(0.2 * qq @ kk.t(), -1).t() @ gg
            got = vd.grad.reshape(4, -1)[h, b].float().cpu().reshape(ref.shape)
            assert (got - ref).abs().max() <= 1e-2 * ref.abs().max()


def test_summary_of_another_plan_is_reported(dev):
    # equal segment count and totals, other smallest K: the per-query arrays sized from the summary are too short for
    # the plan (one block of rows each, K = 16 against 8), and nothing is written to them or behind them
    M = N = np.array([8, 8, 8]); K, K2 = np.array([8, 64, 24]), np.array([16, 64, 16])
    plan, other = make_plan(dev, M, N, K), make_plan(dev, M, N, K2)
    d, do = int((M * K).sum()), int((M * N).sum())
    q, k, v, go = (torch.randn((2, d), generator=torch.Generator().manual_seed(i)).half().to(dev) for i in range(4))
    own, short = capi.attention_rows(plan, d), capi.attention_rows(other, d)
    assert short < own
    info, dims = plan.info, (2, d, d, do, 0.5)
    out, lse, delta = torch.full_like(q, 7.0), torch.full((2, own), 7.0, device=dev), torch.full((2, own), 7.0, device=dev)
    grads = [torch.full_like(q, 7.0) for _ in range(3)]
    plan.info = other.info
    capi.varlen_attention_train(plan, q, k, v, out, lse, *dims)
    assert plan.read(raise_on_bad=False).run_errors == 1
    plan.info = other.info
    capi.varlen_attention_backward(plan, q, k, v, out, go, lse, delta, *grads, *dims)
    assert plan.read(raise_on_bad=False).run_errors == 2
    for t in (out, lse, delta, *grads):
        assert bool((t == 7.0).all())
    # without a summary the arrays have no size: refused
    plan.info = None
    with pytest.raises(capi.BlockedAttentionError):
        capi.varlen_attention_train(plan, q, k, v, out, lse, *dims)
    with pytest.raises(capi.BlockedAttentionError):
        capi.varlen_attention_backward(plan, q, k, v, out, go, lse, delta, *grads, *dims)
    plan.info = info
