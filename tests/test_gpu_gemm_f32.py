"""fp32 varlen GEMM through the C ABI against float64 products.  Products and sums are fp32: |x - ref| is at most
(K + 2) 2^-24 (|A| |B|^T), whatever the order of the sum."""
import numpy as np
import pytest
import torch

from blockedattention_amd import capi
from _util import make_plan

pytestmark = pytest.mark.gpu


def run(dev, M, N, K, H, t1, t2, seed=0, summary=True):
    M, N, K = (np.asarray(x, np.int64) for x in (M, N, K))
    g = torch.Generator("cpu").manual_seed(seed)
    d1, d2, do = int((M * K).sum()), int((N * K).sum()), int((M * N).sum())
    A, B = torch.randn((H, d1), generator=g), torch.randn((H, d2), generator=g)
    plan = make_plan(dev, M, N, K, read=summary)
    out = torch.full((H, do), float("nan"), device=dev)
    print(f"fp32 case M={M[:6]} N={N[:6]} K={K[:6]} H={H} {t1} {t2}", flush=True)
    capi.varlen_gemm(plan, A.to(dev), B.to(dev), out, H, d1, d2, do, t1, t2)
    got = out.cpu().double()
    o1, o2, oo = (np.concatenate([[0], np.cumsum(x)]) for x in (M * K, N * K, M * N))
    for s in range(len(M)):
        m, n, k = int(M[s]), int(N[s]), int(K[s])
        for h in range(H):
            a = A[h, o1[s]:o1[s + 1]].double(); b = B[h, o2[s]:o2[s + 1]].double()
            a = a.reshape(k, m).t() if t1 else a.reshape(m, k)
            b = b.reshape(k, n) if t2 else b.reshape(n, k).t()
            err = (got[h, oo[s]:oo[s + 1]].reshape(m, n) - a @ b).abs() - (k + 2) * 2.0 ** -24 * (a.abs() @ b.abs())
            assert not torch.isnan(err).any() and (err.numel() == 0 or err.max() <= 0), (m, n, k, h)
    assert plan.read().run_errors == 0


@pytest.mark.parametrize("t1,t2", [(False, False), (True, False), (False, True), (True, True)])
def test_layouts_and_tile_edges(dev, t1, t2):
    # aligned and odd reduction lengths around the 16-, 64- and 128-wide steps, 1..4 column tiles, segments below four elements
    run(dev, [1, 16, 17, 63, 64, 65, 130, 3], [64, 1, 33, 48, 65, 128, 15, 1], [64, 4, 128, 60, 16, 20, 132, 68], 2, t1, t2)
    run(dev, [1, 16, 17, 63, 70, 2, 129], [2, 49, 33, 20, 65, 1, 7], [1, 3, 65, 127, 33, 1, 130], 3, t1, t2, seed=1)


def test_empty_dimensions_and_no_summary(dev):
    for summary in (True, False):
        run(dev, [4, 0, 9, 300, 5], [6, 5, 0, 70, 7], [16, 8, 24, 0, 3], 2, False, False, seed=2, summary=summary)
        run(dev, [700, 65], [20, 130], [17, 64], 3, True, True, seed=3, summary=summary)


@pytest.mark.parametrize("t1,t2", [(False, False), (True, False), (False, True), (True, True)])
def test_segments_below_four_elements(dev, t1, t2):
    # every shape whose operands have one to three elements, each between larger neighbours: a piece of such an operand
    # that does not exist (k past K above all, where both operands would have to be wrong) adds nothing
    shapes = [(m, n, k) for m in (1, 2, 3) for n in (1, 2, 3) for k in (1, 2, 3)]
    M, N, K = (np.array([x for s in shapes for x in (s[i], 20)]) for i in range(3))
    run(dev, M, N, K, 2, t1, t2, seed=5)
    run(dev, [2], [3], [1], 1, t1, t2, seed=6)


@pytest.mark.parametrize("t1,t2", [(True, False), (False, True)])
def test_infinity_stays_in_its_row(dev, t1, t2):
    # K = 1, the k-major operand [inf, 2] (and [inf, 2, 3]): the rows or columns without the infinity are finite
    for n in (2, 3):
        x = torch.tensor([[float("inf"), 2.0, 3.0][:n]], device=dev)
        y = torch.tensor([[1.0, -1.0]], device=dev)
        M, N = (n, 2) if t1 else (2, n)
        out = torch.full((1, 2 * n), float("nan"), device=dev)
        print(f"fp32 infinity case {n} {t1} {t2}", flush=True)
        capi.varlen_gemm(make_plan(dev, [M], [N], [1]), x if t1 else y, y if t1 else x, out, 1, M, N, M * N, t1, t2)
        want = torch.outer(x[0], y[0]) if t1 else torch.outer(y[0], x[0])
        assert torch.equal(out.view(M, N), want)


def test_gradients_of_segments_below_four_elements(dev):
    import blockedAttention
    shapes = [(1, 2, 2), (1, 3, 3), (1, 2, 3), (5, 6, 7), (1, 3, 2), (2, 1, 1)]
    M, N, K = (np.array([s[i] for s in shapes]) for i in range(3))
    g = torch.Generator().manual_seed(9)
    a, b, go = (torch.randn((2, int(x.sum())), generator=g) for x in (M * K, N * K, M * N))
    ad, bd = a.to(dev).requires_grad_(), b.to(dev).requires_grad_()
    blockedAttention.blockGEMM(ad, bd, None, None, None, *(torch.from_numpy(x).to(dev) for x in (M, N, K))).backward(go.to(dev))
    o1, o2, oo = (np.concatenate([[0], np.cumsum(x)]) for x in (M * K, N * K, M * N))
    for s, (m, n, k) in enumerate(shapes):
        A, B, G = (t[:, o[s]:o[s + 1]].double().reshape(2, r, -1) for t, o, r in ((a, o1, m), (b, o2, n), (go, oo, m)))
        for got, x, y, red in ((ad.grad[:, o1[s]:o1[s + 1]], G, B, n), (bd.grad[:, o2[s]:o2[s + 1]], G.transpose(1, 2), A, m)):
            err = (got.cpu().double().reshape(2, x.shape[1], -1) - x @ y).abs()
            assert (err <= (red + 2) * 2.0 ** -24 * (x.abs() @ y.abs())).all()
