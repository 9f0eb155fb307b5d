"""The 64 x 64 build of the any-layout GEMM with one LDS buffer (at most four steps a round on average) and with two
(more), every layout: one and several k chunks, column blocks and row rounds, edges of 64, against fp32 matmul."""
import numpy as np
import pytest
import torch

from _util import assert_scores_close, make_plan, random_operands
from blockedattention_amd import capi

pytestmark = pytest.mark.gpu

BATCHES = {                                  # steps of a mean row's round: blocks of 64 columns x chunks of 64 k
    "one step": ([1, 17, 64, 40], [1, 63, 64, 33], [1, 7, 64, 61]),
    "four steps": ([65, 128, 129, 100], [65, 128, 100, 127], [65, 127, 128, 101]),
    "eight steps": ([3, 64, 190, 200], [200, 250, 129, 193], [129, 100, 101, 127]),
    "few steps but for one segment": ([64, 64, 64, 64, 64, 64, 10], [30] * 6 + [300], [61] * 6 + [333]),
}


@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16])
@pytest.mark.parametrize("t1,t2", [(False, False), (False, True), (True, False), (True, True)])
@pytest.mark.parametrize("batch", list(BATCHES))
def test_layouts(dev, dtype, t1, t2, batch):
    M, N, K = (np.asarray(v, np.int64) for v in BATCHES[batch])
    H = 3
    A, B = random_operands(M, N, K, H, dtype, 4)
    dims = (H, A.shape[1], B.shape[1], int((M * N).sum()))
    out = torch.full((H, dims[3]), float("nan"), dtype=dtype, device=dev)
    capi.varlen_gemm(make_plan(dev, M, N, K), A.to(dev), B.to(dev), out, *dims, t1, t2)
    torch.cuda.synchronize()
    o1 = o2 = oo = 0
    for m, n, k in zip(M, N, K):
        a, b = A[:, o1:o1 + m * k].float(), B[:, o2:o2 + n * k].float()
        a = a.reshape(H, k, m).transpose(1, 2) if t1 else a.reshape(H, m, k)
        b = b.reshape(H, k, n) if t2 else b.reshape(H, n, k).transpose(1, 2)
        assert_scores_close(out[:, oo:oo + m * n], torch.matmul(a, b).reshape(H, -1), f"{m} {n} {k}")
        o1 += m * k; o2 += n * k; oo += m * n
