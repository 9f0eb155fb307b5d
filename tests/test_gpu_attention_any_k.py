"""One-pass attention with head dimensions that are no multiple of eight: every build (head dimension up to 32, 64, 96,
128; one and two strips per wavefront), rows of fewer than eight elements, segments of fewer than eight elements, edges
of the key blocks.  Bound and oracle: see test_gpu_attention."""
import numpy as np
import pytest
import torch

from test_gpu_attention import run

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16])
@pytest.mark.parametrize("K", [1, 3, 7, 9, 31, 33, 63, 65, 95, 97, 127])
def test_short_segments(dev, dtype, K):
    M = [1, 1, 2, 16, 17, 64, 65, 130, 3]
    N = [1, 2, 1, 63, 64, 65, 128, 129, 200]
    run(dev, M, N, [K] * len(M), 2, dtype, 0.2, seed=K)


@pytest.mark.parametrize("K", [5, 45, 77, 125])
def test_tall_segments(dev, K):
    run(dev, [300, 511, 700], [129, 320, 64], [K] * 3, 1, torch.bfloat16, -0.1, seed=K)
