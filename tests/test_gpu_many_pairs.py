"""More (segment, head) pairs than one grid dimension can count threads for (2^24 workgroups of 256): every launch that
gives each row block a workgroup of its own, on segments of one row and one column, where the results are closed forms."""
import numpy as np
import pytest
import torch

import blockedAttention

pytestmark = pytest.mark.gpu

NSEG, H = (1 << 20) + 8, 16


def batch(dev, k, dtype, n):
    one = torch.ones(NSEG, dtype=torch.int64, device=dev)
    g = torch.Generator(device=dev).manual_seed(k)
    print(f"many pairs: {NSEG} x {H}, K = {k}, {dtype}", flush=True)
    return one, k * one, [torch.randn((H, NSEG * k), generator=g, device=dev).to(dtype) for _ in range(n)]


def test_fp32_product(dev):
    one, K, (a, b) = batch(dev, 4, torch.float32, 2)
    out = blockedAttention.blockGEMM(a, b, None, None, None, one, one, K)
    x = (a.double() * b.double()).view(H, NSEG, 4)
    # fp32 products and sums in any order: (K + 2) 2^-24 of the sum of sizes
    assert bool(((out.double() - x.sum(-1)).abs() <= 6 * 2.0 ** -24 * x.abs().sum(-1)).all())


def test_any_layout_product_and_gradients(dev):
    one, K, (a, b, _) = batch(dev, 5, torch.float16, 3)
    a.requires_grad_(); b.requires_grad_()
    out = blockedAttention.blockGEMM(a, b, None, None, None, one, one, K)
    x = (a.float() * b.float()).view(H, NSEG, 5).detach()
    # one rounding to 16 bits; below the normal range (2^-14) half a step of 2^-24; fp32 sums below that
    assert bool(((out.float() - x.sum(-1)).abs() <= 2.0 ** -11 * x.sum(-1).abs() + 2.0 ** -25 + 2.0 ** -21 * x.abs().sum(-1)).all())
    out.backward(torch.ones_like(out))
    assert torch.equal(a.grad, b.detach()) and torch.equal(b.grad, a.detach())     # dA = 1 * B, dB = 1 * A


def test_attention_and_gradients(dev):
    one, K, (q, k, v) = batch(dev, 8, torch.float16, 3)
    go = torch.randn(q.shape, generator=torch.Generator(device=dev).manual_seed(1), device=dev).half()
    for t in (q, k, v):
        t.requires_grad_()
    out = blockedAttention.blockFusedAttention(q, k, v, one, one, K, scale=0.3)
    assert torch.equal(out.detach(), v.detach())                # one key: its probability is 1
    dq, dk, dv = torch.autograd.grad(out, (q, k, v), go)
    assert torch.equal(dv, go)
    # dS = dO V - dO O is zero but for the order of two fp32 sums of eight products
    assert float(dq.abs().max()) <= 1e-3 and float(dk.abs().max()) <= 1e-3


def test_softmax_with_one_wide_segment(dev):
    M = np.ones(NSEG, np.int64); N = np.ones(NSEG, np.int64)
    M[-1], N[-1] = 3, 300
    src = torch.randn((H, int((M * N).sum())), generator=torch.Generator(device=dev).manual_seed(2), device=dev)
    print(f"many pairs: softmax {NSEG} x {H}", flush=True)
    got = blockedAttention.blockSoftmax(src, torch.from_numpy(M).to(dev), torch.from_numpy(N).to(dev))
    assert bool((got[:, :NSEG - 1] == 1).all())
    ref = torch.softmax(src[:, NSEG - 1:].double().view(H, 3, 300), -1).view(H, -1)
    assert bool(((got[:, NSEG - 1:].double() - ref).abs() <= 1e-6).all())
