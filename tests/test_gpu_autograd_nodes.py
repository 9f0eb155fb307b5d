"""What the operators' autograd nodes keep between the passes: compiled autograd takes it, saved-tensor hooks may move it,
and what hooks bring back changed is refused before a kernel sees it."""
import pytest
import torch

import blockedAttention
from blockedattention_amd import blockAttention

pytestmark = pytest.mark.gpu

M, N, K = [5, 70, 9], [7, 40, 4], [16, 8, 24]


def meta(dev):
    return [torch.tensor(x, device=dev) for x in (M, N, K)]


def operands(dev, n, dtype=torch.float16):
    g = torch.Generator().manual_seed(3)
    sizes = [sum(m * k for m, k in zip(M, K)), sum(a * k for a, k in zip(N, K))]
    return [torch.randn((2, sizes[min(i, 1)]), generator=g).to(dtype).to(dev).requires_grad_() for i in range(n)]


def product(q, k, m):
    return blockedAttention.blockGEMM(q, k, None, None, None, *m)


def pair(q, k, m):
    return blockedAttention.blockSoftmax(product(q, k, m), m[0], m[1], scale=0.3)


def attention(q, k, v, m):
    return blockedAttention.blockFusedAttention(q, k, v, *m, scale=0.3)


OPS = {"product": (product, 2), "pair": (pair, 2), "attention": (attention, 3)}


def gradients(dev, op, backward=torch.Tensor.backward, hooks=None, m=None):
    f, n = OPS[op]
    ts = operands(dev, n)
    m = m or meta(dev)
    if hooks is None:
        out = f(*ts, m)
    else:
        with torch.autograd.graph.saved_tensors_hooks(*hooks):
            out = f(*ts, m)
    backward(out.float().pow(2).sum())
    return [t.grad for t in ts]


@pytest.mark.parametrize("op", list(OPS))
def test_compiled_autograd(dev, op):
    import torch._dynamo.compiled_autograd as compiled

    def backward(loss):
        with compiled._enable(torch.compile(backend="eager")):
            loss.backward()

    want = gradients(dev, op)
    for _ in range(2):                                         # new metadata, then again
        assert all(torch.equal(a, b) for a, b in zip(gradients(dev, op, backward), want))


@pytest.mark.parametrize("op", list(OPS))
def test_hooks_that_move_and_copy(dev, op):
    want = gradients(dev, op)
    for hooks in ((lambda t: t.cpu(), lambda t: t.to(dev)),     # everything comes back on the GPU, the summary too
                  (lambda t: t.clone(), lambda t: t.clone()),
                  (lambda t: (t.cpu(), t.device), lambda p: p[0].to(p[1]))):
        assert all(torch.equal(a, b) for a, b in zip(gradients(dev, op, hooks=hooks), want))


@pytest.mark.parametrize("op", list(OPS))
@pytest.mark.parametrize("change", ["strided", "short", "wide type"])
def test_hooks_that_change_are_refused(dev, op, change):
    shorter = change == "short"
    change = {"strided": lambda t: torch.stack([t, t], -1)[..., 0], "short": lambda t: t[..., :-1].contiguous(),
              "wide type": lambda t: t.double() if t.is_floating_point() else t}[change]
    # one saved tensor at a time (operands, results, row sums, plans, summaries; not the metadata, which no kernel reads):
    # the backward pass refuses it or makes the same gradients of it
    f, n = OPS[op]
    want, counted = gradients(dev, op), []
    with torch.autograd.graph.saved_tensors_hooks(counted.append, lambda t: t):
        f(*operands(dev, n), meta(dev))
    refused = 0
    for victim in range(len(counted)):
        seen = []

        def pack(t):
            seen.append(t)
            return (t, len(seen) - 1 == victim and t.dtype != torch.int64)

        try:
            got = gradients(dev, op, hooks=(pack, lambda p: change(p[0]) if p[1] else p[0]))
        except RuntimeError:
            refused += 1
            continue
        assert all(torch.equal(a, b) for a, b in zip(got, want)), victim
    if shorter:
        assert refused == sum(t.dtype != torch.int64 for t in counted)


@pytest.mark.parametrize("op", list(OPS))
def test_more_batches_in_flight_than_the_cache_holds(dev, op):
    f, n = OPS[op]
    want = gradients(dev, op)
    for capacity in (0, 2, 8):
        blockAttention.set_schedule_cache(capacity)
        try:
            passes = []
            for _ in range(5):
                ts = operands(dev, n)
                passes.append((ts, f(*ts, meta(dev))))
            for ts, out in passes:
                out.float().pow(2).sum().backward()
                assert all(torch.equal(t.grad, b) for t, b in zip(ts, want))
        finally:
            blockAttention.set_schedule_cache(8)


@pytest.mark.parametrize("op", list(OPS))
def test_gradients_after_a_call_without(dev, op):
    # the schedule of the first call has no plans for the gradients; two passes with gradients on the same metadata
    f, n = OPS[op]
    want, m = gradients(dev, op), meta(dev)
    with torch.no_grad():
        f(*operands(dev, n), m)
    for _ in range(3):
        assert all(torch.equal(a, b) for a, b in zip(gradients(dev, op, m=m), want))


@pytest.mark.parametrize("how", ["plain", "compiled", "checkpoint"])
def test_attention_result_changed_in_place(dev, how):
    # masking or dropout on the attention's own result: its value before the change is what the gradients need
    import torch._dynamo.compiled_autograd as compiled
    from torch.utils.checkpoint import checkpoint

    mask = (torch.arange(2 * sum(a * b for a, b in zip(M, K)), device=dev) % 3).reshape(2, -1).half()

    def step(in_place):
        ts, m = operands(dev, 3), meta(dev)

        def layer(*qkv):
            y = attention(*qkv, m)
            return y.mul_(mask) if in_place else y * mask

        out = checkpoint(layer, *ts, use_reentrant=False) if how == "checkpoint" else layer(*ts)
        loss = out.float().pow(2).sum()
        if how == "compiled":
            with compiled._enable(torch.compile(backend="eager")):
                loss.backward()
        else:
            loss.backward()
        return [t.grad for t in ts]

    assert all(torch.equal(a, b) for a, b in zip(step(True), step(False)))


def test_attention_result_overwritten(dev):
    want = gradients(dev, "attention", backward=lambda loss: loss.backward())
    ts = operands(dev, 3)
    y = attention(*ts, meta(dev))
    grad = (2 * y.float()).half()
    with torch.no_grad():
        y.zero_()
    assert all(torch.equal(a, b) for a, b in zip(torch.autograd.grad(y, ts, grad), want))


@pytest.mark.parametrize("op", list(OPS))
def test_metadata_first_seen_in_inference_mode(dev, op):
    f, n = OPS[op]
    want = gradients(dev, op)
    m = meta(dev)
    with torch.inference_mode():
        f(*[t.detach() for t in operands(dev, n)], m)
    for got, ref in zip(gradients(dev, op, m=m), want):          # the schedule kept from the first call
        assert torch.equal(got, ref)
