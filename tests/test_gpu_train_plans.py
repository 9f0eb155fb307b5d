"""The three plans of a training step in one launch (ba_plan_gemm_train_notify) against the same plans made one by one."""
import ctypes

import numpy as np
import pytest
import torch

import oracle
from blockedattention_amd import capi
from _util import dev_i64

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("nseg", [1, 64, 65, 257, 600, 1500])
@pytest.mark.parametrize("mode", [capi.META_FROM_LISTS, capi.META_FROM_ACCUM, capi.META_GIVEN])
def test_three_plans_in_one_launch(dev, nseg, mode):
    rng = np.random.default_rng(nseg)
    M, N, K = rng.integers(1, 300, nseg), rng.integers(1, 40, nseg), rng.integers(1, 9, nseg) * 8
    M[0] = 700
    lists = [dev_i64(x, dev) for x in (M, N, K)]
    acc = [dev_i64(x, dev) for x in oracle.lists_to_accum(M, N, K)]
    given_lists = lists if mode != capi.META_FROM_ACCUM else [torch.empty_like(x) for x in lists]
    given_acc = acc if mode != capi.META_FROM_LISTS else [torch.empty_like(x) for x in acc]
    plans = [capi.Plan(nseg, dev) for _ in range(3)]
    box = torch.zeros(3 * capi.MAILBOX_BYTES, dtype=torch.uint8, pin_memory=True)
    st = capi.load().ba_plan_gemm_train_notify(*(p.ptr for p in plans), plans[0].bytes, nseg, mode,
                                               *(capi._ptr(x) for x in given_lists + given_acc),
                                               ctypes.c_void_p(box.data_ptr()), 7, capi._stream())
    capi.check(st, "ba_plan_gemm_train_notify")
    order = [(0, 1, 2), (0, 2, 1), (1, 2, 0)]                       # lists of each plan
    accum = [(0, 1, 2), (2, 1, 0), (2, 0, 1)]                       # its operands' and result's prefix sums
    for i, plan in enumerate(plans):
        info = plan.wait(box[i * capi.MAILBOX_BYTES:], 7)
        want = capi.plan_gemm(nseg, dev, *(lists[j] for j in order[i]), *(acc[j] for j in accum[i]), mode=capi.META_GIVEN)
        assert info.as_dict() == want.read().as_dict()
        # header (216 bytes used, the rest is never written) and records; the lists by their counts
        assert torch.equal(plan.buf[:216], want.buf[:216])
        assert torch.equal(plan.buf[256:256 + 48 * nseg], want.buf[256:256 + 48 * nseg])
        cap = (nseg + 4) & ~3
        pfx = 256 + 6 * 48 * cap
        for which in range(4):
            a = pfx + 4 * which * (cap + 4)
            assert torch.equal(plan.buf[a:a + 4 * (nseg + 1)], want.buf[a:a + 4 * (nseg + 1)])
        words = plan.buf.cpu().numpy()[pfx:].view(np.int32)
        blocks = -(-(np.stack([M, N, K])[order[i][1]]) // 128)     # blocks of 128 columns
        assert np.array_equal(words[3 * (cap + 4):][:nseg + 1], np.concatenate([[0], np.cumsum(blocks)]))
    for got, ref in zip(given_lists + given_acc, lists + acc):
        assert torch.equal(got, ref)
