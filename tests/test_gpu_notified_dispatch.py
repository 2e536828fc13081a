"""Notify and dispatch in one launch against the two launches: the same rows, scales, offsets and counts, for expert counts
around one and several per lane of the wave that sums them, from one token on, with and without the host's read-back."""
import ctypes

import numpy as np
import pytest
import torch

from memfabric_hybrid_amd import capi
from memfabric_hybrid_amd.operators import OperatorBuffer
from zbal_testlib import dev, host, rng

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def buf():
    b = OperatorBuffer()
    yield b
    torch.cuda.synchronize()
    b.close()


@pytest.mark.parametrize("qm", [capi.NO_QUANT, capi.QUANT_INT8, capi.QUANT_FP8_B128])
@pytest.mark.parametrize("T,K,E", [(1, 1, 1), (1, 2, 64), (37, 8, 65), (600, 6, 200), (300, 70, 1024), (1100, 8, 32)])
def test_notified_dispatch(buf, qm, T, K, E):
    H = 256
    x = dev(rng(1).standard_normal((T, H)).astype(np.float32)).to(torch.bfloat16)
    ids = rng(2).integers(0, E, (T, K)).astype(np.int64)
    ids[rng(3).random((T, K)) < 0.1] = -1
    idx = dev(ids)
    _, _, per_expert, _, _ = buf.get_dispatch_layout(idx, E)
    note = buf.notify(per_expert, K)
    want, want_scales, counts, _ = buf.dispatch(x, idx, None, per_expert, quant_mode=qm, notified=note)
    total = int(counts.sum())
    assert total == int((ids >= 0).sum())
    for worst in (0, T * K, max(total // 2, 1)):          # read back; all rows; rows past the receive tensor's end are dropped
        recv, scales, received, put_offset, balance = buf.dispatch_counts(x, idx, per_expert, qm, worst, False)
        rows = min(total, worst) if worst else total
        assert received == ([] if worst else host(counts).tolist())
        assert recv.shape[0] == (worst or max(total, 1))
        assert torch.equal(recv[:rows].view(torch.uint8), want[:rows].view(torch.uint8))
        if qm != capi.NO_QUANT:
            assert torch.equal(scales[:rows], want_scales[:rows])
        assert torch.equal(put_offset, note["put_offset"]) and torch.equal(balance, note["balance_matrix"])
