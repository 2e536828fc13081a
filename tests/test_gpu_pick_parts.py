"""Small batches, whose tokens' picks several workgroups share: either side of where a token has eight, four, two and one of them, and
numbers of picks that they do not share evenly or that leave some without any."""
import numpy as np
import pytest
import torch

from memfabric_hybrid_amd import capi
from oracle import oracle as zo
from test_gpu_inline_layout import dispatch
from zbal_testlib import bf16_normal, dev, host, rng

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("T", [1, 32, 33, 64, 65, 128, 129])
@pytest.mark.parametrize("K", [1, 3, 8, 11, 31])
@pytest.mark.parametrize("H", [128, 4096, 7168])
@pytest.mark.parametrize("quant", [0, 1])
def test_rows_of_shared_tokens(T, K, H, quant):
    E = 64
    lib = capi.load()
    idx = np.stack([rng(t + K).permutation(E)[:K] for t in range(T)]).astype(np.int32)
    idx[rng(7).random((T, K)) < 0.1] = -1
    x, ids = bf16_normal((T, H), T), dev(idx)
    got = dispatch(lib, dev(x), ids.data_ptr(), False, T, H, K, E, quant)
    want = zo.dispatch_low_latency(x, zo.DT_BF16, idx, E, quant, T * K)
    rows = int(want[4][-1])
    assert all(np.array_equal(host(got[i]), want[i]) for i in (2, 3, 4))
    assert np.array_equal(host(got[0])[:rows].view(want[0].dtype), want[0][:rows])
    if quant:
        assert np.array_equal(host(got[1])[:rows].view(np.uint32), want[1][:rows].view(np.uint32))
    torch.cuda.synchronize()
