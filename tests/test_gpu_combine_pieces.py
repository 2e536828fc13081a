"""The combine where a token's row goes to one, two, four or eight workgroups: numbers of tokens on either side of each line, rows that the
pieces do not share evenly."""
import numpy as np
import pytest
import torch

from memfabric_hybrid_amd import capi
from oracle import oracle as zo
from zbal_testlib import bf16_normal, dev, host, rng

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("T", [127, 128, 255, 256, 511, 512, 1023, 1024])
@pytest.mark.parametrize("H", [2040, 4096, 7176])
def test_rows_in_pieces(T, H):
    import ctypes
    K, E, lib = 3, 16, capi.load()
    idx = rng(T + H).integers(-1, E, size=(T, K)).astype(np.int64)
    _, counts, send = zo.dispatch_layout(idx, E, 1)
    base = (np.cumsum(counts) - counts).astype(np.int32)
    y, w = bf16_normal((T * K, H), T), rng(T).random((T, K), dtype=np.float32)
    d = [dev(a) for a in (y, base, w, idx.astype(np.int32), send)]
    out = torch.zeros((T, H), dtype=torch.int16, device="cuda")
    windows = (ctypes.c_void_p * 1)(d[0].data_ptr())
    capi.check("combine", lib.zbalhip_combine(windows, 1, 0, T * K, capi.DT_BF16, d[1].data_ptr(), 0, d[2].data_ptr(), d[3].data_ptr(),
                                              d[4].data_ptr(), T, H, K, E, out.data_ptr(), capi.stream_ptr()))
    assert np.array_equal(host(out).view(np.uint16), zo.combine(y, zo.DT_BF16, base, w, idx.astype(np.int32), send, E))
