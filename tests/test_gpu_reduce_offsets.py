"""The reduction in one launch: leading and trailing elements around the vectors, inputs at any offset from a 16-byte
boundary, lengths around a vector and a workgroup, and the layout of large outputs."""
import ctypes

import numpy as np
import pytest
import torch

from memfabric_hybrid_amd import capi
from oracle import oracle as zo
from zbal_testlib import rng

pytestmark = pytest.mark.gpu

TYPES = {capi.DT_INT8: (np.int8, 1), capi.DT_FP16: (np.uint16, 2), capi.DT_BF16: (np.uint16, 2), capi.DT_FP32: (np.float32, 4),
         capi.DT_INT64: (np.int64, 8)}


def reduce(ins, count, dt, op, out):
    arr = (ctypes.c_void_p * len(ins))(*ins)
    return capi.load().zbalhip_reduce(arr, len(ins), count, dt, op, out, 0, None, 0, capi.stream_ptr())


@pytest.mark.parametrize("dt", sorted(TYPES))
@pytest.mark.parametrize("n_in,in_off,out_off", [(3, (0, 1, 2), 0), (8, (1, 1, 1, 1, 1, 1, 1, 1), 0), (2, (0, 0), 1), (4, (1, 1, 1, 1), 1),
                                                 (16, tuple(range(16)), 3)])
def test_offsets_and_lengths(dt, n_in, in_off, out_off):
    npdt, size = TYPES[dt]
    for count in (1, 2, 15, 16, 17, 255 * 16 + 3, 4096 + 5, 100003):
        if npdt == np.uint16:
            conv = zo.f32_to_fp16 if dt == capi.DT_FP16 else zo.f32_to_bf16
            data = [conv(rng(p).standard_normal(count).astype(np.float32)) for p in range(n_in)]
        elif npdt == np.float32:
            data = [rng(p).standard_normal(count).astype(np.float32) for p in range(n_in)]
        else:
            data = [rng(p).integers(-100, 100, count).astype(npdt) for p in range(n_in)]
        bufs = []
        for d, off in zip(data, in_off):
            b = torch.zeros((count + 64) * size, dtype=torch.uint8, device="cuda")
            b[off * size:(off + count) * size] = torch.from_numpy(d.view(np.uint8).copy()).cuda()
            bufs.append(b)
        out = torch.full(((count + 64) * size,), 0x5a, dtype=torch.uint8, device="cuda")
        assert reduce([b.data_ptr() + o * size for b, o in zip(bufs, in_off)], count, dt, capi.REDUCE_SUM, out.data_ptr() + out_off * size) == 0
        got = out.cpu().numpy()
        want = zo.reduce(data, dt, capi.REDUCE_SUM)
        assert np.array_equal(got[out_off * size:(out_off + count) * size], want.view(np.uint8)), (count, in_off)
        assert (got[:out_off * size] == 0x5a).all() and (got[(out_off + count) * size:] == 0x5a).all()


@pytest.mark.parametrize("count", [(64 << 20) - 8, (64 << 20), (64 << 20) + 8 * 1024 * 33 + 5])
def test_large_outputs_cover_every_element(count):
    ins = [torch.randint(-1000, 1000, (count,), device="cuda", dtype=torch.int16) for _ in range(2)]
    out = torch.zeros((count,), device="cuda", dtype=torch.int16)
    assert reduce([t.data_ptr() for t in ins], count, capi.DT_INT16, capi.REDUCE_SUM, out.data_ptr()) == 0
    assert torch.equal(out, ins[0] + ins[1])
