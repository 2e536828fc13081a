"""The permute kernel that works the layout out itself: numbers of picks that are no whole number of its four-pick loads, fewer and more
than a workgroup takes at a time, either side of where it brings more threads than a row has pieces, ids at any 4-byte address;
and int8 bytes of rows with infinities and NaN."""
import numpy as np
import pytest
import torch

from memfabric_hybrid_amd import capi
from oracle import oracle as zo
from zbal_testlib import bf16_normal, dev, host, rng

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def lib():
    return capi.load()


def dispatch(lib, x, ids, is64, T, H, K, E, quant):
    """zbalhip_dispatch_low_latency: rows, scales, expand_idx, counts, running sums"""
    ex = torch.zeros((T * K, H), dtype=torch.int16 if quant == 0 else torch.int8, device="cuda")
    sc, eidx = torch.zeros((T * K,), device="cuda"), torch.full((T, K), -9, dtype=torch.int32, device="cuda")
    nums, sums = torch.zeros((E,), dtype=torch.int64, device="cuda"), torch.zeros((E,), dtype=torch.int32, device="cuda")
    scratch = torch.zeros((50 * E,), dtype=torch.int32, device="cuda")
    flag = quant | (0x400 if is64 else 0)                        # ZBALHIP_IDS_ARE_I64
    capi.check("dispatch", lib.zbalhip_dispatch_low_latency(
        x.data_ptr(), capi.DT_BF16, ids, T, H, K, E, flag, 1, ex.data_ptr(), sc.data_ptr(), eidx.data_ptr(), nums.data_ptr(), sums.data_ptr(),
        scratch.data_ptr(), 50, capi.stream_ptr()))
    return ex, sc, eidx, nums, sums


@pytest.mark.parametrize("T,K", [(1, 1), (1, 3), (5, 1), (73, 7), (128, 4), (171, 3), (257, 1), (341, 3), (585, 7), (1365, 3), (512, 8), (4096, 1)])
@pytest.mark.parametrize("H", [32, 2048, 7168])
@pytest.mark.parametrize("npdt", [np.int32, np.int64])
def test_rows_of_any_number_of_picks(lib, T, K, H, npdt):
    E = 37
    idx = rng(T * K + H).integers(-1, E + 1, size=(T, K)).astype(npdt)
    x = bf16_normal((T, H), T)
    # one element into an allocation: 4-byte (int32) or 8-byte (int64) alignment, nothing behind the last id but the end
    held = torch.zeros((T * K + 1,), dtype=torch.int64 if npdt == np.int64 else torch.int32, device="cuda")
    held[1:] = dev(idx.ravel())
    for quant in (0, 1):
        got = dispatch(lib, dev(x), held[1:].data_ptr(), npdt == np.int64, T, H, K, E, quant)
        want = zo.dispatch_low_latency(x, zo.DT_BF16, idx.astype(np.int32), E, quant, T * K)
        rows = int(want[4][-1])
        assert np.array_equal(host(got[2]), want[2]) and np.array_equal(host(got[3]), want[3]) and np.array_equal(host(got[4]), want[4])
        assert np.array_equal(host(got[0])[:rows].view(want[0].dtype), want[0][:rows])
        if quant:
            assert np.array_equal(host(got[1])[:rows].view(np.uint32), want[1][:rows].view(np.uint32))


def test_bytes_of_infinities_and_nan(lib):
    """A NaN quotient is -128; an infinity makes the scale of its row 0, and 0 times an infinity is one."""
    T, H, E = 4, 512, 4
    x = torch.randn((T, H), device="cuda").to(torch.bfloat16)
    x[0, 7], x[1, 300], x[2, 5], x[2, 6] = float("nan"), float("inf"), float("-inf"), float("nan")
    ids = torch.arange(T, dtype=torch.int32, device="cuda").reshape(T, 1)
    ex, sc, _, _, _ = dispatch(lib, x, ids.data_ptr(), False, T, H, 1, E, 1)
    q, v = host(ex), x.float().cpu().numpy()
    for t in range(T):
        amax = np.float32(np.nanmax(np.abs(v[t])))
        with np.errstate(all="ignore"):
            p = v[t] * (np.float32(127.0) / amax)
        want = np.where(np.isnan(p), -128, np.clip(np.rint(p), -128, 127)).astype(np.int8)
        assert np.array_equal(q[t], want), t
