"""The second GEMM of the int modes from the first one's fp32 values: the same bits as from the bytes that the requantisation
launch makes of them, which the oracle pins elsewhere. Rows at the edges of its tiles (32 rows, 16 where two workgroups share a
tile), K of one group of slabs and of several, rows of zeros, and what the C ABI refuses."""
import numpy as np
import pytest
import torch

from memfabric_hybrid_amd import capi
from memfabric_hybrid_amd.operators import OperatorBuffer
from test_gpu_gemm import row_off_dev
from zbal_testlib import rng

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def buf():
    b = OperatorBuffer()
    yield b
    torch.cuda.synchronize()
    b.close()


def second(buf, mode, a, scale, w, ws, ws_dt, off, E, R, K, N, dt):
    y = torch.full((R, N), 7.0, dtype=torch.bfloat16 if dt == capi.DT_BF16 else torch.float16, device="cuda")
    capi.check("gmm2", buf.lib.zbalhip_gmm2_dequant(a.data_ptr(), scale.data_ptr(), w.data_ptr(), ws.data_ptr(), ws_dt, off.data_ptr(), E, R, K,
                                                    N, mode, dt, y.data_ptr(), capi.stream_ptr()))
    return y.view(torch.int16)


# edges of 16 and 32 rows; one or two rows, whose tiles two workgroups share; K: one group of slabs (up to 16 or 32), two, five
@pytest.mark.parametrize("counts", [[1, 16, 17, 31, 32, 33, 64, 65, 0, 5], [0, 1, 0, 1], [2], [3, 0, 16]], ids=str)
@pytest.mark.parametrize("K,N", [(512, 512), (1536, 768), (2048, 256), (4608, 512), (8704, 256)])
@pytest.mark.parametrize("mode,dt", [(1, capi.DT_BF16), (3, capi.DT_BF16), (1, capi.DT_FP16), (3, capi.DT_FP16)])
def test_second_gemm_from_values(buf, mode, dt, counts, K, N):
    E, R = len(counts), sum(counts)
    g = torch.Generator(device="cuda").manual_seed(K + R)
    k1, n1 = 512, 2 * K                                         # a first GEMM that makes K values of a row
    a = torch.randint(-127, 128, (R, k1), dtype=torch.int8, device="cuda", generator=g)
    a[R // 2] = 0                                               # a row of zeros: maximum 0
    xs = torch.rand((R,), device="cuda", generator=g) * 0.05 + 0.005
    shape = (lambda k, n: (E, n * k // 2)) if mode == 3 else (lambda k, n: (E, n * k))
    w1, w2 = (torch.randint(-128, 128, shape(k, n), dtype=torch.int8, device="cuda", generator=g) for k, n in ((k1, n1), (K, N)))
    if mode == 1:
        s1 = torch.rand((E, n1), device="cuda", generator=g) * 0.003 + 0.0015
        s2, s2_dt = (torch.rand((E, N), device="cuda", generator=g) * 0.003).to(torch.bfloat16), capi.DT_BF16
    else:
        s1, s2 = ((torch.rand((E, k // 128, n), device="cuda", generator=g) * 0.01).to(torch.float16) for k, n in ((k1, n1), (K, N)))
        s2_dt = capi.DT_FP16
    off = row_off_dev(np.array(counts, dtype=np.int64))

    def first(flag):
        q2, scale2, sgl = torch.zeros((R, K), dtype=torch.int8, device="cuda"), torch.zeros((R,), device="cuda"), torch.zeros((R * (K + 1),), device="cuda")
        capi.check("gmm1", buf.lib.zbalhip_gmm1_swiglu_quant(a.data_ptr(), xs.data_ptr(), w1.data_ptr(), s1.data_ptr(), off.data_ptr(), E, R, k1, n1,
                                                             mode | flag, q2.data_ptr(), scale2.data_ptr(), sgl.data_ptr(), capi.stream_ptr()))
        return q2, scale2, sgl

    q2, scale2, _ = first(0)
    none, no_scale, sgl = first(capi.SWIGLU_VALUES)
    assert not none.any() and not no_scale.any()
    want = second(buf, mode, q2, scale2, w2, s2, s2_dt, off, E, R, K, N, dt)
    got = second(buf, mode | capi.SWIGLU_VALUES, sgl, sgl[R * K:], w2, s2, s2_dt, off, E, R, K, N, dt)
    assert torch.equal(got, want)


def test_values_are_for_the_int_modes_and_whole_chunks(buf):
    t = torch.zeros((1 << 16,), device="cuda")
    p, off = t.data_ptr(), row_off_dev(np.array([4]))
    gmm2 = lambda k, mode: buf.lib.zbalhip_gmm2_dequant(p, p, p, p, capi.DT_FP32, off.data_ptr(), 1, 4, k, 256, mode | capi.SWIGLU_VALUES,
                                                        capi.DT_BF16, p, capi.stream_ptr())
    assert gmm2(512, 2) == gmm2(640, 1) == gmm2(640, 3) == -2
    assert buf.lib.zbalhip_gmm1_swiglu_quant(p, p, p, p, off.data_ptr(), 1, 4, 512, 256, 2 | capi.SWIGLU_VALUES, p, p, p, capi.stream_ptr()) == -2
    takes = buf.lib.zbalhip_gmm2_takes_values
    assert takes(32, 80, 2048, 1) and takes(32, 80, 2048, 3)
    assert not takes(32, 81, 2048, 1) and not takes(32, 80, 2048, 2) and not takes(32, 8, 640, 1)
