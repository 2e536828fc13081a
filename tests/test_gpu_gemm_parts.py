"""Tiles of the first GEMM that several workgroups share along K: one or two tiles more per XCD than a whole number per CU, with
room for their sums, with exactly enough and with a row too little. The bits are those of the launch that shares none. fp8
shares none whatever memory it is given: its sums depend on their order."""
import pytest
import torch

from memfabric_hybrid_amd import capi
from memfabric_hybrid_amd.operators import OperatorBuffer
from test_gpu_gemm import row_off_dev
from zbal_testlib import rng

pytestmark = pytest.mark.gpu

WORDS, PARTS = 512, 4


@pytest.fixture(scope="module")
def buf():
    b = OperatorBuffer()
    yield b
    torch.cuda.synchronize()
    b.close()


# K: nine and ten chunks of four slabs, which four parts cannot have alike
@pytest.mark.parametrize("mode", [1, 2])
@pytest.mark.parametrize("K,rest,rows,room", [(4608, 1, 13, 64), (4608, 1, 16, 16), (4608, 1, 17, 16), (5120, 2, 1, 40), (5120, 2, 35, 35)])
def test_tiles_shared_along_k(buf, mode, K, rest, rows, room):
    cus = torch.cuda.get_device_properties(0).multi_processor_count // 8
    E, N = cus + rest, 2048                                    # eight columns per expert: one per XCD
    counts = rng(K + rest).integers(1, 20, E)
    counts[cus:] = rows
    counts[cus - 1] = 30
    R, I = int(counts.sum()), N // 2
    g = torch.Generator(device="cuda").manual_seed(rest)
    w = torch.randint(-128, 128, (E, N, K), dtype=torch.int8, device="cuda", generator=g)      # any bytes are a pre-packed weight
    a = torch.randint(-127, 128, (R, K), dtype=torch.int8, device="cuda", generator=g)
    if mode == 1:
        xs = torch.rand((R,), device="cuda", generator=g) * 0.05 + 0.005
        ws = torch.rand((E, N), device="cuda", generator=g) * 0.003 + 0.0015
    else:
        a, w = a & 0x7e ^ (a & -128), w & 0x7e ^ (w & -128)                                  # no NaN
        xs = torch.rand((R, K // 128), device="cuda", generator=g) * 2e-4 + 1e-4
        ws = torch.rand((E, K // 128, N // 128), device="cuda", generator=g) * 2e-4 + 1e-4
    off = row_off_dev(counts)
    sgl = torch.empty((R * (I + 1),), device="cuda")
    scratch = torch.full((WORDS + 8 * rest * PARTS * room * 256,), float("nan"), device="cuda")

    def run(parts):
        q2 = torch.empty((R, I), dtype=torch.uint8, device="cuda")
        s2 = torch.empty((R,) if mode == 1 else (R, N // 256), device="cuda")
        scratch[:WORDS].view(torch.int32).zero_()
        capi.check("gmm1", buf.lib.zbalhip_gmm1_swiglu_quant_parts(
            a.data_ptr(), xs.data_ptr(), w.data_ptr(), ws.data_ptr(), off.data_ptr(), E, R, K, N, mode, q2.data_ptr(), s2.data_ptr(),
            sgl.data_ptr(), None, scratch.data_ptr() if parts else None, scratch.numel() * 4 if parts else 0, capi.stream_ptr()))
        return q2, s2, int((scratch[:WORDS].view(torch.int32) == PARTS).sum()) if parts else 0

    want_q2, want_s2, _ = run(False)
    for _ in range(2):
        got_q2, got_s2, shared = run(True)
        assert shared == (8 * rest if mode == 1 and rows <= room else 0)
        assert torch.equal(got_q2, want_q2) and torch.equal(got_s2, want_s2)
