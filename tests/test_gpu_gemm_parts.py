"""Tiles of the first GEMM that several workgroups share along K: one or two tiles more per XCD than a whole number per CU, with
room for their sums, with exactly enough and with a row too little. The bits are those of the launch that shares none. fp8
shares none whatever memory it is given: its sums depend on their order."""
import ctypes

import pytest
import torch

from memfabric_hybrid_amd import capi
from memfabric_hybrid_amd.operators import OperatorBuffer
from test_gpu_gemm import row_off_dev
from test_gpu_shared_expert import SharedExpert
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


def tiles_of(rows, tall):
    """Heights of an expert's row tiles, as the kernel cuts them."""
    tm = 96 if tall else 64
    n = -(-rows // tm)
    height = (-(-rows // max(n, 1)) + 15) & ~15
    return [min(height, rows - i * height) for i in range(n)]


def rows_shared(K, rest):
    """Rows up to which `rest` tiles are shared (shared_rows beside the kernel)."""
    return 0 if rest > 10 else (K // 128 - 24) * (11 - rest) // 4


# The last experts' rows and the room for a shared tile's. Workgroups per tile: four up to 8 tiles over, three of 9 and 10, none beyond.
# All tiles are shared or none: heights on either side of the line, of the room, and one of them too tall; an expert of two row tiles; a
# shared expert (the first tile of all); `tall`: 48 rows per expert and more on average, the tile of 96 rows and two slabs in flight.
@pytest.mark.parametrize("K,last,room,tall,shared", [
    (4608, [3] * 8, 64, False, 0), (4608, [9] * 8, 64, False, 0), (4608, [9] * 7 + [10], 64, False, 0), (5120, list(range(8)) + [8, 8], 8, False, 20),
    (7168, [8] * 9 + [1], 24, False, 0), (7168, [9] * 10, 64, False, 0), (14336, [1] * 11, 64, False, 0), (4608, [1, 2], 1, False, 0),
    (4608, [30], 30, False, 64), (4608, [31], 64, False, 64), (7168, [1, 64], 64, False, 64), (7168, [1, 64, 33], 48, False, 0),
    (7168, [100], 64, False, 0), (14336, [5, 64] * 4, 64, False, 17),
    (7168, [80], 80, True, 0), (7168, [81], 96, True, 0), (7168, [40, 96, 1], 96, True, 70), (14336, [96, 3, 95] * 2, 96, True, 96),
    (14336, [20] * 9, 20, True, 0), (14336, [130, 20], 80, True, 0), (14336, [130, 20], 79, True, 0)])
def test_numbers_of_parts_and_heights_of_tiles(buf, K, last, room, tall, shared):
    heights = [h for rows in last for h in tiles_of(rows, tall)]
    rest, N = len(heights), 2048
    cus = torch.cuda.get_device_properties(0).multi_processor_count // 8
    first = cus - (1 if shared else 0)
    counts = rng(K + rest).integers(60, 97, first) if tall else rng(K + rest).integers(1, 20, first)
    counts = [int(c) for c in counts] + last
    E, R, I = len(counts), sum(counts), N // 2
    parts = min(4, cus // rest) if max(heights) <= min(room, rows_shared(K, rest)) else 0
    assert (R + shared > 48 * (E + bool(shared))) == tall and R + shared <= 87 * E
    g = torch.Generator(device="cuda").manual_seed(rest)
    w = torch.randint(-128, 128, (E + 1, N, K), dtype=torch.int8, device="cuda", generator=g)
    a = torch.randint(-127, 128, (R + shared, K), dtype=torch.int8, device="cuda", generator=g)
    xs = torch.rand((R + shared,), device="cuda", generator=g) * 0.05 + 0.005
    ws = torch.rand((E + 1, N), device="cuda", generator=g) * 0.003 + 0.0015
    off = row_off_dev(counts + [shared])
    along = SharedExpert(w[E].data_ptr(), ws[E].data_ptr(), shared, None)
    scratch = torch.full((WORDS + 8 * rest * min(4, cus // rest) * room * 256,), float("nan"), device="cuda")

    def run(share):
        q2, s2 = torch.zeros((R + shared, I), dtype=torch.int8, device="cuda"), torch.zeros((R + shared,), device="cuda")
        sgl = torch.empty(((R + shared) * (I + 1),), device="cuda")
        scratch[:WORDS].view(torch.int32).zero_()
        capi.check("gmm1", buf.lib.zbalhip_gmm1_swiglu_quant_parts(
            a.data_ptr(), xs.data_ptr(), w.data_ptr(), ws.data_ptr(), off.data_ptr(), E, R, K, N, 1, q2.data_ptr(), s2.data_ptr(), sgl.data_ptr(),
            ctypes.byref(along) if shared else None, scratch.data_ptr() if share else None, scratch.numel() * 4 if share else 0,
            capi.stream_ptr()))
        return q2, s2, scratch[:WORDS].view(torch.int32).clone()

    want_q2, want_s2, _ = run(False)
    assert int((want_q2 != 0).any(dim=1).sum()) == R + shared
    for _ in range(2):
        got_q2, got_s2, arrived = run(True)
        assert arrived.tolist() == ([parts] * rest + [0] * (cus - rest)) * 8 + [0] * (WORDS - 8 * cus)
        assert torch.equal(got_q2, want_q2) and torch.equal(got_s2, want_s2)
