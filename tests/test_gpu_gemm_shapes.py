"""Every shape the grouped GEMMs choose by rows per expert, with row counts at the edges of its tiles (sub-tiles of 16
rows, one or two row groups of waves, one tile more), against the oracle. The K loops run at their shortest (as many
slabs as the pipeline has stages ahead) and longer."""
import numpy as np
import pytest
import torch

from memfabric_hybrid_amd import capi
from memfabric_hybrid_amd.operators import OperatorBuffer
from oracle import oracle as zo
from test_gpu_gemm import assert_requant_close, fp8_operands, gmm1, gmm2
from zbal_testlib import FP8_GEMM_ELEM_TOL, assert_fp8_close, dev, host, rng

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def buf():
    b = OperatorBuffer()
    yield b
    torch.cuda.synchronize()
    b.close()


# rows per expert on average: the classes of W4A8 end at 48, 100, 160, 224 and 640, those of the 8-bit modes at 8, 84-100
EDGES = {"few": [0, 1, 15, 16, 17, 2, 8, 5, 0, 3], "64": [1, 0, 16, 31, 33, 63, 64, 65, 80, 127],
         "100": [0, 96, 97, 127, 128, 129, 112, 64, 1, 200], "160": [191, 192, 193, 176, 177, 0, 30, 160, 161, 256],
         "47": [47, 48, 49, 33, 32, 31, 0, 17, 64, 1], "53": [63, 64, 65, 49, 48, 128, 50, 0, 20, 33],
         "sparse": [0] * 63 + [5, 70] + [0] * 66 + [16, 1] + [0] * 60 + [33, 2], "1000": [1000, 769, 96, 97, 1151, 1153, 767, 800, 0, 700],
         "900": [128, 129, 127, 112, 113, 1024, 1025, 3001, 2945, 1], "224": [128, 129, 256, 257, 192, 255, 0, 144, 300, 250], "640": [384, 385, 192, 577, 1, 0, 600, 383, 500, 191]}


# whole chunks of the streaming kernel's slabs, channel tiles in eighths and not
STREAM_SHAPES = [(512, 512), (1024, 2304), (1536, 768)]


@pytest.mark.parametrize("edges", sorted(EDGES))
@pytest.mark.parametrize("K,N", [(256, 512), (384, 256), (640, 1280)] + STREAM_SHAPES)
def test_w4a8_shapes_bit_exact(buf, edges, K, N):
    counts = np.array(EDGES[edges], dtype=np.int64)
    E, rows = len(counts), int(counts.sum())
    a = rng(1).integers(-128, 128, (rows, K)).astype(np.int8)
    a[:3] = -128                                    # with -8 below: the largest sums a scale group can have
    xs = rng(2).uniform(0.005, 0.05, rows).astype(np.float32)
    w = rng(3).integers(-8, 8, (E, K, N)).astype(np.int8)
    w[:, :, :40] = -8
    gs = rng(4).uniform(0.001, 0.01, (E, K // 128, N)).astype(np.float16).view(np.uint16)
    packed = buf.prepack_weight(dev(w), int4=True)
    assert np.array_equal(host(gmm2(buf, dev(a), dev(xs), packed, dev(gs), capi.DT_FP16, counts, K, N, 3)),
                          zo.gmm2_w4a8(a, xs, w, gs, counts))
    q2, s2, _ = gmm1(buf, dev(a), dev(xs), packed, dev(gs), counts, K, N, 3)
    r_q2, r_s2, _ = zo.gmm1_swiglu_quant_w4a8(a, xs, w, gs, counts)
    assert np.array_equal(host(s2).view(np.uint32), r_s2.view(np.uint32)) and np.array_equal(host(q2), r_q2)


@pytest.mark.parametrize("edges", ["few", "47", "53", "64", "100", "160", "sparse"])
@pytest.mark.parametrize("K,N", [(256, 512), (640, 1280)] + STREAM_SHAPES)
def test_8_bit_shapes(buf, edges, K, N):
    counts = np.array(EDGES[edges], dtype=np.int64)
    E, rows = len(counts), int(counts.sum())
    a = rng(1).integers(-127, 128, (rows, K)).astype(np.int8)
    xs = rng(2).uniform(0.005, 0.05, rows).astype(np.float32)
    w = rng(3).integers(-128, 128, (E, K, N)).astype(np.int8)
    ws = rng(4).uniform(0.0015, 0.0045, (E, N)).astype(np.float32)
    packed = buf.prepack_weight(dev(w))
    assert np.array_equal(host(gmm2(buf, dev(a), dev(xs), packed, dev(ws), capi.DT_FP32, counts, K, N, 1)),
                          zo.grouped_gemm_w8a8_dequant(a, xs, w, ws, counts))
    q2, s2, _ = gmm1(buf, dev(a), dev(xs), packed, dev(ws), counts, K, N, 1)
    r_q2, r_s2 = zo.gmm1_swiglu_quant_w8a8(a, xs, w, ws, counts)[:2]
    assert np.array_equal(host(s2).view(np.uint32), r_s2.view(np.uint32)) and np.array_equal(host(q2), r_q2)

    a, sa, w, sw = fp8_operands(E, K, N, rows, 20)
    packed = buf.prepack_weight(dev(w))
    y = gmm2(buf, dev(a), dev(sa), packed, dev(sw), capi.DT_FP32, counts, K, N, 2)
    assert_fp8_close(zo.bf16_to_f32(host(y)), zo.bf16_to_f32(zo.gmm2_fp8(a, sa, w, sw, counts)), "fp8 GEMM", FP8_GEMM_ELEM_TOL)
    q2, s2, _ = gmm1(buf, dev(a), dev(sa), packed, dev(sw), counts, K, N, 2)
    r_q2, r_s2, _ = zo.gmm1_swiglu_quant_fp8(a, sa, w, sw, counts)
    blocks = (rows, N // 256, 128)
    assert np.allclose(host(s2), r_s2, rtol=1e-4)
    assert_requant_close(zo.e4m3_to_f32(host(q2)).reshape(blocks) * host(s2)[:, :, None],
                         zo.e4m3_to_f32(r_q2).reshape(blocks) * r_s2[:, :, None], host(q2), r_q2)


# averages either side of the lines that `stream_rows` draws by K and rows per expert; the second GEMM runs with the shorter K too
LINES = [(2560, 87), (2560, 88), (2560, 108), (2560, 109), (2560, 112), (2560, 113), (2560, 160), (2560, 184), (2560, 185), (8704, 150),
         (8704, 151), (8704, 192), (8704, 193), (8704, 352), (8704, 353), (1024, 520), (1024, 521)]


@pytest.mark.parametrize("K,avg", LINES)
def test_8_bit_lines_of_the_dispatch(buf, K, avg):
    N, counts = 512, np.array([avg - 40, avg + 40, 2 * avg, 0], dtype=np.int64)
    E, rows = len(counts), int(counts.sum())
    assert rows == avg * E
    a = rng(1).integers(-127, 128, (rows, K)).astype(np.int8)
    xs = rng(2).uniform(0.005, 0.05, rows).astype(np.float32)
    w = rng(3).integers(-128, 128, (E, K, N)).astype(np.int8)
    ws = rng(4).uniform(0.0015, 0.0045, (E, N)).astype(np.float32)
    packed = buf.prepack_weight(dev(w))
    q2, s2, _ = gmm1(buf, dev(a), dev(xs), packed, dev(ws), counts, K, N, 1)
    r_q2, r_s2 = zo.gmm1_swiglu_quant_w8a8(a, xs, w, ws, counts)[:2]
    assert np.array_equal(host(s2).view(np.uint32), r_s2.view(np.uint32)) and np.array_equal(host(q2), r_q2)

    a, sa, w, sw = fp8_operands(E, K, N, rows, 20)
    packed = buf.prepack_weight(dev(w))
    y = gmm2(buf, dev(a), dev(sa), packed, dev(sw), capi.DT_FP32, counts, K, N, 2)
    assert_fp8_close(zo.bf16_to_f32(host(y)), zo.bf16_to_f32(zo.gmm2_fp8(a, sa, w, sw, counts)), "fp8 GEMM", FP8_GEMM_ELEM_TOL)
    q2, s2, _ = gmm1(buf, dev(a), dev(sa), packed, dev(sw), counts, K, N, 2)
    r_q2, r_s2, _ = zo.gmm1_swiglu_quant_fp8(a, sa, w, sw, counts)
    blocks = (rows, N // 256, 128)
    assert np.allclose(host(s2), r_s2, rtol=1e-4)
    assert_requant_close(zo.e4m3_to_f32(host(q2)).reshape(blocks) * host(s2)[:, :, None],
                         zo.e4m3_to_f32(r_q2).reshape(blocks) * r_s2[:, :, None], host(q2), r_q2)


@pytest.mark.parametrize("avg", [192, 193])
def test_many_tiles_are_the_same_rows_as_few(buf, avg):
    """1024 experts of four channel tiles are many tiles, 64 are not: the second GEMM gives the same bits either way."""
    K, N, E, part = 512, 1024, 1024, 64
    counts = rng(5).multinomial(avg * part, np.full(part, 1.0 / part), size=E // part).reshape(-1).astype(np.int64)
    rows = int(counts.sum())
    a = torch.randint(-127, 128, (rows, K), dtype=torch.int8, device="cuda")
    xs = torch.rand((rows,), device="cuda") + 0.5
    w = torch.randint(-128, 128, (E, N, K), dtype=torch.int8, device="cuda")         # any bytes are a pre-packed weight
    ws = torch.rand((E, N), device="cuda") + 0.5
    whole = gmm2(buf, a, xs, w, ws, capi.DT_FP32, counts, K, N, 1)
    off = np.concatenate([[0], np.cumsum(counts)])
    for e in range(0, E, part):
        r = slice(int(off[e]), int(off[e + part]))
        got = gmm2(buf, a[r].contiguous(), xs[r].contiguous(), w[e:e + part], ws[e:e + part], capi.DT_FP32, counts[e:e + part], K, N, 1)
        assert torch.equal(whole[r].view(torch.int16), got.view(torch.int16))


# either side of 112 rows per expert, of the tiles that all but fill the chip twice (up to 640 rows) and once; experts whose tiles have
# one to eight sub-tiles of 16 rows, five and six (65 to 96 rows) among them, and none
@pytest.mark.parametrize("E,avg,N", [(64, 112, 4864), (64, 113, 4864), (8, 640, 6144), (8, 640, 6400), (8, 641, 3072), (8, 641, 3328)])
def test_w4a8_lines_of_the_dispatch(buf, E, avg, N):
    """The same bits as expert by expert, where the tiles are of 64 rows."""
    K, rows = 512, avg * E
    edges = [0, 70, 161, 192] if E == 8 else [0, 70, 161, 192, 1, 96, 127, 128]
    counts = np.array(edges + [(rows - sum(edges)) // (E - len(edges))] * (E - len(edges)), dtype=np.int64)
    counts[-1] += rows - counts.sum()
    assert (counts >= 0).all() and counts.max() * (N // 256) < 65536
    a = torch.randint(-128, 128, (rows, K), dtype=torch.int8, device="cuda")
    xs = torch.rand((rows,), device="cuda") + 0.5
    w = torch.randint(-128, 128, (E, N, K // 2), dtype=torch.int8, device="cuda")      # any bytes are a pre-packed weight
    gs = ((torch.rand((E, K // 128, N), device="cuda") + 0.5) * 1e-3).to(torch.float16)
    whole = gmm2(buf, a, xs, w, gs, capi.DT_FP16, counts, K, N, 3)
    q2, s2, _ = gmm1(buf, a, xs, w, gs, counts, K, N, 3)
    off = np.concatenate([[0], np.cumsum(counts)])
    for e in range(E):
        r = slice(int(off[e]), int(off[e + 1]))
        if counts[e] == 0:
            continue
        one = (buf, a[r].contiguous(), xs[r].contiguous(), w[e:e + 1], gs[e:e + 1])
        assert torch.equal(whole[r].view(torch.int16), gmm2(*one, capi.DT_FP16, counts[e:e + 1], K, N, 3).view(torch.int16)), e
        want_q2, want_s2, _ = gmm1(*one, counts[e:e + 1], K, N, 3)
        assert torch.equal(q2[r], want_q2) and torch.equal(s2[r], want_s2), e


@pytest.mark.parametrize("mode", [1, 3])
@pytest.mark.parametrize("spread", [0.2, 30.0, 70.0, 400.0])
@pytest.mark.parametrize("avg", [20, 500])
def test_swiglu_either_side_of_the_short_form(buf, mode, spread, avg):
    """Gate values (standard deviation `spread`) that stay within the short form's 80, straddle it and leave exp()'s range; both kernels."""
    K, N, counts = 512, 512, np.array([avg, 0, avg + 17, avg - 17], dtype=np.int64)
    E, rows = len(counts), int(counts.sum())
    a = rng(1).integers(-127, 128, (rows, K)).astype(np.int8)
    a[5] = 0                                                       # gate and up are 0
    xs = rng(2).uniform(0.5, 1.5, rows).astype(np.float32)
    lo, hi = (-128, 128) if mode == 1 else (-8, 8)
    w = rng(3).integers(lo, hi, (E, K, N)).astype(np.int8)
    per_unit = spread / (73.0 * (hi - lo) * 0.29 * K ** 0.5)
    if mode == 1:
        ws = rng(4).uniform(0.5 * per_unit, 1.5 * per_unit, (E, N)).astype(np.float32)
        want = zo.gmm1_swiglu_quant_w8a8(a, xs, w, ws, counts)[:2]
    else:
        ws = rng(4).uniform(0.5 * per_unit, 1.5 * per_unit, (E, K // 128, N)).astype(np.float16).view(np.uint16)
        want = zo.gmm1_swiglu_quant_w4a8(a, xs, w, ws, counts)[:2]
    q2, s2, _ = gmm1(buf, dev(a), dev(xs), buf.prepack_weight(dev(w), int4=mode == 3), dev(ws), counts, K, N, mode)
    assert np.array_equal(host(s2).view(np.uint32), want[1].view(np.uint32)) and np.array_equal(host(q2), want[0])


@pytest.mark.parametrize("sign", [1.0, -1.0])
def test_swiglu_short_form_over_every_float(buf, sign):
    """Every gate value of at most 80: a dot product of 1 and an up value that is a power of two leave the SwiGLU of channel scale
    times token scale, mantissa times 2^e. The launch is made twice, the second time with an infinity in every sixteenth row, which
    sends its wave to the general form: the same bits, and of the two only the general one keeps the sign of -0."""
    K, I, rows = 128, 1 << 20, 16
    a = torch.zeros((rows, K), dtype=torch.int8, device="cuda")
    a[:, 0] = 1
    w = torch.zeros((1, K, 2 * I), dtype=torch.int8, device="cuda")
    w[:, 0] = 1
    packed = buf.prepack_weight(w)
    # subnormal values, then fifteen exponents at a time
    groups = [(None, [-126] * 15)] + [(e, list(range(e, e + 15))) for e in range(-126, 7, 15)]
    for lowest, exponents in groups:
        xs = torch.tensor([2.0 ** min(e, 6) for e in exponents] + [1.0], dtype=torch.float32, device="cuda")
        far = xs.clone()
        far[-1] = float("inf")
        for m in range(0, 1 << 23, I):
            ws = torch.empty((1, 2 * I), dtype=torch.float32, device="cuda")
            ws[0, :I] = torch.arange(m, m + I, device="cuda", dtype=torch.float32) * 2.0 ** -23 + (0.0 if lowest is None else 1.0)
            ws[0, :I] *= sign
            ws[0, I:] = 2.0 ** -(-126 if lowest is None else lowest)                     # an up value of 1 in the first row
            short, general = [gmm1(buf, a, x, packed, ws, [rows], K, 2 * I, 1)[2][:15 * I].view(torch.int32) for x in (xs, far)]
            if lowest is None and m == 0:
                zeros = slice(0, 15 * I, I)
                assert (short[zeros] == 0).all() and (general[zeros] == (0 if sign > 0 else -2 ** 31)).all()
                general[zeros] = 0
            assert torch.equal(short, general), (lowest, m)


# K slabs of the many-row kernel: scales of four steps in whole groups (4, 8), with two and three steps left over (6, 11), with one,
# which makes the last two groups of three and two (5, 9), and rows of less than one group (2, 3)
@pytest.mark.parametrize("slabs", [2, 3, 4, 5, 6, 8, 9, 11])
@pytest.mark.parametrize("avg", [200, 900])
def test_many_rows_fp8(buf, slabs, avg):
    K, N = 128 * slabs, 768
    counts = np.array([avg + 21, 0, 1, 320, 321, 3 * avg, avg + 60, 257], dtype=np.int64)
    E, rows = len(counts), int(counts.sum())
    counts[0] += max(0, 900 * E - rows) if avg == 900 else max(0, 200 * E - rows)      # more than any line to the kernels for fewer rows
    check_fp8_gemms(buf, counts, K, N, 20 + slabs)


def check_fp8_gemms(buf, counts, K, N, seed):
    E, rows = len(counts), int(counts.sum())
    a, sa, w, sw = fp8_operands(E, K, N, rows, seed)
    packed = buf.prepack_weight(dev(w))
    y = gmm2(buf, dev(a), dev(sa), packed, dev(sw), capi.DT_FP32, counts, K, N, 2)
    assert_fp8_close(zo.bf16_to_f32(host(y)), zo.bf16_to_f32(zo.gmm2_fp8(a, sa, w, sw, counts)), "fp8 GEMM", FP8_GEMM_ELEM_TOL)
    q2, s2, _ = gmm1(buf, dev(a), dev(sa), packed, dev(sw), counts, K, N, 2)
    r_q2, r_s2, _ = zo.gmm1_swiglu_quant_fp8(a, sa, w, sw, counts)
    blocks = (rows, N // 256, 128)
    assert np.allclose(host(s2), r_s2, rtol=1e-4)
    assert_requant_close(zo.e4m3_to_f32(host(q2)).reshape(blocks) * host(s2)[:, :, None],
                         zo.e4m3_to_f32(r_q2).reshape(blocks) * r_s2[:, :, None], host(q2), r_q2)


# weight block scales of 128 steps in turns of tiles, of more than that from where the last tile's were
@pytest.mark.parametrize("slabs", [128, 129, 131, 256])
def test_many_rows_fp8_long_k(buf, slabs):
    K, N, counts = 128 * slabs, 512, np.array([401, 0, 700], dtype=np.int64)
    E, rows = len(counts), int(counts.sum())
    assert rows > 352 * E
    check_fp8_gemms(buf, counts, K, N, 30)


@pytest.mark.parametrize("mode", [1, 2])
def test_many_tiles_per_workgroup_are_the_same_rows(buf, mode):
    """More tiles than a workgroup works out at once (32 of them): the same bits as expert by expert, where it has a few."""
    K, N, E, avg = 512, 16384, 32, 1300
    counts = np.array([avg - 16 * e if e % 2 else avg + 16 * e for e in range(E)], dtype=np.int64)
    rows = int(counts.sum())
    assert (rows // 320) * (N // 256) > 32 * 256
    a = torch.randint(0, 256, (rows, K), dtype=torch.uint8, device="cuda")
    w = torch.randint(0, 256, (E, N, K), dtype=torch.uint8, device="cuda")           # any bytes are a pre-packed weight
    if mode == 2:
        a, w = a & 0x77, w & 0x77                                                    # no NaN codes
        xs, ws = torch.rand((rows, K // 128), device="cuda") + 0.5, torch.rand((E, K // 128, N // 128), device="cuda") + 0.5
    else:
        xs, ws = torch.rand((rows,), device="cuda") + 0.5, torch.rand((E, N), device="cuda") + 0.5
    whole = gmm2(buf, a, xs, w, ws, capi.DT_FP32, counts, K, N, mode)
    off = np.concatenate([[0], np.cumsum(counts)])
    for e in range(E):
        r = slice(int(off[e]), int(off[e + 1]))
        got = gmm2(buf, a[r].contiguous(), xs[r].contiguous(), w[e:e + 1], ws[e:e + 1], capi.DT_FP32, counts[e:e + 1], K, N, mode)
        assert torch.equal(whole[r].view(torch.int16), got.view(torch.int16)), e


@pytest.mark.parametrize("counts", [[1], [16], [0, 17, 1], [0] * 20 + [1] + [0] * 50 + [2, 1] + [0] * 57, [3, 0, 8, 33]])
@pytest.mark.parametrize("K,N", STREAM_SHAPES)
def test_tiles_shared_by_two_workgroups(buf, counts, K, N):
    """A handful of rows: every mode, channel scales of either type, experts without rows and just past a tile's 16."""
    counts = np.array(counts, dtype=np.int64)
    E, rows = len(counts), int(counts.sum())
    a = rng(1).integers(-128, 128, (rows, K)).astype(np.int8)
    xs = rng(2).uniform(0.005, 0.05, rows).astype(np.float32)
    w = rng(3).integers(-128, 128, (E, K, N)).astype(np.int8)
    ws = rng(4).uniform(0.0015, 0.0045, (E, N)).astype(np.float32)
    packed = buf.prepack_weight(dev(w))
    for dt, s in ((capi.DT_FP32, ws), (capi.DT_BF16, zo.f32_to_bf16(ws))):
        assert np.array_equal(host(gmm2(buf, dev(a), dev(xs), packed, dev(s), dt, counts, K, N, 1)),
                              zo.grouped_gemm_w8a8_dequant(a, xs, w, s, counts))
    q2, s2, _ = gmm1(buf, dev(a), dev(xs), packed, dev(ws), counts, K, N, 1)
    r_q2, r_s2 = zo.gmm1_swiglu_quant_w8a8(a, xs, w, ws, counts)[:2]
    assert np.array_equal(host(s2).view(np.uint32), r_s2.view(np.uint32)) and np.array_equal(host(q2), r_q2)

    w = rng(5).integers(-8, 8, (E, K, N)).astype(np.int8)
    gs = rng(6).uniform(0.001, 0.01, (E, K // 128, N)).astype(np.float16).view(np.uint16)
    packed = buf.prepack_weight(dev(w), int4=True)
    assert np.array_equal(host(gmm2(buf, dev(a), dev(xs), packed, dev(gs), capi.DT_FP16, counts, K, N, 3)),
                          zo.gmm2_w4a8(a, xs, w, gs, counts))
    q2, s2, _ = gmm1(buf, dev(a), dev(xs), packed, dev(gs), counts, K, N, 3)
    r_q2, r_s2, _ = zo.gmm1_swiglu_quant_w4a8(a, xs, w, gs, counts)
    assert np.array_equal(host(s2).view(np.uint32), r_s2.view(np.uint32)) and np.array_equal(host(q2), r_q2)

    a, sa, w, sw = fp8_operands(E, K, N, rows, 20)
    y = gmm2(buf, dev(a), dev(sa), buf.prepack_weight(dev(w)), dev(sw), capi.DT_FP32, counts, K, N, 2)
    assert_fp8_close(zo.bf16_to_f32(host(y)), zo.bf16_to_f32(zo.gmm2_fp8(a, sa, w, sw, counts)), "fp8 GEMM", FP8_GEMM_ELEM_TOL)
