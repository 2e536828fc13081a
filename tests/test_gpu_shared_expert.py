"""A shared expert of the routed experts' width runs in their launches: every way the layout is worked out (inside the
permute launch, from range histograms, from a launch of its own), x_active_mask, smooth scales and tensor lists, against
the oracle, which runs it as a one-expert layer; so does every kernel shape that its rows can bring a launch to. A
workspace without room for its rows gives the same results."""
import ctypes

import numpy as np
import pytest
import torch

from memfabric_hybrid_amd import capi
from memfabric_hybrid_amd.operators import OperatorBuffer
from oracle import oracle as zo
from test_gpu_gemm import fp8_operands, fused_inputs, gmm1, gmm2, row_off_dev
from zbal_testlib import dev, host, max_rel_err, rng

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def buf():
    b = OperatorBuffer()
    yield b
    torch.cuda.synchronize()
    b.close()


@pytest.mark.parametrize("mode", [0, 2, 3])
@pytest.mark.parametrize("T,H,K,E,I,active,smooth", [(1, 512, 2, 8, 512, None, False), (70, 512, 4, 8, 512, 37, True),
                                                      (1200, 256, 4, 8, 128, None, False), (1200, 256, 4, 8, 128, 0, True),
                                                      (1100, 256, 4, 8, 128, 1001, True), (600, 256, 8, 300, 128, 555, False)])
def test_shared_expert_in_the_routed_launches(buf, mode, T, H, K, E, I, active, smooth):
    check_shared_expert(buf, mode, T, H, K, E, I, active, smooth)


# the tall tiles of the weight stream (150 rows per expert, the shared one's among them; W4A8's want the chip full: 711 rows), the
# lower W4A8 ones with as many rows, and the many-row kernel with the K of a prefill layer in both GEMMs (480 rows)
@pytest.mark.parametrize("mode,T,H,K,E,I,active,smooth", [(0, 300, 512, 4, 8, 512, None, False), (2, 300, 512, 4, 8, 512, 200, False),
                                                           (3, 300, 512, 4, 8, 512, None, True), (3, 1280, 512, 4, 8, 512, 1200, False),
                                                           (3, 1280, 3072, 4, 8, 1536, 1200, False),
                                                           (0, 800, 7168, 2, 4, 2048, None, False), (2, 800, 7168, 2, 4, 2048, 777, False)])
def test_shared_expert_in_tall_tiles(buf, mode, T, H, K, E, I, active, smooth):
    check_shared_expert(buf, mode, T, H, K, E, I, active, smooth)


@pytest.mark.parametrize("mode", [0, 2, 3])
@pytest.mark.parametrize("T,active,smooth", [(1, None, False), (70, 37, True), (300, None, False), (1200, 1100, False)])
def test_shared_expert_in_the_smallest_workspace(buf, mode, T, active, smooth):
    check_shared_expert(buf, mode, T, 512, 4, 8, 256, active, smooth, smallest=True)


@pytest.mark.parametrize("mode", [0, 2, 3])
@pytest.mark.parametrize("T,active,smooth", [(1, None, False), (70, 37, True), (300, None, False)])
def test_shared_expert_with_tensor_lists(buf, mode, T, active, smooth):
    """The routed experts' operands as lists of tensors, the shared expert's a tensor each."""
    check_shared_expert(buf, mode, T, 512, 4, 8, 512, active, smooth, lists=True)


def check_shared_expert(buf, mode, T, H, K, E, I, active, smooth, lists=False, smallest=False):
    smooth = smooth and mode != 2
    x, ids, es, w1, s1, w2, s2 = fused_inputs(T, H, K, E, I, mode, 200 + mode)
    _, _, _, sw1, ss1, sw2, ss2 = fused_inputs(T, H, 1, 1, I, mode, 210 + mode)
    sm = rng(7).uniform(0.2, 1.0, (E, H)).astype(np.float32) if smooth else None
    ssm = rng(8).uniform(0.2, 1.0, (1, H)).astype(np.float32) if smooth else None
    sdt1 = torch.float16 if mode == 3 else None
    sdt2 = {0: torch.bfloat16, 2: None, 3: torch.float16}[mode]
    pack = lambda w: buf.prepack_weight(dev(w), int4=mode == 3)
    n = T if active is None else active
    more = {}
    if active is not None:
        more["x_active_mask"] = dev(np.arange(T) < active)
    if smooth:
        more.update(expert_smooth_scales=dev(sm), share_smooth_scales=dev(ssm[0]))
    seven = lambda: torch.full((T, H), 7.0, dtype=torch.bfloat16, device="cuda")
    routed = (pack(w1), dev(s1, sdt1), pack(w2), dev(s2, sdt2))
    if lists:
        routed = [[t[e].clone() for e in range(E)] for t in routed]
        more["is_tensor_list"] = True
    args = (dev(x, torch.bfloat16), dev(ids), *routed, dev(es), E)
    share = dict(share_gmm1_weight=pack(sw1), share_gmm1_scale=dev(ss1, sdt1), share_gmm2_weight=pack(sw2), share_gmm2_scale=dev(ss2, sdt2))
    out, shared, nums = buf.fused_deep_moe(*args, quant_mode=mode, out=seven(), share_out=seven(), **share, **more)
    untouched = host(torch.full((T - n, H), 7.0, dtype=torch.bfloat16))
    assert np.array_equal(host(out)[n:], untouched) and np.array_equal(host(shared)[n:], untouched)
    if n:
        ref, counts = zo.fused_moe(x[:n], zo.DT_BF16, ids[:n], es[:n], w1, s1, w2, s2, E, mode, smooth=sm)
        ref_share, _ = zo.fused_moe(x[:n], zo.DT_BF16, np.zeros((n, 1), np.int64), np.ones((n, 1), np.float32), sw1, ss1, sw2, ss2, 1,
                                    mode, smooth=ssm)
        assert np.array_equal(host(nums), counts)
        for got, want in ((out, ref), (shared, ref_share)):
            if mode == 2:
                assert max_rel_err(zo.bf16_to_f32(host(got)[:n]), zo.bf16_to_f32(want)) < 2e-2
            else:
                assert np.array_equal(host(got)[:n], want)
    # a byte less: packed more tightly, or without room for its rows, when it takes turns with the routed experts
    tight = buf.fused_workspace_bytes(T, H, K, E, 2 * I, mode, 2 * I) - 1
    run = lambda ws: buf.fused_deep_moe(*args, quant_mode=mode, out=seven(), share_out=seven(), workspace=ws, **share, **more)
    out2, shared2, _ = run(torch.empty((tight,), dtype=torch.uint8, device="cuda"))
    assert np.array_equal(host(out2), host(out)) and np.array_equal(host(shared2), host(shared))
    if not smallest:
        return
    # the smallest that is accepted: turns, in every mode
    whole, low, high = torch.empty((tight,), dtype=torch.uint8, device="cuda"), 0, tight
    while high - low > 1:
        mid = (low + high) // 2
        try:
            out3, shared3, _ = run(whole[:mid])
            high = mid
        except capi.ZbalError:
            low = mid
    out3, shared3, _ = run(whole[:high])
    assert np.array_equal(host(out3), host(out)) and np.array_equal(host(shared3), host(shared))
    # no room for its rows in q1 and q2 (each rounded up to 256 bytes)
    assert high <= buf.fused_workspace_bytes(T, H, K, E, 2 * I, mode, 2 * I) - T * (H + I) + 2 * 255


class SharedExpert(ctypes.Structure):
    """zbalhip_shared_expert_t"""
    _fields_ = [("weight", ctypes.c_void_p), ("scale", ctypes.c_void_p), ("rows", ctypes.c_int64), ("out", ctypes.c_void_p)]


# a K of one slab: the 256-row shape; of three: the many-row kernel
@pytest.mark.parametrize("K", [128, 384])
@pytest.mark.parametrize("R,S", [(2000, 1600), (1601, 1537)])
def test_shared_expert_in_many_rows(buf, R, S, K):
    """More rows than the fused layer brings there with a shared expert: the bits are those of a launch for either expert by
    itself, which in the 256-row shape is a kernel that knows of no shared expert."""
    N = 512
    a, sa, w, sw = fp8_operands(2, K, N, R + S, 40)
    a, sa, w, sw = dev(a), dev(sa), buf.prepack_weight(dev(w)), dev(sw)
    off = row_off_dev([R, S])
    alone = [(slice(0, R), 0), (slice(R, R + S), 1)]
    y, y_shared = torch.empty((R, N), dtype=torch.bfloat16, device="cuda"), torch.empty((S, N), dtype=torch.bfloat16, device="cuda")
    sh = SharedExpert(w[1].data_ptr(), sw[1].data_ptr(), S, y_shared.data_ptr())
    capi.check("gmm2", buf.lib.zbalhip_gmm2_dequant_shared(
        a.data_ptr(), sa.data_ptr(), w.data_ptr(), sw.data_ptr(), capi.DT_FP32, off.data_ptr(), 1, R, K, N, 2, capi.DT_BF16,
        y.data_ptr(), ctypes.byref(sh), capi.stream_ptr()))
    q2 = torch.empty((R + S, N // 2), dtype=torch.uint8, device="cuda")
    s2 = torch.empty((R + S, N // 256), dtype=torch.float32, device="cuda")
    sh.out = None
    capi.check("gmm1", buf.lib.zbalhip_gmm1_swiglu_quant_shared(
        a.data_ptr(), sa.data_ptr(), w.data_ptr(), sw.data_ptr(), off.data_ptr(), 1, R, K, N, 2, q2.data_ptr(), s2.data_ptr(), None,
        ctypes.byref(sh), capi.stream_ptr()))
    for (r, e), got in zip(alone, (y, y_shared)):
        n = r.stop - r.start
        one = (buf, a[r].contiguous(), sa[r].contiguous(), w[e:e + 1], sw[e:e + 1])
        want = gmm2(*one, capi.DT_FP32, [n], K, N, 2)
        assert torch.equal(got.view(torch.int16), want.view(torch.int16))
        want_q2, want_s2, _ = gmm1(*one, [n], K, N, 2)
        assert torch.equal(q2[r], want_q2) and torch.equal(s2[r], want_s2)
