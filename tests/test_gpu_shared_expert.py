"""A shared expert of the routed experts' width runs in their launches: every way the layout is worked out (inside the
permute launch, from range histograms, from a launch of its own), x_active_mask, smooth scales and tensor lists, against
the oracle, which runs it as a one-expert layer. A workspace without room for its rows gives the same results."""
import numpy as np
import pytest
import torch

from memfabric_hybrid_amd.operators import OperatorBuffer
from oracle import oracle as zo
from test_gpu_gemm import fused_inputs
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
    args = (dev(x, torch.bfloat16), dev(ids), pack(w1), dev(s1, sdt1), pack(w2), dev(s2, sdt2), dev(es), E)
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
    # no room for its rows: it takes turns with the routed experts
    tight = buf.fused_workspace_bytes(T, H, K, E, 2 * I, mode, 2 * I) - 1
    ws = torch.empty((tight,), dtype=torch.uint8, device="cuda")
    out2, shared2, _ = buf.fused_deep_moe(*args, quant_mode=mode, out=seven(), share_out=seven(), workspace=ws, **share, **more)
    assert np.array_equal(host(out2), host(out)) and np.array_equal(host(shared2), host(shared))
