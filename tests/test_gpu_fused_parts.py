"""Fused layers in which a tile of the first GEMM is left over when every CU has as many (K > 4096, one expert more than CUs of an XCD,
one tile of every expert per XCD)."""
import numpy as np
import pytest
import torch

from memfabric_hybrid_amd import capi
from memfabric_hybrid_amd.operators import OperatorBuffer
from oracle import oracle as zo
from zbal_testlib import dev, distinct_topk, host

pytestmark = pytest.mark.gpu

H, I, K = 4608, 1024, 4


@pytest.fixture(scope="module")
def buf():
    b = OperatorBuffer()
    yield b
    torch.cuda.synchronize()
    b.close()


def experts():
    return torch.cuda.get_device_properties(0).multi_processor_count // 8


def weights(mode, n, seed):
    """Of n experts, as the entry point takes them unpacked: w1 [n, H, 2 * I], its scales, w2 [n, I, H], its scales."""
    g = torch.Generator(device="cuda").manual_seed(seed)
    if mode == 1:
        w1, w2 = (torch.randint(-16, 16, s, dtype=torch.int8, device="cuda", generator=g) for s in ((n, H, 2 * I), (n, I, H)))
        s1 = torch.rand((n, 2 * I), device="cuda", generator=g) * 0.003 + 0.0015
        return w1, s1, w2, (torch.rand((n, H), device="cuda", generator=g) * 0.003 + 0.0015).to(torch.bfloat16)
    out = []
    for k, width in ((H, 2 * I), (I, H)):
        w = torch.empty((n, k, width), device="cuda", dtype=torch.float8_e4m3fn)
        for e in range(n):
            w[e] = (torch.randn((k, width), device="cuda", generator=g) * 100.0).clamp_(-448, 448).to(torch.float8_e4m3fn)
        out += [w, (torch.rand((n, k // 128, width // 128), device="cuda", generator=g) + 0.5) / (100.0 * k ** 0.5)]
    return tuple(out)


def packed(buf, w):
    return buf.prepack_weight(w[0]), w[1], buf.prepack_weight(w[2]), w[3]


def share_args(buf, w):
    return dict(zip(("share_gmm1_weight", "share_gmm1_scale", "share_gmm2_weight", "share_gmm2_scale"), packed(buf, w)))


def inputs(T, E, seed):
    g = torch.Generator(device="cuda").manual_seed(seed)
    ids = distinct_topk(T, E, K, seed).astype(np.int32)
    assert len(np.unique(ids)) == E                              # every expert has a tile
    return (torch.randn((T, H), device="cuda", generator=g).to(torch.bfloat16), dev(ids), torch.rand((T, K), device="cuda", generator=g))


def test_fp8_row_depends_on_its_token_alone(buf):
    """The bits of a token's fp8 row are the same whoever is in the batch beside it, with a shared expert (whose tile is the one that
    leaves one over) and without, and in a workspace of any size: every sum over K is one chain."""
    E, T = experts(), 64
    routed, share = packed(buf, weights(2, E, 1)), share_args(buf, weights(2, 1, 2))
    x, ids, es = inputs(T, E, 3)
    run = lambda n, **more: buf.fused_deep_moe(x[:n], ids[:n], *routed, es[:n], E, quant_mode=2, **more)
    alone, _, _ = run(T)
    assert float(alone.abs().max()) > 1e-3
    beside, shared, _ = run(T, **share)
    assert torch.equal(alone, beside)
    few, few_shared, _ = run(40, **share)
    assert torch.equal(few, alone[:40]) and torch.equal(few_shared, shared[:40])
    whole = buf.fused_workspace_bytes(T, H, K, E, 2 * I, 2, 2 * I)
    turns = buf.fused_workspace_bytes(T, H, K, E, 2 * I, 2)      # no room for the shared expert's rows beside the others
    assert turns < whole
    for size in (whole, turns):
        out, out_shared, _ = run(T, workspace=torch.empty((size,), dtype=torch.uint8, device="cuda"), **share)
        assert torch.equal(out, alone) and torch.equal(out_shared, shared), size


def regions(T, n_experts):
    """W8A8 workspace in which a shared expert rides along: where the fp32 values and y (apart) begin, y's bytes and those of the values."""
    rows, all_rows = T * K, T * K + T
    align = lambda n: (n + 255) // 256 * 256
    values = sum(align(n) for n in (rows * 4, n_experts * 8, (n_experts + 2) * 4, 50 * n_experts * 4, all_rows * I, all_rows * 4, all_rows * H,
                                    all_rows * 4))
    return values, values + align(all_rows * (I + 1) * 4), align(rows * H * 2), align(all_rows * (I + 1) * 4)


@pytest.mark.parametrize("together", [False, True])
def test_w8a8_layer_with_a_tile_shared_along_k(buf, together):
    """A routed expert's tile on every XCD is left over behind the shared expert's and is shared along K, in the part of y that the second GEMM
    does not write for the tokens that the mask leaves out: the sums are still there afterwards. Every call on a workspace that the call
    before has left as it is, and replays of a graph with new inputs, against the oracle; y beside the fp32 values and in their place."""
    E, T, n = experts(), 96, 56
    routed, share = weights(1, E, 5), weights(1, 1, 6)
    args, share_kw = packed(buf, routed), share_args(buf, share)
    mask = torch.arange(T, device="cuda") < n
    values, apart, y_bytes, value_bytes = regions(T, E)
    size, y = (values + max(y_bytes, value_bytes), values) if together else (apart + y_bytes, apart)
    unwritten = slice(max(y + n * K * H * 2, values + value_bytes if together else 0), y + y_bytes)      # of y, behind the values and the routed rows

    def layer(x, ids, es, out, share_out, ws):
        return buf.fused_deep_moe(x, ids, *args, es, E, quant_mode=1, x_active_mask=mask, out=out, share_out=share_out, workspace=ws, **share_kw)

    seven = lambda: torch.full((T, H), 7.0, dtype=torch.bfloat16, device="cuda")
    ws, g_ws = (torch.full((size,), 0x5a, dtype=torch.uint8, device="cuda") for _ in range(2))
    x, ids, es = inputs(T, E, 30)
    s_out, s_share = seven(), seven()
    layer(x, ids, es, s_out, s_share, g_ws)              # first call outside the capture
    torch.cuda.synchronize()
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        layer(x, ids, es, s_out, s_share, g_ws)
    hosted = [host(t) for t in routed], [host(t) for t in share]
    for seed in (31, 32, 33):
        nx, nids, nes = inputs(T, E, seed)
        assert len(np.unique(host(nids)[:n])) == E
        ws[unwritten].fill_(0x5a)
        out, shared, nums = layer(nx, nids, nes, seven(), seven(), ws)
        assert bool((ws[unwritten] != 0x5a).any()), "no tile was shared"
        xh, idh, esh = host(nx)[:n], host(nids)[:n].astype(np.int64), host(nes)[:n]
        want, counts = zo.fused_moe(xh, zo.DT_BF16, idh, esh, *hosted[0], E, 1)
        want_share, _ = zo.fused_moe(xh, zo.DT_BF16, np.zeros((n, 1), np.int64), np.ones((n, 1), np.float32), *hosted[1], 1, 1)
        assert np.array_equal(host(nums), counts)
        assert np.array_equal(host(out)[:n], want) and np.array_equal(host(shared)[:n], want_share)
        x.copy_(nx), ids.copy_(nids), es.copy_(nes)
        s_out.fill_(7.0), s_share.fill_(7.0)
        graph.replay()
        torch.cuda.synchronize()
        assert torch.equal(s_out, out) and torch.equal(s_share, shared), seed
