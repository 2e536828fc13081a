"""Expert ids of either width, the one-launch layout and the counts read back by the notify kernel, at the sizes where
the paths change: layouts worked out by the permute kernel itself (up to 4096 picks), by token ranges, by one launch."""
import numpy as np
import pytest
import torch

from memfabric_hybrid_amd import capi
from oracle import oracle as zo
from zbal_testlib import dev, host, rng

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def buf():
    from memfabric_hybrid_amd.operators import OperatorBuffer
    b = OperatorBuffer()
    yield b
    b.close()


@pytest.mark.parametrize("T,K,E", [(1, 1, 1), (5, 3, 8), (512, 8, 32), (513, 8, 32), (700, 6, 300), (1500, 3, 1000)])
@pytest.mark.parametrize("use_fp8", [False, True])
def test_int64_ids_give_the_int32_results(buf, T, K, E, use_fp8):
    H = 256
    idx = rng(T + E).integers(0, E, size=(T, K)).astype(np.int64)
    x = torch.randn((T, H), device="cuda").to(torch.bfloat16)
    y = torch.randn((T * K, H), device="cuda").to(torch.bfloat16)
    w = torch.rand((T, K), device="cuda")
    outs = []
    for ids in (dev(idx), dev(idx.astype(np.int32))):
        recv, scales, nums, h = buf.low_latency_dispatch(x, ids, T, E, use_fp8=use_fp8)
        outs.append((recv, nums, h["expand_idx"], h["ep_recv_count"], buf.low_latency_combine(y, w, h)) +
                    ((scales,) if use_fp8 else ()))
    for a, b in zip(*outs):
        assert torch.equal(a, b)
    assert np.array_equal(host(outs[0][1]), np.bincount(idx.ravel(), minlength=E))


@pytest.mark.parametrize("T,K,E,R", [(0, 4, 8, 1), (1, 1, 1, 1), (3, 5, 7, 7), (1025, 8, 32, 1), (999, 7, 96, 4), (4097, 3, 1000, 40)])
@pytest.mark.parametrize("npdt", [np.int64, np.int32])
def test_layout_in_one_launch(buf, T, K, E, R, npdt):
    idx = rng(T * 7 + E).integers(-1, E + 1, size=(T, K)).astype(npdt)
    d = dev(idx) if T else torch.empty((1, K), dtype=torch.int64, device="cuda")
    per_rank, per_expert, send, in_rank = (torch.full(s, -7, dtype=torch.int32, device="cuda")
                                           for s in ((R,), (E,), (max(T, 1), K), (max(T, 1), R)))
    rc = buf.lib.zbalhip_dispatch_layout_in_rank(d.data_ptr(), int(npdt == np.int64), T, E, K, R, per_rank.data_ptr(),
                                                 per_expert.data_ptr(), send.data_ptr(), in_rank.data_ptr(),
                                                 capi.stream_ptr())
    assert rc == 0
    want_rank, want_expert, want_send = zo.dispatch_layout(idx.astype(np.int64), E, R)
    assert np.array_equal(host(per_rank), want_rank) and np.array_equal(host(per_expert), want_expert)
    assert T == 0 or np.array_equal(host(send), want_send)
    valid = (idx >= 0) & (idx < E)
    want_in = np.stack([(valid & (idx // (E // R) == r)).any(axis=1) for r in range(R)], axis=1).astype(np.int32)
    assert T == 0 or np.array_equal(host(in_rank), want_in)


# whole tokens per wave: 64, 21, 10, one, one, and more picks than a wave has lanes; tokens either side of a block's eight steps of them
@pytest.mark.parametrize("K", [1, 3, 6, 33, 64, 65])
@pytest.mark.parametrize("T", [1, 127, 128, 129, 1345])
@pytest.mark.parametrize("npdt", [np.int64, np.int32])
def test_tokens_of_one_rank(buf, T, K, npdt):
    E = 40
    idx = rng(T + K).integers(-1, E + 1, size=(T, K)).astype(npdt)
    idx[::3] = E                                                                # tokens without a valid pick
    idx[::6, K - 1] = E - 1                                                     # or with the last one only
    d = dev(idx)
    per_rank, per_expert, send, in_rank = (torch.full(s, -7, dtype=torch.int32, device="cuda") for s in ((1,), (E,), (T, K), (T, 1)))
    assert buf.lib.zbalhip_dispatch_layout_in_rank(d.data_ptr(), int(npdt == np.int64), T, E, K, 1, per_rank.data_ptr(),
                                                   per_expert.data_ptr(), send.data_ptr(), in_rank.data_ptr(), capi.stream_ptr()) == 0
    want = ((idx >= 0) & (idx < E)).any(axis=1)
    assert np.array_equal(host(in_rank)[:, 0], want.astype(np.int32)) and host(per_rank)[0] == want.sum()
    _, want_expert, want_send = zo.dispatch_layout(idx.astype(np.int64), E, 1)
    assert np.array_equal(host(per_expert), want_expert) and np.array_equal(host(send), want_send)


@pytest.mark.parametrize("E", [1, 63, 64, 65, 1024])
def test_counts_read_back_by_the_notify_kernel(buf, E):
    """Several calls in a row, with work queued in front and behind, give the counts of that call."""
    out = {k: torch.empty(n, dtype=t, device="cuda") for k, n, t in
           (("recv", E, torch.int32), ("put", E, torch.int32), ("total", 1, torch.int32), ("per", E, torch.int64),
            ("bal", 2, torch.int32))}
    ti, ref = capi.tensor_info, lambda t: __import__("ctypes").byref(t)
    for rep in range(3):
        c = rng(E + rep).integers(0, 50, size=E).astype(np.int32)
        counts, got = dev(c), np.full(E, -1, dtype=np.int64)
        busy = torch.randn((2048, 2048), device="cuda")
        for _ in range(10 * rep):
            busy = busy @ busy * 1e-3
        pending = capi.PendingCounts()
        capi.check("begin", buf.lib.zbal_dispatch_normal_notify_begin(
            ref(ti(counts)), E, 4, ref(ti(out["recv"])), ref(ti(out["total"])), ref(ti(out["per"])), ref(ti(out["put"])),
            ref(ti(out["bal"])), ref(pending), buf.comm, capi.stream_ptr(), 0))
        busy = busy @ busy                                   # work behind the notify
        capi.check("end", buf.lib.zbal_dispatch_normal_notify_end(ref(pending), E, got.ctypes.data, buf.comm,
                                                                  capi.stream_ptr(), 0))
        assert np.array_equal(got, c)
        assert np.array_equal(host(out["put"]), np.cumsum(c) - c) and host(out["total"])[0] == c.sum()
        assert np.array_equal(host(out["per"]), c)
