"""The router where its ranks change to rounds of arg-max (experts > 4 * topk), at whole and ragged numbers of 64 experts, with ties, with
experts ruled out by minus infinity, and down to the last expert that is left."""
import numpy as np
import pytest
import torch

from memfabric_hybrid_amd import capi
from memfabric_hybrid_amd.operators import OperatorBuffer
from oracle import oracle as zo
from zbal_testlib import dev, host, rng

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def buf():
    b = OperatorBuffer()
    yield b
    torch.cuda.synchronize()
    b.close()


@pytest.mark.parametrize("E,K", [(4, 1), (5, 1), (24, 6), (25, 6), (32, 8), (33, 8), (63, 8), (64, 8), (64, 15), (64, 16), (64, 32), (65, 8), (127, 31),
                                 (128, 8), (129, 8), (256, 32), (257, 3), (1024, 16)])
@pytest.mark.parametrize("style", ["normal", "ties", "ruled out"])
def test_picks_and_weights(buf, E, K, style):
    g = rng(E * 64 + K)
    T = 70
    logits = g.integers(-2, 3, (T, E)).astype(np.float32) if style == "ties" else g.standard_normal((T, E)).astype(np.float32)
    if style == "ruled out":                     # all but one expert, all but K - 1 of them, or every other one
        for t in range(T):
            kept = g.permutation(E)[:(1, max(K - 1, 1), max(E // 2, 1))[t % 3]]
            logits[t, np.setdiff1d(np.arange(E), kept)] = -np.inf
    idx, w = buf.topk_route(dev(logits), K)
    ridx, rw = zo.topk_route(logits, K)
    assert np.array_equal(host(idx), ridx)
    assert np.allclose(host(w), rw, rtol=1e-6, atol=0)       # the router's bound: weights within 1e-6 relative


# ranks, rounds of one logit per lane, and rounds of two and of sixteen
@pytest.mark.parametrize("E,K", [(8, 8), (32, 8), (33, 8), (64, 8), (65, 8), (128, 8), (1000, 16)])
@pytest.mark.parametrize("dt", [torch.int64, torch.int32])
def test_nan_logits_are_no_picks(buf, E, K, dt):
    """A NaN is never picked: a row's picks are its other logits in their order, and where there are fewer of them than picks the rest of
    the row is an id that no expert has. No slot keeps what the memory held. One NaN makes the row's softmax, and so every weight, NaN."""
    g = rng(E + K)
    T = 4 * K + 6
    logits = g.standard_normal((T, E)).astype(np.float32)
    left = [min(E, max(0, n)) for n in range(-1, K + 3)] + [E - 1, E - 2]
    for t in range(T):
        if t % 4:                                # every fourth row as it is
            logits[t, g.permutation(E)[left[t % len(left)]:]] = np.nan
    lg = dev(logits)
    idx, w = torch.full((T, K), 5, dtype=dt, device="cuda"), torch.full((T, K), 0.25, device="cuda")
    capi.check("route", buf.lib.zbalhip_topk_route(lg.data_ptr(), T, E, K, idx.data_ptr(), int(dt == torch.int64), w.data_ptr(), capi.stream_ptr()))
    idx, w = host(idx), host(w)
    for t in range(T):
        numbers = np.flatnonzero(~np.isnan(logits[t]))
        want = numbers[np.argsort(-logits[t, numbers], kind="stable")][:K]
        assert np.array_equal(idx[t, :len(want)], want), (t, idx[t])
        assert ((idx[t, len(want):] < 0) | (idx[t, len(want):] >= E)).all(), (t, idx[t])
        assert np.isnan(w[t]).all() if len(numbers) < E else abs(w[t].sum() - 1) < 1e-5, (t, w[t])
