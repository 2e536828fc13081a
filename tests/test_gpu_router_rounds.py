"""The router where its ranks change to rounds of arg-max (experts > 4 * topk), at whole and ragged numbers of 64 experts, with ties, with
experts ruled out by minus infinity, and down to the last expert that is left."""
import numpy as np
import pytest
import torch

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
