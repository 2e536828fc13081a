"""Where the operators' outputs come from: torch's allocator, of the stream and the mode that the call runs under."""
import numpy as np
import pytest
import torch

from memfabric_hybrid_amd import capi
from memfabric_hybrid_amd.operators import OperatorBuffer
from zbal_testlib import dev, rng

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def buf():
    b = OperatorBuffer()
    yield b
    torch.cuda.synchronize()
    b.close()


def inputs(T, H, K, E):
    x = dev(rng(1).standard_normal((T, H)).astype(np.float32)).to(torch.bfloat16)
    return x, dev(np.stack([rng(t).permutation(E)[:K] for t in range(T)]).astype(np.int64))


@pytest.mark.parametrize("fill", [False, True])
def test_deterministic_mode_fills_what_is_not_written(buf, fill):
    """Rows that nobody sends to are NaN, as torch.empty would have them, where deterministic algorithms are asked for."""
    T, H, K, E = 5, 256, 4, 16
    x, idx = inputs(T, H, K, E)
    idx[2:] = -1
    torch.use_deterministic_algorithms(fill)
    try:
        recv, _, count, h = buf.low_latency_dispatch(x, idx, T, E, use_fp8=False)
    finally:
        torch.use_deterministic_algorithms(False)
    assert int(count.sum()) == 2 * K and recv[:2 * K].isfinite().all()
    if fill:
        assert recv[2 * K:].isnan().all()


@pytest.mark.parametrize("use_fp8", [False, True])
def test_outputs_are_counted_and_given_back(buf, use_fp8):
    T, H, K, E = 9, 512, 4, 16
    x, idx = inputs(T, H, K, E)
    before = torch.cuda.memory_allocated()
    out = buf.low_latency_dispatch(x, idx, T, E, use_fp8=use_fp8)
    held = torch.cuda.memory_allocated() - before
    assert held >= T * K * H * (1 if use_fp8 else 2) + 4 * 512       # pieces of 512 bytes at least
    assert all(t.is_cuda and t.device == x.device for t in (out[0], out[1], out[2], out[3]["expand_idx"]))
    del out
    assert torch.cuda.memory_allocated() == before


def test_outputs_belong_to_the_stream_of_the_call(buf):
    """A block that is freed on a side stream is handed out to that stream's next call and not to another stream's."""
    T, H, K, E = 9, 512, 4, 16
    x, idx = inputs(T, H, K, E)
    torch.cuda.synchronize()
    side = torch.cuda.Stream()
    with torch.cuda.stream(side):
        recv = buf.low_latency_dispatch(x, idx, T, E, use_fp8=False)[0]
        want, at = recv.clone(), recv.data_ptr()
        recv.record_stream(torch.cuda.current_stream())
        del recv
    other = buf.low_latency_dispatch(x, idx, T, E, use_fp8=False)[0]
    assert other.data_ptr() != at
    torch.cuda.synchronize()
    assert torch.equal(other, want)
