"""What a caller holds with a result: the operators' outputs take the memory of their own values and no more."""
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


def owns_its_values(t):
    return t.untyped_storage().nbytes() == max(t.numel(), 1) * t.element_size() and t.storage_offset() == 0


@pytest.mark.parametrize("qm", [capi.NO_QUANT, capi.QUANT_INT8, capi.QUANT_FP8_B128])
@pytest.mark.parametrize("T,share", [(1, 1.0), (1, 0.0), (300, 0.0), (300, 0.1), (300, 1.0)])
def test_received_rows_alone(buf, qm, T, share):
    """Counts read back by the host: recv and its scales are the received rows, not a row for every pick."""
    H, K, E = 256, 8, 32
    x = dev(rng(1).standard_normal((T, H)).astype(np.float32)).to(torch.bfloat16)
    ids = np.stack([rng(t).permutation(E)[:K] for t in range(T)]).astype(np.int64)
    ids[rng(2).random((T, K)) >= share] = -1
    idx = dev(ids)
    _, _, per_expert, _, _ = buf.get_dispatch_layout(idx, E)
    recv, scales, received, _, _ = buf.dispatch_counts(x, idx, per_expert, qm, 0, False)
    assert sum(received) == int((ids >= 0).sum()) and recv.shape == (max(sum(received), 1), H)
    assert owns_its_values(recv) and owns_its_values(scales)


@pytest.mark.parametrize("T", [1, 7, 300])
@pytest.mark.parametrize("use_fp8,blocks", [(False, False), (True, False), (True, True)])
def test_every_output_has_an_allocation_of_its_own(buf, T, use_fp8, blocks):
    """Small ones too: freeing, saving or keeping one output leaves the others alone."""
    H, K, E = 256, 4, 16
    x = dev(rng(1).standard_normal((T, H)).astype(np.float32)).to(torch.bfloat16)
    idx, weights = buf.topk_route(dev(rng(2).random((T, E), dtype=np.float32)), K)
    per_rank, _, per_expert, in_rank, _ = buf.get_dispatch_layout(idx, E)
    note = buf.notify(per_expert, K)
    qm = capi.NO_QUANT if not use_fp8 else capi.QUANT_FP8_B128 if blocks else capi.QUANT_INT8
    recv, scales, received, put_offset, balance = buf.dispatch_counts(x, idx, per_expert, qm, 0, False)
    ll_recv, ll_scales, ll_count, h = buf.low_latency_dispatch(x, idx, T, E, use_fp8=use_fp8, fp8_block_scale=blocks)
    outputs = [idx, weights, per_rank, per_expert, in_rank, buf.send_token_idx, *note.values(), recv, scales, put_offset, balance,
               ll_recv, ll_scales, ll_count, h["expand_idx"], h["ep_recv_count"]]
    assert all(owns_its_values(t) for t in outputs)
    assert len({t.untyped_storage().data_ptr() for t in outputs}) == len(outputs)
    kept = [t.clone() for t in outputs[1:]]
    idx.untyped_storage().resize_(0)
    assert all(torch.equal(a.view(torch.uint8), b.view(torch.uint8)) for a, b in zip(outputs[1:], kept))
