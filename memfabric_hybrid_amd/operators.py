"""The operator layer under `memfabric_hybrid_amd.buffer.Buffer`: one method per zbal operator.

`OperatorBuffer` plays the part of adaptor::deep_ep::Buffer (reference
app/zbal/src/csrc/adaptor/deepep/zbal_deepep.cpp), the C++ object the
reference's Python `Buffer` keeps as `self.runtime`: it allocates the
operators' tensors with the reference's shapes and dtypes and makes one or
more calls through the zbal C ABI per method, in native code
(csrc/torch/zbal_torch.cpp). Nothing here synchronises with
the host; the DeepEP-compatible signatures, handle tuples and Python lists
live in buffer.py. Differences from the reference's adaptor, all deliberate:
  * no host synchronisation between notify and dispatch (the reference reads
    the received-token count back with .item(), zbal_deepep.cpp:359): outputs
    are sized for the worst case tokens * topk rows;
  * one process: MoE operators run on a group of one rank; further "ranks" exist only as HBM windows
    for the reductions;
  * `use_fp8` selects real e4m3 with 1x128 scales when fp8_block_scale=True
    (the reference maps the flag to int8, zbal_deepep.cpp:514,525).
torch is used for device memory and streams only.
"""
import ctypes
import threading

import torch

from . import capi

_LOCK = threading.Lock()
_STATE = {"world": None, "local": None, "users": 0}

# The process models this many "ranks" as local HBM windows; reductions may use groups up to this size.
MODEL_WORLD_SIZE = 16


def _create_comm(lib, name, world, size, rank):
    co = capi.CommOptions(name=name, backendType=capi.BACKEND_GPU, isWorldGroup=world, groupSize=size,
                          groupRankId=rank)
    comm = ctypes.c_void_p()
    capi.check("zbal_comm_create", lib.zbal_comm_create(ctypes.byref(co), ctypes.byref(comm)))
    return comm


def _acquire(device_index):
    """Bootstrap once per process; returns the one-rank group the MoE operators run on."""
    lib = capi.load()
    with _LOCK:
        if _STATE["world"] is None:
            opts = capi.BootstrapOptions()
            capi.check("zbal_bootstrap_options_init", lib.zbal_bootstrap_options_init(ctypes.byref(opts)))
            opts.worldSize, opts.rankId, opts.deviceId = MODEL_WORLD_SIZE, 0, device_index
            capi.check("zbal_bootstrap", lib.zbal_bootstrap(ctypes.byref(opts), None))
            _STATE["world"] = _create_comm(lib, b"world", 1, MODEL_WORLD_SIZE, 0)
            _STATE["local"] = _create_comm(lib, b"local", 0, 1, 0)
        _STATE["users"] += 1
        return _STATE["local"]


def _release():
    lib = capi.load()
    with _LOCK:
        _STATE["users"] -= 1
        if _STATE["users"] == 0 and _STATE["world"] is not None:
            lib.zbal_comm_destroy_all(0)
            lib.zbal_unbootstrap(0)
            _STATE["world"] = _STATE["local"] = None


def create_group(name, size, rank):
    """A sub-group of `size` modelled ranks in which this process is `rank` (needs a live Buffer)."""
    if _STATE["world"] is None:
        raise RuntimeError("create a Buffer first: it bootstraps the library")
    return _create_comm(capi.load(), name.encode(), 0, size, rank)


def destroy_group(comm):
    capi.check("zbal_comm_destroy", capi.load().zbal_comm_destroy(comm, 0))


class OperatorBuffer:
    """One-rank MoE layout / dispatch / combine / fused-MoE operators on worst-case-sized tensors."""

    num_ranks = 1
    rank = 0

    def __init__(self, device=None):
        if not torch.cuda.is_available():
            raise RuntimeError("memfabric_hybrid_amd needs a GPU; there is no CPU path")
        self.device = torch.device("cuda", torch.cuda.current_device()) if device is None else torch.device(device)
        self.lib = capi.load()
        self.native = capi.native()
        self.comm = _acquire(self.device.index or 0)
        self._comm, self._dev = self.comm.value, self.device.index or 0      # as the native calls take them
        self.send_token_idx = None       # kept between layout, dispatch and combine (zbal_deepep.cpp:254,305,423)
        self._tables = {}                # device address tables of tensor-list operands
        self._closed = False

    def close(self):
        if not self._closed:
            self._closed = True
            _release()

    def __del__(self):
        try:
            self.close()
        except Exception:
            pass

    # -- helpers ---------------------------------------------------------------------------
    def _empty(self, shape, dtype):
        return torch.empty(shape, dtype=dtype, device=self.device)

    @staticmethod
    def _ti(t, **kw):
        return ctypes.byref(capi.tensor_info(t, **kw))

    # -- router (extension) ------------------------------------------------------------------
    def topk_route(self, logits, num_topk, idx_dtype=torch.int64):
        """idx_dtype: torch.int64 (what get_dispatch_layout takes) or torch.int32 (what dispatch / fused_deep_moe take)"""
        return self.native.topk_route(self._comm, self._dev, logits, num_topk, idx_dtype == torch.int64)

    # -- normal mode -------------------------------------------------------------------------
    def get_dispatch_layout(self, topk_idx, num_experts):
        """zbal_deepep.cpp:209-257. Returns (num_tokens_per_rank, None, num_tokens_per_expert, is_token_in_rank, None)."""
        assert topk_idx.dim() == 2 and topk_idx.is_contiguous() and topk_idx.dtype == torch.int64
        # (the reference leaves is_token_in_rank unwritten)
        per_rank, per_expert, self.send_token_idx, is_token_in_rank = self.native.layout(self._comm, self._dev, topk_idx,
                                                                                         num_experts)
        return per_rank, None, per_expert, is_token_in_rank, None

    def notify(self, num_tokens_per_expert, num_topk):
        """zbal_deepep.cpp:318-357: received counts, exclusive put offsets and the balance matrix, left on the device."""
        recv_data, recv_per_expert, put_offset, balance, total = self.native.notify(self._comm, self._dev,
                                                                                    num_tokens_per_expert, num_topk)
        return dict(recv_data=recv_data, recv_per_expert=recv_per_expert, put_offset=put_offset, balance_matrix=balance,
                    total_recv=total)

    def dispatch(self, x, topk_idx, topk_weights, num_tokens_per_expert, quant_mode=capi.NO_QUANT, recv_rows=None,
                 notified=None):
        """zbal_deepep.cpp:259-393. Returns (recv_x, recv_x_scales, num_recv_tokens_per_expert (device int64), handle).
        recv_rows: rows of the receive tensors (default: the worst case tokens * topk; rows past a smaller tensor's
        end are dropped); notified: the result of notify() when the caller has already run it."""
        assert self.send_token_idx is not None, "call get_dispatch_layout first"
        T, H = x.shape
        K = topk_idx.shape[1]
        E = num_tokens_per_expert.shape[0]
        expert_ids = topk_idx.to(torch.int32)
        note = self.notify(num_tokens_per_expert, K) if notified is None else notified
        put_offset, balance = note["put_offset"], note["balance_matrix"]
        rows = max(T * K, 1) if recv_rows is None else max(int(recv_rows), 1)
        recv_x, scales = self.native.dispatch(self._comm, self._dev, x, expert_ids, self.send_token_idx, put_offset, balance,
                                              E, quant_mode, rows)
        handle = dict(put_offset=put_offset, balance_matrix=balance, expert_ids=expert_ids,
                      send_token_idx=self.send_token_idx, total_recv=note["total_recv"], num_experts=E)
        return recv_x, scales, note["recv_per_expert"], handle

    def dispatch_counts(self, x, topk_idx, num_tokens_per_expert, quant_mode, num_worst_tokens, running_sums):
        """notify() and dispatch() as one native call, the counts read back unless num_worst_tokens says how many rows
        to allow for. Returns (recv_x, recv_x_scales, list of received counts, put_offset, balance_matrix)."""
        assert self.send_token_idx is not None, "call get_dispatch_layout first"
        return self.native.dispatch_counts(self._comm, self._dev, x, topk_idx, self.send_token_idx, num_tokens_per_expert,
                                           quant_mode, num_worst_tokens, running_sums)

    def combine(self, x, handle, topk_weights):
        """zbal_deepep.cpp:395-452."""
        return self.native.combine(self._comm, self._dev, x, handle["put_offset"], topk_weights, handle["expert_ids"],
                                   handle["send_token_idx"], handle["balance_matrix"], handle["num_experts"])

    # -- low-latency mode ----------------------------------------------------------------------
    def low_latency_dispatch(self, x, topk_idx, num_max_dispatch_tokens_per_rank, num_experts, use_fp8=True,
                             fp8_block_scale=False):
        """zbal_deepep.cpp:454-565. Returns (packed_recv_x, packed_recv_x_scales, packed_recv_count, handle)."""
        qm = capi.NO_QUANT if not use_fp8 else capi.QUANT_FP8_B128 if fp8_block_scale else capi.QUANT_INT8
        recv, scales, packed_recv_count, expand_idx, ep_recv_count = self.native.ll_dispatch(
            self._comm, self._dev, x, topk_idx, num_max_dispatch_tokens_per_rank, num_experts, qm)
        handle = dict(expert_ids=topk_idx, expand_idx=expand_idx, ep_recv_count=ep_recv_count, num_experts=num_experts)
        return recv, scales, packed_recv_count, handle

    def low_latency_combine(self, x, topk_weights, handle):
        """zbal_deepep.cpp:567-656."""
        return self.native.ll_combine(self._comm, self._dev, x, handle["expert_ids"], handle["expand_idx"],
                                      handle["ep_recv_count"], topk_weights, handle["num_experts"])

    # -- fused MoE ------------------------------------------------------------------------------
    def prepack_weight(self, w, int4=False):
        """[E,K,N] one byte per element -> the library's pre-packed layout (the reference's format cast); shape stays [E,N,K]."""
        E, K, N = w.shape
        if int4:
            dst = self._empty((E, N, K // 2), torch.uint8)
            capi.check("zbal_moe_weight_prepack", self.lib.zbal_moe_weight_prepack(
                self._ti(w), self._ti(dst, dtype=capi.DT_INT4X2), self.comm, capi.stream_ptr(), 0))
        else:
            dst = self._empty((E, N, K), w.dtype)
            capi.check("zbal_moe_weight_prepack", self.lib.zbal_moe_weight_prepack(
                self._ti(w), self._ti(dst), self.comm, capi.stream_ptr(), 0))
        return dst

    def fused_workspace_bytes(self, tokens, hidden, topk, num_experts, gmm1_h_len, quant_mode, share_gmm1_h_len=0):
        n = self.lib.zbal_fused_deep_moe_workspace_size(tokens, hidden, topk, num_experts, gmm1_h_len, share_gmm1_h_len,
                                                        quant_mode)
        if n == 0:
            raise ValueError("invalid fused MoE shape")
        return int(n)

    def fused_deep_moe(self, x, topk_idx, gmm1_permuted_weight, gmm1_permuted_weight_scale, gmm2_weight,
                       gmm2_weight_scale, topk_weights, num_experts, quant_mode=0, expert_smooth_scales=None,
                       share_gmm1_weight=None, share_gmm1_scale=None, share_gmm2_weight=None, share_gmm2_scale=None,
                       share_smooth_scales=None, x_active_mask=None, workspace=None, out=None, is_tensor_list=False,
                       share_out=None):
        """zbal_deepep.cpp:658-802. Weights are pre-packed (prepack_weight; shared-expert weights as [1,N,K]).
        Returns (output, share_output, expert_token_nums) like the reference; share_output is None without a shared
        expert. x_active_mask [T] bool: only the first sum(mask) tokens are routed; the other rows of `out` keep
        their contents. is_tensor_list: the four routed-expert operands are sequences of per-expert tensors (each
        pre-packed on its own, [1,N,K] or [N,K]); the library receives one device table of addresses per operand."""
        return self.native.fused(
            self._comm, self._dev, x, topk_idx, gmm1_permuted_weight, gmm1_permuted_weight_scale, gmm2_weight,
            gmm2_weight_scale, topk_weights, num_experts, quant_mode, expert_smooth_scales, share_gmm1_weight,
            share_gmm1_scale, share_gmm2_weight, share_gmm2_scale, share_smooth_scales, x_active_mask, workspace, out,
            share_out, is_tensor_list, self._tables)
