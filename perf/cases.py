"""The work whose speed matters to a program that uses this library on one MI355X, as cases that can be timed.

Four kinds of pass, each through the library's public entry points:
  layer    one MoE layer of a serving engine: Buffer.topk_route, then Buffer.fused_deep_moe on pre-packed weights;
  lowlat   the decode-side exchange of an engine with expert GEMMs of its own: Buffer.low_latency_dispatch, then
           Buffer.low_latency_combine of the experts' outputs;
  normal   the prefill / training-side exchange: Buffer.get_dispatch_layout, Buffer.dispatch, then Buffer.combine of
           the experts' outputs;
  reduce   the local compute of zbal_all_reduce / zbal_reduce_scatter over the windows of a group.

Layer shapes: 7168 x 2048 with 32 local experts and 4096 x 1536 with 128 are this repository's benchmark layers;
2048 x 1024 with 64 experts, top-6, is a generic small one.
"""
import math
import os

import numpy as np
import torch

from memfabric_hybrid_amd import capi
from memfabric_hybrid_amd.buffer import Buffer
from memfabric_hybrid_amd.operators import create_group, destroy_group

# hidden, experts, top-k, intermediate size of an expert
SHAPES = {"wide": (7168, 32, 8, 2048), "many": (4096, 128, 8, 1536), "small": (2048, 64, 6, 1024)}
# fused_deep_moe's quant_mode
MODES = {"w8a8": 1, "fp8": 2, "w4a8": 3}
HALVES = {"bf16": torch.bfloat16, "fp16": torch.float16}
REDUCE_TYPES = {"bf16": (torch.bfloat16, capi.DT_BF16, 2), "fp16": (torch.float16, capi.DT_FP16, 2),
                "fp32": (torch.float32, capi.DT_FP32, 4), "int32": (torch.int32, capi.DT_INT32, 4)}
REDUCE_OPS = {"sum": capi.REDUCE_SUM, "max": capi.REDUCE_MAX}


def _layer(name, shape, mode, tokens, zipf=False, shared=False, lists=False, dtype="bf16"):
    return {"name": name, "kind": "layer", "shape": shape, "mode": mode, "tokens": tokens, "zipf": zipf, "shared": shared,
            "lists": lists, "dtype": dtype}


def _lowlat(name, hidden, experts, topk, tokens, int8):
    return {"name": name, "kind": "lowlat", "hidden": hidden, "experts": experts, "topk": topk, "tokens": tokens,
            "int8": int8}


def _normal(name, hidden, experts, topk, tokens, int8, host_counts):
    return {"name": name, "kind": "normal", "hidden": hidden, "experts": experts, "topk": topk, "tokens": tokens,
            "int8": int8, "host_counts": host_counts}


def _reduce(name, scatter, ranks, rank, count, dtype, op):
    return {"name": name, "kind": "reduce", "scatter": scatter, "ranks": ranks, "rank": rank, "count": count,
            "dtype": dtype, "op": op}


def listed():
    return [
        # a single sequence being decoded: eight expert rows, nothing but latency and the weights of eight experts
        _layer("layer w8a8 1", "wide", "w8a8", 1),
        # the decode step of a full batch, some experts popular
        _layer("layer w8a8 128 zipf", "wide", "w8a8", 128, zipf=True),
        # a decode step of a half-empty batch, with the shared expert such models have
        _layer("layer fp8 37 shared", "wide", "fp8", 37, shared=True),
        # the benchmark's prefill batch
        _layer("layer fp8 4096", "wide", "fp8", 4096),
        # chunked prefill mixed with decoding: a ragged token count over many experts
        _layer("layer w4a8 509", "many", "w4a8", 509),
        # the largest prefill batch
        _layer("layer w4a8 16384", "many", "w4a8", 16384),
        # decode exchange of a nearly idle engine, rows sent as they are
        _lowlat("lowlat bf16 7", 7168, 32, 8, 7, False),
        # decode exchange of a full batch, rows quantised (the default)
        _lowlat("lowlat int8 128", 7168, 32, 8, 128, True),
        # prefill exchange with the default host read-back of the received counts
        _normal("normal bf16 4096", 7168, 32, 8, 4096, False, True),
        # the same without the read-back, quantised, on a ragged batch
        _normal("normal int8 1021", 4096, 128, 8, 1021, True, False),
        # an odd gradient shard in half precision: slices off the 16-byte boundary
        _reduce("reduce_scatter fp16 odd", True, 8, 3, 100003, "fp16", "sum"),
        # the benchmark's reduction: eight buffers of 256 MiB
        _reduce("all_reduce bf16 8x256MiB", False, 8, 0, 128 << 20, "bf16", "sum"),
    ]


def _log_int(rng, lo, hi):
    return min(hi, max(lo, int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))))


def draw(rng):
    u = rng.random()
    if u < 0.5:
        shape, mode = rng.choice([("wide", "w8a8"), ("wide", "fp8"), ("many", "w4a8"), ("many", "w8a8"), ("small", "w8a8"),
                                  ("small", "fp8"), ("small", "w4a8")])
        case = _layer(None, shape, mode, _log_int(rng, 1, 4096 if shape == "wide" else 8192), zipf=rng.random() < 0.3,
                      shared=shape == "wide" and rng.random() < 0.4, lists=rng.random() < 0.15,
                      dtype="fp16" if rng.random() < 0.15 else "bf16")
    elif u < 0.7:
        hidden, experts, topk, _ = SHAPES[rng.choice(sorted(SHAPES))]
        case = _lowlat(None, hidden, experts, topk, _log_int(rng, 1, 512), rng.random() < 0.6)
    elif u < 0.85:
        hidden, experts, topk, _ = SHAPES[rng.choice(sorted(SHAPES))]
        case = _normal(None, hidden, experts, topk, _log_int(rng, 64, 8192), rng.random() < 0.5, rng.random() < 0.5)
    else:
        ranks = rng.choice([2, 4, 8, 16])
        dtype = rng.choice(["bf16", "bf16", "fp16", "fp32", "fp32", "int32"])
        scatter = rng.random() < 0.5
        # a reduce-scatter's windows hold `ranks` slices each; together no more memory than the largest listed case
        most = (2 << 30) // (ranks * (ranks if scatter else 1) * REDUCE_TYPES[dtype][2])
        case = _reduce(None, scatter, ranks, rng.randrange(ranks), _log_int(rng, 1 << 10, most), dtype,
                       "max" if rng.random() < 0.15 else "sum")
    del case["name"]
    return case


# ---- what a user's program has in hand before the call ---------------------------------------------------------------

_buffer = None


def buffer():
    """The one Buffer a program keeps."""
    global _buffer
    if _buffer is None:
        _buffer = Buffer()
    return _buffer


def _generator(seed):
    return torch.Generator(device="cuda").manual_seed(seed)


def _logits(g, tokens, experts, zipf):
    """Router logits whose top-k is a draw of distinct experts, uniform or with Zipf(1.2) popularity (log p plus Gumbel
    noise)."""
    u = torch.rand((tokens, experts), device="cuda", generator=g)
    if not zipf:
        return u
    p = 1.0 / torch.arange(1, experts + 1, device="cuda", dtype=torch.float32) ** 1.2
    p = p[torch.randperm(experts, device="cuda", generator=g)]
    return (torch.log(p / p.sum())[None, :] - torch.log(-torch.log(u.clamp_(1e-9, 1 - 1e-7)))).contiguous()


def _weights(g, mode, experts, k, n):
    """Expert weights [experts, k, n], pre-packed, with scales that keep the layer's values of order one."""
    shape, norm = (experts, k, n), k ** 0.5
    if mode == "fp8":
        w = torch.empty(shape, device="cuda", dtype=torch.float8_e4m3fn)
        for e in range(experts):
            w[e] = (torch.randn((k, n), device="cuda", generator=g) * 100.0).clamp_(-448, 448).to(torch.float8_e4m3fn)
        s = (torch.rand((experts, k // 128, n // 128), device="cuda", generator=g) + 0.5) / (100.0 * norm)
    elif mode == "w8a8":
        w = torch.randint(-127, 128, shape, device="cuda", dtype=torch.int8, generator=g)
        s = (torch.rand((experts, n), device="cuda", generator=g) + 0.5) / (73.0 * norm)
    else:
        w = torch.randint(-8, 8, shape, device="cuda", dtype=torch.int8, generator=g)
        s = ((torch.rand((experts, k // 128, n), device="cuda", generator=g) + 0.5) / (4.6 * norm)).to(torch.float16)
    return buffer().prepack_weight(w, int4=mode == "w4a8"), s


def _prepare_layer(case, g):
    hidden, experts, topk, inter = SHAPES[case["shape"]]
    mode, tokens = case["mode"], case["tokens"]
    w1, s1 = _weights(g, mode, experts, hidden, 2 * inter)
    w2, s2 = _weights(g, mode, experts, inter, hidden)
    if mode == "w8a8":
        s2 = s2.to(torch.bfloat16)
    more = {"quant_mode": MODES[mode]}
    if case["lists"]:
        def split(t):
            out = [t[e:e + 1] for e in range(experts)]
            for v in out:
                v.zbal_prepacked = True
            return out
        w1, w2 = split(w1), split(w2)
        s1, s2 = [s1[e] for e in range(experts)], [s2[e] for e in range(experts)]
        more["is_tensor_list"] = True
    if case["shared"]:
        sw1, ss1 = _weights(g, mode, 1, hidden, 2 * inter)
        sw2, ss2 = _weights(g, mode, 1, inter, hidden)
        more.update(share_gmm1_weight=sw1, share_gmm1_scale=ss1, share_gmm2_weight=sw2,
                    share_gmm2_scale=ss2.to(torch.bfloat16) if mode == "w8a8" else ss2, share_gmm1_h_len=2 * inter)
    x = torch.randn((tokens, hidden), device="cuda", generator=g).to(HALVES[case["dtype"]])
    return dict(kind="layer", x=x, logits=_logits(g, tokens, experts, case["zipf"]), w=(w1, s1, w2, s2), more=more,
                experts=experts, topk=topk)


def _prepare_exchange(case, g):
    tokens, hidden, experts, topk = case["tokens"], case["hidden"], case["experts"], case["topk"]
    if case["kind"] == "normal":
        os.environ["DEEP_NORMAL_MODE_USE_INT8_QUANT"] = "1" if case["int8"] else "0"
    w, idx = torch.topk(torch.softmax(_logits(g, tokens, experts, False), dim=-1), topk, dim=-1)
    return dict(kind=case["kind"], x=torch.randn((tokens, hidden), device="cuda", generator=g).to(torch.bfloat16),
                idx=idx.contiguous(), w=(w / w.sum(dim=-1, keepdim=True)).contiguous(),
                y=torch.randn((tokens * topk, hidden), device="cuda", generator=g).to(torch.bfloat16), tokens=tokens,
                experts=experts, int8=case["int8"], worst=0 if case.get("host_counts") else tokens * topk)


class _Group:
    """A group of modelled ranks with a send window each, and this rank's receive buffer."""

    serial = 0

    def __init__(self, case, g):
        buffer()
        _Group.serial += 1
        dtype, self.dt, size = REDUCE_TYPES[case["dtype"]]
        self.op, self.count, self.scatter = REDUCE_OPS[case["op"]], case["count"], case["scatter"]
        elems = self.count * (case["ranks"] if self.scatter else 1)
        self.lib = capi.load()
        self.comm = create_group("perf%d" % _Group.serial, case["ranks"], case["rank"])
        self.windows = []
        for r in range(case["ranks"]):
            if dtype == torch.int32:
                w = torch.randint(-1000, 1000, (elems,), device="cuda", dtype=dtype, generator=g)
            else:
                w = torch.empty((elems,), device="cuda", dtype=dtype).normal_(generator=g)
            capi.check("window", self.lib.zbal_comm_register_peer_window(self.comm, r, w.data_ptr(), elems * size))
            self.windows.append(w)
        self.send = self.windows[case["rank"]]
        self.recv = torch.empty((self.count,), device="cuda", dtype=dtype)
        self.tmp = None if self.scatter else torch.empty_like(self.recv)        # zbal_all_reduce asks for one

    def run(self):
        stream = capi.stream_ptr()
        if self.scatter:
            rc = self.lib.zbal_reduce_scatter(self.send.data_ptr(), self.recv.data_ptr(), self.count, self.dt, self.op,
                                              self.comm, stream)
        else:
            rc = self.lib.zbal_all_reduce(self.send.data_ptr(), self.recv.data_ptr(), self.tmp.data_ptr(), self.count,
                                          self.dt, self.op, self.comm, stream)
        capi.check("reduce", rc)
        return self.recv

    def __del__(self):
        torch.cuda.synchronize()
        destroy_group(self.comm)


def prepare(case, seed):
    g = _generator(seed)
    if case["kind"] == "layer":
        return _prepare_layer(case, g)
    if case["kind"] == "reduce":
        return dict(kind="reduce", group=_Group(case, g))
    return _prepare_exchange(case, g)


# ---- one pass ------------------------------------------------------------------------------------------------------

def run(state):
    kind = state["kind"]
    if kind == "reduce":
        return state["group"].run()
    buf, x = buffer(), state["x"]
    if kind == "layer":
        w1, s1, w2, s2 = state["w"]
        idx, w = buf.topk_route(state["logits"], state["topk"], torch.int32)
        out, counts = buf.fused_deep_moe(x, idx, w1, s1, w2, s2, w, state["experts"], **state["more"])
        return idx, w, out, counts, buf.last_share_output
    idx, w = state["idx"], state["w"]
    if kind == "lowlat":
        recv, counts, handle, _, _ = buf.low_latency_dispatch(x, idx, state["tokens"], state["experts"],
                                                              use_fp8=state["int8"])
        out, _, _ = buf.low_latency_combine(state["y"], idx, w, handle)
        return recv, counts, out
    per_rank, _, per_expert, in_rank, _ = buf.get_dispatch_layout(idx, state["experts"])
    recv, _, _, received, handle, _ = buf.dispatch(x, num_tokens_per_rank=per_rank, is_token_in_rank=in_rank,
                                                   num_tokens_per_expert=per_expert, topk_idx=idx, topk_weights=w,
                                                   num_worst_tokens=state["worst"])
    out, _, _ = buf.combine(state["y"], handle)
    return per_rank, per_expert, in_rank, recv, np.asarray(received, dtype=np.int64), out


# ---- what a pass cannot do without, and how exact it is ---------------------------------------------------------------

def work(case):
    if case["kind"] == "reduce":
        values = case["ranks"] * case["count"]
        return {"bytes": (values + case["count"]) * REDUCE_TYPES[case["dtype"]][2], "flops": values}
    tokens = case["tokens"]
    if case["kind"] == "layer":
        hidden, experts, topk, inter = SHAPES[case["shape"]]
        weights = 3 * hidden * inter                            # elements of one expert
        per_weight = 0.5 if case["mode"] == "w4a8" else 1
        per_weight += {"w8a8": 0, "fp8": 4 / 128 ** 2, "w4a8": 2 / 128}[case["mode"]]
        # experts that some token picks, on average over uniform routing
        touched = experts * (1 - (1 - topk / experts) ** tokens) + (1 if case["shared"] else 0)
        outputs = 2 if case["shared"] else 1
        return {"bytes": touched * weights * per_weight + tokens * (hidden * 2 * (1 + outputs) + experts * 4 + topk * 8),
                "flops": 2 * tokens * (topk + (1 if case["shared"] else 0)) * weights}
    hidden, topk = case["hidden"], case["topk"]
    rows = tokens * topk
    sent = rows * (hidden + 4 if case["int8"] else hidden * 2)
    return {"bytes": tokens * hidden * 2 + rows * 12 + sent + rows * hidden * 2 + tokens * hidden * 2,
            "flops": 2 * rows * hidden}


def tolerance(case):
    if case["kind"] == "reduce":
        if case["dtype"] == "int32":
            return "exact"
        # fp32 accumulation in any order, one rounding to the type
        return {"rel": {"bf16": 1e-2, "fp16": 2e-3, "fp32": 1e-5}[case["dtype"]]}
    # half-precision outputs; indices, counts and int8 rows are the same
    return {"rel": 1e-2}
