"""bench.py's workloads, one step each: the stages that it times one by one give what the whole layer gives (bench_moe
asserts it), and every line has its figures."""
import argparse

import numpy as np
import pytest
import torch

import bench
from memfabric_hybrid_amd import capi
from memfabric_hybrid_amd.operators import OperatorBuffer

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("workload", ["prefill", "prefill_w8a8", "decode", "qwen_w4a8", "reduce"])
def test_a_step_of_every_workload(workload):
    args = argparse.Namespace(gpus=1, steps=1, warmup=1, tokens=4096, cpu_sample_tokens=0, workload=workload, no_cpu=True,
                              equal_rows=False, no_others=True)
    buf = OperatorBuffer()
    if workload == "reduce":
        line = bench.bench_reduce(args, torch, np, capi, buf)
        assert all(v["exact"] for v in line["variants"].values())
    else:
        line = bench.bench_moe(args, torch, np, capi, buf, workload)
        assert all(ms > 0 for ms in line["stages"]["ms"].values()) and line["roofline"]["achieved"] > 0
    assert line["value"] > 0 and line["ms_per_step"] > 0 and line["n_gpus"] == 1
    torch.cuda.synchronize()
    buf.close()
    torch.cuda.empty_cache()
