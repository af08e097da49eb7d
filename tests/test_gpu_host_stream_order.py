"""Pinned queries that earlier work on the caller's stream is still writing when a streamed host search is called."""
import numpy as np
import pytest

from harmonia_amd import BPlusTree
from harmonia_amd import workloads as W

pytestmark = pytest.mark.gpu


def test_queries_written_by_the_callers_stream(gpu):
    import torch

    keys, vals = W.gen_keys(1 << 18, 78)
    tree = BPlusTree.from_keys(keys, vals)
    n = (1 << 22) + 4099
    hq = torch.zeros(n, dtype=torch.int64).pin_memory()
    hv = torch.zeros(n, dtype=torch.int64).pin_memory()
    hf = torch.zeros(n, dtype=torch.uint8).pin_memory()
    s = torch.cuda.Stream()
    x = torch.randn(4096, 4096, device="cuda")
    g = torch.Generator(device="cuda")
    for step in range(3):
        g.manual_seed(step)
        torch.cuda.synchronize()
        with torch.cuda.stream(s):
            for _ in range(20):  # a few milliseconds before the queries are there
                x = torch.tanh(x @ x)
            pick = torch.randint(0, len(keys), (n,), device="cuda", generator=g)
            hq.copy_(torch.from_numpy(keys.view(np.int64)).cuda()[pick], non_blocking=True)
            tree.search_batch(hq, out_vals=hv, out_found=hf, stream=s)
        assert bool(hf.all()) and np.array_equal(hv.numpy().view(np.uint64), W.splitmix64_mix(hq.numpy().view(np.uint64)))
    tree.close()
