"""Trees that come and go reuse device memory: results stay right when blocks return with other trees' data
in them, from several threads at once, and the memory goes back to the driver when the device is
synchronized."""
import threading

import numpy as np
import pytest

from harmonia_amd import BPlusTree, load
from harmonia_amd import workloads as W

pytestmark = pytest.mark.gpu


def rounds(seed, out):
    try:
        g = np.random.RandomState(seed)
        for i in range(12):
            n = int(g.choice([0, 1, 7, 900, 5000, 40000, 120001]))
            F = int(g.choice([32, 64, 128]))
            keys, vals = W.gen_keys(max(n, 1), seed * 100 + i)
            keys, vals = keys[:n], vals[:n]
            t = BPlusTree.from_keys(keys, vals, fanout=F, leaf_fill=int(g.randint(1, 9)))
            q = np.concatenate([keys, W.gen_misses(max(n, 1), 100, seed * 100 + i)])
            v, f = t.search_batch(q, psa_bits=16 if i % 2 else 0)
            assert f[:n].all() and not f[n:].any() and np.array_equal(v[:n], vals) and not v[n:].any()
            if n:
                t.update(q, q)  # every miss becomes a key
                t.publish()
                v, f = t.search_batch(q)
                assert f.all() and np.array_equal(v, q)
            t.close()
    except BaseException as e:  # reported by the test's own thread
        out.append(e)


def test_reuse_across_threads(gpu):
    out = []
    ts = [threading.Thread(target=rounds, args=(s, out)) for s in range(1, 5)]
    for t in ts:
        t.start()
    for t in ts:
        t.join()
    assert not out, out


def test_memory_goes_back(gpu):
    import torch

    lib = load()
    lib.hm_device_synchronize()
    n = 3_000_000
    keys, vals = W.gen_keys(n, 9)
    free0 = torch.cuda.mem_get_info()[0]
    for _ in range(6):
        t = BPlusTree.from_keys(keys, vals)
        t.search_batch(keys[:1000])
        t.close()
        kept = free0 - torch.cuda.mem_get_info()[0]
        assert kept <= (512 << 20) + (64 << 20)  # the bound, and the runtime's own small blocks
    lib.hm_device_synchronize()
    assert free0 - torch.cuda.mem_get_info()[0] <= 64 << 20
