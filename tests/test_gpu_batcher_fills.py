"""Batchers on the sorted path filled to any part of their capacity, fills of different sizes one after the other:
tiles of 8192 and chunks of 2048 and 4096, their remainders and eighths.  And a small flush takes about as long in a
large batcher as in a small one."""
import time

import numpy as np
import pytest

import oracle
from harmonia_amd import Batcher, BPlusTree
from harmonia_amd import workloads as W

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("cap", [70001, (1 << 22) + 12345])
def test_fills(gpu, cap):
    keys, vals = W.gen_keys(200003, 61)
    sk = np.sort(keys)
    sv = W.splitmix64_mix(sk)
    tree = BPlusTree.from_keys(keys, vals)
    q = W.point_queries(sk, cap, 62)
    ev, ef = oracle.search_sorted(sk, sv, q)
    b = Batcher(tree, cap, psa_bits=16)
    fills = [cap, 1, cap // 8, cap // 8 + 1, 8191, 8192, 8193, 2049, 4097, 65536, 65537, cap // 2, cap - 1, 63, cap]
    for m in fills:
        at = (cap - m) // 3
        off = b.add(q[at:at + m])
        b.flush()
        v, f = b.copy_out(off, m)
        assert np.array_equal(f, ef[at:at + m]) and np.array_equal(v, ev[at:at + m])
    b.close()
    tree.close()


def test_small_flush_of_a_large_batcher(gpu):
    import torch

    keys, vals = W.gen_keys(1 << 22, 63)
    tree = BPlusTree.from_keys(keys, vals)
    n = 1 << 20
    q = torch.from_numpy(W.point_queries(np.sort(keys), n, 64).view(np.int64)).cuda()
    torch.cuda.synchronize()
    times = {}
    for cap in (n, n << 7):
        b = Batcher(tree, cap, psa_bits=16)
        best = []
        for _ in range(12):
            t0 = time.perf_counter()
            for _ in range(10):
                b.add(q)
                b.flush()
            b.sync()
            best.append(time.perf_counter() - t0)
        times[cap] = min(best) / 10
        b.close()
    print({c: round(t * 1e6, 1) for c, t in times.items()})
    assert times[n << 7] < 3 * times[n]
    tree.close()
