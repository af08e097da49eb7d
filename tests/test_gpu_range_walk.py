"""Range scans at the sizes where the wave walk and its launch rules change: one range per wave and eight,
offsets computed in the kernel and by the scan, lengths around a leaf and a step, leaves with free slots,
output capacities that cut a pair of stores, and lengths past every key.  Whole numbers: equal."""
import ctypes

import numpy as np
import pytest

import oracle
from harmonia_amd import BPlusTree, load
from harmonia_amd import workloads as W

pytestmark = pytest.mark.gpu


def scan(tree, starts, lens, cap):
    import torch

    n = len(starts)
    d = lambda a, t: torch.from_numpy(np.ascontiguousarray(a).view(t)).cuda()
    s, ln = d(starts, np.int64), d(lens, np.int32)
    off = torch.full((n + 1,), -1, dtype=torch.int64, device="cuda")
    k, v = (torch.zeros(max(cap, 1) + 2, dtype=torch.int64, device="cuda") for _ in range(2))
    c = torch.full((n,), -1, dtype=torch.int32, device="cuda")
    torch.cuda.synchronize()
    assert load().hm_range(tree._handle(), s.data_ptr(), ln.data_ptr(), n, off.data_ptr(), k.data_ptr(), v.data_ptr(),
                           c.data_ptr(), ctypes.c_uint64(cap), None) == 0
    torch.cuda.synchronize()
    return (off.cpu().numpy().view(np.uint64), k.cpu().numpy().view(np.uint64), v.cpu().numpy().view(np.uint64),
            c.cpu().numpy().view(np.uint32))


@pytest.mark.parametrize("F,fill", [(32, 8), (64, 5), (128, 8), (128, 1)])
@pytest.mark.parametrize("n", [1, 3, 2048, 2049, 16384, 16387])
def test_range_walk_sizes(gpu, F, fill, n):
    keys, vals = W.gen_keys(30011, 5)
    sk = np.sort(keys)
    sv = W.splitmix64_mix(sk)
    g = np.random.RandomState(n)
    starts = np.where(g.rand(n) < 0.5, sk[g.randint(0, len(sk), n)], g.randint(0, 1 << 63, n).astype(np.uint64))
    lens = g.choice([0, 1, 2, 7, 8, 9, 63, 64, 65, 247, 257], n).astype(np.uint32)
    starts[0], lens[0] = sk[-1], 9
    tree = BPlusTree.from_keys(keys, vals, fanout=F, leaf_fill=fill)
    total = int(lens.sum())
    eo, ek, ev, ec = oracle.range_sorted(sk, sv, starts, lens=lens)
    off, k, v, c = scan(tree, starts, lens, total)
    assert np.array_equal(off, eo) and np.array_equal(c, ec)
    for cap in (total, total // 2 | 1):  # an odd capacity ends inside a two-pair store
        if cap != total:
            off, k, v, c = scan(tree, starts, lens, cap)
            assert np.array_equal(off, eo) and np.array_equal(c, ec)
        written = np.concatenate([np.arange(o, o + m) for o, m in zip(eo[:-1].astype(np.int64), ec.astype(np.int64))])
        written = written[written < cap]
        exp = np.zeros(len(k), dtype=np.uint64)
        exp[written] = ek[written]
        assert np.array_equal(k, exp)  # and nothing anywhere else
        exp[written] = ev[written]
        assert np.array_equal(v, exp)
    tree.close()


@pytest.mark.parametrize("fill", [3, 8])
def test_range_longer_than_tree(gpu, fill):
    """A length near 2^32 from the first key returns every key, whatever the leaves' fill."""
    keys, vals = W.gen_keys(1001, 6)
    sk = np.sort(keys)
    tree = BPlusTree.from_keys(keys, vals, fanout=32, leaf_fill=fill)
    off, k, v, c = scan(tree, np.zeros(1, dtype=np.uint64), np.array([0xFFFFFFFF], dtype=np.uint32), 1001)
    assert int(c[0]) == 1001 and int(off[1]) == 0xFFFFFFFF
    assert np.array_equal(k[:1001], sk) and np.array_equal(v[:1001], W.splitmix64_mix(sk))
    lo, hi = sk[[10, 500, 1000]], sk[[17, 500, 1000]]
    bk, bv, bc = tree.range_between(lo, hi, 9)
    assert bc.tolist() == [8, 1, 1] and np.array_equal(bk[:8], sk[10:18]) and bk[9] == sk[500] and bk[18] == sk[1000]
    tree.close()
