"""Searches through the one-pass partition (PSA on, results in input order) at the sizes where its pieces
change: one query, a wave's 64, a wave's 512, chunks of 4096, tiles of 8192, the batch sizes where a digit
bit is added, results at odd addresses, every query equal, clustered keys, misses outside the key range, and
trees of one to four levels.  Against the oracle's sorted-array search; whole numbers, equal."""
import numpy as np
import pytest

import oracle
from harmonia_amd import BPlusTree, HM_KEY_MAX
from harmonia_amd import workloads as W

pytestmark = pytest.mark.gpu


def check(tree, sk, sv, q, odd=False, **opts):
    import torch

    n = len(q)
    o = 1 if odd else 0  # an odd element offset: 8-byte aligned keys and values, unaligned flags
    dq = torch.from_numpy(np.concatenate([np.zeros(o, np.uint64), q]).view(np.int64)).cuda()[o:]
    v = torch.full((n + 2,), -1, dtype=torch.int64, device="cuda")
    f = torch.full((n + 2,), 7, dtype=torch.uint8, device="cuda")
    torch.cuda.synchronize()
    tree.search_batch(dq, out_vals=v[o:o + n], out_found=f[o:o + n], psa_bits=16, **opts)
    torch.cuda.synchronize()
    ev, ef = oracle.search_sorted(sk, sv, q)
    v, f = v.cpu().numpy().view(np.uint64), f.cpu().numpy()
    assert np.array_equal(f[o:o + n], ef) and np.array_equal(v[o:o + n], ev)
    rest = np.r_[0:o, o + n:n + 2]
    assert (f[rest] == 7).all() and (v[rest] == HM_KEY_MAX).all()  # nothing beside the results


@pytest.mark.parametrize("F,n_keys", [(32, 1), (32, 200), (64, 9000), (64, 300007), (128, 70001)])
@pytest.mark.parametrize("odd", [False, True])
def test_partition_sizes(gpu, F, n_keys, odd):
    keys, vals = W.gen_keys(n_keys, 21)
    sk = np.sort(keys)
    sv = W.splitmix64_mix(sk)
    tree = BPlusTree.from_keys(keys, vals, fanout=F, leaf_fill=8 if F != 64 else 6)
    q = W.point_queries(sk, 30000, 5)
    for n in (1, 2, 63, 64, 65, 511, 513, 4095, 4096, 4097, 8191, 8192, 8193, 16385, 30000):
        check(tree, sk, sv, q[:n], odd)
    tree.close()


@pytest.mark.parametrize("n", [(1 << 20) - 3, (1 << 20) + 1, (1 << 21) + 1, (1 << 23) + 5])
def test_partition_digit_bits(gpu, n):
    keys, vals = W.gen_keys(1 << 18, 22)
    sk = np.sort(keys)
    sv = W.splitmix64_mix(sk)
    tree = BPlusTree.from_keys(keys, vals)
    check(tree, sk, sv, W.point_queries(sk, n, 6), odd=True)
    tree.close()


@pytest.mark.parametrize("F", [32, 64, 128])
@pytest.mark.parametrize("kind", ["equal", "clustered", "outside", "sorted", "dense ids", "key max"])
def test_partition_shapes(gpu, F, kind):
    g = np.random.RandomState(7)
    n_keys, n = 200003, 70001
    if kind == "clustered":  # half of the keys in a 2^-40 part of the range
        keys = np.unique(np.concatenate([g.randint(0, 1 << 62, n_keys // 2), (1 << 61) + g.randint(0, 1 << 22, n_keys // 2)]))
    elif kind == "dense ids":
        keys = np.arange(5000, 5000 + n_keys)
    else:
        keys = np.unique(g.randint(1 << 40, 1 << 50, n_keys))
    sk = keys.astype(np.uint64)
    sv = W.splitmix64_mix(sk)
    q = np.where(g.rand(n) < 0.8, sk[g.randint(0, len(sk), n)], g.randint(0, 1 << 51, n).astype(np.uint64))
    if kind == "equal":
        q[:] = sk[len(sk) // 2]
    elif kind == "outside":  # below, above, and with bits above the key range's top bit
        q = np.where(g.rand(n) < 0.5, q | np.uint64(1 << 62), q & np.uint64((1 << 30) - 1))
    elif kind == "sorted":
        q = np.sort(q)
    elif kind == "key max":
        q[g.rand(n) < 0.3] = np.uint64(HM_KEY_MAX)
        q[:100] = np.uint64(HM_KEY_MAX - 1)
    tree = BPlusTree.from_keys(sk, sv, keys_sorted=True, fanout=F, leaf_fill=8)
    check(tree, sk, sv, q)
    check(tree, sk, sv, q, lds_levels=0)
    tree.close()
