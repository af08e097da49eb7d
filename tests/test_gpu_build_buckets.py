"""Bulk builds at the sizes and key distributions where the bucket path changes: two keys, a wave, a tile of
8192, each number of digit bits, few varying bits, keys that crowd into one bucket (the radix path), equal
and reserved keys.  The device layout equals the oracle's build bit for bit."""
import numpy as np
import pytest

import oracle
from harmonia_amd import BPlusTree, HM_KEY_MAX, HarmoniaError
from harmonia_amd import workloads as W

pytestmark = pytest.mark.gpu


def check(keys, F, fill, device):
    vals = W.splitmix64_mix(keys)
    if device:
        import torch

        k, v = (torch.from_numpy(x.view(np.int64)).cuda() for x in (keys, vals))
        torch.cuda.synchronize()
    else:
        k, v = keys, vals
    t = BPlusTree.from_keys(k, v, fanout=F, leaf_fill=fill)
    e = t.export()
    sk = np.sort(keys)
    lay = oracle.build_bfs(sk, W.splitmix64_mix(sk), F, fill)
    assert np.array_equal(e["leaves"].reshape(-1), np.asarray(lay.leaves).reshape(-1).view(np.uint64))
    assert np.array_equal(e["inner"], lay.inner) and np.array_equal(e["prefix"], lay.prefix)
    s = t.stats()
    assert s.key_min == sk[0] and s.key_max == sk[-1] and s.n_keys == len(sk)
    t.close()


@pytest.mark.parametrize("n", [2, 3, 9, 63, 65, 1023, 8191, 8193, 50001, 1179648, 1179650, 2400001])
@pytest.mark.parametrize("fill,device", [(8, True), (5, False)])
def test_build_sizes(gpu, n, fill, device):
    check(W.gen_keys(n, 31)[0], 64, fill, device)


@pytest.mark.parametrize("F", [32, 64, 128])
@pytest.mark.parametrize("kind", ["crowded", "half crowded", "few bits", "dense", "low bits", "descending"])
def test_build_distributions(gpu, F, kind):
    g = np.random.RandomState(3)
    n = 60000
    keys = {"crowded": lambda: np.r_[np.uint64(1 << 60), np.arange(n, dtype=np.uint64)],
            "half crowded": lambda: np.r_[g.randint(1 << 50, 1 << 62, n // 2).astype(np.uint64), np.arange(n, dtype=np.uint64)],
            "few bits": lambda: np.arange(200, dtype=np.uint64) + np.uint64(5 << 40),
            "dense": lambda: np.arange(n, dtype=np.uint64) + np.uint64(12345),
            "low bits": lambda: np.unique(g.randint(0, 1 << 20, n).astype(np.uint64)) | np.uint64(0xABC << 50),
            "descending": lambda: np.sort(np.unique(g.randint(0, 1 << 62, n).astype(np.uint64)))[::-1].copy()}[kind]()
    keys = np.unique(keys)
    if kind != "descending":
        g.shuffle(keys)
    check(keys, F, 7, True)


@pytest.mark.parametrize("n", [3, 5000, 200000])
@pytest.mark.parametrize("where", [0, 1])
def test_build_rejects(gpu, n, where):
    keys = W.gen_keys(n, 33)[0]
    bad = keys.copy()
    bad[-1 if where else 0] = bad[n // 2]
    with pytest.raises(HarmoniaError, match="duplicate"):
        BPlusTree.from_keys(bad, bad)
    bad = keys.copy()
    bad[-1 if where else 0] = np.uint64(HM_KEY_MAX)
    with pytest.raises(HarmoniaError, match="reserved"):
        BPlusTree.from_keys(bad, bad)
