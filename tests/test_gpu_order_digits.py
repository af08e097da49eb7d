"""Sorting by one digit in LDS, around the number of keys that may share a digit (32): upsert batches (equal
keys: the last write wins) and builds with that many keys crowded into a small part of their range."""
import numpy as np
import pytest

from harmonia_amd import BPlusTree
from test_gpu_update_batches import check, epoch

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("crowd", [1, 31, 32, 33, 500])
@pytest.mark.parametrize("n", [4097, 20001])
@pytest.mark.parametrize("equal", [False, True])
def test_upsert_batches(gpu, crowd, n, equal):
    g = np.random.RandomState(crowd + n)
    keys = np.arange(1, 2001, dtype=np.uint64) * np.uint64(1 << 50)
    want = dict(zip(keys.tolist(), keys.tolist()))
    tree = BPlusTree.from_keys(keys, keys, keys_sorted=True, fanout=64, leaf_fill=6)
    k = g.randint(1, 1 << 62, n).astype(np.uint64)
    for c in range(0, n - crowd, 4096):  # in every chunk
        near = np.uint64(5 << 56) + g.randint(0, 1 if equal else 1 << 20, crowd).astype(np.uint64)
        k[c + g.choice(min(4096, n - c), crowd, replace=False)] = near
    v = g.randint(0, 1 << 63, n, dtype=np.uint64)
    epoch(tree, k, v, True)
    want.update(zip(k.tolist(), v.tolist()))
    check(tree, want)
    tree.close()


@pytest.mark.parametrize("crowd", [31, 32, 33, 2000])
@pytest.mark.parametrize("n", [3000, 60001])
def test_builds(gpu, crowd, n):
    import torch

    g = np.random.RandomState(crowd + n)
    near = (np.uint64(5 << 56) + g.choice(1 << 22, crowd, replace=False).astype(np.uint64))
    k = np.unique(np.concatenate([g.randint(1, 1 << 62, n - crowd).astype(np.uint64), near]))
    g.shuffle(k)
    v = g.randint(0, 1 << 63, len(k), dtype=np.uint64)
    dk, dv = (torch.from_numpy(x.view(np.int64)).cuda() for x in (k, v))
    torch.cuda.synchronize()
    tree = BPlusTree.from_keys(dk, dv, fanout=64, leaf_fill=7)
    check(tree, dict(zip(k.tolist(), v.tolist())))
    tree.close()
