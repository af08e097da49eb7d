"""Upsert epochs at the batch sizes where the sort, the de-duplication and the plan change: one key, the
blocks of 16 and 32 entries, the tiles of 2048 and 4096 and their remainders, batches of one repeated key,
keys that all fall into one leaf or past every stored key.  The tree after the epoch holds exactly the
dictionary's keys and values (last write wins)."""
import numpy as np
import pytest

from harmonia_amd import BPlusTree
from harmonia_amd import workloads as W

pytestmark = pytest.mark.gpu


def epoch(tree, k, v, device):
    if device:
        import torch

        dk, dv = (torch.from_numpy(x.view(np.int64)).cuda() for x in (k, v))
        torch.cuda.synchronize()
        tree.update(dk, dv)
    else:
        tree.update(k, v)
    tree.publish()


def check(tree, want):
    k = np.array(sorted(want), dtype=np.uint64)
    v = np.array([want[int(x)] for x in k], dtype=np.uint64)
    leaves = tree.export()["leaves"]
    got_k, got_v = leaves[:, :8].reshape(-1), leaves[:, 8:].reshape(-1)
    stored = got_k != np.uint64(0xFFFFFFFFFFFFFFFF)
    assert np.array_equal(got_k[stored], k) and np.array_equal(got_v[stored], v)
    ov, of = tree.search_batch(k)
    assert of.all() and np.array_equal(ov, v)


@pytest.mark.parametrize("n", [1, 2, 15, 17, 31, 33, 2047, 4095, 4096, 4097, 6143, 8193, 20001])
@pytest.mark.parametrize("device", [False, True])
def test_epoch_sizes(gpu, n, device):
    keys, _ = W.gen_keys(9001, 11)
    g = np.random.RandomState(n)
    want = dict(zip(keys.tolist(), W.splitmix64_mix(keys).tolist()))
    tree = BPlusTree.from_keys(keys, W.splitmix64_mix(keys), fanout=32, leaf_fill=5)
    miss = W.gen_misses(len(keys), 3 * n, 11)
    for step in range(3):  # stored keys, new ones, and a third of the batch written twice
        k = np.where(g.rand(n) < 0.9, keys[g.randint(0, len(keys), n)], miss[step * n:(step + 1) * n])
        k = np.where(g.rand(n) < 0.3, k[g.randint(0, n, n)], k)
        v = g.randint(0, 1 << 63, n, dtype=np.uint64)
        epoch(tree, k, v, device)
        want.update(zip(k.tolist(), v.tolist()))
        check(tree, want)
    tree.close()


@pytest.mark.parametrize("n", [40, 4096, 5000, 12289])
@pytest.mark.parametrize("kind", ["one key", "one leaf", "past the end", "below", "descending"])
def test_epoch_shapes(gpu, n, kind):
    keys = np.arange(1, 3001, dtype=np.uint64) * np.uint64(1 << 40)
    want = dict(zip(keys.tolist(), keys.tolist()))
    tree = BPlusTree.from_keys(keys, keys, fanout=64, leaf_fill=8)
    i = np.arange(n, dtype=np.uint64)
    g = np.random.RandomState(n)
    k = {"one key": np.full(n, keys[77]), "one leaf": keys[1600] + np.uint64(1) + i, "past the end": keys[-1] + i,
         "below": i, "descending": (keys[-1] + np.uint64(n) - i)}[kind]
    if kind != "descending":
        k = k[g.permutation(n)]
    v = g.randint(0, 1 << 63, n, dtype=np.uint64)
    epoch(tree, k, v, True)
    want.update(zip(k.tolist(), v.tolist()))
    check(tree, want)
    tree.close()
