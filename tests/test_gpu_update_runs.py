"""Upsert epochs whose batch crowds: long runs of new keys between and over one leaf's keys (splits counted in
32 and in 64 bits), appended runs, overflowing leaves at every place of their node's entries, and more nodes
to re-spread than a block of the plan lists.  The tree holds exactly the dictionary's keys and values."""
import numpy as np
import pytest

from harmonia_amd import BPlusTree
from test_gpu_update_batches import check, epoch

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("F,fill", [(32, 1), (64, 5), (128, 8)])
@pytest.mark.parametrize("n", [9, 200, 65530, 70003])
@pytest.mark.parametrize("kind", ["between", "over", "append", "all below"])
def test_long_runs(gpu, F, fill, n, kind):
    keys = (np.arange(1, 2501, dtype=np.uint64)) * np.uint64(1 << 20)
    want = dict(zip(keys.tolist(), keys.tolist()))
    tree = BPlusTree.from_keys(keys, keys, keys_sorted=True, fanout=F, leaf_fill=fill)
    g = np.random.RandomState(n)
    i = np.arange(n, dtype=np.uint64)
    for step in range(2):
        if kind == "between":  # one leaf, between two of its keys
            k = keys[1200] + np.uint64(1) + i + np.uint64(step * n)
        elif kind == "over":  # four keys of one leaf or two, each overwritten, and new keys around them
            k = np.concatenate([keys[1200:1204], keys[1199] + np.uint64(5 + step) + i * np.uint64((5 << 20) // n)])
        elif kind == "append":
            k = np.concatenate([keys[-2:], keys[-1] + np.uint64(1) + i + np.uint64(step * n)])
        else:
            k = np.uint64(step * n) + i
        k = k[g.permutation(len(k))]
        v = g.randint(0, 1 << 63, len(k), dtype=np.uint64)
        epoch(tree, k, v, True)
        want.update(zip(k.tolist(), v.tolist()))
        check(tree, want)
    tree.close()


@pytest.mark.parametrize("F", [32, 64, 128])
@pytest.mark.parametrize("at", [0, 1, 17, -1])
@pytest.mark.parametrize("per_leaf", [0, 1, 2])
def test_overflow_at_each_place_of_a_node(gpu, F, at, per_leaf):
    """Leaf `at` of three nodes gets three keys for two free slots, every leaf `per_leaf` besides."""
    nodes = 7
    keys = np.arange(1, nodes * F * 6 + 1, dtype=np.uint64) * np.uint64(100)  # 6 keys to a leaf
    want = dict(zip(keys.tolist(), keys.tolist()))
    tree = BPlusTree.from_keys(keys, keys, keys_sorted=True, fanout=F, leaf_fill=6)
    first = keys[::6]
    over = np.concatenate([first[n * F + at % F] + np.array([1, 2, 3], np.uint64) for n in (0, 3, 6)])
    k = np.concatenate([over] + [first + np.uint64(50 + j) for j in range(per_leaf)])
    epoch(tree, k, k, True)
    assert tree.stats().relayouts == (1 if F * (6 + per_leaf) + 3 > 8 * F else 0)
    want.update(zip(k.tolist(), k.tolist()))
    check(tree, want)
    tree.close()


def test_more_nodes_than_a_block_lists(gpu):
    """Two new keys for one free slot in a leaf of each of 300000 nodes: a block of the plan sees 293."""
    import torch

    F, fill, nodes = 32, 7, 300000
    keys = torch.arange(1, nodes * F * fill + 1, dtype=torch.int64, device="cuda") * 16
    torch.cuda.synchronize()
    tree = BPlusTree.from_keys(keys, keys, keys_sorted=True, fanout=F, leaf_fill=fill)
    at = keys[3 * fill::F * fill]
    new = torch.stack([at + 1, at + 2], 1).reshape(-1).contiguous()
    torch.cuda.synchronize()
    tree.update(new, new)
    tree.publish()
    assert tree.stats().relayouts == 0
    for q in (new, keys):
        v, f = torch.empty_like(q), torch.empty(q.numel(), dtype=torch.uint8, device="cuda")
        torch.cuda.synchronize()
        tree.search_batch(q, out_vals=v, out_found=f)
        torch.cuda.synchronize()
        assert bool(f.all()) and torch.equal(v, q)
    tree.close()
