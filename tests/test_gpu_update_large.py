"""Epochs on both sides of the size where the batch's keys are located by the sorted searches' kernel, every fanout, few and
many repeated keys; and so many overflowing nodes that the blocks of the plan list more than fit in LDS.  The tree
holds exactly what a dictionary would."""
import numpy as np
import pytest

from harmonia_amd import BPlusTree

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("F", [32, 64, 128])
@pytest.mark.parametrize("n", [(1 << 17) - 1, 1 << 17, (1 << 17) + 1, (1 << 20) + 3])
@pytest.mark.parametrize("repeats", [False, True])
def test_located_batches(gpu, F, n, repeats):
    import torch

    g = np.random.RandomState(n % 1000 + F)
    stored = np.unique(g.randint(0, 1 << 62, 400000)).astype(np.uint64)
    tree = BPlusTree.from_keys(stored, stored, keys_sorted=True, fanout=F, leaf_fill=5)
    k = np.where(g.rand(n) < 0.8, stored[g.randint(0, len(stored), n)], g.randint(0, 1 << 62, n).astype(np.uint64))
    k[:2] = [0, np.uint64(2**64 - 2)]  # below and above every stored key
    if repeats:
        k = k[g.randint(0, n // 50, n)]
    v = g.randint(0, 1 << 63, n).astype(np.uint64)
    dk, dv = (torch.from_numpy(x.view(np.int64)).cuda() for x in (k, v))
    torch.cuda.synchronize()
    tree.update(dk, dv)
    tree.publish()
    new_k, last = np.unique(k[::-1], return_index=True)  # the last write of each key
    want_k = np.union1d(stored, new_k)
    want_v = want_k.copy()
    want_v[np.searchsorted(want_k, new_k)] = v[::-1][last]
    leaves = tree.export()["leaves"]
    got_k, got_v = leaves[:, :8].reshape(-1), leaves[:, 8:].reshape(-1)
    there = got_k != np.uint64(2**64 - 1)
    assert np.array_equal(got_k[there], want_k) and np.array_equal(got_v[there], want_v)
    assert tree.stats().n_keys == len(want_k)
    ov, of = tree.search_batch(want_k)
    assert of.all() and np.array_equal(ov, want_v)
    tree.close()


def test_plan_lists_that_spill(gpu):
    """Eight new keys for the seven free slots of a leaf in each of 300000 nodes: each of the plan's 256 blocks finds
    some 1170 of them, and its list in LDS holds 1024."""
    import torch

    F, nodes = 32, 300000
    keys = torch.arange(1, nodes * F + 1, dtype=torch.int64, device="cuda") * 16
    at = keys[5::F]
    new = (at[:, None] + torch.arange(1, 9, device="cuda")).reshape(-1).contiguous()
    torch.cuda.synchronize()
    tree = BPlusTree.from_keys(keys, keys, keys_sorted=True, fanout=F, leaf_fill=1)
    tree.update(new, new)
    assert not tree.publish()
    assert tree.stats().respreads == nodes and tree.stats().n_keys == len(keys) + len(new)
    for q in (new, keys):
        v, f = torch.zeros_like(q), torch.zeros(q.numel(), dtype=torch.uint8, device="cuda")
        torch.cuda.synchronize()
        tree.search_batch(q, out_vals=v, out_found=f)
        torch.cuda.synchronize()
        assert bool(f.all()) and torch.equal(v, q)
    tree.close()
