"""Searches sorted by few bits, results in input order, of trees whose keys differ only in a few low bits: the
partition's digit may be wider than the bits that order the tree's keys, or than the bits asked for."""
import numpy as np
import pytest

import oracle
from harmonia_amd import Batcher, BPlusTree, HM_KEY_MAX
from harmonia_amd import workloads as W

pytestmark = pytest.mark.gpu


def inputs(n_keys, base, n):
    sk = np.uint64(base) + np.arange(n_keys, dtype=np.uint64)
    g = np.random.RandomState(n & 0xFFFF)
    q = np.uint64(base) + g.randint(0, 2 * n_keys, n).astype(np.uint64)
    far = g.randint(0, n, 1000)  # bits above every key's
    q[far] = g.randint(0, 1 << 62, 1000).astype(np.uint64)
    q[far[:50]] = np.uint64(HM_KEY_MAX)
    return sk, W.splitmix64_mix(sk), q


@pytest.mark.parametrize("bits", [9, 10, 11, 12, 16])
@pytest.mark.parametrize("n", [1000, (1 << 21) + 512, (1 << 22) + (1 << 13)])
@pytest.mark.parametrize("n_keys,base", [(1, 0), (500, 0), (1000, 0), (500, 7 << 40)])
def test_few_bits(gpu, bits, n, n_keys, base):
    import torch

    sk, sv, q = inputs(n_keys, base, n)
    tree = BPlusTree.from_keys(sk, sv, keys_sorted=True, fanout=64, leaf_fill=6)
    dq = torch.from_numpy(q.view(np.int64)).cuda()
    v, f = torch.full_like(dq, -1), torch.full((n,), 7, dtype=torch.uint8, device="cuda")
    torch.cuda.synchronize()
    tree.search_batch(dq, out_vals=v, out_found=f, psa_bits=bits)
    torch.cuda.synchronize()
    ev, ef = oracle.search_sorted(sk, sv, q)
    assert np.array_equal(f.cpu().numpy(), ef) and np.array_equal(v.cpu().numpy().view(np.uint64), ev)
    tree.close()


def test_few_bits_in_a_captured_pipeline(gpu):
    sk, sv, q = inputs(500, 0, 70001)
    tree = BPlusTree.from_keys(sk, sv, keys_sorted=True)
    b = Batcher(tree, (1 << 22) + (1 << 13), psa_bits=9)
    ev, ef = oracle.search_sorted(sk, sv, q)
    for m in (70001, 300, 70001):
        off = b.add(q[:m])
        b.flush()
        v, f = b.copy_out(off, m)
        assert np.array_equal(f, ef[:m]) and np.array_equal(v, ev[:m])
    b.close()
    tree.close()
