"""Closed intervals on both sides of the sizes where their kernel changes, capacities below and above the line
for long ones, trees with full and with half-empty leaves.  Against numpy's searchsorted."""
import numpy as np
import pytest

from harmonia_amd import BPlusTree, HM_KEY_MAX
from harmonia_amd import workloads as W

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("F,fill", [(32, 8), (64, 4), (128, 7)])
@pytest.mark.parametrize("n,cap", [(12288, 9), (12289, 9), (12289, 63), (12289, 64), (49152, 64), (49153, 64), (49153, 70)])
def test_intervals(gpu, F, fill, n, cap):
    g = np.random.RandomState(n + cap)
    sk = np.unique(g.randint(1, 1 << 62, 40011)).astype(np.uint64)
    sv = W.splitmix64_mix(sk)
    tree = BPlusTree.from_keys(sk, sv, keys_sorted=True, fanout=F, leaf_fill=fill)
    a = g.randint(0, len(sk), n)
    b = np.minimum(a + g.randint(0, 2 * cap, n), len(sk) - 1)
    lo, hi = sk[a].copy(), sk[b].copy()
    lo[::3] += np.uint64(1)  # between keys
    hi[::5] -= np.uint64(1)
    lo[0], hi[0] = 0, HM_KEY_MAX - 1
    lo[1], hi[1] = hi[2], lo[2]
    lo[3], hi[3] = sk[-1] + np.uint64(1), HM_KEY_MAX
    lo[4], hi[4] = HM_KEY_MAX, HM_KEY_MAX
    lo[n - 1], hi[n - 1] = sk[-3], HM_KEY_MAX
    k, v, c = tree.range_between(lo, hi, cap)
    k, v = np.asarray(k).reshape(n, cap), np.asarray(v).reshape(n, cap)
    i = np.searchsorted(sk, lo, "left")
    e = np.searchsorted(sk, hi, "right")
    want = np.minimum(np.maximum(e - i, 0), cap)
    assert np.array_equal(np.asarray(c), want)
    slot = np.arange(cap)
    on = slot < want[:, None]
    at = np.minimum(i[:, None] + slot, len(sk) - 1)
    assert np.array_equal(k[on], sk[at][on]) and np.array_equal(v[on], sv[at][on])
    tree.close()
