"""A search that names one descent per query, or the shape of that kernel, gets it: two sort passes in front of it
and two behind, where the tree's own choice makes one partition pass.  Results are the same."""
import ctypes

import numpy as np
import pytest

import oracle
from harmonia_amd import BPlusTree, load
from harmonia_amd import workloads as W

pytestmark = pytest.mark.gpu

NAMED = [dict(sorted_kernel=1), dict(group_size=2), dict(queries_per_group=4), dict(blocks_per_cu=5), dict(lds_levels=0),
         dict(group_size=2, queries_per_group=4, lds_levels=1, blocks_per_cu=10)]


def launches(lib, stage):
    ms, n = ctypes.c_double(0), ctypes.c_uint64(0)
    lib.hm_profile_get(stage, ctypes.byref(ms), ctypes.byref(n))
    return n.value


@pytest.mark.parametrize("opts,passes", [({}, 1)] + [(o, 2) for o in NAMED])
@pytest.mark.parametrize("bits", [9, 16])
def test_named_kernel(gpu, opts, passes, bits):
    keys, vals = W.gen_keys(40000, 31)
    sk = np.sort(keys)
    q = W.point_queries(sk, 60001, 8)
    tree = BPlusTree.from_keys(keys, vals)
    lib = load()
    lib.hm_profile_reset()
    lib.hm_profile_enable(1)
    try:
        v, f = tree.search_batch(q, psa_bits=bits, **opts)
        assert (launches(lib, b"psa_scatter"), launches(lib, b"search")) == (passes, 1)
    finally:
        lib.hm_profile_enable(0)
        lib.hm_profile_reset()
    ev, ef = oracle.search_sorted(sk, W.splitmix64_mix(sk), q)
    assert np.array_equal(f, ef) and np.array_equal(v, ev)
    tree.close()
