"""The tuner times a pipeline that has neither a sort width nor blocks per CU of its own once, so that noise does not
pick those: where the partitioned search wins, they are the defaults."""
import numpy as np
import pytest

from harmonia_amd import BPlusTree
from harmonia_amd import workloads as W

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("seed", range(4))
def test_partitioned_search_is_timed_once(gpu, seed):
    n = 1 << 20
    keys, vals = W.gen_keys(n, 51)
    sk = np.sort(keys)
    q = W.point_queries(sk, n, seed)
    tree = BPlusTree.from_keys(keys, vals)
    r = tree.autotune(q, quick=True)
    shape = (r["psa_group"], r["psa_queries_per_group"], r["output_mode"])
    print(shape, r["psa_bits"], r["psa_blocks_per_cu"], r["psa_ms"], r["direct_ms"])
    if shape == (2, 4, 1) and r["psa_bits"] <= 16:
        assert (r["psa_bits"], r["psa_blocks_per_cu"]) == (16, 10)
    v, f = tree.search_batch(q[:5000])
    i = np.searchsorted(sk, q[:5000]).clip(0, n - 1)
    assert np.array_equal(f == 1, sk[i] == q[:5000])
    tree.close()
