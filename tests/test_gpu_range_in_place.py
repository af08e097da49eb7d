"""Range scans whose counts take the place of their lengths in device memory: the offsets are those of the lengths, at
the sizes where the offsets' kernel changes."""
import numpy as np
import pytest

from harmonia_amd import BPlusTree, load

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n", [1, 2, 65, 300, 2048, 2049, 20000])
@pytest.mark.parametrize("F", [32, 64, 128])
def test_counts_over_lengths(gpu, F, n):
    import torch

    n_keys = 100000
    sk = np.arange(1, n_keys + 1, dtype=np.uint64) * np.uint64(10)
    tree = BPlusTree.from_keys(sk, sk + np.uint64(3), keys_sorted=True, fanout=F, leaf_fill=7)
    g = np.random.RandomState(n)
    lens = g.randint(0, 90, n).astype(np.uint32)
    # every second range starts near the last key or past it, so that its count is below its length
    start = np.where(np.arange(n) % 2 == 0, g.randint(0, 10 * n_keys, n), 10 * n_keys - 200 + g.randint(0, 400, n))
    first = np.searchsorted(sk, start.astype(np.uint64))
    want_n = np.minimum(lens, n_keys - first).astype(np.uint32)
    want_off = np.concatenate([[0], np.cumsum(lens, dtype=np.int64)])
    cap = int(want_off[-1])
    ds = torch.from_numpy(start.astype(np.int64)).cuda()
    lc = torch.from_numpy(lens.view(np.int32)).cuda()
    off = torch.zeros(n + 1, dtype=torch.int64, device="cuda")
    k, v = (torch.zeros(max(cap, 1), dtype=torch.int64, device="cuda") for _ in range(2))
    torch.cuda.synchronize()
    rc = load().hm_range(tree._handle(), ds.data_ptr(), lc.data_ptr(), n, off.data_ptr(), k.data_ptr(), v.data_ptr(),
                         lc.data_ptr(), cap, None)
    torch.cuda.synchronize()
    assert rc == 0
    assert np.array_equal(off.cpu().numpy(), want_off) and np.array_equal(lc.cpu().numpy().view(np.uint32), want_n)
    want = np.zeros(cap, dtype=np.int64)
    for i in range(n):
        want[want_off[i]:want_off[i] + want_n[i]] = sk[first[i]:first[i] + want_n[i]].astype(np.int64)
    assert np.array_equal(k.cpu().numpy()[:cap], want)
    assert np.array_equal(v.cpu().numpy()[:cap], np.where(want, want + 3, 0))
    tree.close()
