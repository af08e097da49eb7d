"""Range scans and closed intervals on both sides of the sizes where another kernel takes them, ranges that are short,
long, empty or past the last key, leaves full and nearly empty.  And fewer closed intervals do not take longer than
more of them."""
import numpy as np
import pytest

from harmonia_amd import BPlusTree, load

pytestmark = pytest.mark.gpu
N_KEYS = 60000
SK = np.arange(1, N_KEYS + 1, dtype=np.uint64) * np.uint64(10)


def zeros(n, dtype):
    import torch

    return torch.zeros(max(int(n), 1), dtype=dtype, device="cuda")


def expect(first, count, offset, cap):
    """Keys at their places: count[i] keys from SK[first[i]] at offset[i]."""
    j = np.arange(int(count.sum())) - np.repeat(np.cumsum(count) - count, count)
    want = np.zeros(cap, dtype=np.int64)
    want[np.repeat(offset, count) + j] = SK[np.repeat(first, count) + j].astype(np.int64)
    return want


@pytest.mark.parametrize("F,fill", [(32, 1), (64, 8), (128, 5)])
@pytest.mark.parametrize("n", [4096, 4097, 16384, 16385, 65536, 65537])
@pytest.mark.parametrize("most", [3, 140])
def test_ranges(gpu, F, fill, n, most):
    import torch

    tree = BPlusTree.from_keys(SK, SK + np.uint64(1), keys_sorted=True, fanout=F, leaf_fill=fill)
    g = np.random.RandomState(n + most)
    lens = g.randint(0, most + 1, n).astype(np.uint32)
    start = g.randint(0, 10 * N_KEYS + 50, n).astype(np.uint64)
    start[:3] = [0, 10 * N_KEYS, np.uint64(2**64 - 1)]
    first = np.searchsorted(SK, start)
    count = np.minimum(lens, N_KEYS - first).astype(np.int64)
    off = np.concatenate([[0], np.cumsum(lens, dtype=np.int64)])
    cap = int(off[-1])
    ds = torch.from_numpy(start.view(np.int64)).cuda()
    dl = torch.from_numpy(lens.view(np.int32)).cuda()
    do, dk, dv, dc = zeros(n + 1, torch.int64), zeros(cap, torch.int64), zeros(cap, torch.int64), zeros(n, torch.int32)
    torch.cuda.synchronize()
    rc = load().hm_range(tree._handle(), ds.data_ptr(), dl.data_ptr(), n, do.data_ptr(), dk.data_ptr(), dv.data_ptr(),
                         dc.data_ptr(), cap, None)
    torch.cuda.synchronize()
    assert rc == 0 and np.array_equal(do.cpu().numpy(), off) and np.array_equal(dc.cpu().numpy(), count)
    want = expect(first, count, off[:-1], cap)
    assert np.array_equal(dk.cpu().numpy(), want) and np.array_equal(dv.cpu().numpy(), np.where(want, want + 1, 0))
    tree.close()


@pytest.mark.parametrize("F,fill", [(32, 1), (64, 8), (128, 5)])
@pytest.mark.parametrize("n", [4096, 4097, 20000])
@pytest.mark.parametrize("most,cap", [(3, 3), (40, 256), (300, 256)])
def test_intervals(gpu, F, fill, n, most, cap):
    import torch

    tree = BPlusTree.from_keys(SK, SK + np.uint64(1), keys_sorted=True, fanout=F, leaf_fill=fill)
    g = np.random.RandomState(n + most)
    lo = g.randint(0, 10 * N_KEYS + 50, n).astype(np.uint64)
    hi = lo + g.randint(0, 10 * most, n).astype(np.uint64)
    lo[:2], hi[:2] = [30, np.uint64(2**64 - 1)], [20, np.uint64(2**64 - 1)]
    first = np.searchsorted(SK, lo)
    count = np.clip(np.searchsorted(SK, hi, side="right") - first, 0, cap)
    dlo, dhi = (torch.from_numpy(x.view(np.int64)).cuda() for x in (lo, hi))
    dk, dv, dc = zeros(n * cap, torch.int64), zeros(n * cap, torch.int64), zeros(n, torch.int32)
    torch.cuda.synchronize()
    rc = load().hm_range_between(tree._handle(), dlo.data_ptr(), dhi.data_ptr(), n, cap, dk.data_ptr(), dv.data_ptr(),
                                 dc.data_ptr(), None)
    torch.cuda.synchronize()
    assert rc == 0 and np.array_equal(dc.cpu().numpy(), count)
    want = expect(first, count, np.arange(n) * cap, n * cap)
    assert np.array_equal(dk.cpu().numpy(), want) and np.array_equal(dv.cpu().numpy(), np.where(want, want + 1, 0))
    tree.close()


def test_fewer_intervals_take_no_longer(gpu):
    """Intervals of up to 40 keys with room for 256: by a graph of 20 calls, so that device time counts."""
    import torch

    lib, cap, calls = load(), 256, 20
    keys = torch.arange(1, (1 << 22) + 1, dtype=torch.int64, device="cuda") * 10
    torch.cuda.synchronize()
    tree = BPlusTree.from_keys(keys, keys, keys_sorted=True)
    s = torch.cuda.Stream()
    us = {}
    for n in (4097, 12289, 24576, 49152, 60000):
        i = torch.randint(0, len(keys) - 40, (n,), device="cuda")
        lo, hi = keys[i], keys[i + torch.randint(0, 40, (n,), device="cuda")]
        dk, dv, dc = zeros(n * cap, torch.int64), zeros(n * cap, torch.int64), zeros(n, torch.int32)
        a = (tree._handle(), lo.data_ptr(), hi.data_ptr(), n, cap, dk.data_ptr(), dv.data_ptr(), dc.data_ptr(), s.cuda_stream)
        torch.cuda.synchronize()
        assert lib.hm_range_between(*a) == 0  # the stream's workspace is there
        s.synchronize()
        g = torch.cuda.CUDAGraph()
        with torch.cuda.graph(g, stream=s):
            for _ in range(calls):
                assert lib.hm_range_between(*a) == 0
        t = []
        for _ in range(6):
            e0, e1 = (torch.cuda.Event(enable_timing=True) for _ in range(2))
            with torch.cuda.stream(s):
                e0.record()
                g.replay()
                e1.record()
            s.synchronize()
            t.append(e0.elapsed_time(e1) * 1e3 / calls)
        us[n] = min(t)
        del g
    print({n: round(t, 1) for n, t in us.items()})
    sizes = sorted(us)
    assert all(us[a] < 1.4 * us[b] for a, b in zip(sizes, sizes[1:]))
    tree.close()
