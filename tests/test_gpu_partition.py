"""Searches through the one-pass partition (PSA on, results in input order) at the sizes where its pieces
change: one query, a wave's 64, a wave's 512, chunks of 2048 and 4096, tiles of 8192, the batch sizes where a digit
bit is added, results at odd addresses, every query equal, clustered keys, misses outside the key range, and
trees of one to four levels.  Against the oracle's sorted-array search; whole numbers, equal."""
import numpy as np
import pytest

import oracle
from harmonia_amd import BPlusTree, HM_KEY_MAX
from harmonia_amd import workloads as W

pytestmark = pytest.mark.gpu


def check(tree, sk, sv, q, odd=False, **opts):
    import torch

    n = len(q)
    o = 1 if odd else 0  # an odd element offset: 8-byte aligned keys and values, unaligned flags
    dq = torch.from_numpy(np.concatenate([np.zeros(o, np.uint64), q]).view(np.int64)).cuda()[o:]
    v = torch.full((n + 2,), -1, dtype=torch.int64, device="cuda")
    f = torch.full((n + 2,), 7, dtype=torch.uint8, device="cuda")
    torch.cuda.synchronize()
    tree.search_batch(dq, out_vals=v[o:o + n], out_found=f[o:o + n], psa_bits=16, **opts)
    torch.cuda.synchronize()
    ev, ef = oracle.search_sorted(sk, sv, q)
    v, f = v.cpu().numpy().view(np.uint64), f.cpu().numpy()
    assert np.array_equal(f[o:o + n], ef) and np.array_equal(v[o:o + n], ev)
    rest = np.r_[0:o, o + n:n + 2]
    assert (f[rest] == 7).all() and (v[rest] == HM_KEY_MAX).all()  # nothing beside the results


@pytest.mark.parametrize("F,n_keys", [(32, 1), (32, 200), (64, 9000), (64, 300007), (128, 70001)])
@pytest.mark.parametrize("odd", [False, True])
def test_partition_sizes(gpu, F, n_keys, odd):
    keys, vals = W.gen_keys(n_keys, 21)
    sk = np.sort(keys)
    sv = W.splitmix64_mix(sk)
    tree = BPlusTree.from_keys(keys, vals, fanout=F, leaf_fill=8 if F != 64 else 6)
    q = W.point_queries(sk, 30000, 5)
    for n in (1, 2, 63, 64, 65, 511, 513, 4095, 4096, 4097, 8191, 8192, 8193, 16385, 30000):
        check(tree, sk, sv, q[:n], odd)
    tree.close()


@pytest.mark.parametrize("n", [(1 << 20) - 3, (1 << 20) + 1, (1 << 21) + 1, (1 << 23) + 5])
def test_partition_digit_bits(gpu, n):
    keys, vals = W.gen_keys(1 << 18, 22)
    sk = np.sort(keys)
    sv = W.splitmix64_mix(sk)
    tree = BPlusTree.from_keys(keys, vals)
    check(tree, sk, sv, W.point_queries(sk, n, 6), odd=True)
    tree.close()


@pytest.mark.parametrize("F", [32, 64, 128])
@pytest.mark.parametrize("kind", ["equal", "clustered", "outside", "sorted", "dense ids", "key max"])
def test_partition_shapes(gpu, F, kind):
    g = np.random.RandomState(7)
    n_keys, n = 200003, 70001
    if kind == "clustered":  # half of the keys in a 2^-40 part of the range
        keys = np.unique(np.concatenate([g.randint(0, 1 << 62, n_keys // 2), (1 << 61) + g.randint(0, 1 << 22, n_keys // 2)]))
    elif kind == "dense ids":
        keys = np.arange(5000, 5000 + n_keys)
    else:
        keys = np.unique(g.randint(1 << 40, 1 << 50, n_keys))
    sk = keys.astype(np.uint64)
    sv = W.splitmix64_mix(sk)
    q = np.where(g.rand(n) < 0.8, sk[g.randint(0, len(sk), n)], g.randint(0, 1 << 51, n).astype(np.uint64))
    if kind == "equal":
        q[:] = sk[len(sk) // 2]
    elif kind == "outside":  # below, above, and with bits above the key range's top bit
        q = np.where(g.rand(n) < 0.5, q | np.uint64(1 << 62), q & np.uint64((1 << 30) - 1))
    elif kind == "sorted":
        q = np.sort(q)
    elif kind == "key max":
        q[g.rand(n) < 0.3] = np.uint64(HM_KEY_MAX)
        q[:100] = np.uint64(HM_KEY_MAX - 1)
    tree = BPlusTree.from_keys(sk, sv, keys_sorted=True, fanout=F, leaf_fill=8)
    check(tree, sk, sv, q)
    check(tree, sk, sv, q, lds_levels=0)
    tree.close()


@pytest.mark.parametrize("psa", [True, False])
def test_captured_search_after_the_key_range_widens(gpu, psa):
    """A batcher's captured searches see keys that an in-place epoch adds outside the old key range."""
    from harmonia_amd import Batcher

    keys = (np.uint64(3) << np.uint64(40)) + np.arange(50000, dtype=np.uint64) * np.uint64(16)
    tree = BPlusTree.from_keys(keys, keys, keys_sorted=True, fanout=64, leaf_fill=5)
    b = Batcher(tree, 60000, psa_bits=16 if psa else 0)
    new = np.array([5, 1 << 20, (3 << 40) + 7, (5 << 40) + 1, (1 << 60) + 3, HM_KEY_MAX - 1], dtype=np.uint64)
    q = np.concatenate([keys, new])
    want = np.zeros(len(q), dtype=np.uint8)
    want[:len(keys)] = 1
    for step in range(4):
        off = b.add(q)
        b.flush()
        v, f = b.copy_out(off, len(q))
        assert np.array_equal(f, want) and np.array_equal(v, np.where(want == 1, q, 0))
        if step % 2 == 0:  # an epoch between flushes: two keys further out each time
            k = new[step + 1:step + 4]
            before = tree.stats().relayouts
            tree.update(k, k)
            tree.publish()
            assert tree.stats().relayouts == before
            want[len(keys) + step + 1:len(keys) + step + 4] = 1
    b.close()
    tree.close()


@pytest.mark.parametrize("F", [32, 64, 128])
@pytest.mark.parametrize("n", [70001, 3 * (1 << 20), 3 * (1 << 20) + 1])
def test_partition_by_bits_that_order_nothing(gpu, F, n):
    """One key far from dense ids: every query falls into one bucket, and each quad reads its nodes."""
    sk = np.append(np.arange(1, 200000, dtype=np.uint64) * np.uint64(3), np.uint64((1 << 63) + 5))
    sv = W.splitmix64_mix(sk)
    tree = BPlusTree.from_keys(sk, sv, keys_sorted=True, fanout=F, leaf_fill=5)
    g = np.random.RandomState(9)
    q = g.randint(0, 610000, n).astype(np.uint64)
    q[g.randint(0, n, 50)] = np.uint64((1 << 63) + 5)
    q[-1] = np.uint64(HM_KEY_MAX)
    check(tree, sk, sv, q)
    tree.close()


@pytest.mark.parametrize("F", [32, 64, 128])
@pytest.mark.parametrize("n", [3 * (1 << 19) - 1, 3 * (1 << 19), 3 * (1 << 20) + 1])
@pytest.mark.parametrize("low", [False, True])
def test_psa_order_results(gpu, F, n, low):
    """Results in PSA order where the searching kernel changes: the batch's size, and keys below the window."""
    import torch

    g = np.random.RandomState(10)
    sk = np.unique(g.randint(0, 1 << (47 if low else 62), 300007)).astype(np.uint64)
    sv = W.splitmix64_mix(sk)
    tree = BPlusTree.from_keys(sk, sv, keys_sorted=True, fanout=F, leaf_fill=7)
    q = np.where(g.rand(n) < 0.8, sk[g.randint(0, len(sk), n)], g.randint(0, 1 << 63, n).astype(np.uint64))
    q[g.randint(0, n, 100)] = np.uint64(HM_KEY_MAX)
    dq = torch.from_numpy(q.view(np.int64)).cuda()
    v, f = torch.empty_like(dq), torch.empty(n, dtype=torch.uint8, device="cuda")
    pos = torch.empty(n, dtype=torch.int32, device="cuda")
    torch.cuda.synchronize()
    tree.search_batch(dq, out_vals=v, out_found=f, out_pos=pos, psa_bits=16, sorted_output=True)
    torch.cuda.synchronize()
    want = np.argsort(q >> np.uint64(48), kind="stable")
    ev, ef = oracle.search_sorted(sk, sv, q[want])
    assert np.array_equal(pos.cpu().numpy(), want)
    assert np.array_equal(f.cpu().numpy(), ef) and np.array_equal(v.cpu().numpy().view(np.uint64), ev)
    tree.close()


@pytest.mark.parametrize("n", [70001, 3 * (1 << 20) + 1])
@pytest.mark.parametrize("share", [0.0001, 0.3])
def test_partition_found_values_like_the_miss_mark(gpu, n, share):
    """Stored values equal to the one that stands for a miss on the way back."""
    g = np.random.RandomState(11)
    sk = np.unique(g.randint(0, 1 << 62, 50003)).astype(np.uint64)
    sv = W.splitmix64_mix(sk)
    sv[g.rand(len(sk)) < share] = np.uint64(0xB5D19F6E03C7A28D)
    sv[7] = np.uint64(0)
    sv[len(sk) // 2] = np.uint64(0xB5D19F6E03C7A28D)
    tree = BPlusTree.from_keys(sk, sv, keys_sorted=True, fanout=64, leaf_fill=8)
    q = np.where(g.rand(n) < 0.7, sk[g.randint(0, len(sk), n)], g.randint(0, 1 << 62, n).astype(np.uint64))
    q[:2] = sk[[7, len(sk) // 2]]
    check(tree, sk, sv, q)
    check(tree, sk, sv, q, odd=True)
    tree.close()


@pytest.mark.parametrize("bits", [1, 8, 9, 16, 17, 25])
def test_psa_order_positions(gpu, bits):
    """Positions of PSA-order results, odd places in memory: one, two (written in place), three and four passes."""
    import torch

    g = np.random.RandomState(12)
    sk = np.unique(g.randint(0, 1 << 62, 30007)).astype(np.uint64)
    tree = BPlusTree.from_keys(sk, sk, keys_sorted=True, fanout=64, leaf_fill=8)
    for n in (1, 4097, 60001):
        q = g.randint(0, 1 << 63, n).astype(np.uint64)
        dq = torch.from_numpy(q.view(np.int64)).cuda()
        v, f = torch.empty_like(dq), torch.empty(n, dtype=torch.uint8, device="cuda")
        pos = torch.full((n + 2,), -1, dtype=torch.int32, device="cuda")
        torch.cuda.synchronize()
        tree.search_batch(dq, out_vals=v, out_found=f, out_pos=pos[1:n + 1], psa_bits=bits, sorted_output=True)
        torch.cuda.synchronize()
        want = np.argsort(q >> np.uint64(64 - bits), kind="stable")
        pos = pos.cpu().numpy()
        assert np.array_equal(pos[1:n + 1], want) and pos[0] == -1 and pos[n + 1] == -1
        ev, ef = oracle.search_sorted(sk, sk, q[want])
        assert np.array_equal(f.cpu().numpy(), ef) and np.array_equal(v.cpu().numpy().view(np.uint64), ev)
    tree.close()
