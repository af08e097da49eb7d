"""Memory that closed trees left for reuse is there for whatever the library allocates next: with the GPU nearly
full, a batcher, a tuner and a server get what the pool keeps."""
import numpy as np
import pytest

from harmonia_amd import Batcher, BPlusTree, load
from harmonia_amd import workloads as W

pytestmark = pytest.mark.gpu
MIB = 1 << 20


def fill_gpu(leave):
    """Tensors that take all device memory but `leave` bytes or a little more."""
    import torch

    held, size = [], 8 << 30
    while size >= 32 * MIB:
        free = torch.cuda.mem_get_info()[0]
        if free < leave + size:
            size //= 2
            continue
        try:
            held.append(torch.empty(size, dtype=torch.uint8, device="cuda"))
        except torch.OutOfMemoryError:
            size //= 2
    return held


@pytest.mark.parametrize("what", ["batcher", "tuner"])
def test_pool_gives_way(gpu, what):
    import torch

    torch.cuda.empty_cache()
    load().hm_device_synchronize()
    keys, vals = W.gen_keys(100000, 5)
    tree = BPlusTree.from_keys(keys, vals)
    n = 6 << 20  # a batcher or tuner of n queries: scratch of 43 bytes each, buffers of 17
    q = torch.from_numpy(np.resize(keys, n).view(np.int64)).cuda()
    if what == "tuner":  # its first run loads every kernel
        tree.autotune(keys[:4096], quick=True)
    big = torch.arange(1, (7 << 20) + 1, dtype=torch.int64, device="cuda")
    torch.cuda.synchronize()
    for t in [BPlusTree.from_keys(big, big, keys_sorted=True) for _ in range(4)]:
        t.close()  # about 120 MiB each
    held = fill_gpu(280 * MIB)
    try:
        assert torch.cuda.mem_get_info()[0] < 340 * MIB
        if what == "batcher":
            b = Batcher(tree, n)
            off = b.add(q[:50000])
            b.flush()
            v, f = b.copy_out(off, 50000)
            assert f.all() and np.array_equal(v, vals[:50000])
            b.close()
        else:
            assert tree.autotune(q, quick=True)["trials"] > 100
    finally:
        del held
        torch.cuda.empty_cache()
        tree.close()
