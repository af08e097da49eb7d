"""What a tree holds on the device does not depend on the trees that were closed before it: after a larger one,
it takes the bytes that it counts against its budget and reports, no more."""
import pytest

from harmonia_amd import BPlusTree, load

pytestmark = pytest.mark.gpu
SLACK = 12 << 20  # arrays of a few bytes take whole pages, at most 2 MiB each


@pytest.mark.parametrize("budget", [False, True])
@pytest.mark.parametrize("n", [2_200_003, 3_900_001])
def test_held_bytes_after_a_larger_tree(gpu, budget, n):
    import torch

    lib = load()
    keys = torch.arange(1, 4_000_001, dtype=torch.int64, device="cuda") * 7
    torch.cuda.synchronize()
    alone = BPlusTree.from_keys(keys[:n], keys[:n])
    base = alone.stats().bytes_device
    alone.close()
    lib.hm_device_synchronize()
    free0 = torch.cuda.mem_get_info()[0]
    for _ in range(2):
        BPlusTree.from_keys(keys, keys).close()
    tree = BPlusTree.from_keys(keys[:n], keys[:n], mem_budget=base + (1 << 20) if budget else 0)
    assert tree.stats().bytes_device == base
    lib.hm_device_synchronize()  # what the pool still keeps goes back
    assert free0 - torch.cuda.mem_get_info()[0] <= base + SLACK
    tree.close()
