"""A closed tree's memory is other programs' again after harmonia_amd.device_synchronize()."""
import pytest

import harmonia_amd
from harmonia_amd import BPlusTree

pytestmark = pytest.mark.gpu


def test_closed_trees_memory_goes_back(gpu):
    import torch

    keys = torch.arange(1, 3_000_001, dtype=torch.int64, device="cuda")
    torch.cuda.synchronize()
    BPlusTree.from_keys(keys[:1000], keys[:1000]).close()
    harmonia_amd.device_synchronize()
    free0 = torch.cuda.mem_get_info()[0]
    BPlusTree.from_keys(keys, keys).close()
    harmonia_amd.device_synchronize()
    assert free0 - torch.cuda.mem_get_info()[0] <= 4 << 20
