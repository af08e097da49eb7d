"""What one wave of a large epoch's plan finds reaches the host, wherever in the grid it stands: a leaf that
overflows in a node with room (a re-spread), one in a full node (a re-layout), both, or neither, in a batch of
300000 overwrites (256 blocks of the plan, some with a second round)."""
import pytest

from harmonia_amd import BPlusTree

pytestmark = pytest.mark.gpu

N = 300000


@pytest.mark.parametrize("place", [0, 1023, 131072, 262143, 262144, N - 9])
@pytest.mark.parametrize("kind", ["nothing", "listed", "full", "both"])
def test_plan_summary(gpu, place, kind):
    import torch

    F, fill = 32, 7
    keys = torch.arange(1, N + 1, dtype=torch.int64, device="cuda") * 1024
    torch.cuda.synchronize()
    tree = BPlusTree.from_keys(keys, keys, keys_sorted=True, fanout=F, leaf_fill=fill)
    at = place // fill * fill  # the first key of the leaf
    far = (at + N // 2) % N // fill * fill
    new = []
    if kind in ("listed", "both"):  # two keys for one free slot
        new += [keys[at] + torch.arange(1, 3, device="cuda")]
    if kind in ("full", "both"):  # more than the node's free slots
        new += [keys[far if kind == "both" else at] + torch.arange(1, F + 10, device="cuda")]
    k = torch.cat([keys] + new)
    k = k[torch.randperm(len(k), device="cuda")]
    v = k ^ 0x5555
    torch.cuda.synchronize()
    tree.update(k, v)
    relaid = tree.publish()
    st = tree.stats()
    assert relaid == (kind in ("full", "both"))
    assert (st.relayouts, st.respreads) == (int(relaid), int(kind == "listed"))
    assert st.n_keys == len(k)
    out, found = torch.empty_like(k), torch.empty(len(k), dtype=torch.uint8, device="cuda")
    torch.cuda.synchronize()
    tree.search_batch(k, out_vals=out, out_found=found)
    torch.cuda.synchronize()
    assert bool(found.all()) and torch.equal(out, v)
    leaves = torch.from_numpy(tree.export()["leaves"][:, :8].reshape(-1).view("int64"))
    assert torch.equal(leaves[leaves != -1], torch.sort(k).values.cpu())
    tree.close()
