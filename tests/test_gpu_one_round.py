"""Unsorted batches take one query per group only where one round of resident blocks holds them: the default is no
slower than four queries per group at the sizes where that changes, and the results are the same."""
import pytest

from harmonia_amd import BPlusTree

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("F,log_keys", [(32, 20), (32, 25), (64, 25), (128, 25)])
def test_default_shape(gpu, F, log_keys):
    import torch

    keys = torch.arange(1, (1 << log_keys) + 1, dtype=torch.int64, device="cuda") * 3
    torch.cuda.synchronize()
    tree = BPlusTree.from_keys(keys, keys ^ 77, keys_sorted=True, fanout=F)
    s = torch.cuda.Stream()
    for n in (49152, 49153, 65536, 65537):
        q = torch.randint(0, 4 << log_keys, (n,), device="cuda")
        v, f = torch.zeros_like(q), torch.zeros(n, dtype=torch.uint8, device="cuda")
        torch.cuda.synchronize()
        us = {}
        for qpg in (0, 4):
            call = lambda: tree.search_batch(q, out_vals=v, out_found=f, psa_bits=0, stream=s, queries_per_group=qpg)
            call()
            s.synchronize()
            g = torch.cuda.CUDAGraph()
            with torch.cuda.graph(g, stream=s):
                for _ in range(20):
                    call()
            t = []
            for _ in range(8):
                e0, e1 = (torch.cuda.Event(enable_timing=True) for _ in range(2))
                with torch.cuda.stream(s):
                    e0.record()
                    g.replay()
                    e1.record()
                s.synchronize()
                t.append(e0.elapsed_time(e1) * 50)
            us[qpg] = min(t)
            hit = (q % 3 == 0) & (q > 0) & (q <= 3 << log_keys)
            assert torch.equal(f.bool(), hit) and torch.equal(v, torch.where(hit, q ^ 77, 0))
            v.zero_(), f.zero_()
            torch.cuda.synchronize()
            del g
        print(F, log_keys, n, {k: round(x, 2) for k, x in us.items()})
        assert us[0] < 1.25 * us[4]
    tree.close()
