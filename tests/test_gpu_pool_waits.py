"""Trees are built, searched, updated and closed in one thread while another thread captures a graph: the
capture stays valid, whatever waits for device memory the library makes, and results are right."""
import threading

import numpy as np
import pytest

from harmonia_amd import BPlusTree
from harmonia_amd import workloads as W

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("update", [False, True])
def test_capture_in_another_thread_survives(gpu, update):
    import torch

    keys, vals = W.gen_keys(50000, 3)
    new = W.gen_misses(50000, 9000, 3)
    BPlusTree.from_keys(keys, vals).close()  # code objects are loaded
    x = torch.zeros(1000, device="cuda")
    errors = []

    def trees():
        try:
            for n in (700, 50000):
                t = BPlusTree.from_keys(keys[:n], vals[:n])
                for m in (100, n):  # the second grows the stream's workspace
                    v, f = t.search_batch(keys[:m], psa_bits=16)
                    assert f.all() and np.array_equal(v, vals[:m])
                if update:
                    t.update(new, new)
                    t.publish()
                    v, f = t.search_batch(new)
                    assert f.all() and np.array_equal(v, new)
                t.close()
        except BaseException as e:  # reported by the test's own thread
            errors.append(e)

    g = torch.cuda.CUDAGraph()
    torch.cuda.synchronize()
    with torch.cuda.graph(g, capture_error_mode="thread_local"):
        x += 1
        th = threading.Thread(target=trees)
        th.start()
        th.join()
        x *= 2
    assert not errors, errors
    for want in (2.0, 6.0, 14.0):
        g.replay()
        torch.cuda.synchronize()
        assert bool((x == want).all())
