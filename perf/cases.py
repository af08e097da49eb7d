"""What a program has this library do, as measurable cases: lookups, range scans, upsert epochs, bulk
builds and packed uneven batches over device-resident buffers, from one request's worth of keys to the
largest batches, through the package's public entry points (and, for range scans into device memory,
the C ABI that `harmonia_amd.load()` returns).

A case is a dict with "op" and sizes; `prepare` makes its inputs on the GPU from the seed alone.
Every output is a whole number (values, found flags, positions, counts, offsets), so there is no
64-bit reference to give: equal results are equal bits.

Keys are a bijective scramble of consecutive integers into [0, 2^63) ("uniform"), or ascending ids
with small gaps ("ids", loaded already sorted); a key's value is a hash of it.
"""
import math

import numpy as np
import torch

from harmonia_amd import Batcher, BPlusTree, load

MASK63 = (1 << 63) - 1


# ---- inputs ---------------------------------------------------------------------------------
def _signed(x):
    return x - (1 << 64) if x >= (1 << 63) else x


def _shr(z, k):
    """Logical right shift of int64."""
    return (z >> k) & ((1 << (64 - k)) - 1)


def _mix(z):
    """splitmix64's output function (int64 arithmetic wraps)."""
    z = z + _signed(0x9E3779B97F4A7C15)
    z = (z ^ _shr(z, 30)) * _signed(0xBF58476D1CE4E5B9)
    z = (z ^ _shr(z, 27)) * _signed(0x94D049BB133111EB)
    return z ^ _shr(z, 31)


def _scramble(x, salt):
    """A seeded bijection of [0, 2^63): odd multipliers and xor-shifts, each invertible."""
    x = (x ^ salt) & MASK63
    x = (x * _signed(0x9E3779B97F4A7C15)) & MASK63
    x = x ^ (x >> 31)
    x = (x * _signed(0xBF58476D1CE4E5B9)) & MASK63
    x = x ^ (x >> 29)
    x = (x * _signed(0x94D049BB133111EB)) & MASK63
    return x ^ (x >> 32)


def _salt(seed):
    return int(np.random.RandomState(seed & 0x7FFFFFFF).randint(1 << 62, dtype=np.int64))


def _keys(case, seed, lo, hi):
    """Keys number lo .. hi - 1 of the case's key space; numbers past case["keys"] are never stored."""
    i = torch.arange(lo, hi, dtype=torch.int64, device="cuda")
    if case.get("space", "uniform") == "ids":
        # ascending, gaps of 9 to 23; numbers past the end give keys that stand between stored ids
        n = case["keys"]
        past = i >= n
        j = torch.where(past, (i - n) % n, i)
        k = (_salt(seed) >> 24) + 16 * j + (_mix(j) & 7)
        return torch.where(past, k + 8, k)
    return _scramble(i, _salt(seed))


def _tree(case, seed):
    n = case["keys"]
    k = _keys(case, seed, 0, n)
    v = _mix(k)
    torch.cuda.synchronize()  # a build takes no stream: its inputs have to be there when it is called
    return BPlusTree.from_keys(k, v, keys_sorted=case.get("space") == "ids", fanout=case.get("fanout", 64),
                               leaf_fill=case.get("fill", 8)), k


def _gen(seed):
    g = torch.Generator(device="cuda")
    g.manual_seed(seed)
    return g


def _queries(case, seed, n, keys, g):
    """n lookups, 9 in 10 of them stored keys: uniform, Zipf(0.99) over the key order, or ascending runs of 4096."""
    total, order = case["keys"], case.get("order", "unsorted")
    if order == "zipf":  # every query a stored key; rank 1 is the smallest
        u = torch.rand(n, dtype=torch.float64, device="cuda", generator=g)
        r = ((float(total) ** 0.01 - 1.0) * u + 1.0).pow(100.0).long().clamp_(1, total) - 1
        return torch.sort(keys).values[r]
    pick = torch.randint(0, total, (n,), device="cuda", generator=g)
    miss = torch.rand(n, device="cuda", generator=g) >= 0.9
    q = torch.where(miss, _keys(case, seed, total, total + n), keys[pick])
    if order == "runs" and n > 4096:
        s = torch.sort(q).values
        m = n // 4096
        runs = s[: m * 4096].view(m, 4096)[torch.randperm(m, device="cuda", generator=g)]
        q = torch.cat([runs.reshape(-1), s[m * 4096:]])
    return q


def _results(n):
    return torch.zeros(n, dtype=torch.int64, device="cuda"), torch.zeros(n, dtype=torch.uint8, device="cuda")


def _batch_sizes(case):
    """Uneven batch sizes, log-uniform in [32, case["most"]]."""
    r = np.random.RandomState(case["batches"])
    return np.exp(r.uniform(math.log(32), math.log(case["most"] + 1), case["batches"])).astype(np.int64)


# ---- the cases ------------------------------------------------------------------------------
def listed():
    return [
        # one request's keys against a small tree: launch and descent latency
        {"name": "lookup_64", "op": "search", "keys": 1 << 20, "n": 64},
        # a burst of requests against a large tree, below the sort threshold; a ragged count
        {"name": "lookup_20k", "op": "search", "keys": 1 << 25, "n": 20011},
        # the small benchmark configuration: 2^20 lookups on 2^20 keys, the smallest batch that is sorted first
        {"name": "lookup_1m_of_1m", "op": "search", "keys": 1 << 20, "n": 1 << 20},
        # the benchmark's workload: 2^24 unsorted lookups on 2^26 keys
        {"name": "lookup_16m_of_64m", "op": "search", "keys": 1 << 26, "n": 1 << 24},
        # skewed lookups on the wide-fanout tree, as in the benchmark
        {"name": "lookup_zipf_f128", "op": "search", "keys": 1 << 26, "n": 1 << 24, "order": "zipf", "fanout": 128},
        # results in sorted order with their positions, as a join consumes them; an odd count
        {"name": "lookup_psa_order", "op": "search", "keys": 1 << 25, "n": 3000001, "out": "psa"},
        # a request's worth of short scans
        {"name": "range_300", "op": "range", "keys": 1 << 22, "n": 300, "lo": 16, "hi": 256},
        # the benchmark's scans: 2^20 ranges of 16 to 256 pairs on the wide-fanout tree
        {"name": "range_1m_f128", "op": "range", "keys": 1 << 26, "n": 1 << 20, "lo": 16, "hi": 256, "fanout": 128},
        # a serving epoch: a few thousand upserts, one in twenty a new key, then read back
        {"name": "upsert_4k", "op": "update", "keys": 1 << 24, "n": 4001, "fill": 6},
        # a large epoch on a large tree
        {"name": "upsert_1m", "op": "update", "keys": 1 << 26, "n": 1 << 20, "fill": 6},
        # a bulk build from unsorted pairs, then one lookup of every key
        {"name": "build_4m", "op": "build", "keys": 4000037},
        # uneven batches packed into one graph replay
        {"name": "batches_96", "op": "batch", "keys": 1 << 25, "batches": 96, "most": 1 << 18},
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    op = rng.choice(["search", "search", "search", "range", "update", "build", "batch"])
    c = {"op": op, "fanout": rng.choice([32, 64, 64, 128]), "space": rng.choice(["uniform", "uniform", "ids"])}
    if op == "search":
        c.update(keys=_log_int(rng, 1 << 16, 1 << 26), n=_log_int(rng, 32, 1 << 24),
                 order=rng.choice(["unsorted", "unsorted", "runs", "zipf"]))
        if c["n"] >= 1 << 20 and rng.random() < 0.3:
            c["out"] = "psa"
    elif op == "range":
        c.update(keys=_log_int(rng, 1 << 18, 1 << 26), n=_log_int(rng, 32, 1 << 20), lo=rng.choice([1, 16]),
                 hi=rng.choice([40, 256]), between=rng.random() < 0.25)
    elif op == "update":
        c.update(keys=_log_int(rng, 1 << 18, 1 << 26), n=_log_int(rng, 256, 1 << 20), fill=rng.choice([5, 6]))
    elif op == "build":
        c.update(keys=_log_int(rng, 1 << 14, 4000037), fill=rng.choice([6, 8]))
    else:
        c.update(keys=_log_int(rng, 1 << 18, 1 << 25), batches=rng.randrange(16, 97), most=_log_int(rng, 1 << 12, 1 << 18))
    return c


def prepare(case, seed):
    op, g = case["op"], _gen(seed)
    if op == "build":
        k = _keys(case, seed, 0, case["keys"])
        v, f = _results(case["keys"])
        return {"case": case, "keys": k, "vals": _mix(k), "v": v, "f": f}
    tree, keys = _tree(case, seed)
    s = {"case": case, "tree": tree}
    if op == "search":
        s["q"] = _queries(case, seed, case["n"], keys, g)
        s["v"], s["f"] = _results(case["n"])
        if case.get("out") == "psa":
            s["pos"] = torch.zeros(case["n"], dtype=torch.int32, device="cuda")
    elif op == "range":
        n, lo, hi = case["n"], case["lo"], case["hi"]
        even = torch.arange(n, device="cuda") % (hi - lo + 1) + lo  # every length as often as the next one
        s["len"] = even[torch.randperm(n, device="cuda", generator=g)].int()
        if case.get("between"):  # closed intervals that hold lo .. hi keys
            sk = torch.sort(keys).values
            i = torch.randint(0, case["keys"] - hi, (n,), device="cuda", generator=g)
            s["start"], s["end"] = sk[i], sk[i + s["len"].long() - 1]
            s["cap"] = n * hi
        else:
            span = int(keys.max()) - int(keys.min())
            s["start"] = int(keys.min()) + (torch.rand(n, dtype=torch.float64, device="cuda", generator=g) * span).long()
            s["cap"] = int(s["len"].sum())
        s["off"] = torch.zeros(n + 1, dtype=torch.int64, device="cuda")
        s["k"], s["v"] = (torch.zeros(s["cap"], dtype=torch.int64, device="cuda") for _ in range(2))
        s["count"] = torch.zeros(n, dtype=torch.int32, device="cuda")
        s["lib"] = load()
    elif op == "update":  # 19 in 20 stored keys (a few of them written twice), the rest new
        n = case["n"]
        pick = torch.randint(0, case["keys"], (n,), device="cuda", generator=g)
        new = torch.rand(n, device="cuda", generator=g) < 0.05
        s["uk"] = torch.where(new, _keys(case, seed, case["keys"], case["keys"] + n), keys[pick])
        s["uv"] = torch.randint(-(1 << 62), 1 << 62, (n,), device="cuda", generator=g)
        s["v"], s["f"] = _results(n)
    else:
        sizes = _batch_sizes(case)
        total = int(sizes.sum())
        s["q"] = _queries(case, seed, total, keys, g)
        starts = np.concatenate([[0], np.cumsum(sizes)[:-1]])
        order = np.random.RandomState(seed & 0x7FFFFFFF).permutation(len(sizes))  # batches come from anywhere
        s["ptrs"] = (s["q"].data_ptr() + 8 * starts[order]).astype(np.uint64)
        s["sizes"] = sizes[order].astype(np.uint64)
        s["stream"] = torch.cuda.Stream()
        torch.cuda.synchronize()
        s["batcher"] = Batcher(tree, total, stream=s["stream"])
        s["total"] = total
        s["v"], s["f"] = _results(total)
    return s


def run(s):
    case = s["case"]
    op = case["op"]
    if op == "search":
        if "pos" in s:
            s["tree"].search_batch(s["q"], out_vals=s["v"], out_found=s["f"], psa_bits=16, sorted_output=True,
                                   out_pos=s["pos"])
            return s["v"], s["f"], s["pos"]
        s["tree"].search_batch(s["q"], out_vals=s["v"], out_found=s["f"])
        return s["v"], s["f"]
    if op == "range":
        lib, h, n = s["lib"], s["tree"]._handle(), case["n"]
        k, v, c = s["k"].data_ptr(), s["v"].data_ptr(), s["count"].data_ptr()
        if "end" in s:
            rc = lib.hm_range_between(h, s["start"].data_ptr(), s["end"].data_ptr(), n, case["hi"], k, v, c, None)
        else:
            rc = lib.hm_range(h, s["start"].data_ptr(), s["len"].data_ptr(), n, s["off"].data_ptr(), k, v, c, s["cap"],
                              None)
        if rc:
            raise RuntimeError(f"range scan failed: {rc}")
        return s["k"], s["v"], s["count"], s["off"]
    if op == "update":
        s["tree"].update(s["uk"], s["uv"])
        s["tree"].publish()
        s["tree"].search_batch(s["uk"], out_vals=s["v"], out_found=s["f"])
        return s["v"], s["f"]
    if op == "build":
        t = BPlusTree.from_keys(s["keys"], s["vals"], keys_sorted=case.get("space") == "ids",
                                fanout=case.get("fanout", 64), leaf_fill=case.get("fill", 8))
        t.search_batch(s["keys"], out_vals=s["v"], out_found=s["f"])
        t.close()
        return s["v"], s["f"]
    b = s["batcher"]
    b.add_many(s["ptrs"], s["sizes"])
    b.flush()
    b.copy_out(0, s["total"], out_vals=s["v"], out_found=s["f"])
    torch.cuda.current_stream().wait_stream(s["stream"])
    return s["v"], s["f"]


# ---- what a pass cannot do without ------------------------------------------------------------
def _leaves_touched(n_leaves, n, order="unsorted"):
    """Expected number of distinct 128-byte leaves that n lookups reach."""
    if order == "zipf":
        e = np.geomspace(1, n_leaves + 1, 4096)
        z = (float(n_leaves) ** 0.01 - 1) / 0.01
        mid = np.sqrt(e[1:] * e[:-1])
        return float((np.diff(e) * -np.expm1(-n * mid ** -0.99 / z)).sum())
    return n_leaves * -math.expm1(-n / n_leaves)


def work(case):
    op, keys = case["op"], case["keys"]
    leaves = max(1, math.ceil(keys / case.get("fill", 8)))
    if op == "batch":
        n = int(_batch_sizes(case).sum())
        b = 17 * n + 128 * _leaves_touched(leaves, n)
    elif op == "search":
        n = case["n"]
        b = 17 * n + 128 * _leaves_touched(leaves, n, case.get("order", "unsorted"))
        if case.get("out") == "psa":
            b += 4 * n
    elif op == "range":
        n, pairs = case["n"], case["n"] * (case["lo"] + case["hi"]) / 2
        b = 24 * n + 16 * pairs + min(128.0 * leaves, 16 * pairs + 128 * n)
    elif op == "update":  # batch in; its leaves read and written; then read back
        n = case["n"]
        b = 16 * n + 3 * 128 * _leaves_touched(leaves, n) + 17 * n
    else:  # pairs in, leaves and inner levels out, then every key looked up
        b = 16 * keys + 2 * 128 * leaves * (1 + 1.125 / 16) + 17 * keys
    return {"bytes": float(b), "flops": 0.0}
