"""The work a program has this library do, as cases that can be timed and compared.

Every case goes through the package's public entry points: one batch on a device-resident tree
(StmTree.run_batch_device, and its form that allocates nothing), a stream of batches
(run_batches_device), range scans (run_batch_scan_device), a batch of host arrays (run_batch),
a tree's whole life (create, bulk load, batches, close) and requests through the serving loop
(eirene_amd.serving.Server).  Keys are drawn from the benchmark's distributions (uniform, Normal,
Gamma, Zipf ranks with inserts beside hot keys); batches mix lookups of loaded and of absent keys
with inserts.  A kept tree takes the same batch again on each pass, so after the first pass its
inserts are updates of keys it holds; the cases that make their tree anew insert new keys (and
split leaves) on every pass.

    listed()             the named cases
    draw(rng)            one more case of the same ranges
    prepare(case, seed)  inputs, trees and handles a program holds before the call
    run(state)           one pass; returns every answer
    work(case)           the bytes a pass cannot do without
"""
import math

import numpy as np
import torch

import eirene_amd as ea
from eirene_amd import serving

ROUTES = {"descent": ea.ROUTE_DESCENT, "learned": ea.ROUTE_LEARNED, "index": ea.ROUTE_INDEX}
KEY_LIMIT = 1 << 63


def listed():
    return [
        # A latency-bound caller: one small batch at a time on a small index.
        dict(name="call_1000", kind="call", dist="uniform", load=1 << 20, ops=1000, insert=0.05,
             route="descent", fanout=64, noalloc=False),
        # A serving engine's own loop: middle-sized batches through the call that allocates nothing.
        dict(name="call_40k_noalloc", kind="call", dist="uniform", load=1 << 23, ops=40001,
             insert=0.10, route="learned", fanout=64, noalloc=True),
        # The headline workload, one synchronous call per batch: 2^26 Gamma keys, learned routing.
        dict(name="call_4m_learned", kind="call", dist="gamma", load=1 << 26, ops=1 << 22,
             insert=0.05, route="learned", fanout=64, noalloc=False),
        # The same mix as one device-resident stream: each batch's front half overlaps the one before.
        dict(name="stream_2m_learned", kind="stream", dist="gamma", load=1 << 25, lo=1 << 21,
             hi=1 << 21, batches=8, insert=0.05, route="learned", fanout=64),
        # Uneven batching: sizes log-uniform over 2^10..2^20 on Normal keys.
        dict(name="stream_uneven", kind="stream", dist="normal", load=1 << 24, lo=1 << 10,
             hi=1 << 20, batches=24, insert=0.05, route="descent", fanout=64),
        # A batch of mixed requests with short range scans (90 % lookups, 8 % inserts, 2 % scans).
        dict(name="scan_short", kind="scan", dist="uniform", load=1 << 23, ops=131075, insert=0.08,
             scans=0.02, len_lo=16, len_hi=256, route="descent", fanout=64),
        # Analytics beside point reads: a few thousand long range scans.
        dict(name="scan_long", kind="scan", dist="uniform", load=1 << 23, ops=4099, insert=0.0,
             scans=0.5, len_lo=500, len_hi=8000, route="descent", fanout=64),
        # The caller keeps its ops in host memory: the call copies in, runs and copies out.
        dict(name="host_1m", kind="host", dist="uniform", load=1 << 22, ops=1 << 20, insert=0.05,
             route="descent", fanout=64),
        # Building an index: create, bulk load, first lookups, close.
        dict(name="build_4m", kind="life", dist="uniform", load=1 << 22, lo=1 << 16, hi=1 << 16,
             batches=2, insert=0.0, route="learned", fanout=64),
        # Growth of a fresh tree: half of a large batch's ops insert new keys, most leaves split.
        dict(name="grow_uniform", kind="life", dist="uniform", load=1 << 20, lo=1 << 19, hi=1 << 19,
             batches=6, insert=0.5, route="descent", fanout=64),
        # Contended growth: half the ops insert new keys beside Zipf-hot ones, in small batches.
        dict(name="grow_zipf", kind="life", dist="zipf", load=1 << 20, lo=1 << 14, hi=1 << 14,
             batches=16, insert=0.5, route="descent", fanout=64),
        # Requests of 1..2^14 ops handed to the continuous-batching server and awaited.
        dict(name="serve_16", kind="serve", dist="uniform", load=1 << 22, lo=1, hi=1 << 14,
             batches=16, insert=0.08, scans=0.02, len_lo=16, len_hi=256, route="descent",
             fanout=64),
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["call", "call", "call", "stream", "stream", "scan", "scan", "host", "life",
                       "life", "serve"])
    c = dict(kind=kind, dist=rng.choice(["uniform", "normal", "gamma", "zipf"]),
             load=_log_int(rng, 1 << 18, 1 << 24), insert=rng.choice([0.0, 0.05, 0.05, 0.1, 0.5]),
             route=rng.choice(["descent", "learned", "learned", "index"]),
             fanout=rng.choice([32, 64, 64, 128]))
    # A batch's inserts beside one Zipf-hot key all meet in one leaf: such batches stay small.
    most = 1 << 14 if c["dist"] == "zipf" else 1 << 22
    if kind == "call":
        c["ops"] = _log_int(rng, 300, most)
        c["noalloc"] = c["ops"] <= ea.NOALLOC_MAX_OPS and rng.random() < 0.5
    elif kind == "stream":
        c["lo"] = _log_int(rng, 1 << 9, min(most, 1 << 18))
        c["hi"] = _log_int(rng, c["lo"], min(most, 1 << 20))
        c["batches"] = rng.randint(3, 24)
    elif kind == "scan":
        c["ops"] = _log_int(rng, 1 << 10, min(most, 1 << 18))
        c["len_lo"] = _log_int(rng, 1, 500)
        c["len_hi"] = _log_int(rng, c["len_lo"], 4000)
        c["scans"] = min(0.5, 4e6 / (c["ops"] * (c["len_lo"] + c["len_hi"])))
        c["insert"] = min(c["insert"], 0.1)
    elif kind == "host":
        c["ops"] = _log_int(rng, 1 << 10, min(most, 1 << 20))
    elif kind == "life":
        c["load"] = min(c["load"], 1 << 22)
        c["lo"] = _log_int(rng, 1 << 12, min(most, 1 << 18))
        c["hi"] = _log_int(rng, c["lo"], min(most, 1 << 20))
        c["batches"] = rng.randint(1, 12)
    else:
        c["lo"], c["hi"], c["batches"] = 1, _log_int(rng, 1 << 8, 1 << 15), rng.randint(4, 16)
        c.update(insert=0.08, scans=0.02, len_lo=16, len_hi=256)
    return c


# ---------------------------------------------------------------- inputs
class _Array:
    """A torch tensor in the place of a DeviceBuffer: the batch calls take its address and length."""

    def __init__(self, tensor):
        self.tensor = tensor
        self.ptr = tensor.data_ptr()
        self.n = tensor.numel()


class _State:
    pass


def _random(gen, n, lo=0, hi=KEY_LIMIT - 1):
    return torch.randint(lo, hi, (n,), generator=gen, device="cuda", dtype=torch.int64)


def _unit(gen, n):
    return torch.rand(n, generator=gen, device="cuda", dtype=torch.float64)


def _draw_keys(gen, dist, n):
    """n keys of the distribution, as non-negative int64 (the library reads them as u64)."""
    if dist == "normal":
        x = torch.randn(n, generator=gen, device="cuda", dtype=torch.float64) * 2.0 ** 58 + 2.0 ** 62
    elif dist == "gamma":  # k = 2: the sum of two exponentials
        x = -(torch.log1p(-_unit(gen, n)) + torch.log1p(-_unit(gen, n))) * 2.0 ** 56
    else:
        return _random(gen, n)
    # The doubles leave the lowest bits empty.
    return x.clamp(0, 2.0 ** 62 * 1.99).to(torch.int64) ^ _random(gen, n, 0, 1 << 9)


def _load(gen, case):
    """(sorted distinct keys, the same keys in loading order, their values)."""
    dist = "uniform" if case["dist"] == "zipf" else case["dist"]
    srt = torch.unique(_draw_keys(gen, dist, case["load"]))
    keys = srt[torch.randperm(srt.numel(), generator=gen, device="cuda")]
    return srt, keys, _random(gen, keys.numel(), -KEY_LIMIT)


def _sizes(case):
    """Batch sizes of a stream, spread over the logarithm of [lo, hi], in a mixed order."""
    b, lo, hi = case["batches"], math.log(case["lo"]), math.log(case["hi"])
    mixed = [(i * 7 + 3) % b if b % 7 else (i * 5 + 3) % b for i in range(b)]
    return [int(round(math.exp(lo + (hi - lo) * (i + 0.5) / b))) for i in mixed]


def _ops(gen, case, srt, n):
    """(keys, vals, ops) of n mixed ops: lookups (nine in ten of them of loaded keys), inserts of
    new keys, and scans of lengths spread over [len_lo, len_hi] where the case has them."""
    u = _unit(gen, n)
    insert = u < case["insert"]
    if case["dist"] == "zipf":  # ranks of Zipf(0.99) over the sorted keys, by the continuous inverse
        m = srt.numel()
        r = ((m ** 0.01 - 1.0) * _unit(gen, n) + 1.0).pow(100.0).to(torch.int64).sub(1).clamp(0, m - 2)
        hot = srt[r]
        beside = hot + 1 + _random(gen, n) % (srt[r + 1] - hot - 1).clamp(min=1)
        keys = torch.where(insert, beside, hot)
    else:
        held = srt[_random(gen, n) % srt.numel()]
        fresh = _draw_keys(gen, case["dist"], n)
        keys = torch.where(insert | (_unit(gen, n) >= 0.9), fresh, held)
    vals = _random(gen, n, -KEY_LIMIT)
    ops = torch.where(insert, ea.OP_INSERT, ea.OP_GET).to(torch.uint8)
    if case.get("scans"):  # evenly spread; which ops scan, and how far, is the case's alone
        at = torch.arange(0, n, max(1, round(1 / case["scans"])), device="cuda")
        ops[at] = ea.OP_RANGE
        vals[at] = case["len_lo"] + at * 40503 % (case["len_hi"] - case["len_lo"] + 1)
    return keys, vals, ops


def _config(case, n_load, n_ops, max_batch):
    return ea.StmConfig(fanout=case["fanout"], route=ROUTES[case["route"]],
                        max_keys=n_load + n_ops + (1 << 18), max_batch=max(1 << 16, max_batch))


def prepare(case, seed):
    gen = torch.Generator(device="cuda")
    gen.manual_seed(seed)
    srt, keys, vals = _load(gen, case)
    s = _State()
    s.kind = case["kind"]
    if "batches" in case:
        sizes = _sizes(case)
        s.offsets = np.cumsum([0] + sizes).astype(np.uint64)
    else:
        sizes = [case["ops"]]
    n = sum(sizes)
    s.noalloc = case.get("noalloc", False)
    s.config = _config(case, keys.numel(), n, max(sizes))
    batch = _ops(gen, case, srt, n)
    if s.kind == "life":
        s.load_keys, s.load_vals = _Array(keys), _Array(vals)
    else:
        s.tree = ea.StmTree(s.config)
        torch.cuda.synchronize()
        s.tree.bulk_load_device(_Array(keys), _Array(vals))
        if s.config.route != ea.ROUTE_DESCENT:
            s.tree.retrain()
    if s.kind in ("host", "serve"):
        k, v, o = (x.cpu().numpy() for x in batch)
        s.batch = (k.view(np.uint64), v.view(np.uint64), o)
        if s.kind == "serve":
            at = s.offsets
            s.requests = [tuple(x[int(a):int(b)] for x in s.batch) for a, b in zip(at, at[1:])]
            s.server = serving.Server(s.tree, hbm_budget=256 << 20)
        return s
    s.batch = [_Array(x) for x in batch]
    s.out_vals = _Array(torch.zeros(n, dtype=torch.int64, device="cuda"))
    s.out_found = _Array(torch.zeros(n, dtype=torch.uint8, device="cuda"))
    if s.kind == "scan":
        pairs = int(batch[1][batch[2] == ea.OP_RANGE].sum())
        s.scan_keys = _Array(torch.zeros(max(pairs, 1), dtype=torch.int64, device="cuda"))
        s.scan_vals = _Array(torch.zeros(max(pairs, 1), dtype=torch.int64, device="cuda"))
    torch.cuda.synchronize()
    return s


# ---------------------------------------------------------------- one pass
def run(s):
    if s.kind == "host":
        return s.tree.run_batch(*s.batch)
    if s.kind == "serve":
        tickets = [s.server.submit(*r) for r in s.requests]
        return [s.server.wait(t)[:4] for t in tickets]
    out = (s.out_vals, s.out_found)
    if s.kind == "call":
        call = s.tree.run_batch_device_noalloc if s.noalloc else s.tree.run_batch_device
        call(*s.batch, *out)
    elif s.kind == "stream":
        s.tree.run_batches_device(*s.batch, *out, s.offsets)
    elif s.kind == "scan":
        s.tree.run_batch_scan_device(*s.batch, *out, s.scan_keys, s.scan_vals)
        return [x.tensor for x in (*out, s.scan_keys, s.scan_vals)]
    else:
        with ea.StmTree(s.config) as tree:
            tree.bulk_load_device(s.load_keys, s.load_vals)
            tree.run_batches_device(*s.batch, *out, s.offsets)
            return s.out_vals.tensor, s.out_found.tensor, tree.size()
    return s.out_vals.tensor, s.out_found.tensor


def work(case):
    """Per op: key and op code read (and an insert's value), the entry it meets read or written
    (16 B), the answer written (9 B); per scanned pair 16 B read and written; per loaded key 16 B
    read and written where the tree is made in the pass."""
    n = sum(_sizes(case)) if "batches" in case else case["ops"]
    scans = case.get("scans", 0.0)
    pairs = n * scans * (case.get("len_lo", 0) + case.get("len_hi", 0)) / 2
    b = n * (9 + 8 * (case["insert"] + scans) + 16 + 9) + 32 * pairs
    if case["kind"] == "life":
        b += 32 * case["load"]
    return {"bytes": int(b), "flops": 0}
