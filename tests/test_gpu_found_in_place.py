"""Batches whose found flags take the place of their op codes, against the oracle: every form of the
sort, also where the batch is sorted a second time from its input, streams, scans and the call that
allocates nothing."""
import numpy as np
import pytest

from test_gpu_sample_sort import crafted
from test_gpu_small_batches import sample_positions

pytestmark = pytest.mark.gpu

OP_INSERT, OP_GET, OP_RANGE = 0, 1, 3


def uniform(n, rng):
    return rng.integers(0, 1 << 62, n, dtype=np.uint64)


def misleading(n, rng):
    """Keys that the small-batch sort's sample of a 12000-op batch misleads."""
    keys = np.uint64(1 << 61) + rng.integers(0, 1 << 30, n, dtype=np.uint64)
    at = sample_positions(n, 256)
    keys[at] = np.sort(rng.choice(1 << 40, at.size, replace=False).astype(np.uint64))
    return keys


def hot_neighbours(n, rng):
    """A quarter beside one key: the normalized sort's buckets overflow with distinct keys."""
    keys = uniform(n, rng)
    keys[:n // 4] = np.uint64(1 << 60) + rng.integers(1, 1 << 30, n // 4, dtype=np.uint64)
    return rng.permutation(keys)


def crowded_interval(n, rng):
    return crafted(n, rng, 1)


NOALLOC_MOST = 65536
CASES = pytest.mark.parametrize("n,keys_of,again,call", [
    (n, keys_of, again, call)
    for n, keys_of, again in [(1000, uniform, 0), (12000, uniform, 0), (12000, misleading, 1),
                              (300000, hot_neighbours, 1), (400000, uniform, 0),
                              (400000, crowded_interval, 1)]
    for call in ("batch", "stream", "noalloc") if call != "noalloc" or n <= NOALLOC_MOST])


def batch(n, keys_of, rng):
    keys = keys_of(n, rng)
    load = np.unique(rng.choice(keys, 5000))
    ops = np.where(rng.random(n) < 0.4, OP_INSERT, OP_GET).astype(np.uint8)
    return load, keys, rng.integers(0, 1 << 62, n, dtype=np.uint64), ops


def check_tree(t, o):
    k, v = t.dump()
    ek, ev = o.dump()
    np.testing.assert_array_equal(k, ek)
    np.testing.assert_array_equal(v, ev)
    assert t.check() == 0


@CASES
def test_found_flags_in_place_of_op_codes(oracle_mod, n, keys_of, again, call):
    from eirene_amd import DeviceBuffer, StmTree
    rng = np.random.default_rng(n)
    load, keys, vals, ops = batch(n, keys_of, rng)
    o = oracle_mod.Oracle()
    o.bulk_load(load, load)
    with StmTree(max_keys=1 << 20, max_batch=1 << 19) as t:
        t.bulk_load(load, load)
        t.capture_graphs()
        dk, dv = DeviceBuffer.from_array(keys), DeviceBuffer.from_array(vals)
        ov = DeviceBuffer(n, np.uint64)
        for b in range(2):
            do = DeviceBuffer.from_array(ops)
            if call == "stream":
                cut = np.array([0, n, n], np.uint64)
                t.run_batches_device(dk, dv, do, ov, do, cut)
            else:
                run = t.run_batch_device if call == "batch" else t.run_batch_device_noalloc
                run(dk, dv, do, ov, do)
            want = o.run_batch(keys, vals, ops)
            np.testing.assert_array_equal(do.download(), want[1])
            np.testing.assert_array_equal(ov.download(), want[0])
        assert t.stats()["sort_fallbacks"] >= again
        check_tree(t, o)


def test_stream_of_batches_in_place(oracle_mod):
    """A misleading sample in mid-stream: what is run again still has its op codes."""
    from eirene_amd import DeviceBuffer, StmTree
    rng = np.random.default_rng(2)
    n, batches = 12000, 8
    parts = [batch(n, misleading if b == 4 else uniform, rng) for b in range(batches)]
    load = np.unique(np.concatenate([p[0] for p in parts]))
    keys, vals, ops = (np.concatenate([p[i] for p in parts]) for i in (1, 2, 3))
    o = oracle_mod.Oracle()
    o.bulk_load(load, load)
    want = [o.run_batch(*p[1:]) for p in parts]
    with StmTree(max_keys=1 << 20, max_batch=1 << 16) as t:
        t.bulk_load(load, load)
        t.capture_graphs()
        dk, dv, do = (DeviceBuffer.from_array(x) for x in (keys, vals, ops))
        ov = DeviceBuffer(keys.size, np.uint64)
        t.run_batches_device(dk, dv, do, ov, do, (np.arange(batches + 1) * n).astype(np.uint64))
        np.testing.assert_array_equal(do.download(), np.concatenate([w[1] for w in want]))
        np.testing.assert_array_equal(ov.download(), np.concatenate([w[0] for w in want]))
        check_tree(t, o)


def test_scans_in_place(oracle_mod):
    from eirene_amd import DeviceBuffer, StmTree
    rng = np.random.default_rng(4)
    load, keys, vals, ops = batch(12000, misleading, rng)
    at = rng.choice(keys.size, 60, replace=False)
    ops[at], vals[at] = OP_RANGE, rng.integers(1, 300, at.size)
    pairs = int(vals[at].sum())
    o = oracle_mod.Oracle()
    o.bulk_load(load, load)
    ev, ef, esk, esv = o.run_batch_scan(keys, vals, ops)
    with StmTree(max_keys=1 << 20, max_batch=1 << 16) as t:
        t.bulk_load(load, load)
        dk, dv, do = (DeviceBuffer.from_array(x) for x in (keys, vals, ops))
        ov = DeviceBuffer(keys.size, np.uint64)
        sk, sv = DeviceBuffer(pairs, np.uint64), DeviceBuffer(pairs, np.uint64)
        t.run_batch_scan_device(dk, dv, do, ov, do, sk, sv)
        np.testing.assert_array_equal(ov.download(), ev)
        np.testing.assert_array_equal(do.download(), ef)
        first = 0
        for i in np.flatnonzero(ops == OP_RANGE):
            m = int(ev[i])
            np.testing.assert_array_equal(sk.download(m, first), esk[first:first + m])
            np.testing.assert_array_equal(sv.download(m, first), esv[first:first + m])
            first += int(vals[i])
        check_tree(t, o)
