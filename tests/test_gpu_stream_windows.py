"""Replayed batch streams of more batches than one descriptor window (4096) holds, with batches
between them that are launched, against the oracle."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def test_replays_over_several_windows(oracle_mod):
    from eirene_amd import DeviceBuffer, StmTree
    rng = np.random.default_rng(71)
    load = np.unique(rng.integers(0, 1 << 40, 20000, dtype=np.uint64))
    sizes = rng.integers(1, 6, 9000)
    sizes[[5, 4095, 4096, 8191]] = [1024, 1025, 4096, 4097]  # the last one has no graph
    n = int(sizes.sum())
    keys = np.where(rng.random(n) < 0.5, rng.choice(load, n),
                    rng.integers(0, 1 << 40, n, dtype=np.uint64)).astype(np.uint64)
    vals = rng.integers(0, 1 << 62, n, dtype=np.uint64)
    ops = (rng.random(n) < 0.6).astype(np.uint8)  # 1: GET, 0: INSERT
    offsets = np.concatenate([[0], np.cumsum(sizes)]).astype(np.uint64)
    o = oracle_mod.Oracle()
    o.bulk_load(load, load)
    want = [o.run_batch(keys[a:z], vals[a:z], ops[a:z])
            for a, z in zip(offsets[:-1].astype(int), offsets[1:].astype(int))]
    with StmTree(max_keys=1 << 18, max_batch=1 << 13) as t:
        t.bulk_load(load, load)
        t.capture_graphs()
        dk, dv, do = (DeviceBuffer.from_array(x) for x in (keys, vals, ops))
        ov, of = DeviceBuffer(n, np.uint64), DeviceBuffer(n, np.uint8)
        t.run_batches_device(dk, dv, do, ov, of, offsets)
        np.testing.assert_array_equal(ov.download(), np.concatenate([w[0] for w in want]))
        np.testing.assert_array_equal(of.download(), np.concatenate([w[1] for w in want]))
        k, v = t.dump()
        ek, ev = o.dump()
        np.testing.assert_array_equal(k, ek)
        np.testing.assert_array_equal(v, ev)
        assert t.check() == 0
