"""Batch streams on a tree for whose second batch scratch the GPU has no memory: they run on one
stream, as they did before the tree had seen enough batches for two."""
import ctypes as C

import numpy as np
import pytest

pytestmark = pytest.mark.gpu

GIB = 1 << 30


def test_streams_without_memory_for_the_second_scratch(oracle_mod):
    from eirene_amd import DeviceBuffer, StmError, StmTree
    rng = np.random.default_rng(13)
    load = np.unique(rng.integers(0, 1 << 40, 20000, dtype=np.uint64))
    sizes = np.array([2049] * 40 + [30, 5000])
    n = int(sizes.sum())
    keys = np.where(rng.random(n) < 0.5, rng.choice(load, n),
                    rng.integers(0, 1 << 40, n, dtype=np.uint64)).astype(np.uint64)
    ops = (rng.random(n) < 0.7).astype(np.uint8)  # 1: GET, 0: INSERT
    offsets = np.concatenate([[0], np.cumsum(sizes)]).astype(np.uint64)
    o = oracle_mod.Oracle()
    o.bulk_load(load, load)
    with StmTree(max_keys=1 << 18, max_batch=1 << 30) as t:  # a scratch of some 140 GiB, unused
        t.bulk_load(load, load)
        dk, dv, do = (DeviceBuffer.from_array(x) for x in (keys, keys, ops))
        ov, of = DeviceBuffer(n, np.uint64), DeviceBuffer(n, np.uint8)
        free, total = C.c_size_t(), C.c_size_t()
        assert t._lib.hipMemGetInfo(C.byref(free), C.byref(total)) == 0
        ballast = DeviceBuffer(max(free.value - 64 * GIB, 1), np.uint8)
        for _ in range(2):
            t.run_batches_device(dk, dv, do, ov, of, offsets)
            want = [o.run_batch(keys[a:z], keys[a:z], ops[a:z])
                    for a, z in zip(offsets[:-1].astype(int), offsets[1:].astype(int))]
            np.testing.assert_array_equal(ov.download(), np.concatenate([w[0] for w in want]))
            np.testing.assert_array_equal(of.download(), np.concatenate([w[1] for w in want]))
        with pytest.raises(StmError) as e:  # asked for by name, it is an error
            t.capture_graphs()
        assert e.value.code == 2
        v, f = t.run_batch(load[:100], load[:100], np.ones(100, np.uint8))
        assert f.all()
        ballast.free()
