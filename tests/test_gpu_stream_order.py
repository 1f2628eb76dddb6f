"""A batch stream starts after whatever the caller has queued on the tree's stream, also once its
sorts run on a second stream: inputs that a queued copy has yet to bring, answers that a queued copy
has yet to take away."""
import ctypes as C

import numpy as np
import pytest

pytestmark = pytest.mark.gpu

DEVICE_TO_DEVICE = 3


@pytest.mark.parametrize("size", [2049, 40000])
def test_stream_waits_for_queued_copies(oracle_mod, size):
    from eirene_amd import DeviceBuffer, StmTree
    rng = np.random.default_rng(size)
    load = np.unique(rng.integers(0, 1 << 50, 60000, dtype=np.uint64))
    n = 4 * size
    offsets = (np.arange(5) * size).astype(np.uint64)

    def batch():
        keys = np.where(rng.random(n) < 0.6, rng.choice(load, n),
                        rng.integers(0, 1 << 50, n, dtype=np.uint64)).astype(np.uint64)
        return (keys, rng.integers(0, 1 << 62, n, dtype=np.uint64),
                (rng.random(n) < 0.7).astype(np.uint8))  # 1: GET, 0: INSERT

    o = oracle_mod.Oracle()
    o.bulk_load(load, load)

    def replay(b):
        parts = [o.run_batch(*(x[i:i + size] for x in b)) for i in range(0, n, size)]
        return np.concatenate([p[0] for p in parts]), np.concatenate([p[1] for p in parts])

    with StmTree(max_keys=1 << 20, max_batch=1 << 16) as t:
        t.bulk_load(load, load)

        def queue_copy(dst, src):
            item = np.dtype(src.dtype).itemsize
            assert t._lib.hipMemcpyAsync(C.c_void_p(dst.ptr), C.c_void_p(src.ptr),
                                         C.c_size_t(src.n * item), DEVICE_TO_DEVICE,
                                         C.c_void_p(t.stream())) == 0

        busy = DeviceBuffer(1 << 28, np.uint8), DeviceBuffer(1 << 28, np.uint8)
        first = batch()
        first[2][:] = 1  # lookups only: they leave the tree as it is
        cur = [DeviceBuffer.from_array(x) for x in first]
        out = DeviceBuffer(n, np.uint64), DeviceBuffer(n, np.uint8)
        for _ in range(8):  # enough batches for the second stream
            t.run_batches_device(*cur, *out, offsets)
        before = None
        for _ in range(3):
            b = batch()
            new = [DeviceBuffer.from_array(x) for x in b]
            kept = DeviceBuffer(n, np.uint64), DeviceBuffer(n, np.uint8)
            for _ in range(40):  # some milliseconds
                queue_copy(*busy)
            for dst, src in list(zip(kept, out)) + list(zip(cur, new)):
                queue_copy(dst, src)
            t.run_batches_device(*cur, *out, offsets)
            want = replay(b)
            for x, w in zip(out, want):
                np.testing.assert_array_equal(x.download(), w)
            if before is not None:
                for x, w in zip(kept, before):
                    np.testing.assert_array_equal(x.download(), w)
            before = want
        k, v = t.dump()
        ek, ev = o.dump()
        np.testing.assert_array_equal(k, ek)
        np.testing.assert_array_equal(v, ev)
        assert t.check() == 0
