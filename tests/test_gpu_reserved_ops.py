"""Ops with the reserved key in device batches: the call reports them, the other ops run, and the
refused ones are answered as absent, in every form of the sort and fold."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

RESERVED = np.uint64(0xFFFFFFFFFFFFFFFF)


@pytest.mark.parametrize("n", [1, 900, 2000, 30000, 250000, 300000, 400000])
@pytest.mark.parametrize("share", [0.3, 1.0])
def test_reserved_ops_are_absent(oracle_mod, n, share):
    from eirene_amd import DeviceBuffer, StmError, StmTree
    rng = np.random.default_rng(n)
    load = np.unique(rng.integers(0, 1 << 62, 20000, dtype=np.uint64))
    keys = rng.choice(load, n).astype(np.uint64)
    bad = rng.random(n) < share
    bad[0] = True
    keys[bad] = RESERVED
    ops = (rng.random(n) < 0.5).astype(np.uint8)  # 1: GET, 0: INSERT
    vals = rng.integers(1, 1 << 62, n, dtype=np.uint64)
    o = oracle_mod.Oracle()
    o.bulk_load(load, load)
    want = np.zeros(n, np.uint64), np.zeros(n, np.uint8)
    if not bad.all():
        want[0][~bad], want[1][~bad] = o.run_batch(keys[~bad], vals[~bad], ops[~bad])
    with StmTree(max_keys=1 << 17, max_batch=1 << 19) as t:
        t.bulk_load(load, load)
        dk, dv, do = (DeviceBuffer.from_array(x) for x in (keys, vals, ops))
        ov = DeviceBuffer.from_array(np.full(n, 9, np.uint64))
        of = DeviceBuffer.from_array(np.full(n, 9, np.uint8))
        with pytest.raises(StmError) as e:
            t.run_batch_device(dk, dv, do, ov, of)
        assert e.value.code == 1
        np.testing.assert_array_equal(of.download(), want[1])
        np.testing.assert_array_equal(ov.download(), want[0])
        k, v = t.dump()
        ek, ev = o.dump()
        np.testing.assert_array_equal(k, ek)
        np.testing.assert_array_equal(v, ev)
        assert t.check() == 0
