"""Batches at the end of the node pool.  What needs no node is done whatever the pool holds: every
update of a held key, every lookup, new keys while their leaf has room.  An insert that finds no
node is dropped, answered as absent (as it is), and the call reports the full pool."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

STALE = np.uint64(0x5151515151515151)


def fresh_keys(rng, held, n, crowded):
    """n keys the tree does not hold; crowded: hundreds of them between two held keys."""
    if crowded:
        at = rng.choice(held, max(n // 300, 1))
        k = rng.choice(at, 2 * n) + rng.integers(1, 1 << 14, 2 * n).astype(np.uint64)
    else:
        k = rng.integers(0, 1 << 44, 2 * n, dtype=np.uint64)
    return rng.permutation(np.setdiff1d(k, held))[:n]


@pytest.mark.parametrize("fanout", [32, 64, 128])
@pytest.mark.parametrize("n", [600, 2000, 5000, 60000])
@pytest.mark.parametrize("crowded", [False, True])
def test_full_pool(fanout, n, crowded):
    from eirene_amd import DeviceBuffer, StmError, StmTree
    rng = np.random.default_rng(fanout + n + crowded)
    load = np.unique(rng.integers(0, 1 << 44, 40000, dtype=np.uint64))
    with StmTree(fanout=fanout, max_keys=1 << 14, max_batch=1 << 16) as t:
        t.bulk_load(load, load)
        held, vals = load, load
        full = 0
        for _ in range(300):
            upd = rng.permutation(held.size)[:n // 3]
            get = rng.permutation(held.size)[:n // 20]
            get = np.setdiff1d(get, upd)
            new = fresh_keys(rng, held, n - upd.size - get.size, crowded)
            keys = np.concatenate([held[upd], held[get], new])
            ops = np.zeros(keys.size, np.uint8)  # 0: INSERT, 1: GET
            ops[upd.size:upd.size + get.size] = 1
            put = rng.integers(0, 1 << 62, keys.size, dtype=np.uint64)
            order = rng.permutation(keys.size)
            dk, dv, do = (DeviceBuffer.from_array(x[order]) for x in (keys, put, ops))
            ov = DeviceBuffer.from_array(np.full(keys.size, STALE))
            of = DeviceBuffer.from_array(np.full(keys.size, 7, np.uint8))
            try:
                t.run_batch_device(dk, dv, do, ov, of)
            except StmError as e:
                assert e.code == 2, e
                full += 1
            want_v = np.concatenate([vals[upd], vals[get], np.zeros(new.size, np.uint64)])[order]
            want_f = np.concatenate([np.ones(upd.size + get.size), np.zeros(new.size)])[order]
            np.testing.assert_array_equal(of.download(), want_f)
            np.testing.assert_array_equal(ov.download(), want_v)
            k, v = t.dump()
            assert t.size() == k.size and t.check() == 0
            # The state the batch should leave, and which of its new keys it left out.
            vals = vals.copy()
            vals[upd] = put[:upd.size]
            allk = np.concatenate([held, new])
            allv = np.concatenate([vals, put[upd.size + get.size:]])
            o = np.argsort(allk)
            allk, allv = allk[o], allv[o]
            kept = np.isin(allk, k, assume_unique=True)
            np.testing.assert_array_equal(allk[kept], k)
            np.testing.assert_array_equal(allv[kept], v)
            assert np.isin(held, k, assume_unique=True).all()
            if not full:
                assert kept.all()
            held, vals = k, v
            if full == 3:
                break
        assert full == 3
