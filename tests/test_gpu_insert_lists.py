"""Batches of inserts alone, at the sizes where the insert list is dealt out differently (64, 65536
merged INSERTs) and with parts that end inside a leaf's run, against the oracle."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

OP_INSERT = 0


@pytest.mark.parametrize("fanout", [32, 64, 128])
@pytest.mark.parametrize("n", [7, 8, 9, 63, 64, 65, 2047, 2049, 16385, 65535, 65536, 65537])
@pytest.mark.parametrize("dense", [False, True])
def test_lists_of_inserts(oracle_mod, fanout, n, dense):
    from eirene_amd import StmConfig, StmTree
    rng = np.random.default_rng(n + fanout)
    load = np.unique(rng.integers(0, 1 << 40, 30000, dtype=np.uint64))
    o = oracle_mod.Oracle()
    o.bulk_load(load, load)
    held = load.size
    with StmTree(StmConfig(fanout=fanout, max_keys=1 << 19, max_batch=1 << 17)) as t:
        t.bulk_load(load, load)
        for b in range(2):
            keys = rng.integers(0, 1 << 40, 2 * n + 64, dtype=np.uint64)
            if dense:  # half of them in runs of up to 200 beside some of the held keys
                at = rng.choice(load, n // 100 + 1)
                keys[::2] = rng.choice(at, keys[::2].size) + rng.integers(1, 1 << 20, keys[::2].size).astype(np.uint64)
            keys = rng.permutation(np.unique(keys))[:n]
            keys[:n // 8] = rng.permutation(load)[:n // 8]  # some are updates
            keys = np.unique(keys)
            keys = rng.permutation(keys)
            vals = rng.integers(0, 1 << 63, keys.size, dtype=np.uint64)
            before = t.stats()["upserts"]
            ops = np.full(keys.size, OP_INSERT, dtype=np.uint8)
            want = o.run_batch(keys, vals, ops)
            got = t.run_batch(keys, vals, ops)
            assert np.array_equal(got[0], want[0]) and np.array_equal(got[1], want[1]), b
            assert t.stats()["upserts"] - before == keys.size
            held += int((want[1] == 0).sum())
            assert t.size() == held
        if n > 20000:
            assert t.stats()["leaf_splits"] > 0
        k, v = t.dump()
        ek, ev = o.dump()
        assert np.array_equal(k, ek) and np.array_equal(v, ev)
        assert t.check() == 0
