"""Small and middle-sized batches against the oracle, bit-exact: the sizes at which the batch
kernels change how they divide their work (one op, a lane group, a wavefront, a workgroup, the
lane groups the device holds at once, each side of a boundary), over key distributions that
give few and many ops per key, for each route and node size.  Inserts return the previous value,
so a second batch of the same keys also checks what the first one stored."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

SIZES = [1, 2, 63, 65, 255, 1000, 2047, 2048, 2049, 4097, 16384, 16385, 28673, 65537, 114689]


def batch(rng, dist, n, load):
    if dist == "spread":
        keys = np.where(rng.random(n) < 0.6, rng.choice(load, n),
                        rng.integers(0, 1 << 63, n, dtype=np.uint64))
    elif dist == "few":  # many ops per key
        keys = rng.choice(load[: max(1, n // 50)], n)
    else:  # one key takes a third, distinct keys just above it another third
        keys = rng.choice(load, n)
        m = n // 3
        keys[:m] = load[0]
        keys[m: 2 * m] = load[0] + rng.integers(1, 1 << 20, m).astype(np.uint64)
        rng.shuffle(keys)
    return (keys, rng.integers(0, 1 << 63, n, dtype=np.uint64),
            rng.choice(4, n, p=[0.3, 0.6, 0.05, 0.05]).astype(np.uint8))


@pytest.mark.parametrize("n", SIZES)
@pytest.mark.parametrize("dist,route,fanout,lanes", [
    ("spread", 0, 64, 16), ("few", 1, 64, 16), ("hot", 2, 32, 8), ("spread", 1, 128, 64)])
def test_batch_sizes(oracle_mod, n, dist, route, fanout, lanes):
    from eirene_amd import StmConfig, StmTree
    rng = np.random.default_rng(n * 31 + fanout)
    load = np.unique(rng.integers(0, 1 << 62, 40000, dtype=np.uint64))
    rng.shuffle(load)
    lv = rng.integers(0, 1 << 63, load.size, dtype=np.uint64)
    o = oracle_mod.Oracle()
    o.bulk_load(load, lv)
    with StmTree(StmConfig(max_keys=1 << 20, max_batch=1 << 17, route=route, fanout=fanout,
                           lanes_per_op=lanes, train_steps=20)) as t:
        t.bulk_load(load, lv)
        keys, vals, ops = batch(rng, dist, n, load)
        for _ in range(2):
            got, want = t.run_batch(keys, vals, ops), o.run_batch(keys, vals, ops)
            assert np.array_equal(got[1], want[1]) and np.array_equal(got[0], want[0])
            vals = vals + np.uint64(1)
        k, v = t.dump()
        ek, ev = o.dump()
        assert np.array_equal(k, ek) and np.array_equal(v, ev)
        assert t.check() == 0
