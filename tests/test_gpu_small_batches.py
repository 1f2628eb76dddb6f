"""Small and middle-sized batches against the oracle, bit-exact: the sizes at which the batch
kernels change how they divide their work (one op, a lane group, a wavefront, a workgroup, the
lane groups the device holds at once, each side of a boundary), over key distributions that
give few and many ops per key, for each route and node size.  Inserts return the previous value,
so a second batch of the same keys also checks what the first one stored."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

SIZES = [1, 2, 63, 65, 255, 1000, 1024, 1025, 2047, 2048, 2049, 4097, 16384, 16385, 28673, 32769,
         65536, 65537, 114689, 262144, 262145]


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
    with StmTree(StmConfig(max_keys=1 << 20, max_batch=1 << 19, route=route, fanout=fanout,
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


def sample_positions(n, s):
    """Input positions the small-batch sort samples: a hashed place in each of s equal stretches."""
    def h(x):
        x = np.uint32(x)
        x = np.uint32(((int(x) ^ (int(x) >> 16)) * 0x7FEB352D) & 0xFFFFFFFF)
        x = np.uint32(((int(x) ^ (int(x) >> 15)) * 0x846CA68B) & 0xFFFFFFFF)
        return int(x) ^ (int(x) >> 16)
    lo = [j * n // s for j in range(s + 1)]
    return np.array([lo[j] + ((h(j) * (lo[j + 1] - lo[j])) >> 32) for j in range(s)])


@pytest.mark.parametrize("stream", [False, True])
def test_misleading_sample_sorts_again(oracle_mod, stream):
    """A batch whose sampled ops all hold low keys puts the rest into one bucket of the small-batch
    sort: it is sorted again exactly (sort_fallbacks = 1), the batches after it at once."""
    from eirene_amd import DeviceBuffer, StmConfig, StmTree
    rng = np.random.default_rng(5)
    n = 20000
    load = np.unique(rng.integers(0, 1 << 62, 30000, dtype=np.uint64))
    o = oracle_mod.Oracle()
    o.bulk_load(load, load)
    with StmTree(StmConfig(max_keys=1 << 20, max_batch=1 << 16)) as t:
        t.bulk_load(load, load)
        keys, vals, ops = batch(rng, "spread", 4 * n, load)
        for s in (512, 1024):  # the bucket counts of a 20000-op call and of its replayed size class
            low = sample_positions(n, s) + n
            keys[low] = np.sort(rng.choice(1 << 40, low.size, replace=False).astype(np.uint64))
        rest = np.setdiff1d(np.arange(n, 2 * n), np.concatenate(
            [sample_positions(n, s) + n for s in (512, 1024)]))
        keys[rest] = load[100] + rng.integers(0, 1 << 30, rest.size, dtype=np.uint64)
        offsets = np.arange(0, 4 * n + 1, n).astype(np.uint64)
        want = [o.run_batch(keys[a:a + n], vals[a:a + n], ops[a:a + n]) for a in range(0, 4 * n, n)]
        bufs = [DeviceBuffer.from_array(x) for x in (keys, vals, ops)]
        ov, of = DeviceBuffer(4 * n, np.uint64), DeviceBuffer(4 * n, np.uint8)
        if stream:
            t.run_batches_device(*bufs, ov, of, offsets)
        else:
            for b in range(4):
                t.run_batch_device(*bufs, ov, of, n=n, offset=b * n)
        assert np.array_equal(ov.download(), np.concatenate([w[0] for w in want]))
        assert np.array_equal(of.download(), np.concatenate([w[1] for w in want]))
        st = t.stats()
        assert st["sort_fallbacks"] == 1 and st["batches"] == 4 and st["ops"] == 4 * n
        assert t.check() == 0


def grow(oracle_mod, batches, load, **kw):
    """Runs (keys, ops) batches on a tree and the oracle; answers, dump and invariants must agree."""
    from eirene_amd import StmConfig, StmTree
    rng = np.random.default_rng(3)
    o = oracle_mod.Oracle()
    o.bulk_load(load, load)
    with StmTree(StmConfig(**{**dict(max_keys=1 << 21, max_batch=1 << 19), **kw})) as t:
        if load.size:
            t.bulk_load(load, load)
        for b, (keys, ops) in enumerate(batches):
            vals = rng.integers(0, 1 << 63, keys.size, dtype=np.uint64)
            got, want = t.run_batch(keys, vals, ops), o.run_batch(keys, vals, ops)
            assert np.array_equal(got[1], want[1]) and np.array_equal(got[0], want[0]), b
            assert t.check() == 0
        k, v = t.dump()
        ek, ev = o.dump()
        assert np.array_equal(k, ek) and np.array_equal(v, ev)
        return t.stats()


@pytest.mark.parametrize("fanout", [32, 64, 128])
@pytest.mark.parametrize("run", [1, 2, 16, 17, 63, 64, 65, 100, 1024, 1025, 5000])
def test_runs_of_one_leaf(oracle_mod, fanout, run):
    """Runs of `run` inserts into single leaves, new keys and present ones, beside leaves without
    any: leaves that fill exactly, overfill by one, split into two and into hundreds, under
    parents that overfill in turn."""
    rng = np.random.default_rng(run * 7 + fanout)
    load = np.arange(1, 6001, dtype=np.uint64) << np.uint64(40)
    batches = []
    for b in range(3):
        at = rng.choice(5990, 40 if run < 1000 else 6, replace=False)
        new = (load[at][:, None] + rng.integers(1, 1 << 39, (at.size, run), dtype=np.uint64)).ravel()
        old = np.concatenate([load[a: a + 3] for a in at])
        keys = np.concatenate([new, old, rng.choice(load, 500)])
        ops = np.concatenate([np.zeros(new.size + old.size, np.uint8), np.ones(500, np.uint8)])
        order = rng.permutation(keys.size)
        batches.append((keys[order], ops[order]))
    st = grow(oracle_mod, batches, load, fanout=fanout)
    assert st["deferred"] == 0


@pytest.mark.parametrize("fanout", [32, 64, 128])
@pytest.mark.parametrize("n", [1, 32, 33, 64, 65, 129, 3000, 200000])
def test_inserts_into_an_empty_tree(oracle_mod, fanout, n):
    """Every insert goes into the one leaf: the root splits, for the larger batches into more nodes
    than one new root holds."""
    rng = np.random.default_rng(n + fanout)
    batches = [(rng.integers(0, 1 << 63, m, dtype=np.uint64), np.zeros(m, np.uint8))
               for m in (n, max(1, n // 3))]
    st = grow(oracle_mod, batches, np.zeros(0, np.uint64), fanout=fanout)
    assert st["height"] > 1 or n <= fanout


def test_pool_runs_full(oracle_mod):
    """Batches past what the pool holds: the call reports it, and the tree stays well formed and
    keeps every key it had."""
    from eirene_amd import StmConfig, StmError, StmTree
    rng = np.random.default_rng(9)
    with StmTree(StmConfig(max_keys=2000, max_batch=1 << 16)) as t:
        kept = None
        for _ in range(40):
            keys = rng.integers(0, 1 << 63, 4000, dtype=np.uint64)
            try:
                t.run_batch(keys, keys, np.zeros(keys.size, np.uint8))
            except StmError as e:
                assert e.code == 2
                break
            kept = t.dump()[0]
        else:
            pytest.fail("the pool never ran full")
        assert t.check() == 0
        assert np.isin(kept, t.dump()[0]).all()
