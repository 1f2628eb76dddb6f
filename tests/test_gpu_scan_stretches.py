"""Range scans that go from node to node without a merge while the batch inserts nothing into their
way, against the oracle: batches of lookups and scans alone, an insert that ends such a walk in its
first stretch or a later one, more lookups than the walk looks through on its way, leaves with
appended entries and split leaves; four wavefronts per scan (below 8192 ops), one, a tree of one
leaf."""
import numpy as np
import pytest

from test_gpu_scan import check_scan_batch

pytestmark = pytest.mark.gpu

OP_INSERT, OP_GET, OP_RANGE = 0, 1, 3
SPAN = 1 << 40


def lengths_of(fanout):
    per = fanout - fanout // 4  # entries of a leaf as built, children of a node as built
    return np.array([100, 1, 2, per - 1, per, per + 1, 4 * per, 4 * per + 1, 8 * per - 1, 8 * per,
                     8 * per + 1, per * per - 1, per * per, per * per + 1, 3 * per * per + 5, 20, 257,
                     1000])


def loaded(rng, held):
    return np.unique(rng.integers(1, SPAN, held, dtype=np.uint64))


def scan_batch(rng, srt, n, lengths, inserts):
    keys = rng.integers(0, SPAN, n, dtype=np.uint64)
    ops = np.full(n, OP_GET, dtype=np.uint8)
    ops[rng.random(n) < inserts] = OP_INSERT
    vals = rng.integers(0, 1 << 40, n, dtype=np.uint64)
    at = rng.choice(n, lengths.size, replace=False)
    ops[at] = OP_RANGE
    vals[at] = lengths
    keys[at] = rng.choice(srt, lengths.size) + rng.integers(0, 2, lengths.size).astype(np.uint64)
    keys[at[:2]] = [0, srt[-1] + np.uint64(1)]
    if inserts == 0:
        assert (ops == OP_INSERT).sum() == 0
    return keys, vals, ops


@pytest.mark.parametrize("fanout", [32, 64, 128])
@pytest.mark.parametrize("n,inserts,held", [(300, 0.0, 50000), (300, 0.02, 50000), (300, 0.0, 7),
                                            (6000, 0.0, 20000), (6000, 0.001, 20000),
                                            (9000, 0.0, 50000), (9000, 0.001, 20000)])
def test_scans_with_few_inserts(oracle_mod, fanout, n, inserts, held):
    from eirene_amd import StmConfig, StmTree
    rng = np.random.default_rng(fanout * 100 + n)
    load = loaded(rng, held)
    o = oracle_mod.Oracle()
    o.bulk_load(load, load + 1)
    with StmTree(StmConfig(fanout=fanout, max_keys=1 << 18, max_batch=1 << 16)) as t:
        t.bulk_load(load, load + 1)
        for b in range(3):
            batch = scan_batch(rng, load, n, lengths_of(fanout), inserts)
            check_scan_batch(t, o, *batch, f"batch {b}")
            # New keys, half as many as the tree was loaded with in the end: entries out of order,
            # split leaves.
            size = t.size()
            more = rng.integers(1, SPAN, held // 6 + 1, dtype=np.uint64)
            ops = np.full(more.size, OP_INSERT, dtype=np.uint8)
            t.run_batch(more, more, ops)
            o.run_batch(more, more, ops)
            assert t.size() > size
        assert t.check() == 0


@pytest.mark.parametrize("fanout", [32, 64, 128])
@pytest.mark.parametrize("n", [40, 8192])
def test_one_insert_on_the_way(oracle_mod, fanout, n):
    """One insert of a new key at every distance from the scan's start, before and after it in the
    batch, among lookups of keys outside the scan's range."""
    from eirene_amd import StmConfig, StmTree
    rng = np.random.default_rng(fanout + n)
    load = loaded(rng, 40000)
    o = oracle_mod.Oracle()
    o.bulk_load(load, load + 1)
    per = fanout - fanout // 4
    length = 2 * per * per + 3
    start = 1000
    with StmTree(StmConfig(fanout=fanout, max_keys=1 << 18, max_batch=1 << 16)) as t:
        t.bulk_load(load, load + 1)
        for i, d in enumerate([0, 1, per, 3 * per, 9 * per, per * per + 7, 2 * per * per, length,
                               length + 5 * per]):
            key = load[start + d] + np.uint64(1)
            for place in (0, n - 1):
                keys = rng.choice(load[:900], n).astype(np.uint64)
                vals = np.zeros(n, dtype=np.uint64)
                ops = np.full(n, OP_GET, dtype=np.uint8)
                keys[n // 2], vals[n // 2], ops[n // 2] = load[start], length, OP_RANGE
                keys[place], vals[place], ops[place] = key, 7 + i, OP_INSERT
                check_scan_batch(t, o, keys, vals, ops, f"distance {d} place {place}")
        assert t.check() == 0


@pytest.mark.parametrize("lookups", [255, 256, 257, 300, 5000])
def test_lookups_on_the_way(oracle_mod, lookups):
    """Lookups of keys inside the scans' ranges: as many as the walk looks through, and more."""
    from eirene_amd import StmConfig, StmTree
    rng = np.random.default_rng(lookups)
    load = loaded(rng, 60000)
    o = oracle_mod.Oracle()
    o.bulk_load(load, load + 1)
    lengths = np.array([10000, 2500, 48, 3000, 20000])
    with StmTree(StmConfig(max_keys=1 << 18, max_batch=1 << 16)) as t:
        t.bulk_load(load, load + 1)
        n = lookups + lengths.size
        keys = rng.choice(load[2000:4000], n, replace=lookups > 1900).astype(np.uint64)
        vals = np.zeros(n, dtype=np.uint64)
        ops = np.full(n, OP_GET, dtype=np.uint8)
        at = rng.choice(n, lengths.size, replace=False)
        keys[at], vals[at], ops[at] = load[[1990, 1999, 2000, 3000, 1]], lengths, OP_RANGE
        check_scan_batch(t, o, keys, vals, ops)
