"""Range scans that take whole level-1 nodes where the batch inserts nothing, against the oracle:
lengths at the edges of leaves, chunks and nodes, starts before the first and after the last key,
inserts that end the fast form in the first stretch or a later one, more than four windows of
groups inside a scan, leaves with appended entries; four wavefronts per scan (up to 8191 ops), one,
and a tree of one leaf."""
import numpy as np
import pytest

from test_gpu_scan import check_scan_batch

pytestmark = pytest.mark.gpu


def scan_batch(rng, load, n, lengths, inserts, span):
    srt = np.sort(load)
    keys = rng.integers(0, span, n, dtype=np.uint64)
    ops = np.zeros(n, dtype=np.uint8)
    ops[rng.random(n) < inserts] = 1
    vals = rng.integers(0, 1 << 40, n, dtype=np.uint64)
    at = rng.choice(n, lengths.size, replace=False)
    ops[at] = 3
    vals[at] = lengths
    keys[at] = rng.choice(srt, lengths.size) + rng.integers(0, 2, lengths.size).astype(np.uint64)
    keys[at[:2]] = [0, srt[-1] + np.uint64(1)]
    return keys, vals, ops


@pytest.mark.parametrize("fanout", [32, 64, 128])
@pytest.mark.parametrize("n,inserts,held", [(300, 0.0, 50000), (300, 0.02, 50000), (300, 0.0, 7),
                                            (6000, 0.0, 20000), (6000, 0.001, 20000),
                                            (9000, 0.001, 20000)])
def test_scans_by_level_1_nodes(oracle_mod, fanout, n, inserts, held):
    from eirene_amd import StmConfig, StmTree
    rng = np.random.default_rng(fanout * 100 + n)
    span = 1 << 40
    load = np.unique(rng.integers(1, span, held, dtype=np.uint64))
    per = fanout - fanout // 4
    lengths = np.array([100, 1, 2, per - 1, per, per + 1, 4 * per, 8 * per - 1, 8 * per, 8 * per + 1,
                        per * per - 1, per * per, per * per + 1, 3 * per * per + 5, 20, 257, 1000])
    o = oracle_mod.Oracle()
    o.bulk_load(load, load + 1)
    with StmTree(StmConfig(fanout=fanout, max_keys=1 << 18, max_batch=1 << 16)) as t:
        t.bulk_load(load, load + 1)
        for b in range(3):
            keys, vals, ops = scan_batch(rng, load, n, lengths, inserts, span)
            check_scan_batch(t, o, keys, vals, ops, f"batch {b}")
            # New keys of two batches' worth: leaves with entries out of order, and splits.
            more = rng.integers(1, span, held // 10 + 1, dtype=np.uint64)
            one = np.ones(more.size, dtype=np.uint8)
            t.run_batch(more, more, one)
            o.run_batch(more, more, one)
        assert t.check() == 0
