"""The device sort of up to 2^18 keys (one workgroup up to 2048, sampled buckets above) against
numpy's stable argsort: the edges of its shapes and tiles, equal keys, few keys, crowded keys, the
extremes, and keys that mislead its sample, which the exact passes then sort."""
import numpy as np
import pytest

from test_gpu_small_batches import sample_positions

pytestmark = pytest.mark.gpu


def samples_of(n):
    return 256 if n <= 1 << 14 else 512 if n <= 1 << 15 else 1024 if n <= 1 << 16 else 2048


def keys_of(dist, n, rng):
    if dist == "uniform":
        return rng.integers(0, 1 << 63, n, dtype=np.uint64)
    if dist == "sorted":
        return np.sort(rng.integers(0, 1 << 63, n, dtype=np.uint64))
    if dist == "equal":
        return np.full(n, 7, dtype=np.uint64)
    if dist == "few":
        return rng.choice(rng.integers(0, 1 << 63, 5, dtype=np.uint64), n)
    if dist == "crowded":
        return np.uint64(1 << 50) * rng.integers(0, 9, n, dtype=np.uint64) + rng.integers(0, 40, n, dtype=np.uint64)
    if dist == "extremes":
        return np.where(rng.random(n) < 0.5, np.uint64(0), np.uint64(2 ** 64 - 1))
    keys = np.uint64(1 << 61) + rng.integers(0, 1 << 40, n, dtype=np.uint64)  # misleading
    if n > 2048:
        at = sample_positions(n, samples_of(n))
        keys[at] = np.sort(rng.choice(1 << 40, at.size, replace=False).astype(np.uint64))
    return keys


@pytest.mark.parametrize("dist", ["uniform", "sorted", "equal", "few", "crowded", "extremes", "misleading"])
@pytest.mark.parametrize("n", [1, 2, 63, 64, 65, 1023, 1024, 1025, 2047, 2048, 2049, 3071, 16384, 16385,
                               32768, 32769, 65536, 65537, 200001, (1 << 18) - 1, 1 << 18, (1 << 18) + 1])
def test_sorts_like_a_stable_argsort(dist, n):
    from eirene_amd import sort_pairs
    keys = keys_of(dist, n, np.random.default_rng(n))
    got_k, got_i = sort_pairs(keys)
    want = np.argsort(keys, kind="stable")
    assert np.array_equal(got_i, want.astype(np.uint32))
    assert np.array_equal(got_k, keys[want])


@pytest.mark.parametrize("n", [1, 50, 2000, 3000, 150000])
@pytest.mark.parametrize("route", [0, 1, 2])
def test_trees_of_few_leaves(oracle_mod, n, route):
    """Loads, dumps and leaf directories of small trees go through the same sorts."""
    from eirene_amd import StmTree
    rng = np.random.default_rng(n)
    load = rng.integers(0, 1 << 62, n, dtype=np.uint64)
    load[::3] = load[0]  # repeated keys: the last value stays
    vals = rng.integers(0, 1 << 62, n, dtype=np.uint64)
    o = oracle_mod.Oracle()
    o.bulk_load(load, vals)
    with StmTree(max_keys=1 << 18, max_batch=1 << 12, route=route, train_steps=20) as t:
        t.bulk_load(load, vals)
        if route:
            t.retrain()
            fences, _ = t.route_directory()
            assert (np.diff(fences.astype(np.int64)) > 0).all()
        v, f = t.run_batch(load, vals, np.ones(n, np.uint8))
        ev, ef = o.run_batch(load, vals, np.ones(n, np.uint8))
        np.testing.assert_array_equal(v, ev)
        np.testing.assert_array_equal(f, ef)
        k, d = t.dump()
        ek, ed = o.dump()
        np.testing.assert_array_equal(k, ek)
        np.testing.assert_array_equal(d, ed)
        assert t.check() == 0
