"""The sample sort of 393217 .. 2^22 keys against numpy's stable argsort, bit-exact: the edges of
its shapes and tiles, sorted and reversed input (whole tiles in one bucket), hot keys that fill
many buckets, keys that crowd a bin, a bucket too large for one workgroup (taken in groups of its sample
intervals) and a sample that misleads (sorted again by the exact passes)."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

LO, MAX = (3 << 17) + 1, 1 << 22


def samples_of(n):
    return 8 * (512 if n <= 1 << 19 else 1024 if n <= 1 << 20 else 2048)


def sample_positions(n):
    """Where the sort draws its samples: one per equal stretch of the input, at a hashed place."""
    m32 = np.uint64(0xFFFFFFFF)
    s = samples_of(n)
    j = np.arange(s, dtype=np.uint64)
    x = ((j ^ (j >> np.uint64(16))) * np.uint64(0x7FEB352D)) & m32
    x = ((x ^ (x >> np.uint64(15))) * np.uint64(0x846CA68B)) & m32
    x = x ^ (x >> np.uint64(16))
    lo = j * np.uint64(n) // np.uint64(s)
    hi = (j + np.uint64(1)) * np.uint64(n) // np.uint64(s)
    return (lo + ((x * (hi - lo)) >> np.uint64(32))).astype(np.int64)


def crafted(n, rng, width, many=12000):
    """Evenly spread samples; `many` of the other keys within `width` intervals from the 800th on."""
    s = samples_of(n)
    keys = rng.integers(0, s << 40, n, dtype=np.uint64)
    at = sample_positions(n)
    rest = np.setdiff1d(np.arange(n), at)
    dense = rng.choice(rest, many, replace=False)
    keys[dense] = np.uint64(800 << 40) + rng.integers(0, width << 40, dense.size, dtype=np.uint64)
    keys[at] = rng.permutation(s).astype(np.uint64) << np.uint64(40)
    return keys


def keys_of(dist, n, rng):
    if dist == "uniform":
        return rng.integers(0, 1 << 63, n, dtype=np.uint64)
    if dist == "sorted":
        return np.sort(rng.integers(0, 1 << 63, n, dtype=np.uint64))
    if dist == "reversed":
        return np.sort(rng.integers(0, 1 << 63, n, dtype=np.uint64))[::-1].copy()
    if dist == "normal":
        return (rng.normal(2.0 ** 62, 2.0 ** 58, n)).clip(0).astype(np.uint64)
    if dist == "zipf":  # from a key in a twentieth of the places down to single ones
        return (rng.zipf(1.2, n) % 1000003).astype(np.uint64) << np.uint64(40)
    if dist == "crowded":  # keys of 33..4000 places each, some beside a neighbour, some in a row
        sizes = rng.integers(33, 4000, n // 1000 + 1)
        keys = np.repeat(np.sort(rng.integers(0, 1 << 62, sizes.size, dtype=np.uint64)), sizes)[:n]
        keys = np.concatenate([keys, keys[: n - keys.size]])
        near = rng.random(n) < 0.05
        keys[near] += rng.integers(1, 4, int(near.sum()), dtype=np.uint64)
        keys[: n // 2] = rng.permutation(keys[: n // 2])
        return keys
    if dist == "extremes":
        return np.where(rng.random(n) < 0.5, np.uint64(0), np.uint64(2 ** 64 - 1))
    if dist == "overfull":
        return crafted(n, rng, 8)
    return crafted(n, rng, 1)  # misleading


@pytest.mark.parametrize("dist", ["uniform", "sorted", "reversed", "normal", "zipf", "crowded",
                                  "extremes", "overfull", "misleading"])
@pytest.mark.parametrize("n", [LO, 1 << 19, (1 << 19) + 1, (1 << 20) + 4095, 1 << 21, MAX - 1, MAX])
def test_sorts_like_a_stable_argsort(dist, n):
    from eirene_amd import sort_pairs
    keys = keys_of(dist, n, np.random.default_rng(n))
    got_k, got_i = sort_pairs(keys)
    want = np.argsort(keys, kind="stable")
    assert np.array_equal(got_i, want.astype(np.uint32))
    assert np.array_equal(got_k, keys[want])


@pytest.mark.parametrize("dist,fallbacks", [("overfull", 0), ("misleading", 1)])
def test_batches_count_the_exact_sort(oracle_mod, dist, fallbacks):
    from eirene_amd import StmConfig, StmTree
    rng = np.random.default_rng(3)
    n = 400000
    keys = crafted(n, rng, 8 if dist == "overfull" else 1)
    vals = rng.integers(0, 1 << 63, n, dtype=np.uint64)
    ops = (rng.random(n) < 0.9).astype(np.uint8)
    load = np.unique(rng.choice(keys, 50000))
    o = oracle_mod.Oracle()
    o.bulk_load(load, load)
    want = o.run_batch(keys, vals, ops)
    with StmTree(StmConfig(max_keys=1 << 20, max_batch=1 << 19)) as t:
        t.bulk_load(load, load)
        got = t.run_batch(keys, vals, ops)
        assert np.array_equal(got[0], want[0]) and np.array_equal(got[1], want[1])
        assert t.stats()["sort_fallbacks"] == fallbacks
        k, v = t.dump()
        ek, ev = o.dump()
        assert np.array_equal(k, ek) and np.array_equal(v, ev)
        assert t.check() == 0


@pytest.mark.parametrize("n", [400000, MAX])
@pytest.mark.parametrize("equal", [False, True])
def test_one_large_interval_is_halved(n, equal):
    """6000 keys between two samples, spread or all equal to the lower one: no exact sort, checked by
    its results alone where the keys go through sort_pairs."""
    from eirene_amd import sort_pairs
    rng = np.random.default_rng(n + equal)
    keys = crafted(n, rng, 1, 6000)
    if equal:
        inside = (keys >= np.uint64(800 << 40)) & (keys < np.uint64(801 << 40))
        keys[inside] = np.uint64(800 << 40)
    got_k, got_i = sort_pairs(keys)
    want = np.argsort(keys, kind="stable")
    assert np.array_equal(got_i, want.astype(np.uint32))
    assert np.array_equal(got_k, keys[want])


def test_one_large_interval_needs_no_exact_sort(oracle_mod):
    from eirene_amd import StmConfig, StmTree
    rng = np.random.default_rng(4)
    n = 400000
    keys = crafted(n, rng, 1, 6000)
    vals = rng.integers(0, 1 << 63, n, dtype=np.uint64)
    ops = (rng.random(n) < 0.5).astype(np.uint8)
    o = oracle_mod.Oracle()
    want = o.run_batch(keys, vals, ops)
    with StmTree(StmConfig(max_keys=1 << 20, max_batch=1 << 19)) as t:
        got = t.run_batch(keys, vals, ops)
        assert np.array_equal(got[0], want[0]) and np.array_equal(got[1], want[1])
        assert t.stats()["sort_fallbacks"] == 0
