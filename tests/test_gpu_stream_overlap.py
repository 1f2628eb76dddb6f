"""Batch streams whose sorts run on the second stream beside the batch before, against the oracle:
mixed sizes, learned routing that retrains between batches, a reserved key, a full pool and a
misleading sample in mid-stream (with later sorts already done), small batches among overlapped ones.

A tree overlaps once its streams have brought enough large batches ("fed") or stm_capture_graphs has
prepared it ("captured", which also replays the batches of up to 4096 ops)."""
import numpy as np
import pytest

from test_gpu_small_batches import sample_positions
from test_gpu_stream import check_same, make_stream, oracle_replay, run_stream

pytestmark = pytest.mark.gpu

RESERVED = np.uint64(0xFFFFFFFFFFFFFFFF)
OP_INSERT, OP_GET = 0, 1
WAYS = pytest.mark.parametrize("way", ["fed", "captured"])


def prepared(way, load, lv, **kw):
    from eirene_amd import StmTree
    t = StmTree(**{**dict(max_keys=1 << 20, max_batch=1 << 14), **kw})
    t.bulk_load(load, lv)
    if way == "captured":
        t.capture_graphs()
    else:
        n = 40 * 2049
        run_stream(t, np.resize(load, n), np.resize(lv, n), np.full(n, OP_GET, np.uint8),
                   (np.arange(41) * 2049).astype(np.uint64))
    return t


def check_tree(t, o):
    k, v = t.dump()
    ek, ev = o.dump()
    np.testing.assert_array_equal(k, ek)
    np.testing.assert_array_equal(v, ev)
    assert t.check() == 0


@WAYS
@pytest.mark.parametrize("fanout,tile,per_wave", [(32, 8, 512), (64, 16, 512), (64, 16, 32), (128, 16, 512)])
def test_overlapped_stream(oracle_mod, way, fanout, tile, per_wave):
    rng = np.random.default_rng(fanout + tile + per_wave)
    load = rng.integers(0, 1 << 63, size=40000, dtype=np.uint64)
    lv = rng.integers(0, 1 << 63, size=load.size, dtype=np.uint64)
    keys, vals, ops, offsets = make_stream(fanout * 7 + tile, load, 80, 1 << 14)
    o, want_v, want_f = oracle_replay(oracle_mod, load, lv, keys, vals, ops, offsets)
    with prepared(way, load, lv, fanout=fanout, sort_tile_items=tile, upsert_ops_per_wave=per_wave) as t:
        before = t.stats()["ops"]
        check_same(*run_stream(t, keys, vals, ops, offsets, calls=2), want_v, want_f)
        assert t.stats()["ops"] - before == keys.size
        check_tree(t, o)


@WAYS
def test_small_batches_between_large_ones(oracle_mod, way):
    """Large batches alternate between the scratch sets; small ones take the first set between."""
    rng = np.random.default_rng(8)
    load = rng.integers(0, 1 << 44, size=30000, dtype=np.uint64)
    sizes = np.array([5000, 7, 5000, 5000, 2048, 9000, 1, 1, 9000, 16000, 300, 16000, 3000, 16000] * 4)
    n = int(sizes.sum())
    keys = np.where(rng.random(n) < 0.5, rng.choice(load, n),
                    rng.integers(0, 1 << 44, n, dtype=np.uint64)).astype(np.uint64)
    vals = rng.integers(0, 1 << 62, n, dtype=np.uint64)
    ops = np.where(rng.random(n) < 0.3, OP_INSERT, OP_GET).astype(np.uint8)
    offsets = np.concatenate([[0], np.cumsum(sizes)]).astype(np.uint64)
    o, want_v, want_f = oracle_replay(oracle_mod, load, load, keys, vals, ops, offsets)
    with prepared(way, load, load) as t:
        check_same(*run_stream(t, keys, vals, ops, offsets), want_v, want_f)
        check_tree(t, o)


@WAYS
def test_overlapped_learned_stream(oracle_mod, way):
    from eirene_amd import ROUTE_LEARNED
    rng = np.random.default_rng(17)
    load = np.unique(rng.gamma(2.0, 2.0 ** 40, size=60000).astype(np.uint64))
    lv = rng.integers(0, 1 << 63, size=load.size, dtype=np.uint64)
    keys, vals, ops, offsets = make_stream(23, load, 60, 1 << 14)
    o, want_v, want_f = oracle_replay(oracle_mod, load, lv, keys, vals, ops, offsets)
    with prepared(way, load, lv, route=ROUTE_LEARNED, retrain_every=3, train_steps=50, timing=True) as t:
        trained = t.stats()["phase_launches"]["train"]
        check_same(*run_stream(t, keys, vals, ops, offsets), want_v, want_f)
        check_tree(t, o)
        st = t.stats()
        assert st["route_hits"] > 0 and st["phase_launches"]["train"] - trained >= 10


@WAYS
@pytest.mark.parametrize("where", [5, 6])
def test_reserved_key_in_mid_stream(oracle_mod, way, where):
    """The tree holds the batches up to and including the failing one (less its reserved ops)."""
    from eirene_amd import DeviceBuffer, StmError
    rng = np.random.default_rng(29 + where)
    load = rng.integers(0, 1 << 62, size=20000, dtype=np.uint64)
    sizes = np.array([6000, 3000, 5000, 100, 7000, 6000, 900, 6000, 12000, 50, 9000])
    n = int(sizes.sum())
    offsets = np.concatenate([[0], np.cumsum(sizes)]).astype(np.uint64)
    keys = np.where(rng.random(n) < 0.5, rng.choice(load, n),
                    rng.integers(0, 1 << 62, n, dtype=np.uint64)).astype(np.uint64)
    vals = rng.integers(0, 1 << 62, n, dtype=np.uint64)
    ops = np.where(rng.random(n) < 0.3, OP_INSERT, OP_GET).astype(np.uint8)
    a, z = int(offsets[where]), int(offsets[where + 1])
    keys[[a + 3, (a + z) // 2]] = RESERVED
    ops[[a + 3, (a + z) // 2]] = [OP_INSERT, OP_GET]
    real = keys != RESERVED
    # without the two reserved ops
    o, want_v, want_f = oracle_replay(oracle_mod, load, load, keys[:z][real[:z]], vals[:z][real[:z]],
                                      ops[:z][real[:z]],
                                      np.minimum(offsets[:where + 2], z - 2).astype(np.uint64))
    with prepared(way, load, load) as t:
        dk, dv, do = (DeviceBuffer.from_array(x) for x in (keys, vals, ops))
        ov, of = DeviceBuffer(n, np.uint64), DeviceBuffer(n, np.uint8)
        with pytest.raises(StmError) as e:
            t.run_batches_device(dk, dv, do, ov, of, offsets)
        assert e.value.code == 1 and f"{sizes.size - 1 - where} later batches skipped" in str(e.value)
        check_same(ov.download()[:z][real[:z]], of.download()[:z][real[:z]], want_v, want_f)
        check_tree(t, o)


@WAYS
def test_full_pool_in_mid_stream(oracle_mod, way):
    from eirene_amd import DeviceBuffer, StmError
    rng = np.random.default_rng(31)
    load = np.unique(rng.integers(0, 1 << 62, 30000, dtype=np.uint64))
    size, batches = 8000, 24
    keys = rng.permutation(np.setdiff1d(rng.integers(0, 1 << 62, size * batches + 100, dtype=np.uint64),
                                        load))[:size * batches]
    ops = np.full(keys.size, OP_INSERT, np.uint8)
    offsets = (np.arange(batches + 1) * size).astype(np.uint64)
    with prepared(way, load, load, max_keys=1 << 14) as t:
        dk, do = DeviceBuffer.from_array(keys), DeviceBuffer.from_array(ops)
        ov, of = DeviceBuffer(keys.size, np.uint64), DeviceBuffer(keys.size, np.uint8)
        with pytest.raises(StmError) as e:
            t.run_batches_device(dk, dk, do, ov, of, offsets)
        assert e.value.code == 2 and "later batches skipped" in str(e.value)
        k, v = t.dump()
        np.testing.assert_array_equal(k, v)
        assert t.check() == 0 and np.isin(load, k).all()
        # Whole batches, then part of one, then nothing.
        share = np.array([np.isin(keys[i * size:(i + 1) * size], k).mean() for i in range(batches)])
        last = int(np.flatnonzero(share > 0)[-1])
        assert 0 < last < batches - 1 and (share[:last] == 1).all() and 0 < share[last] < 1
        assert not of.download()[:last * size].any() and not ov.download()[:last * size].any()


@WAYS
@pytest.mark.parametrize("at", [1, 4, 9])
def test_misleading_sample_in_mid_stream(oracle_mod, way, at):
    """Batch `at` runs empty and the ones whose sorts were done beside it too; it is run again
    exactly, and the stream goes on."""
    rng = np.random.default_rng(5 + at)
    n, batches = 12000, 12
    load = np.unique(rng.integers(0, 1 << 62, 30000, dtype=np.uint64))
    keys = np.where(rng.random(batches * n) < 0.5, rng.choice(load, batches * n),
                    rng.integers(0, 1 << 62, batches * n, dtype=np.uint64)).astype(np.uint64)
    vals = rng.integers(0, 1 << 62, keys.size, dtype=np.uint64)
    ops = np.where(rng.random(keys.size) < 0.4, OP_INSERT, OP_GET).astype(np.uint8)
    low = sample_positions(n, 256)
    rest = np.setdiff1d(np.arange(n), low)
    keys[at * n + low] = np.sort(rng.choice(1 << 40, low.size, replace=False).astype(np.uint64))
    keys[at * n + rest] = load[100] + rng.integers(0, 1 << 30, rest.size, dtype=np.uint64)
    offsets = (np.arange(batches + 1) * n).astype(np.uint64)
    o, want_v, want_f = oracle_replay(oracle_mod, load, load, keys, vals, ops, offsets)
    with prepared(way, load, load) as t:
        before = t.stats()
        check_same(*run_stream(t, keys, vals, ops, offsets), want_v, want_f)
        check_tree(t, o)
        st = t.stats()
        assert st["sort_fallbacks"] == 1
        assert st["batches"] - before["batches"] == batches and st["ops"] - before["ops"] == keys.size
