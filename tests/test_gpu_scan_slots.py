"""A scan that reaches the end of the key space leaves the rest of its slots as the caller had them.

The device areas that a batch's pairs come from held other batches' pairs before; the caller's
arrays must not receive those.  Scans of whole length stand before, between and after the short
ones, so that every stretch of written slots is checked for its place.
"""
import ctypes as C

import numpy as np
import pytest

pytestmark = pytest.mark.gpu

OP_INSERT, OP_GET, OP_RANGE = 0, 1, 3
LOADED = np.arange(1, 5001, dtype=np.uint64) * np.uint64(10)
FREE = np.uint64(0xABABABABABABABAB)


def tree():
    from eirene_amd import StmTree
    t = StmTree(max_keys=1 << 16, max_batch=1 << 10)
    t.bulk_load(LOADED, LOADED * np.uint64(3))
    return t


def scans_from(starts, lengths):
    return (np.array(starts, np.uint64), np.array(lengths, np.uint64),
            np.full(len(starts), OP_RANGE, np.uint8))


FULL = scans_from([10] * 40, [200] * 40)  # every slot of the area is written
# (start, length): 50000 is the last key
SHORT = scans_from([49910, 100, 50001, 49500, 50000, 20, 49990], [50, 30, 70, 40, 1, 25, 300])


def expected(keys, lengths):
    """(area keys, area values, pairs per scan) with FREE in the slots no scan writes."""
    area_k, area_v, pairs = [], [], []
    for k, n in zip(keys, lengths):
        x = LOADED[LOADED >= k][:int(n)]
        pad = np.full(int(n) - x.size, FREE, np.uint64)
        area_k += [x, pad]
        area_v += [x * np.uint64(3), pad]
        pairs.append(x.size)
    return np.concatenate(area_k), np.concatenate(area_v), pairs


def outputs(n, slots):
    return (np.zeros(n, np.uint64), np.zeros(n, np.uint8), np.full(slots, FREE, np.uint64),
            np.full(slots, FREE, np.uint64))


def check(batch, out):
    keys, lengths, _ = batch
    ek, ev, pairs = expected(keys, lengths)
    assert out[0].tolist() == pairs
    assert out[1].tolist() == [1 if p else 0 for p in pairs]
    np.testing.assert_array_equal(out[2], ek)
    np.testing.assert_array_equal(out[3], ev)


def test_server_leaves_unwritten_slots():
    from eirene_amd import serving
    lib = serving._lib()
    with tree() as t, serving.Server(t, hbm_budget=64 << 20) as srv:
        def request(batch):
            keys, lengths, ops = batch
            out = outputs(keys.size, int(lengths.sum()))
            ticket = C.c_uint64()
            assert lib.stm_server_submit(
                srv._h, keys.ctypes.data, lengths.ctypes.data, ops.ctypes.data, keys.size,
                out[0].ctypes.data, out[1].ctypes.data, out[2].ctypes.data, out[3].ctypes.data,
                out[2].size, -1.0, C.byref(ticket)) == 0
            assert lib.stm_server_wait(srv._h, ticket, None) == 0
            check(batch, out)

        for _ in range(4):  # every batch slot has held pairs
            request(FULL)
        for _ in range(4):
            request(SHORT)
        request(scans_from([60000], [20]))  # writes nothing at all


def test_run_batch_scan_leaves_unwritten_slots():
    with tree() as t:
        def call(batch):
            keys, lengths, ops = batch
            out = outputs(keys.size, int(lengths.sum()))
            assert t._lib.stm_run_batch_scan(
                t._h, keys.ctypes.data, lengths.ctypes.data, ops.ctypes.data, keys.size,
                out[0].ctypes.data, out[1].ctypes.data, out[2].ctypes.data, out[3].ctypes.data,
                out[2].size) == 0
            check(batch, out)

        call(FULL)
        call(SHORT)
        call(scans_from([60000], [20]))
        # More ops than one chunk holds: whole scans first, short ones in the later chunks.
        rng = np.random.default_rng(5)
        starts = np.concatenate([np.full(1024, 500), rng.integers(49000, 50100, 1500)])
        call(scans_from(starts, rng.integers(1, 60, starts.size)))


def test_in_place_answers_of_a_short_scan():
    """The answers may take the place of the lengths: the slots' places are known from before."""
    with tree() as t:
        keys, lengths, ops = (x.copy() for x in SHORT)
        out = outputs(keys.size, int(lengths.sum()))
        assert t._lib.stm_run_batch_scan(
            t._h, keys.ctypes.data, lengths.ctypes.data, ops.ctypes.data, keys.size,
            lengths.ctypes.data, out[1].ctypes.data, out[2].ctypes.data, out[3].ctypes.data,
            out[2].size) == 0
        check(SHORT, (lengths,) + out[1:])
