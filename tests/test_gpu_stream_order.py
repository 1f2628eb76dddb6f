"""A batch stream starts after whatever the caller has queued on the tree's stream, also once its
sorts run on a second stream: inputs that a queued copy has yet to bring, answers that a queued copy
has yet to take away."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


class Array:
    """A torch tensor in the place of a DeviceBuffer."""

    def __init__(self, tensor):
        self.tensor, self.ptr, self.n = tensor, tensor.data_ptr(), tensor.numel()


def device(x):
    import torch
    return torch.from_numpy(x.view(np.int64) if x.dtype == np.uint64 else x).cuda()


@pytest.mark.parametrize("size", [2049, 40000])
def test_stream_waits_for_queued_copies(oracle_mod, size):
    import torch
    from eirene_amd import StmTree
    rng = np.random.default_rng(size)
    load = np.unique(rng.integers(0, 1 << 50, 60000, dtype=np.uint64))
    n = 4 * size
    offsets = (np.arange(5) * size).astype(np.uint64)

    def batch():
        keys = np.where(rng.random(n) < 0.6, rng.choice(load, n),
                        rng.integers(0, 1 << 50, n, dtype=np.uint64)).astype(np.uint64)
        return (keys, rng.integers(0, 1 << 62, n, dtype=np.uint64),
                (rng.random(n) < 0.7).astype(np.uint8))  # 1: GET, 0: INSERT

    o = oracle_mod.Oracle()
    o.bulk_load(load, load)

    def replay(b):
        parts = [o.run_batch(*(x[i:i + size] for x in b)) for i in range(0, n, size)]
        return np.concatenate([p[0] for p in parts]), np.concatenate([p[1] for p in parts])

    with StmTree(max_keys=1 << 20, max_batch=1 << 16) as t:
        t.bulk_load(load, load)
        stream = torch.cuda.ExternalStream(t.stream())
        busy = torch.zeros(2, 1 << 28, dtype=torch.uint8, device="cuda")
        cur = [Array(device(x)) for x in batch()]
        cur[2].tensor.fill_(1)  # lookups only: they leave the tree as it is
        out = Array(torch.zeros(n, dtype=torch.int64, device="cuda"))
        found = Array(torch.zeros(n, dtype=torch.uint8, device="cuda"))
        torch.cuda.synchronize()
        for _ in range(8):  # enough batches for the second stream
            t.run_batches_device(*cur, out, found, offsets)
        before = None
        for _ in range(3):
            b = batch()
            new = [device(x) for x in b]
            kept = torch.zeros_like(out.tensor), torch.zeros_like(found.tensor)
            torch.cuda.synchronize()
            with torch.cuda.stream(stream):
                for _ in range(40):  # some milliseconds
                    busy[0].copy_(busy[1])
                kept[0].copy_(out.tensor)
                kept[1].copy_(found.tensor)
                for a, x in zip(cur, new):
                    a.tensor.copy_(x)
            t.run_batches_device(*cur, out, found, offsets)
            want = replay(b)
            got = out.tensor.cpu().numpy().view(np.uint64), found.tensor.cpu().numpy()
            np.testing.assert_array_equal(got[0], want[0])
            np.testing.assert_array_equal(got[1], want[1])
            if before is not None:
                np.testing.assert_array_equal(kept[0].cpu().numpy().view(np.uint64), before[0])
                np.testing.assert_array_equal(kept[1].cpu().numpy(), before[1])
            before = want
        k, v = t.dump()
        ek, ev = o.dump()
        np.testing.assert_array_equal(k, ek)
        np.testing.assert_array_equal(v, ev)
        assert t.check() == 0
