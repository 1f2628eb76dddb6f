"""The device sort with its keys in place of its input, at the sizes of each of its forms, against
numpy's stable argsort; also keys that the exact passes sort again, from the input."""
import numpy as np
import pytest

from test_gpu_sample_sort import keys_of

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dist", ["uniform", "misleading"])
@pytest.mark.parametrize("n", [40000, 1 << 18, 3 << 17, (3 << 17) + 1, 1 << 19, (1 << 19) + 1, 1 << 20,
                               (1 << 20) + 1, 1 << 22, (1 << 22) + 1])
def test_sorts_in_place(n, dist):
    from eirene_amd import DeviceBuffer, load_library
    keys = keys_of(dist, n, np.random.default_rng(n))
    d, idx = DeviceBuffer.from_array(keys), DeviceBuffer(n, np.uint32)
    assert load_library().stm_sort_pairs_device(0, d.ptr, n, d.ptr, idx.ptr) == 0
    want = np.argsort(keys, kind="stable")
    assert np.array_equal(idx.download(), want.astype(np.uint32))
    assert np.array_equal(d.download(), keys[want])
