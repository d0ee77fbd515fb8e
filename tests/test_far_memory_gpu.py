"""Inputs in pinned host memory: the same results, by the route that reads them over the link once."""
import ctypes

import numpy as np
import pytest

from thrust_amd import datagen

pytestmark = pytest.mark.gpu


def _placed(x, kind):
    import torch
    t = torch.from_numpy(x)
    return t.cuda() if kind == "device" else t.pin_memory()


def _kernels(dev, call):
    """Labels of the kernels that call(temp, bytes) launches, with the storage it asks for."""
    import torch
    need = ctypes.c_size_t(0)
    dev.check(call(None, ctypes.byref(need)), "size query")
    temp = torch.full((max(need.value, 256),), 255, dtype=torch.uint8, device="cuda")
    dev.profile_collect()
    dev.profile_enable()
    dev.check(call(temp.data_ptr(), ctypes.byref(need)), "call")
    dev.profile_enable(False)
    return set(dev.profile_collect())


@pytest.mark.parametrize("dtype", [np.int32, np.uint8, np.float64])
@pytest.mark.parametrize("kind", ["device", "pinned"])
def test_reduce(dev, dtype, kind):
    size, code = np.dtype(dtype).itemsize, dev.DTYPE_OF_NP[np.dtype(dtype)]
    near_most = (256 << 10 if size == 1 else 512 << 10) // size
    far_most = (128 << 10) // size
    init = ctypes.create_string_buffer(8)
    for n in (far_most, far_most + 1, near_most, near_most + 1):
        x = (datagen.splitmix64(3, n) % np.uint64(8)).astype(dtype)
        src, out = _placed(x, kind), dev.DeviceArray(1, code)
        kernels = _kernels(dev, lambda t, b: dev.load().thrust_amd_reduce(t, b, src.data_ptr(), n, code, dev.PLUS, init, out.ptr,
                                                                         dev.stream_ptr()))
        assert out.numpy()[0] == x.sum(dtype=dtype), n
        assert ("reduce_one" in kernels) == (n <= (near_most if kind == "device" else far_most)), (n, kernels)


@pytest.mark.parametrize("places", [("device", "device"), ("pinned", "device"), ("device", "pinned")])
def test_merge(dev, places):
    for n in (1 << 18, (1 << 18) + 1, (1 << 20) + 3, (1 << 23) + 5):
        raw = (datagen.splitmix64(5, n) >> np.uint64(33)).astype(np.uint32)
        na = n // 2 + 7
        a, b = np.sort(raw[:na]), np.sort(raw[na:])
        da, db, out = _placed(a.view(np.int32), places[0]), _placed(b.view(np.int32), places[1]), dev.DeviceArray(n, dev.U32)
        kernels = _kernels(dev, lambda t, s: dev.load().thrust_amd_merge(t, s, da.data_ptr(), na, db.data_ptr(), n - na, out.ptr,
                                                                        dev.U32, 0, dev.stream_ptr()))
        assert np.array_equal(out.numpy(), np.sort(raw)), n
        searched_inside = n <= (1 << 23 if places == ("device", "device") else 1 << 18)
        assert ("merge_partition" in kernels) != searched_inside, (n, kernels)
