"""The one-workgroup sort (up to 8192 keys): the edges of its two workgroup sizes, and inputs that take
each of its ways: few varying bits, top 16 bits that tell the keys apart, groups that share them up to and
beyond the size sorted by counting, bit ranges, both directions."""
import numpy as np
import pytest

from thrust_amd import datagen

pytestmark = pytest.mark.gpu

SIZES = [2, 63, 65, 255, 257, 1023, 1024, 1025, 2047, 2048, 2049, 4095, 4096, 4097, 8191, 8192, 8193]


def _keys(kind, dtype, n):
    r = datagen.splitmix64(77, n)
    bits = np.dtype(dtype).itemsize * 8
    if kind == "full":
        u = r
    elif kind == "equal":
        u = np.zeros_like(r) + np.uint64(5)
    elif kind == "low":          # two low bytes vary
        u = r & np.uint64(0xFFFF)
    elif kind == "groups16":     # about 16 keys share their upper half
        u = ((r >> np.uint64(32)) % np.uint64(max(n // 16, 1))) << np.uint64(bits // 2) | (r & np.uint64(0xFF))
    elif kind == "groups200":    # about 200 do
        u = ((r >> np.uint64(32)) % np.uint64(max(n // 200, 1))) << np.uint64(bits // 2) | (r & np.uint64(0xFF))
    elif kind == "skewed":       # most keys equal
        u = np.where(r % np.uint64(10) != 0, np.uint64(1 << 6), r)
    u = u.astype({8: np.uint8, 16: np.uint16, 32: np.uint32, 64: np.uint64}[bits])
    x = u.view(dtype)
    return np.where(np.isnan(x), dtype(1), x) if np.dtype(dtype).kind == "f" else x


def _order(x, descending, begin, end):
    """Stable order by bits [begin, end) of the radix code."""
    bits = x.dtype.itemsize * 8
    u = x.view(f"u{x.dtype.itemsize}").copy()
    top = u.dtype.type(1 << (bits - 1))
    if x.dtype.kind == "f":
        u = np.where(u & top, ~u, u | top)
    elif x.dtype.kind == "i":
        u = u ^ top
    u = (u.astype(np.uint64) >> np.uint64(begin)) & np.uint64((1 << (end - begin)) - 1)
    if descending:
        u = np.uint64((1 << (end - begin)) - 1) - u
    return np.argsort(u, kind="stable")


@pytest.mark.parametrize("dtype", [np.uint8, np.int16, np.uint32, np.int32, np.float32, np.uint64, np.float64])
@pytest.mark.parametrize("kind", ["full", "equal", "low", "groups16", "groups200", "skewed"])
def test_small_sorts(dev, dtype, kind):
    bits = np.dtype(dtype).itemsize * 8
    for n in SIZES:
        x = _keys(kind, dtype, n)
        for descending, begin, end in ((False, 0, bits), (True, 0, bits), (False, bits // 4, bits - 1)):
            order = _order(x, descending, begin, end)
            k = dev.DeviceArray.from_numpy(x)
            dev.sort_keys(k, descending=descending, begin_bit=begin, end_bit=end)
            assert np.array_equal(k.numpy().view(np.uint8), x[order].view(np.uint8)), (n, descending, begin)
            for vdtype in (np.uint8, np.uint32, np.uint64):
                v = np.arange(n).astype(vdtype)
                k, w = dev.DeviceArray.from_numpy(x), dev.DeviceArray.from_numpy(v)
                dev.sort_pairs(k, w, descending=descending, begin_bit=begin, end_bit=end)
                assert np.array_equal(k.numpy().view(np.uint8), x[order].view(np.uint8)), (n, vdtype)
                assert np.array_equal(w.numpy(), v[order]), (n, vdtype, descending, begin)
