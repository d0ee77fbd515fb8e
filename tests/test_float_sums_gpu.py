"""Short sums of floats in one workgroup are no less exact than the same sums by several workgroups.

The order of addition of the several workgroups is restated here; its own error on the same arrays, against sums in wider
floats, is the bound for what the device computes.
"""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def _in_a_row(a):
    r = a[..., 0]
    for i in range(1, a.shape[-1]):
        r = r + a[..., i]
    return r


def _wave_sum(v):
    """64 lanes by a tree."""
    while v.shape[-1] > 1:
        v = v[..., 0::2] + v[..., 1::2]
    return v[..., 0]


def _reduce_by_two_launches(x):
    """reduce_partials_kernel and reduce_final_kernel: workgroups of 256 lanes with 8 vectors of 16 bytes each per tile,
    at most 256 tiles here."""
    rows, n = x.shape
    vec = 16 // x.dtype.itemsize
    tile = 256 * 8 * vec
    full, tiles = n // tile, -(-n // tile)
    acc = np.zeros((rows, tiles, 256), x.dtype)
    own = x[:, :full * tile].reshape(rows, full, 8, 256, vec).transpose(0, 1, 3, 2, 4).reshape(rows, full, 256, 8 * vec)
    for i in range(8 * vec):
        acc[:, :full] += own[..., i]
    rest = x[:, full * tile:]
    for k in range(0, rest.shape[1], tiles * 256):
        part = np.zeros((rows, tiles * 256), x.dtype)
        part[:, :rest[:, k:k + tiles * 256].shape[1]] = rest[:, k:k + tiles * 256]
        acc += part.reshape(rows, tiles, 256)
    final = np.zeros((rows, 256), x.dtype)
    final[:, :tiles] = _in_a_row(_wave_sum(acc.reshape(rows, tiles, 4, 64)))
    return _in_a_row(_wave_sum(final.reshape(rows, 4, 64)))


def _wave_scan(v):
    """wave_inclusive_scan: rows of 16 lanes by shifts of 1, 2, 4 and 8, then the rows."""
    v = v.reshape(*v.shape[:-1], 4, 16)
    for k in (1, 2, 4, 8):
        left = np.zeros_like(v)
        left[..., k:] = v[..., :-k]
        v = left + v
    v[..., 1::2, :] = v[..., 0::2, 15:] + v[..., 1::2, :]
    v[..., 2:, :] = v[..., 1:2, 15:] + v[..., 2:, :]
    return v.reshape(*v.shape[:-2], 64)


def _scan_by_tiles(x):
    """scan_kernel with tiles of 256 lanes and 4 vectors of 16 bytes each, every tile behind the one before it."""
    rows, n = x.shape
    vec = 16 // x.dtype.itemsize
    tile = 256 * 4 * vec
    tiles = -(-n // tile)
    y = np.zeros((rows, tiles * tile), x.dtype)
    y[:, :n] = x
    y = y.reshape(rows, tiles, 4, 4, 64, vec)  # wave, vector, lane, place
    carry = np.zeros((rows, tiles, 4), x.dtype)
    for j in range(4):
        incl = _wave_scan(_in_a_row(y[:, :, :, j]))
        run = np.zeros_like(incl)
        run[..., 1:] = incl[..., :-1]
        run = carry[..., None] + run
        carry = carry + incl[..., 63]
        for i in range(vec):
            run = run + y[:, :, :, j, :, i]
            y[:, :, :, j, :, i] = run
    before = np.zeros_like(carry)
    for w in range(1, 4):
        before[..., w] = before[..., w - 1] + carry[..., w - 1]
    total = before[..., 3] + carry[..., 3]
    prefix = np.zeros_like(total)
    for t in range(1, tiles):
        prefix[:, t] = prefix[:, t - 1] + total[:, t - 1]
    return ((prefix[..., None] + before)[..., None, None, None] + y).reshape(rows, -1)[:, :n]


def _error(got, exact):
    """Per row, 2-norm of the difference over 2-norm of the result."""
    got, exact = got.reshape(len(exact), -1).astype(np.longdouble), exact.reshape(len(exact), -1)
    return np.sqrt(((got - exact) ** 2).sum(1) / (exact ** 2).sum(1))


def _rms(errors):
    return float(np.sqrt((np.concatenate(errors) ** 2).mean()))


@pytest.mark.parametrize("dtype,sizes", [(np.float32, (5003, 20011, 50021, 100003)), (np.float64, (5003, 20011, 50021))])
def test_reduce_in_one_workgroup(dev, dtype, sizes):
    rng = np.random.default_rng(11)
    here, there = [], []
    for n in sizes:
        x = rng.random((40, n)).astype(dtype)
        exact = x.astype(np.longdouble).sum(1)
        got = np.array([dev.reduce(dev.DeviceArray.from_numpy(row)).numpy()[0] for row in x])
        here.append(_error(got, exact))
        there.append(_error(_reduce_by_two_launches(x), exact))
    assert _rms(here) <= _rms(there), (_rms(here), _rms(there))


@pytest.mark.parametrize("dtype,sizes", [(np.float32, (8001, 12007, 16384)), (np.float64, (5003, 8192))])
def test_scan_in_one_workgroup(dev, dtype, sizes):
    rng = np.random.default_rng(13)
    here, there = [], []
    for n in sizes:
        x = rng.random((400, n)).astype(dtype)
        exact = x.astype(np.longdouble).cumsum(1)
        got = np.array([dev.inclusive_scan(dev.DeviceArray.from_numpy(row)).numpy() for row in x])
        here.append(_error(got, exact))
        there.append(_error(_scan_by_tiles(x), exact))
    assert _rms(here) <= _rms(there), (_rms(here), _rms(there))
