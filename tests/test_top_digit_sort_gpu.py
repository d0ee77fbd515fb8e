"""The sort that runs its passes over the top digits only and orders the stretches of equal prefixes in
one workgroup each: inputs that take it with one digit and with two, whose bins are full or too full for counting,
with stretches too long for a workgroup that the samples see (long_stretch: all digits get their pass) or do not see (the
tail sorts them), and that never take it."""
import numpy as np
import pytest

from thrust_amd import datagen

pytestmark = pytest.mark.gpu

SIZES = [8193, 20_001, 300_007, 1_000_003, 2_500_001]


def _keys(kind, dtype, n):
    r = datagen.splitmix64(99, n)
    bits = np.dtype(dtype).itemsize * 8
    u = np.uint64
    if kind == "uniform":
        k = r
    elif kind == "repeated":      # the low half takes four values: many equal keys in every stretch
        k = (r >> u(64 - bits)) & ~u((1 << (bits // 2)) - 1) | (r & u(3))
    elif kind == "clusters":      # low bits in clusters far apart: the bins of a stretch overflow
        k = (r >> u(64 - bits)) & ~u((1 << (bits - 16)) - 1) | (r & u(1)) << u(bits - 20) | (r >> u(3)) & u(63)
    elif kind == "long_stretch":  # uniform but for one prefix held by more keys than a workgroup takes
        k = r >> u(64 - bits)
        k[n // 3:n // 3 + 9000] = (k[n // 3:n // 3 + 9000] & u((1 << (bits - 16)) - 1)) | u(0x1234) << u(bits - 16)
    elif kind == "equal":         # no digit moves
        k = np.full(n, 12345, dtype=np.uint64)
    elif kind == "skewed":        # nine in ten equal
        k = np.where(r % u(10) != 0, u(1 << 20), r)
    elif kind in ("tens", "near"):  # about ten keys are equal, or share all but their low bits: bins of 9 to 24
        k = (r >> u(64 - bits))[:max(n // 10, 1)][(datagen.splitmix64(98, n) % u(max(n // 10, 1))).astype(np.int64)]
        if kind == "near":
            low = u((1 << (bits // 3)) - 1)
            k = (k & ~low) | (r & low)
    elif kind == "ids":           # 0 .. n-1 shuffled: constant top digits
        k = np.argsort(r).astype(np.uint64)
    elif kind == "sorted":
        k = np.sort(r >> u(64 - bits))
    if kind == "normal":
        k = np.random.default_rng(5).standard_normal(n) * 1000
        return k.astype(dtype) if np.dtype(dtype).kind == "f" else (k * 1000).astype(np.int64).astype(dtype)
    k = k.astype({32: np.uint32, 64: np.uint64}[bits]).view(dtype)
    return np.where(np.isnan(k), dtype(1), k) if np.dtype(dtype).kind == "f" else k


def _order(x, descending):
    """Stable order by the radix code."""
    bits = x.dtype.itemsize * 8
    u = x.view(f"u{x.dtype.itemsize}")
    top = u.dtype.type(1 << (bits - 1))
    if x.dtype.kind == "f":
        u = np.where(u & top, ~u, u | top)
    elif x.dtype.kind == "i":
        u = u ^ top
    return np.argsort(~u if descending else u, kind="stable")


def _control(temp):
    """The control block of the last sort (thrust_amd/csrc/sort_ctl.hpp), the first thing in its temporary storage."""
    words = temp.buf[:15 * 4].cpu().numpy().view(np.uint32)
    return {"gave_up": int(words[9]), "fast": int(words[10]), "long_windows": int(words[14])}


def _sampled(n):
    """Places the plan of a two-digit sort looks at (Sampling in thrust_amd/csrc/radix_sort.hip)."""
    blocks = min(-(-n // 8192), 256)
    each = max(1, min(min(n // 64, 16384) // blocks, 1024))
    count = each * blocks
    step = n // count
    j = np.arange(count, dtype=np.uint64)
    return j * np.uint64(step) + (((j * np.uint64(2654435769) & np.uint64(0xFFFFFFFF)) * np.uint64(step)) >> np.uint64(32))


# (how many keys, what they are): more than a workgroup of the last step takes, and of one tile, some, and many of the tail's
LONG = [(150_001, "hot", 4100), (150_001, "prefix", 5000), (150_001, "both", 8193), (1_000_003, "hot", 9001),
        (1_000_003, "prefix", 30_001)]


@pytest.mark.parametrize("dtype", [np.uint64, np.int64])
@pytest.mark.parametrize("n,kind,many", LONG)
def test_stretches_too_long_for_the_last_step(dev, dtype, n, kind, many):
    """Stretches of equal top digits that the samples do not see are sorted by the tail."""
    unseen = np.ones(n, dtype=bool)
    unseen[_sampled(n)] = False
    at = np.flatnonzero(unseen)[::3]
    assert len(at) >= 2 * many
    x = datagen.splitmix64(5, n)
    spread = len(at) // (2 * many)
    for i, where in enumerate((at[:many * spread:spread], at[many * spread:2 * many * spread:spread])):
        high = np.uint64(0x1234 + 0x7000 * i) << np.uint64(48)
        if kind == "hot" or (kind == "both" and i == 0):
            x[where] = high | np.uint64(77)
        else:
            x[where] = high | (x[where] & np.uint64((1 << 48) - 1))
    x = x.view(dtype)
    temp = dev.Temp()
    for descending in (False, True):
        order = _order(x, descending)
        k = dev.DeviceArray.from_numpy(x)
        dev.sort_keys(k, descending=descending, temp=temp)
        control = _control(temp)
        assert control["fast"] == 2 and control["long_windows"] >= 2, control
        assert np.array_equal(k.numpy(), x[order]), descending
        for vdtype in (np.uint8, np.uint32, np.uint64):
            v = np.arange(n).astype(vdtype)
            k, w = dev.DeviceArray.from_numpy(x), dev.DeviceArray.from_numpy(v)
            dev.sort_pairs(k, w, descending=descending, temp=temp)
            assert _control(temp)["long_windows"] >= 2
            assert np.array_equal(k.numpy(), x[order]), (vdtype, descending)
            assert np.array_equal(w.numpy(), v[order]), (vdtype, descending)


@pytest.mark.parametrize("n", [1 << 25, (1 << 25) + 4097])
@pytest.mark.parametrize("repeats", [1, 100])
def test_four_byte_keys_never_take_two_digits(dev, n, repeats):
    """With two digits, stretches of keys that repeat outgrow a workgroup after the passes over them have run."""
    temp = dev.Temp()
    values = datagen.splitmix64(3, n // repeats).astype(np.uint32)
    x = values[(datagen.splitmix64(4, n) % np.uint64(len(values))).astype(np.int64)]
    k = dev.DeviceArray.from_numpy(x)
    dev.sort_keys(k, temp=temp)
    assert _control(temp)["fast"] == 0
    assert np.array_equal(k.numpy(), np.sort(x))


@pytest.mark.parametrize("dtype", [np.uint32, np.int32, np.float32, np.uint64, np.float64])
@pytest.mark.parametrize("kind", ["uniform", "normal", "repeated", "clusters", "long_stretch", "equal", "skewed", "tens", "near", "ids", "sorted"])
def test_sorts_by_top_digits(dev, dtype, kind):
    temp = dev.Temp()
    for n in SIZES:
        if kind == "long_stretch" and n < 30_000:
            continue
        x = _keys(kind, dtype, n)
        for descending in (False, True):
            order = _order(x, descending)
            k = dev.DeviceArray.from_numpy(x)
            dev.sort_keys(k, descending=descending, temp=temp)
            assert np.array_equal(k.numpy().view(np.uint8), x[order].view(np.uint8)), (n, descending)
            for vdtype in (np.uint8, np.uint32, np.uint64) if n < 1_000_000 else (np.uint32,):
                v = np.arange(n).astype(vdtype)
                k, w = dev.DeviceArray.from_numpy(x), dev.DeviceArray.from_numpy(v)
                dev.sort_pairs(k, w, descending=descending, temp=temp)
                assert np.array_equal(k.numpy().view(np.uint8), x[order].view(np.uint8)), (n, vdtype, descending)
                assert np.array_equal(w.numpy(), v[order]), (n, vdtype, descending)


# Sizes up to which the last step fits one digit, tiles are small, and tiles of 4-byte keys are of the middle size
# (SortPlan and sort_impl in thrust_amd/csrc/radix_sort.hip), and where the two-digit way ends.
EDGES = [(np.uint32, None, 256 * 6144), (np.int32, np.uint16, 256 * 6144), (np.float32, np.uint32, 8 * 6144),
         (np.int32, np.uint64, 256 * 2560), (np.float64, None, 1 << 19),
         (np.uint8, None, 16384 * 160), (np.uint16, np.uint64, 8192 * 160), (np.uint32, None, 18432 * 160),
         (np.int32, np.uint8, 16384 * 160), (np.uint64, np.uint32, 8192 * 160),
         (np.uint32, np.uint32, 14336 * 160), (np.float32, np.uint8, 14336 * 160), (np.uint32, None, 10240 * 512),
         (np.float32, np.uint32, 10240 * 512), (np.int32, np.uint16, 10240 * 512),
         (np.uint32, np.uint8, 1 << 22), (np.int32, np.uint16, 1 << 22), (np.float32, np.uint32, 1 << 22),
         (np.uint32, np.uint16, (1 << 24) - 1)]


@pytest.mark.parametrize("dtype,vdtype,edge", EDGES)
def test_sizes_where_the_kernels_change(dev, dtype, vdtype, edge):
    for n in (edge, edge + 1):
        bits = np.dtype(dtype).itemsize * 8
        x = (datagen.splitmix64(7, n) >> np.uint64(64 - bits)).astype(f"u{bits // 8}").view(dtype)
        if np.dtype(dtype).kind == "f":
            x = np.where(np.isnan(x), dtype(1), x)
        for descending in (False, True):
            order = _order(x, descending)
            k = dev.DeviceArray.from_numpy(x)
            if vdtype is None:
                dev.sort_keys(k, descending=descending)
            else:
                v = np.arange(n).astype(vdtype)
                w = dev.DeviceArray.from_numpy(v)
                dev.sort_pairs(k, w, descending=descending)
                assert np.array_equal(w.numpy(), v[order]), (n, descending)
            assert np.array_equal(k.numpy().view(np.uint8), x[order].view(np.uint8)), (n, descending)


# (key, value, a length): the longest arrays whose passes behind the short way run in one launch (REST_MAX in
# thrust_amd/csrc/radix_sort.hip), and longer ones of 8-byte keys or values
ONE_LAUNCH = [(np.uint32, None, 1 << 20), (np.int32, np.uint8, 3 << 18), (np.uint32, np.uint64, 3 << 18),
              (np.int64, None, 3 << 15), (np.uint64, np.uint16, 3 << 15), (np.float64, np.uint64, 3 << 15),
              (np.uint32, np.uint64, 1 << 19), (np.int64, None, 1 << 15), (np.uint64, np.uint16, 1 << 15), (np.float64, np.uint64, 1 << 15)]


@pytest.mark.parametrize("dtype,vdtype,edge", ONE_LAUNCH)
@pytest.mark.parametrize("kind", ["skewed", "ids", "normal"])
def test_passes_left_over_in_one_launch(dev, dtype, vdtype, edge, kind):
    """Keys that decline the short way, with an even and an odd number of digits that vary (the result is copied back)."""
    temp = dev.Temp()
    for n in (8193, edge // 2, edge, edge + 1):
        x = _keys(kind, dtype, n)
        for descending in (False, True):
            order = _order(x, descending)
            k = dev.DeviceArray.from_numpy(x)
            if vdtype is None:
                dev.sort_keys(k, descending=descending, temp=temp)
            else:
                v = np.arange(n).astype(vdtype)
                w = dev.DeviceArray.from_numpy(v)
                dev.sort_pairs(k, w, descending=descending, temp=temp)
                assert np.array_equal(w.numpy(), v[order]), (n, descending)
            assert np.array_equal(k.numpy().view(np.uint8), x[order].view(np.uint8)), (n, descending)
            assert _control(temp)["gave_up"] == 0


def test_passes_in_one_launch_on_several_streams(dev):
    """Eight sorts at a time that decline the short way: the workgroups of all of them do not fit the GPU together."""
    import torch
    streams = [torch.cuda.Stream() for _ in range(8)]
    xs = [_keys("skewed", np.uint32, 1_000_000 + i) for i in range(8)]
    orders = [_order(x, False) for x in xs]
    for _ in range(3):
        keys = [dev.DeviceArray.from_numpy(x) for x in xs]
        values = [dev.DeviceArray.from_numpy(np.arange(x.size, dtype=np.uint32)) for x in xs]
        temps = [dev.Temp() for _ in xs]
        torch.cuda.synchronize()
        for i, stream in enumerate(streams):
            with torch.cuda.stream(stream):
                if i % 2:
                    dev.sort_keys(keys[i], temp=temps[i])
                else:
                    small = dev.DeviceArray(780_000, keys[i].dtype, keys[i].storage)
                    dev.sort_pairs(small, values[i], temp=temps[i])
        torch.cuda.synchronize()
        for i, x in enumerate(xs):
            if i % 2:
                assert np.array_equal(keys[i].numpy(), x[orders[i]])
            else:
                order = _order(x[:780_000], False)
                assert np.array_equal(keys[i].numpy(780_000), x[:780_000][order])
                assert np.array_equal(values[i].numpy(780_000), order.astype(np.uint32))


def test_long_stretches_among_many_keys(dev):
    """2^25 eight-byte keys, four values 7000 times: the plan takes two digits, the tail sorts the windows that hold them."""
    n = 1 << 25
    x = datagen.splitmix64(8, n)
    where = (datagen.splitmix64(9, 28_000) % np.uint64(n)).astype(np.int64)
    x[where] = np.repeat(datagen.splitmix64(10, 4), 7000)
    temp = dev.Temp()
    k, w = dev.DeviceArray.from_numpy(x), dev.DeviceArray.from_numpy(np.arange(n, dtype=np.uint32))
    dev.sort_pairs(k, w, temp=temp)
    order = _order(x, False)
    assert np.array_equal(k.numpy(), x[order]) and np.array_equal(w.numpy(), order.astype(np.uint32))
    control = _control(temp)
    assert control["fast"] == 2 and control["long_windows"] >= 4, control
