"""thrust_amd_memcpy, device to device: the copy kernel that takes over at 128 MiB, around its edges."""
import pytest

pytestmark = pytest.mark.gpu

LIMIT = 128 << 20


@pytest.mark.parametrize("nbytes", [1, 4097, LIMIT - 1, LIMIT, LIMIT + 1, LIMIT + 4096 + 15, 2 * LIMIT + 7])
@pytest.mark.parametrize("dst_off,src_off", [(0, 0), (5, 5), (15, 31), (0, 1)])
def test_copy_moves_exactly_its_bytes(dev, nbytes, dst_off, src_off):
    import torch
    src = torch.randint(0, 256, (nbytes + 64,), dtype=torch.uint8, device="cuda")
    dst = torch.zeros_like(src)
    dev.check(dev.load().thrust_amd_memcpy(dst.data_ptr() + dst_off, src.data_ptr() + src_off, nbytes, dev.D2D,
                                           dev.stream_ptr()), "thrust_amd_memcpy")
    assert torch.equal(dst[dst_off:dst_off + nbytes], src[src_off:src_off + nbytes])
    assert not dst[:dst_off].any() and not dst[dst_off + nbytes:].any()  # nothing around it is touched
