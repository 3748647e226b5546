"""GPU check of the strided 4-D copy (vkv_array_copy, and the pair of a cache
update): every unit width from 1 to 16 bytes, misaligned bases and pitches,
transposed, broadcast and unit dims, extents that are powers of two and not
(the quotient by multiplication), and copies of one and of four units a
thread; bytes outside the destination's elements stay as they were."""
import pytest
import torch

import vkv

pytestmark = pytest.mark.gpu


def strided(shape, pitch, off, dtype, perm=None):
    """A [shape] view with row pitch `pitch` at element offset `off` of a
    larger buffer filled with 7, and that buffer."""
    n = off + shape[0] * shape[1] * shape[2] * pitch
    buf = torch.full((n + 8,), 7, dtype=dtype, device="cuda")
    st = [shape[1] * shape[2] * pitch, shape[2] * pitch, pitch, 1]
    return buf.as_strided(shape, st, off), buf


@pytest.mark.parametrize("dtype", [torch.uint8, torch.bfloat16, torch.float32])
@pytest.mark.parametrize("shape,spitch,soff,dpitch,doff", [
    ((1, 1, 1, 1), 1, 0, 1, 0), ((2, 3, 5, 64), 64, 0, 64, 0), ((2, 3, 5, 64), 80, 16, 64, 0),
    ((2, 3, 7, 33), 33, 1, 37, 3), ((1, 8, 1023, 256), 256, 256, 256, 0),
    ((3, 1, 1, 100), 104, 4, 100, 2), ((2, 8, 4097, 128), 128, 0, 144, 16)])
def test_copy_units(dtype, shape, spitch, soff, dpitch, doff):
    src, _ = strided(shape, spitch, soff, dtype)
    src.copy_(torch.randint(0, 100, shape, device="cuda").to(dtype))
    dst, buf = strided(shape, dpitch, doff, dtype)
    want = buf.clone()
    want.as_strided(dst.shape, dst.stride(), doff).copy_(src)
    a, b = vkv.arr(src), vkv.arr(dst)
    vkv._chk(vkv.lib().vkv_array_copy(vkv.C.byref(a), vkv.C.byref(b), vkv.stream_ptr()))
    assert torch.equal(buf, want)


@pytest.mark.parametrize("view", ["transposed", "broadcast", "inner_stride", "rows_swapped"])
def test_copy_orders(view):
    x = torch.randn((3, 5, 6, 40), device="cuda").half()
    src = {"transposed": x.transpose(1, 2), "broadcast": x[:, :1].expand(3, 4, 6, 40),
           "inner_stride": x[..., ::2], "rows_swapped": x.transpose(2, 3)}[view]
    dst = torch.empty(src.shape, dtype=src.dtype, device="cuda")
    a, b = vkv.arr(src), vkv.arr(dst)
    vkv._chk(vkv.lib().vkv_array_copy(vkv.C.byref(a), vkv.C.byref(b), vkv.stream_ptr()))
    assert torch.equal(dst, src)


@pytest.mark.parametrize("D,Dv,off", [(64, 128, 0), (33, 5, 1)])
def test_cache_update_pair(D, Dv, off):
    """K and V of different widths in one launch, rows at an odd offset."""
    def rows(d):
        return torch.randn((2 * 3 * 7 * (d + off) + off,), device="cuda").bfloat16().as_strided(
            (2, 3, 7, d), (3 * 7 * (d + off), 7 * (d + off), d + off, 1), off)
    k, v = rows(D), rows(Dv)
    c = vkv.KVCacheSimple()
    c.update(k, v)
    c.update(k[:, :, :1], v[:, :, :1])
    gk, gv = c.state
    assert torch.equal(gk, torch.cat([k, k[:, :, :1]], 2))
    assert torch.equal(gv, torch.cat([v, v[:, :, :1]], 2))
