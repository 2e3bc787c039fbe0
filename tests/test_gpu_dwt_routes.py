"""The fused x/y passes of one transform level against the one-axis passes, bit for bit.

A call whose source does not meet its output takes the fused pass; the same call on the same values with
the output laid over the source takes the passes per axis.  Both evaluate the same sums in the same
order, so they must agree exactly; the integer transform is also compared with the oracle (exactly) and
the float one within the 1e-6 that the fp32 bars of the transforms use.  Sizes: the shortest fused axis
(8), one that is too short (6), tiles of 60 and 62 pairs and one pair more or less, segments with
remainders.
"""
import numpy as np
import pytest

from cudacompress_amd import synthetic as S
from oracle import pyoracle as o
from tests.gpu_util import log, to_dev, to_host

pytestmark = pytest.mark.gpu

PLANES = [(8, 8), (10, 6), (6, 10), (118, 18), (120, 66), (122, 8), (124, 34), (126, 10), (250, 130)]  # x, y


def same(a, b):
    assert np.array_equal(a.view(np.uint8), b.view(np.uint8))


def close(got, want):
    assert float(np.abs(got.astype(np.float64) - want).max()) <= 1e-6 * max(1.0, float(np.abs(want).max()))


@pytest.mark.parametrize("x,y", PLANES)
@pytest.mark.parametrize("pad", [0, 6])
def test_plane(cc, torch_gpu, x, y, pad):
    torch = torch_gpu
    log("dwt 2d routes", x, y, pad)
    row = x + pad
    img = S.gaussian_field((y, row), x + y)
    src, buf, dst = to_dev(torch, img), to_dev(torch, img * 0), to_dev(torch, img * 0 + 7)
    cc.util.dwtFloat2DForward(dst, buf, src, x, y, 1, row, row)
    over = src.clone()
    cc.util.dwtFloat2DForward(over, buf, over, x, y, 1, row, row)
    torch.cuda.synchronize()
    got = to_host(dst)
    same(got[:, :x].copy(), to_host(over)[:, :x].copy())
    assert np.all(got[:, x:] == 7)
    close(got[:, :x], o.dwt97_forward(np.ascontiguousarray(img[:, :x])))
    rec = to_dev(torch, img * 0 + 7)
    cc.util.dwtFloat2DInverse(rec, buf, dst, x, y, 1, row, row)
    cc.util.dwtFloat2DInverse(over, buf, over, x, y, 1, row, row)
    torch.cuda.synchronize()
    same(to_host(rec)[:, :x].copy(), to_host(over)[:, :x].copy())
    assert np.all(to_host(rec)[:, x:] == 7)


@pytest.mark.parametrize("ch", [1, 2, 3, 4])
@pytest.mark.parametrize("x,y", [(8, 8), (122, 18), (250, 66)])
def test_byte_channels(cc, torch_gpu, ch, x, y):
    """Byte images: each channel against the float transform of its plane, and back."""
    torch = torch_gpu
    log("dwt byte routes", ch, x, y)
    img = np.random.default_rng(x + ch).integers(0, 256, (y, x, ch), dtype=np.uint8)
    src = to_dev(torch, img)
    out = torch.zeros_like(src)
    for c in range(ch):
        plane = to_dev(torch, img[..., c].astype(np.float32) - 128)
        want, dst, buf, rec = (torch.empty_like(plane) for _ in range(4))
        cc.util.dwtFloat2DForward(want, buf, plane, x, y)
        cc.util.dwtFloat2DForwardFromByte(dst, buf, src.reshape(-1)[c:], x, y, ch, x, x * ch)
        cc.util.dwtFloat2DInverseToByte(out.reshape(-1)[c:], buf, dst, x, y, ch, x * ch, x)
        cc.util.dwtFloat2DInverse(rec, buf, dst, x, y)
        torch.cuda.synchronize()
        same(to_host(dst), to_host(want))
        same(to_host(out)[..., c].copy(), np.clip(to_host(rec) + np.float32(128.5), 0, 255).astype(np.uint8))
    assert int(np.abs(to_host(out).astype(int) - img).max()) <= 1


@pytest.mark.parametrize("x,y,z", [(8, 8, 2), (16, 8, 66), (122, 10, 8), (126, 34, 4), (6, 12, 10), (20, 130, 72)])
def test_volume(cc, torch_gpu, x, y, z):
    torch = torch_gpu
    log("dwt 3d routes", x, y, z)
    vol = S.gaussian_field((z, y, x), x + y + z)
    src = to_dev(torch, vol)
    dst, b1, b2, rec, rec2, dst2 = (torch.empty_like(src) for _ in range(6))
    cc.util.dwtFloat3DForward(dst, b2, b1, src, x, y, z)
    over = src.clone()
    cc.util.dwtFloat3DForward(dst2, over, b1, over, x, y, z)  # buffer 2 is the source
    torch.cuda.synchronize()
    same(to_host(dst), to_host(dst2))
    close(to_host(dst), o.dwt97_forward(vol))
    cc.util.dwtFloat3DInverse(rec, b2, b1, dst, x, y, z)
    cc.util.dwtFloat3DInverse(rec2, rec2, b1, dst, x, y, z)  # buffer 2 is the destination
    torch.cuda.synchronize()
    same(to_host(rec), to_host(rec2))

    ints = np.round(vol * 200).astype(np.int16)
    isrc = to_dev(torch, ints)
    idst, ibuf, idst2, irec, irec2 = (torch.empty_like(isrc) for _ in range(5))
    cc.util.dwtIntForward(idst, ibuf, isrc, x, y, z)
    iover = isrc.clone()
    cc.util.dwtIntForward(idst2, iover, iover, x, y, z)
    torch.cuda.synchronize()
    same(to_host(idst), to_host(idst2))
    same(to_host(idst), o.dwt53_forward(ints))
    cc.util.dwtIntInverse(irec, ibuf, idst, x, y, z)
    iover = idst.clone()
    cc.util.dwtIntInverse(irec2, iover, iover, x, y, z)
    torch.cuda.synchronize()
    same(to_host(irec), ints)
    same(to_host(irec2), ints)


@pytest.mark.parametrize("n", [2, 10, 64])
def test_column_pass_within_one_array(cc, torch_gpu, n):
    """buffer == destination: columns of up to 64 samples are read before they are replaced."""
    torch = torch_gpu
    log("dwt in place", n)
    img = S.gaussian_field((n, 70), n)
    src = to_dev(torch, img)
    want, buf, dst = torch.empty_like(src), torch.empty_like(src), torch.empty_like(src)
    cc.util.dwtFloat2DForward(want, buf, src, 70, n)
    cc.util.dwtFloat2DForward(dst, dst, src, 70, n)
    rec, rec2 = torch.empty_like(src), want.clone()
    cc.util.dwtFloat2DInverse(rec, buf, want, 70, n)
    cc.util.dwtFloat2DInverse(dst, rec2, rec2, 70, n)  # columns within the source
    torch.cuda.synchronize()
    same(to_host(rec), to_host(dst))
    ints = to_dev(torch, np.round(img * 200).astype(np.int16))
    iwant, ibuf, idst, irec = (torch.empty_like(ints) for _ in range(4))
    cc.util.dwtIntForward(iwant, ibuf, ints, 70, n, 1)
    cc.util.dwtIntForward(idst, idst, ints, 70, n, 1)
    iover = iwant.clone()
    cc.util.dwtIntInverse(irec, iover, iover, 70, n, 1)
    torch.cuda.synchronize()
    same(to_host(idst), to_host(iwant))
    same(to_host(irec), to_host(ints))
