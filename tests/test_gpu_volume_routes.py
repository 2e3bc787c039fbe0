"""The volume codecs at sizes where their passes change shape: rows that are no multiple of four
values, two-sample axes, rows past the fused transforms, streams split over workgroups; segments that
start inside a word; and damaged bitstreams, which are refused before anything is enqueued."""
import numpy as np
import pytest

from cudacompress_amd import synthetic as S
from oracle import pipeline as P
from oracle import pyoracle as o
from tests.gpu_util import log, to_dev, to_host

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("shape,levels", [((6, 10), 1), ((36, 76), 2), ((8, 2056), 3), ((2, 2, 2), 1), ((12, 4, 20), 2),
                                          ((40, 24, 72), 3)])
def test_lossless_ragged(cc, torch_gpu, shape, levels):
    torch = torch_gpu
    log("lossless ragged", shape, levels)
    rng = np.random.default_rng(sum(shape))
    img = np.cumsum(rng.integers(-9, 10, shape), axis=-1).astype(np.int16)
    sz, sy, sx = shape if len(shape) == 3 else (1,) + shape
    inst = cc.createInstance(0, 7, img.size, 32, 16)
    words = cc.compressVolumeLossless(inst, to_dev(torch, img), sx, sy, sz, levels)
    assert np.array_equal(words, P.compress_lossless(img, levels, log2=16, cbs=32))
    out = torch.full(shape, -7, dtype=torch.int16, device="cuda")
    cc.decompressVolumeLossless(inst, out, sx, sy, sz, levels, words)
    torch.cuda.synchronize()
    assert np.array_equal(to_host(out), img)
    inst.close()


@pytest.mark.parametrize("shape,levels", [((2, 2, 2), 1), ((4, 8, 12), 2), ((8, 16, 1032), 1), ((24, 40, 56), 3)])
@pytest.mark.parametrize("lvl0", [False, True], ids=["rle_all", "rle_lvl0"])
def test_float_and_short_ragged(cc, torch_gpu, shape, levels, lvl0):
    torch = torch_gpu
    log("float ragged", shape, levels, lvl0)
    vol = np.random.default_rng(sum(shape)).standard_normal(shape).astype(np.float32)
    sz, sy, sx = shape
    inst = cc.createInstance(0, 7, vol.size, 64, 14)
    src, out = to_dev(torch, vol), torch.full(shape, 9.0, dtype=torch.float32, device="cuda")
    words = cc.compressVolumeFloat(inst, src, sx, sy, sz, levels, 0.02, lvl0)
    want = P.compress_volume_float(vol, levels, 0.02, cbs=64, rle_only_lvl0=lvl0)
    assert np.array_equal(words, want)
    cc.decompressVolumeFloat(inst, out, sx, sy, sz, levels, words, 0.02, lvl0)
    torch.cuda.synchronize()
    ref = P.decompress_volume_float(want, shape, levels, 0.02, cbs=64, rle_only_lvl0=lvl0)
    assert float(np.abs(to_host(out) - ref).max()) <= 1e-6 * max(1.0, float(np.abs(ref).max()))
    words = cc.compressVolumeFloatQuantFirst(inst, src, sx, sy, sz, levels, 0.02, lvl0)
    assert np.array_equal(words, P.compress_volume_float_quant_first(vol, levels, 0.02, cbs=64, rle_only_lvl0=lvl0))
    cc.decompressVolumeFloatQuantFirst(inst, out, sx, sy, sz, levels, words, 0.02, lvl0)
    torch.cuda.synchronize()
    q = np.trunc(vol * (np.float32(1) / np.float32(0.02)) + np.sign(vol) * np.float32(0.5)).astype(np.float32)
    assert np.array_equal(to_host(out), q * np.float32(0.02))
    inst.close()


@pytest.mark.parametrize("rl", [True, False], ids=["rlhuff", "huff"])
@pytest.mark.parametrize("start", [1, 17, 31])
def test_segment_inside_a_word(cc, torch_gpu, rl, start):
    torch = torch_gpu
    rng = np.random.default_rng(start)
    streams = [rng.integers(0, 40, 5000).astype(np.uint16), np.zeros(5000, np.uint16)]
    inst = cc.createInstance(0, 2, 5000, 128, 14)
    bs = cc.BitStream()
    bs.writeBits(0x5A5A5A5A, start)
    assert (cc.encodeRLHuff if rl else cc.encodeHuff)(inst, bs, [to_dev(torch, s) for s in streams], 5000)
    want, nbits = o.encode(streams, rl=rl, log2=14, cbs=128, start_bit=start)
    got = bs.words().copy()
    mask = np.uint32(0xFFFFFFFF >> start)
    assert bs.getBitSize() == nbits and np.array_equal(got[1:], want[1:]) and (got[0] & mask) == (want[0] & mask)
    rs = cc.BitStream(got, bs.getBitSize())
    rs.setBitPosition(start)
    outs = [torch.full((5000,), -1, dtype=torch.int16, device="cuda") for _ in streams]
    (cc.decodeRLHuff if rl else cc.decodeHuff)(inst, rs, outs, 5000)
    torch.cuda.synchronize()
    assert all(np.array_equal(to_host(a, np.uint16), b) for a, b in zip(outs, streams))
    inst.close()


def test_damaged_volume_streams(cc, torch_gpu):
    torch = torch_gpu
    vol = S.gaussian_field((16, 16, 32), 5)
    inst = cc.createInstance(0, 7, vol.size, 64, 14)
    src = to_dev(torch, vol)
    words = cc.compressVolumeFloat(inst, src, 32, 16, 16, 2, 0.01)
    out = torch.full_like(src, 3.0)
    for cut in (0, 1, 5, words.size // 2, words.size - 1):
        with pytest.raises(cc.CCError) as e:
            cc.decompressVolumeFloat(inst, out, 32, 16, 16, 2, words[:cut], 0.01)
        assert e.value.status == 6, cut
    bad = words.copy()
    bad[0] ^= np.uint32(0xF8000000)  # the number of code lengths
    with pytest.raises(cc.CCError):
        cc.decompressVolumeFloat(inst, out, 32, 16, 16, 2, bad, 0.01)
    torch.cuda.synchronize()
    assert float((out - 3.0).abs().max()) == 0.0
    cc.decompressVolumeFloat(inst, out, 32, 16, 16, 2, words, 0.01)  # the instance goes on
    torch.cuda.synchronize()
    ref = P.decompress_volume_float(words, vol.shape, 2, 0.01, cbs=64)
    assert float(np.abs(to_host(out) - ref).max()) <= 1e-6 * float(np.abs(ref).max())
    inst.close()
