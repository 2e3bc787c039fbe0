"""The route of float volumes past 2^31 voxels (single-volume transforms, level by level, one coder job),
forced at small sizes: its words are the oracle's and its values those of the brick passes, bit for bit,
for axes shorter than the filter, rows past a wave, several levels, both symbol sizes and several channels."""
import numpy as np
import pytest

from oracle import pipeline as P
from tests.gpu_util import log, to_dev, to_host

pytestmark = pytest.mark.gpu

SHAPES = [((2, 2, 2), 1), ((4, 8, 12), 2), ((16, 16, 32), 1), ((8, 16, 1032), 1), ((24, 40, 56), 3), ((64, 48, 32), 2),
          ((48, 96, 80), 4)]


def _volume(shape, seed):
    rng = np.random.default_rng(seed)
    v = rng.standard_normal(shape).astype(np.float32)
    for ax in range(3):
        v = v + np.roll(v, 1, ax)
    return v


@pytest.mark.parametrize("lvl0", [False, True], ids=["rle_all", "rle_lvl0"])
@pytest.mark.parametrize("log2", [14, 20])
@pytest.mark.parametrize("shape,levels", SHAPES)
def test_large_route(cc, torch_gpu, shape, levels, log2, lvl0):
    torch = torch_gpu
    log("large route", shape, levels, log2, lvl0)
    sz, sy, sx = shape
    vol = _volume(shape, sum(shape))
    src = to_dev(torch, vol)
    words, recs = {}, {}
    for route in ("large", "bricks"):
        inst = cc.createInstance(0, 7, max(1, vol.size // 8), 64, log2)
        inst.setBrickVolumeLimit(1 if route == "large" else 0)
        cc.setTimingDetail(inst, cc.TIMING_DETAIL_HIGH)
        words[route] = cc.compressVolumeFloat(inst, src, sx, sy, sz, levels, 0.01, lvl0)
        recs[route] = torch.full(shape, 123.0, dtype=torch.float32, device="cuda")
        cc.decompressVolumeFloat(inst, recs[route], sx, sy, sz, levels, words[route], 0.01, lvl0)
        torch.cuda.synchronize()
        kernels = [k for k in cc.getTimings(inst)[0] if k.startswith("Kernel: ")]
        assert any("dwt97_" in k for k in kernels) == (route == "large"), kernels
        assert any("bricks_" in k for k in kernels) == (route == "bricks"), kernels
        inst.close()
    assert np.array_equal(words["large"], words["bricks"])
    assert torch.equal(recs["large"], recs["bricks"])
    if log2 == 14:
        assert np.array_equal(words["large"], P.compress_volume_float(vol, levels, 0.01, cbs=64, rle_only_lvl0=lvl0))
        ref = P.decompress_volume_float(words["large"], shape, levels, 0.01, cbs=64, rle_only_lvl0=lvl0)
        assert float(np.abs(to_host(recs["large"]) - ref).max()) <= 1e-6 * max(1.0, float(np.abs(ref).max()))


@pytest.mark.parametrize("shape,levels", [((24, 40, 56), 3), ((32, 16, 1040), 2)])
def test_large_route_channels(cc, torch_gpu, shape, levels):
    """Three channels whose voxels together pass the limit, none of them alone."""
    torch = torch_gpu
    log("large route, channels", shape, levels)
    sz, sy, sx = shape
    inst = cc.createInstance(0, 21, int(np.prod(shape)) // 8, 128, 14)
    vols = [_volume(shape, k) for k in range(3)]
    steps = [0.01, 0.02, 0.005]
    bits = [cc.compressVolumeFloat(inst, to_dev(torch, v), sx, sy, sz, levels, q) for v, q in zip(vols, steps)]
    outs = {}
    for limit in (0, 2 * vols[0].size + 1):
        inst.setBrickVolumeLimit(limit)
        outs[limit] = [torch.full(shape, -5.0, dtype=torch.float32, device="cuda") for _ in vols]
        cc.decompressVolumeFloatMultiChannel(inst, list(zip(outs[limit], bits, steps)), sx, sy, sz, levels)
        torch.cuda.synchronize()
    for a, b in zip(*outs.values()):
        assert torch.equal(a, b)
    with pytest.raises(cc.CCError):
        inst.setBrickVolumeLimit((1 << 31) + 1)
    inst.close()
