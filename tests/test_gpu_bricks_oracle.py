"""Batched bricks against the oracle, words and reconstructions, every axis length of the brick workload on
every axis, and against the route of large volumes, whose transforms are other kernels (the plain float calls
of small volumes run the batch's own passes)."""
import numpy as np
import pytest

from cudacompress_amd import synthetic as S
from oracle import pipeline as P
from tests.gpu_util import log, to_dev, to_host

pytestmark = pytest.mark.gpu

AXES = (16, 32, 48, 64, 96, 128)
# each length once on each axis, one way round and the other
SHAPES = [tuple(AXES[(i + d) % 6] for d in order) for order in ((0, 1, 2), (2, 1, 0)) for i in range(6)]


@pytest.mark.parametrize("levels,cbs", [(1, 128), (2, 64), (3, 32)])
def test_batched_bricks_match_oracle(cc, torch_gpu, levels, cbs):
    torch = torch_gpu
    log("bricks against the oracle", levels, cbs)
    field = S.gaussian_field((128, 128, 128), 40 + levels)
    rng = np.random.default_rng(levels)
    bricks = []
    for s in SHAPES:
        z, y, x = (int(rng.integers(0, 128 - d + 1)) for d in s)
        bricks.append(np.ascontiguousarray(field[z:z + s[0], y:y + s[1], x:x + s[2]]))
    steps = [float(np.float32(f * float(field.std()))) for f in rng.choice([0.005, 0.05, 0.5], len(bricks))]
    srcs = [to_dev(torch, b) for b in bricks]
    out = torch.empty(sum(b.size for b in bricks) + 4096 * len(bricks), dtype=torch.int32, device="cuda")
    inst = cc.createInstance(0, 7, 128 ** 3 // 8, cbs, 14)
    large = cc.createInstance(0, 7, 128 ** 3 // 8, cbs, 14)
    large.setBrickVolumeLimit(1)
    offs, stat = cc.compressBricksFloat(inst, srcs, SHAPES, steps, levels, out)
    assert np.all(stat == 0)
    dsts = [torch.full_like(s, 77.0) for s in srcs]
    assert np.all(cc.decompressBricksFloat(inst, dsts, SHAPES, steps, levels, out, offs) == 0)
    torch.cuda.synchronize()
    words = to_host(out[: int(offs[-1])], np.uint32)
    for i, (b, q) in enumerate(zip(bricks, steps)):
        got = words[int(offs[i]):int(offs[i + 1])]
        assert np.array_equal(got, P.compress_volume_float(b, levels, q, cbs=cbs)), f"brick {i} {b.shape}"
        ref = P.decompress_volume_float(got, b.shape, levels, q, cbs=cbs)
        rec = to_host(dsts[i])
        assert float(np.abs(rec - ref).max()) <= 1e-6 * max(1.0, float(np.abs(ref).max())), f"brick {i} {b.shape}"
        z, y, x = b.shape
        assert np.array_equal(got, cc.compressVolumeFloat(large, srcs[i], x, y, z, levels, q))
        other = torch.full_like(srcs[i], 55.0)
        cc.decompressVolumeFloat(large, other, x, y, z, levels, got, q)
        torch.cuda.synchronize()
        assert np.array_equal(to_host(other), rec), f"brick {i} {b.shape}"
    inst.close()
    large.close()
