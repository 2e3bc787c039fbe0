"""Segments of the streaming brick passes: a brick coded alone (short segments, the chip is nearly empty)
and among so many that its level takes long ones gives the same words and the same values."""
import numpy as np
import pytest

from cudacompress_amd import synthetic as S
from tests.gpu_util import log

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("copies", [1, 3, 5, 17])  # 8-pair segments up to 32-pair ones on the first level
def test_segments(cc, torch_gpu, copies):
    torch = torch_gpu
    log("brick segments", copies)
    shapes = [(16, 8, 20), (136, 40, 72), (24, 132, 16)]  # rows, planes and depths with remainders
    field = S.gaussian_field((136, 132, 128), 9)
    bricks = [np.ascontiguousarray(field[:z, :y, :x]) for z, y, x in shapes]
    big = torch.from_numpy(np.ascontiguousarray(field[:128, :128, :128])).cuda()
    srcs = [torch.from_numpy(b).cuda() for b in bricks]
    inst = cc.createInstance(0, 7, 64 ** 3, 64, 14)

    def code(extra):
        all_srcs = srcs + [big] * extra
        all_shapes = [tuple(s.shape) for s in all_srcs]
        steps = [0.02] * len(all_srcs)
        out = torch.zeros(sum(s.numel() for s in all_srcs), dtype=torch.int32, device="cuda")
        offs, stat = cc.compressBricksFloat(inst, all_srcs, all_shapes, steps, 2, out)
        assert np.all(stat == 0)
        dsts = [torch.zeros_like(s) for s in all_srcs]
        cc.decompressBricksFloat(inst, dsts, all_shapes, steps, 2, out, offs)
        torch.cuda.synchronize()
        words = out.cpu().numpy()
        return [words[offs[i]:offs[i + 1]] for i in range(3)], [d.cpu().numpy() for d in dsts[:3]]

    for i in range(3):
        want = cc.compressVolumeFloat(inst, srcs[i], *shapes[i][::-1], 2, 0.02)
        w, v = code(copies)
        w1, v1 = code(0)
        assert np.array_equal(w[i].view(np.uint32), want) and np.array_equal(w1[i].view(np.uint32), want)
        assert np.array_equal(v[i].view(np.uint32), v1[i].view(np.uint32))
    inst.close()
