"""Multi-channel float decodes whose channels take turns with the work buffers: the same values as one
channel at a time, and no more device memory than the channels that are transformed together need."""
import pytest

from tests.gpu_util import log

pytestmark = pytest.mark.gpu

LIMIT = 1 << 27  # bytes of work buffers that channels share


def _fields(torch, shape, channels):
    g = torch.Generator(device="cuda")
    g.manual_seed(channels)
    for _ in range(channels):
        x = torch.randn(shape, generator=g, device="cuda")
        for d in range(3):
            x = x + x.roll(1, d)
            x = x + x.roll(2, d)
        yield x


# 2 + 1/8 floats of work a voxel at two levels: 3.0, 1.5 and 0.9 channels of these sizes fit the limit
@pytest.mark.parametrize("shape,channels", [((160, 128, 256), 4), ((192, 256, 212), 2), ((256, 256, 268), 3)])
def test_channels_in_turn(cc, torch_gpu, shape, channels):
    torch = torch_gpu
    log("channels in turn", shape, channels)
    sz, sy, sx = shape
    voxels = sx * sy * sz
    one = cc.createInstance(0, 7, voxels // 8, 128, 14)
    chans, want = [], []
    for k, x in enumerate(_fields(torch, shape, channels)):
        step = 0.01 * (k + 1)
        chans.append((torch.full_like(x, -9.0), cc.compressVolumeFloat(one, x, sx, sy, sz, 2, step), step))
        want.append(torch.empty_like(x))
        cc.decompressVolumeFloat(one, want[-1], sx, sy, sz, 2, chans[-1][1], step)
    one.close()
    inst = cc.createInstance(0, 7 * channels, voxels // 8, 128, 14)
    torch.cuda.synchronize()
    before = torch.cuda.mem_get_info()[0]
    cc.decompressVolumeFloatMultiChannel(inst, chans, sx, sy, sz, 2)
    torch.cuda.synchronize()
    used = before - torch.cuda.mem_get_info()[0]
    for (out, _, _), w in zip(chans, want):
        assert torch.equal(out, w)
    # work buffers of the channels at once; symbols, words and decode tables of all of them; each buffer is
    # allocated a quarter larger than it has to be, and memory is handed out in pieces of 2 MB
    words = sum(c[1].size for c in chans)
    work = max(1, LIMIT // int(8.5 * voxels)) * 8.5 * voxels
    bound = 1.25 * (work + 2 * channels * voxels + 4 * words + voxels * channels / 8) + 16 * (2 << 20)
    log("device memory", used >> 20, "MB, bound", int(bound) >> 20)
    assert used <= bound
    inst.close()
