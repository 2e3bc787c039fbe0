"""Streams long enough that the device encoder splits them over workgroups: zero runs, coding blocks
and output words that cross segment borders, segments without a nonzero or without a codeword bit.
The words are the oracle's."""
import numpy as np
import pytest

from oracle import pyoracle as o
from tests.gpu_util import laplace_symbols, to_dev, to_host

pytestmark = pytest.mark.gpu

CHUNK = 2048  # symbols a workgroup takes per step; two chunks and more are split in a small job


def _patterns(rng, n):
    sparse = np.zeros(n, np.uint16)
    sparse[rng.integers(0, n, max(1, n // 5000))] = 3
    middle = np.zeros(n, np.uint16)  # leading and trailing segments without a nonzero
    middle[n // 2] = 9
    one = np.full(n, 5, np.uint16)
    tail = np.zeros(n, np.uint16)
    tail[-1] = 1
    return {"laplace": laplace_symbols(rng, n, 6.0, 0.4, maxsym=4000), "dense": rng.integers(1, 300, n).astype(np.uint16),
            "wide": rng.integers(0, 16384, n).astype(np.uint16), "sparse": sparse, "middle": middle, "one": one,
            "zeros": np.zeros(n, np.uint16), "tail": tail}


@pytest.mark.parametrize("rl", [True, False], ids=["rlhuff", "huff"])
@pytest.mark.parametrize("n", [2 * CHUNK, 2 * CHUNK + 1, 4 * CHUNK - 1, 13 * CHUNK + 7, 300001])
def test_split_streams(cc, torch_gpu, n, rl):
    torch = torch_gpu
    print("split coder", n, rl, flush=True)
    rng = np.random.default_rng(n)
    inst = cc.createInstance(0, 8, n, 64, 14)
    pats = _patterns(rng, n)
    groups = [[p] for p in pats] + [list(pats)]  # each alone, then all in one call
    for names in groups:
        streams = [pats[k] for k in names]
        words, _ = o.encode(streams, rl=rl, log2=14, cbs=64)
        dev = [to_dev(torch, s) for s in streams]
        out = torch.full((words.size + 64,), -1, dtype=torch.int32, device="cuda")
        for _ in range(2):  # the buffers of the second call hold the first one's
            nw = cc.encodeDevice(inst, rl, dev, n, out)
            torch.cuda.synchronize()
            got = to_host(out, np.uint32)
            assert nw == words.size, names
            assert np.array_equal(got[:nw], words), (names, np.nonzero(got[:nw] != words)[0][:4])
            assert np.all(got[nw:] == 0xFFFFFFFF), names
    inst.close()


def test_split_symbol32_and_overflow(cc, torch_gpu):
    torch = torch_gpu
    rng = np.random.default_rng(5)
    n = 50001
    inst = cc.createInstance(0, 2, n, 128, 20)
    streams = [rng.integers(0, 1 << 18, n).astype(np.uint32), laplace_symbols(rng, n, 9.0, 0.2, dtype=np.uint32)]
    words, _ = o.encode(streams, rl=True, log2=20, cbs=128)
    out = torch.zeros(words.size, dtype=torch.int32, device="cuda")
    nw = cc.encodeDevice(inst, True, [to_dev(torch, s) for s in streams], n, out)
    torch.cuda.synchronize()
    assert nw == words.size and np.array_equal(to_host(out, np.uint32), words)
    streams[1][n - 3] = 1 << 20
    assert cc.encodeDevice(inst, True, [to_dev(torch, s) for s in streams], n, out) is None
    inst.close()
