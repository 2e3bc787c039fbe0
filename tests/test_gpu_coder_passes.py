"""The device encoder's passes at the edges of their rules: zero runs around the lengths where a filler
pair is due or a faster rule ends (255, 256), across lanes, steps of 512 symbols, the four waves' parts
of a stream and the chunks of 2048; symbols on both sides of the 4096 bins; codewords that fit together
in one word, two or none.  The words are the oracle's."""
import numpy as np
import pytest

from oracle import pyoracle as o
from tests.gpu_util import to_dev, to_host

pytestmark = pytest.mark.gpu


def _streams(n):
    def runs(length, sym=1):  # zero runs of `length` between nonzeros
        a = np.zeros(n, np.uint16)
        a[length::length + 1] = sym
        return a
    edge = np.zeros(n, np.uint16)
    edge[[0, n // 2, n - 1]] = [4095, 4096, 7]
    lead = np.zeros(n, np.uint16)
    lead[n - 1] = 4095
    return [runs(k) for k in (1, 7, 8, 240, 247, 248, 249, 254, 255, 256, 257, 511, 512, 513)] + [
        runs(3, 4095), runs(2, 5000), edge, lead, np.arange(n, dtype=np.uint32).astype(np.uint16) % 4099]


@pytest.mark.parametrize("rl", [True, False], ids=["rlhuff", "huff"])
@pytest.mark.parametrize("n", [1, 8, 511, 512, 513, 1025, 2047, 2048, 2049, 6145, 20000])
def test_zero_runs(cc, torch_gpu, n, rl):
    torch = torch_gpu
    print("zero runs", n, rl, flush=True)
    streams = _streams(n)
    inst = cc.createInstance(0, len(streams), n, 64, 14)
    words, _ = o.encode(streams, rl=rl, log2=14, cbs=64)
    out = torch.full((words.size + 64,), -1, dtype=torch.int32, device="cuda")
    nw = cc.encodeDevice(inst, rl, [to_dev(torch, s) for s in streams], n, out)
    torch.cuda.synchronize()
    got = to_host(out, np.uint32)
    assert nw == words.size
    assert np.array_equal(got[:nw], words), np.nonzero(got[:nw] != words)[0][:4]
    assert np.all(got[nw:] == 0xFFFFFFFF)
    inst.close()


def _skewed(rng, order):
    """Symbols whose counts grow like the Fibonacci numbers: codewords of 1 to 20 bits and more."""
    fib = [1, 1]
    while sum(fib) < 45000:
        fib.append(fib[-1] + fib[-2])
    a = np.repeat(np.arange(1, len(fib) + 1), fib).astype(np.uint16)  # the longest codewords side by side
    if order == "shuffled":
        rng.shuffle(a)
    elif order == "mixed":  # long ones among short ones, a few bits each
        k = 4000
        rng.shuffle(a[:k])
    return a


@pytest.mark.parametrize("rl", [True, False], ids=["rlhuff", "huff"])
@pytest.mark.parametrize("order", ["sorted", "shuffled", "mixed"])
def test_codeword_lengths(cc, torch_gpu, order, rl):
    """A thread's eight codewords of every total length, as streams of their own and as zero counts."""
    torch = torch_gpu
    print("codeword lengths", order, rl, flush=True)
    rng = np.random.default_rng(7)
    a = _skewed(rng, order)
    gaps = np.zeros(int(a.sum()) + a.size, np.uint16)  # a symbol after each run of a[i] - 1 zeros
    gaps[np.cumsum(a.astype(np.int64)) - 1] = 1
    for stream in (a, gaps[:60001]):
        inst = cc.createInstance(0, 1, stream.size, 64, 14)
        words, _ = o.encode([stream], rl=rl, log2=14, cbs=64)
        out = torch.zeros(words.size + 8, dtype=torch.int32, device="cuda")
        nw = cc.encodeDevice(inst, rl, [to_dev(torch, stream)], stream.size, out)
        torch.cuda.synchronize()
        got = to_host(out, np.uint32)
        assert nw == words.size
        assert np.array_equal(got[:nw], words), np.nonzero(got[:nw] != words)[0][:4]
        inst.close()
