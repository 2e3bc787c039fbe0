"""The device block decoder where its codeword copy and its long-code path can go wrong: codes
longer than the 10-bit lookup table in every position of a round, blocks of few and of many words,
streams that end inside a block, short (one wave) and long (four waves) sequences.  The decoder is
compared with the symbols the oracle's own bitstream was made from."""
import numpy as np
import pytest

from oracle import pyoracle as o
from tests.gpu_util import to_dev, to_host

pytestmark = pytest.mark.gpu


def _fibonacci(rng, n, depth, dtype):
    """n symbols whose counts fall off like Fibonacci numbers, so that code lengths reach `depth`."""
    p = np.array([1.618 ** -k for k in range(depth + 1)])
    s = rng.choice(depth + 1, n, p=p / p.sum())
    s[: min(n, depth + 1)] = np.arange(min(n, depth + 1))  # every length occurs
    rng.shuffle(s)
    return (s * 37 % 4093).astype(dtype)


@pytest.mark.parametrize("cbs", [32, 64, 256])
@pytest.mark.parametrize("n,depth", [(63, 12), (64 * 64 + 1, 14), (70001, 20), (300007, 24)])
def test_long_codes(cc, torch_gpu, cbs, n, depth):
    torch = torch_gpu
    print("block decoder", cbs, n, depth, flush=True)
    rng = np.random.default_rng(n + depth)
    sym = _fibonacci(rng, n, depth, np.uint16)
    inst = cc.createInstance(0, 2, n, cbs, 14)
    for rl in (False, True):
        src = sym.copy()
        if rl:
            src[rng.random(n) < 0.4] = 0
        words, nbits = o.encode([src], rl=rl, log2=14, cbs=cbs)
        dev = to_dev(torch, words.astype(np.uint32))
        out = torch.full((n,), -1, dtype=torch.int16, device="cuda")
        used = cc.decodeDevice(inst, rl, dev, [out], n)
        torch.cuda.synchronize()
        assert used == words.size
        assert np.array_equal(to_host(out, np.uint16), src)
    inst.close()


@pytest.mark.parametrize("width", [1, 11, 13])
def test_flat_codes(cc, torch_gpu, width):
    """2^width equally frequent symbols: every code has `width` bits (a round of the widest takes the
    most words of the copy; the 14-bit symbol count of a header allows no 14-bit flat code)."""
    torch = torch_gpu
    rng = np.random.default_rng(width)
    n = (1 << width) * max(1, 40000 >> width)
    sym = rng.permutation(np.arange(n) % (1 << width)).astype(np.uint16)
    inst = cc.createInstance(0, 1, n, 64, 14)
    words, _ = o.encode([sym], rl=False, log2=14, cbs=64)
    out = torch.full((n,), -1, dtype=torch.int16, device="cuda")
    cc.decodeDevice(inst, False, to_dev(torch, words.astype(np.uint32)), [out], n)
    torch.cuda.synchronize()
    assert np.array_equal(to_host(out, np.uint16), sym)
    inst.close()


@pytest.mark.parametrize("runs", [True, False], ids=["runs", "plain"])
@pytest.mark.parametrize("depth,blocks", [(11, 2), (12, 3), (14, 7), (18, 43), (19, 70)])
def test_long_codes_in_a_wave_of_few_blocks(cc, torch_gpu, depth, blocks, runs):
    """Codes of up to `depth` bits (the lookup table holds 10) in blocks of 256 symbols, so that most lanes of
    the last wave have no block of their own: Fibonacci counts, whose codes have every length from one bit on
    (runs of that code are taken at once), or with the commonest symbol as two, which has no such code."""
    torch = torch_gpu
    counts = [1, 1]
    while len(counts) < depth + 1:
        counts.append(counts[-1] + counts[-2])
    if not runs:
        counts[-1:] = [counts[-1] // 2, counts[-1] - counts[-1] // 2]
    rng = np.random.default_rng(depth)
    sym = np.repeat(np.arange(1, len(counts) + 1, dtype=np.uint16) * 37, counts)
    n = sym.size
    assert -(-n // 256) == blocks
    print("block decoder, few blocks", n, depth, runs, flush=True)
    rng.shuffle(sym)
    inst = cc.createInstance(0, 1, n, 256, 14)
    for rl in (False, True):
        words, _ = o.encode([sym], rl=rl, log2=14, cbs=256)
        lengths = words[0 if not rl else 1] >> 27  # a table's header starts with its longest code's length
        assert lengths == depth - (not runs)
        out = torch.full((n,), -1, dtype=torch.int16, device="cuda")
        cc.decodeDevice(inst, rl, to_dev(torch, words.astype(np.uint32)), [out], n)
        torch.cuda.synchronize()
        assert np.array_equal(to_host(out, np.uint16), sym)
    inst.close()
