"""The host calls' decode where the table build of a sequence is split over workgroups: symbol counts around
the lookup table's 1024 and every 2048 past it, block counts around 4096, one symbol size and the other.
The decoder is compared with the symbols that the oracle's bitstream was made from."""
import numpy as np
import pytest

from oracle import pyoracle as o
from tests.gpu_util import log, to_host

pytestmark = pytest.mark.gpu


def _symbols(rng, distinct, n, dtype):
    """n symbols of `distinct` values, all of them there, few of them common."""
    s = (rng.geometric(min(1.0, 8.0 / distinct), n) - 1) % distinct
    s[rng.permutation(n)[:distinct]] = np.arange(distinct)
    return (s + 1).astype(dtype)


@pytest.mark.parametrize("distinct,blocks,log2", [
    (1, 4096, 14), (1023, 4095, 14), (1024, 4096, 14), (1025, 4097, 14), (3071, 300, 14), (3072, 8192, 14),
    (3073, 8193, 14), (16000, 1000, 14), (5121, 12289, 16), (30000, 4097, 20)])
def test_tables_and_offsets_in_parts(cc, torch_gpu, distinct, blocks, log2):
    log("decode in parts", distinct, blocks, log2)
    torch = torch_gpu
    rng = np.random.default_rng(distinct + blocks)
    dtype, tdtype = (np.uint32, torch.int32) if log2 > 16 else (np.uint16, torch.int16)
    n = 32 * blocks - 5
    inst = cc.createInstance(0, 2, n, 32, log2)
    for rl in (False, True):
        streams = [_symbols(rng, distinct, n, dtype), _symbols(rng, 3, n, dtype)]  # a second one after the parts
        if rl:
            streams[0][rng.permutation(n)[distinct:n // 4]] = 0
        words, nbits = o.encode(streams, rl=rl, log2=log2, cbs=32)
        bits = cc.BitStream(words, nbits)
        outs = [torch.full((n,), -1, dtype=tdtype, device="cuda") for _ in streams]
        (cc.decodeRLHuff if rl else cc.decodeHuff)(inst, bits, outs, n)
        torch.cuda.synchronize()
        assert bits.getBitPosition() == nbits
        for s, out in zip(streams, outs):
            assert np.array_equal(to_host(out, dtype), s)
    inst.close()


@pytest.mark.parametrize("streams,distinct,blocks", [(1, 1023, 40), (1, 1024, 40), (1, 1025, 40), (1, 9, 1024), (1, 9, 1025),
                                                     (4, 250, 256), (4, 257, 20), (5, 40, 20), (2, 1, 3)])
def test_tables_made_on_the_host_and_on_the_device(cc, torch_gpu, streams, distinct, blocks):
    """Plain decodes around the sizes up to which the host makes their tables: 4 sequences, 1024 symbols and
    1024 blocks in all."""
    log("tables on the host or the device", streams, distinct, blocks)
    torch = torch_gpu
    rng = np.random.default_rng(distinct * streams)
    n = 64 * blocks - 9
    inst = cc.createInstance(0, streams, n, 64, 14)
    for rl in (False, True):
        syms = [_symbols(rng, distinct, n, np.uint16) for _ in range(streams)]
        words, nbits = o.encode(syms, rl=rl, log2=14, cbs=64)
        outs = [torch.full((n,), -1, dtype=torch.int16, device="cuda") for _ in syms]
        (cc.decodeRLHuff if rl else cc.decodeHuff)(inst, cc.BitStream(words, nbits), outs, n)
        torch.cuda.synchronize()
        for s, out in zip(syms, outs):
            assert np.array_equal(to_host(out, np.uint16), s)
    inst.close()


@pytest.mark.parametrize("seed", range(8))
def test_broken_tables_decode_alike_from_the_host_and_from_the_device(cc, torch_gpu, seed):
    """Code lengths that do not make a prefix code (too many or too few codes) are read the same way by both."""
    torch = torch_gpu
    rng = np.random.default_rng(seed)
    n, nlen = 300, int(rng.integers(2, 15))
    counts = rng.integers(0, 6, nlen)
    counts[-1] = 1 + seed % 3
    bits = cc.BitStream()
    for _ in range(5):
        bits.writeBits(nlen, 5)
        for c in counts:
            bits.writeBits(int(c), 14)
        bits.writeBits(int(counts.sum()), 14)
        bits.writeBits(10, 4)
        for k in range(int(counts.sum())):
            bits.writeBits((37 * k + 5) % 1024, 10)
        bits.writeAligned(np.array([32 * 200], np.uint32))  # 200 words of codewords, three blocks 2000 bits apart
        bits.writeAligned((np.arange(200, dtype=np.uint64) * 2654435761 * (seed + 1) % (1 << 32)).astype(np.uint32))
        bits.writeAligned(np.array([0, 2000, 2000], np.uint16))
    inst = cc.createInstance(0, 5, n, 128, 14)
    outs = [torch.full((n,), -1, dtype=torch.int16, device="cuda") for _ in range(6)]
    bits.setBitPosition(0)
    cc.decodeHuff(inst, bits, outs[:1], n)  # one sequence: tables from the host
    bits.setBitPosition(0)
    cc.decodeHuff(inst, bits, outs[1:], n)  # five: from the device
    torch.cuda.synchronize()
    for out in outs[1:]:
        assert torch.equal(out, outs[0])
    inst.close()
