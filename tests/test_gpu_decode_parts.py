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
