"""emu_dequant around the ends of a wavefront's 64 units (8 blocks of the
K-quants, 32 of Q8_0) and of a workgroup's 256: every value's bits against the
oracle, and nothing written before the first or past the last; the same where the
result is large enough for the other kind of store (above 32 MB; Q2_K 256)."""
import ctypes as C

import numpy as np
import pytest

import oracle
from emufpga_amd import _lib
from tests import npref

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("shift", [1, 4])  # floats before the output: 4-byte and 16-byte alignment
@pytest.mark.parametrize("blocks", [1, 7, 8, 9, 31, 33, 127, 129])
@pytest.mark.parametrize("enc", [_lib.Q6_K, _lib.Q5_K, _lib.Q8_0, _lib.Q2_K])
def test_dequant_at_the_ends_of_wavefronts(ctx, enc, blocks, shift):
    rng = np.random.default_rng(enc * 1000 + blocks)
    raw = npref.random_blocks(enc, blocks, rng)
    ref = oracle.decode(enc, raw)
    src = ctx.upload(raw)
    out = ctx.upload(np.full(shift + ref.size + 64, 12345.0, np.float32))
    ctx.check(ctx.lib.emu_dequant(ctx.h, enc, src.ptr, raw.size, C.c_void_p(out.addr + 4 * shift)), "dequant")
    got = out.read(np.float32)
    assert np.array_equal(got[shift:shift + ref.size].view(np.uint32), np.asarray(ref, np.float32).view(np.uint32))
    assert np.all(got[:shift] == 12345.0) and np.all(got[shift + ref.size:] == 12345.0)


@pytest.mark.parametrize("enc,blocks", [(_lib.Q6_K, 32768), (_lib.Q6_K, 32775), (_lib.Q5_K, 32769), (_lib.Q8_0, 262151),
                                        (_lib.Q2_K, 262144), (_lib.Q2_K, 262145)])
def test_dequant_of_large_results(ctx, enc, blocks):
    rng = np.random.default_rng(enc + blocks)
    bb, n = npref.BLOCK_BYTES[enc], 1009
    raw = npref.random_blocks(enc, n, rng)
    ref = np.asarray(oracle.decode(enc, raw), np.float32).view(np.uint32)
    times = -(-blocks // n)
    src = ctx.upload(np.tile(raw, times)[:blocks * bb])
    size = blocks * ref.size // n
    out = ctx.upload(np.full(size + 64, 12345.0, np.float32))
    ctx.check(ctx.lib.emu_dequant(ctx.h, enc, src.ptr, blocks * bb, out.ptr), "dequant")
    got = out.read(np.float32)
    assert np.array_equal(got[:size].view(np.uint32), np.tile(ref, times)[:size])
    assert np.all(got[size:] == 12345.0)
