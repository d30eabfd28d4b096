"""emu_rms_norm and emu_argmax at the edges of their forms, against the oracle:
rows held in registers (whole float4s, up to 16384 values) and any others; one
workgroup per row and rows in chunks of 4096 or more."""
import ctypes as C

import numpy as np
import pytest

import oracle

pytestmark = pytest.mark.gpu


def at(buf, shift):
    return C.c_void_p(buf.addr + 4 * shift)


@pytest.mark.parametrize("shift", [0, 1])
@pytest.mark.parametrize("rows,width", [(1, 4), (1, 252), (1, 256), (3, 260), (2, 4095), (2, 4096), (2, 4100), (1, 16380),
                                        (1, 16384), (1, 16388), (511, 576), (512, 576), (513, 576), (512, 16384)])
def test_rms_norm_forms(ctx, rows, width, shift):
    """shift: floats by which the rows miss their allocation's alignment.  The
    mean of squares of `width` terms, in whatever order, is within width * 2^-24
    of exact relative to itself (all terms positive; a tree is far below that),
    and two such sums are compared; the root halves it."""
    rng = np.random.default_rng(rows + width)
    x = rng.normal(size=(rows, width)).astype(np.float32)
    g = rng.uniform(0.5, 2, width).astype(np.float32)
    pad = np.zeros(shift, np.float32)
    bx, bg = ctx.upload(np.concatenate([pad, x.reshape(-1)])), ctx.upload(np.concatenate([pad, g]))
    by = ctx.upload(np.full(shift + x.size + 4, 7.0, np.float32))
    ctx.check(ctx.lib.emu_rms_norm(ctx.h, at(bx, shift), at(bg, shift), rows, width, 1e-6, at(by, shift)), "rms")
    got = by.read(np.float32)
    assert np.all(got[:shift] == 7.0) and np.all(got[shift + x.size:] == 7.0)
    exact = x / np.sqrt(np.mean(x.astype(np.float64) ** 2, axis=1, keepdims=True) + 1e-6) * g
    assert np.allclose(got[shift:shift + x.size].reshape(rows, width), exact, rtol=4e-6, atol=0)
    if rows <= 3:
        ref = np.stack([oracle.rms_norm(r, g, 1e-6) for r in x])
        assert np.allclose(got[shift:shift + x.size].reshape(rows, width), ref, rtol=width * 2.0**-24 + 4e-6, atol=0)


def test_rms_norm_in_place(ctx):
    rng = np.random.default_rng(2)
    x = rng.normal(size=(5, 1028)).astype(np.float32)
    g = rng.uniform(0.5, 2, 1028).astype(np.float32)
    bx, bg = ctx.upload(x), ctx.upload(g)
    ctx.check(ctx.lib.emu_rms_norm(ctx.h, bx.ptr, bg.ptr, 5, 1028, 1e-6, bx.ptr), "rms")
    exact = x / np.sqrt(np.mean(x.astype(np.float64) ** 2, axis=1, keepdims=True) + 1e-6) * g
    assert np.allclose(bx.read(np.float32).reshape(5, 1028), exact, rtol=4e-6, atol=0)


@pytest.mark.parametrize("shift", [0, 1, 2, 3])
@pytest.mark.parametrize("rows,width", [(1, 1), (3, 3), (2, 1023), (3, 1025), (2, 32767), (2, 32768), (3, 32769), (2, 49152),
                                        (1, 49155), (32, 32769), (33, 32769), (32, 49153), (33, 49153), (1, 262144),
                                        (2, 262147), (70000, 5)])
def test_argmax_forms(ctx, rows, width, shift):
    """Ties at the ends of rows and chunks under both rules, signed zeros,
    infinities, NaN (under the total order, which only the first-index rule
    has), rows of one value."""
    rng = np.random.default_rng(rows + width)
    x = rng.integers(-8, 9, size=(rows, width)).astype(np.float32)  # ties everywhere
    x[0, rng.integers(width, size=2)] = 9.0
    x[-1] = rng.choice([0.0, -0.0], size=width)
    if rows > 2:
        x[1] = -np.inf
        x[1, width // 2] = np.nan if width % 2 else -1.0
    buf, out = ctx.upload(np.concatenate([np.zeros(shift, np.float32), x.reshape(-1)])), ctx.alloc(4 * rows)
    check = range(rows) if rows <= 300 else [0, 1, 65534, 65535, 65536, rows - 1]
    for tie_last in (False, True):
        ctx.check(ctx.lib.emu_argmax(ctx.h, at(buf, shift), rows, width, int(tie_last), out.ptr), "argmax")
        got = out.read(np.int32)
        for r in check:
            if not (tie_last and np.isnan(x[r]).any()):
                assert got[r] == oracle.argmax(x[r], tie_last), (r, tie_last)


class Capture:
    """What the context's stream is given inside `with` goes into a graph."""

    def __init__(self, ctx):
        self.hip, self.stream = C.CDLL(ctx.lib._name), C.c_void_p()  # the HIP runtime it is linked to
        ctx.check(ctx.lib.emu_ctx_stream(ctx.h, C.byref(self.stream)), "stream")
        self.graph, self.exec = C.c_void_p(), C.c_void_p()

    def call(self, name, *args):
        assert getattr(self.hip, name)(*args) == 0, name

    def __enter__(self):
        self.call("hipStreamBeginCapture", self.stream, C.c_int(2))  # relaxed
        return self

    def __exit__(self, *exc):
        self.call("hipStreamEndCapture", self.stream, C.byref(self.graph))
        if exc[0] is None:
            self.call("hipGraphInstantiate", C.byref(self.exec), self.graph, None, None, C.c_size_t(0))

    def nodes(self):
        n = C.c_size_t()
        self.call("hipGraphGetNodes", self.graph, None, C.byref(n))
        return n.value

    def replay(self, stream):
        self.call("hipGraphLaunch", self.exec, stream)
        self.call("hipStreamSynchronize", stream)


def test_captured_calls_hold_no_scratch_of_the_context(ctx):
    """A graph with an argmax over long rows and an attention over a long prefix
    is one launch each, replayed on a stream of its own between the context's
    eager calls of the same kinds, and once more when its context is gone."""
    from emufpga_amd.device import Context

    own = Context(0)
    rng = np.random.default_rng(8)
    rows, width, heads, hd, positions = 4, 100_001, 8, 64, 1000
    x = rng.normal(size=(rows, width)).astype(np.float32)
    q = rng.normal(size=heads * hd).astype(np.float32)
    kv = rng.normal(size=(2, positions, 2 * hd)).astype(np.float16)
    bx, bq, bk, bv = (ctx.upload(a) for a in (x, q, kv[0], kv[1]))
    bi, bo, be, bf = ctx.alloc(4 * rows), ctx.alloc(4 * q.size), ctx.alloc(4 * rows), ctx.alloc(4 * q.size)

    def calls(c, i, o):
        c.check(c.lib.emu_argmax(c.h, bx.ptr, rows, width, 0, i.ptr), "argmax")
        c.check(c.lib.emu_attend_cached(c.h, bq.ptr, bk.ptr, bv.ptr, 1, positions, heads, 2, hd, 0.125, o.ptr), "attend")

    with Capture(own) as g:
        calls(own, bi, bo)
    assert g.nodes() == 2
    beside = C.c_void_p()
    g.call("hipStreamCreate", C.byref(beside))
    k, v = (np.repeat(a.reshape(positions, 2, hd).astype(np.float64), heads // 2, axis=1) for a in kv)
    p = np.exp(np.einsum("phd,hd->ph", k, q.reshape(heads, hd)) * 0.125)
    want = np.einsum("ph,phd->hd", p / p.sum(0), v)
    for last in (False, False, True):
        bi.zero()
        bo.zero()
        ctx.sync()
        if last:
            own.close()
        else:
            calls(own, be, bf)  # the context's own, beside the replay
        g.replay(beside)
        if not last:
            own.sync()
            assert np.array_equal(be.read(np.int32), np.argmax(x, axis=1))
            assert np.allclose(bf.read(np.float32), want.reshape(-1), rtol=2e-5, atol=2e-6)
        assert np.array_equal(bi.read(np.int32), np.argmax(x, axis=1))
        assert np.allclose(bo.read(np.float32), want.reshape(-1), rtol=2e-5, atol=2e-6)
    g.call("hipGraphExecDestroy", g.exec)
    g.call("hipGraphDestroy", g.graph)
    g.call("hipStreamDestroy", beside)
