"""Multi-token matvecs of Q8_0, Q5_K and Q2_K on the f16 matrix cores
(csrc/qsplit.hip) and the vector form beside them, through every epilogue,
against the oracle: |gpu - ref| <= 1e-5 sum |w x|, the bar of
test_qmatvec_random_within_tolerance (an f32 sum in another order).  Sizes: a
row and a half tile, one span and less (32 columns), a last span of one block,
eight wavefronts' spans and one more, two tiles per workgroup, and the sizes on
both sides of the dispatch rule."""
from dataclasses import replace

import numpy as np
import pytest

import oracle
from emufpga_amd import _lib
from emufpga_amd.linear import QuantMatrix, streamed
from emufpga_amd.serve import Model, Session
from tests import npref
from tests.test_gpu_model import SMALL_QWEN3, SMALL_SMOL

pytestmark = pytest.mark.gpu

FORMATS = [_lib.Q8_0, _lib.Q5_K, _lib.Q2_K]


def weights(dtype, raw, rows, cols):
    return npref.DECODERS[dtype](raw).reshape(rows, cols).astype(np.float64)


def blocks(dtype, rows, cols, rng):
    return npref.random_blocks(dtype, rows * cols // npref.BLOCK_ELEMS[dtype], rng)


@pytest.mark.parametrize("n_tok", [2, 4, 5, 8])
@pytest.mark.parametrize("dtype,rows,cols", [
    (_lib.Q8_0, 1, 32), (_lib.Q8_0, 17, 288), (_lib.Q8_0, 40, 480), (_lib.Q8_0, 33, 2336), (_lib.Q5_K, 16, 256),
    (_lib.Q5_K, 31, 2304), (_lib.Q2_K, 1, 256), (_lib.Q2_K, 50, 2560), (_lib.Q8_0, 8193, 1024), (_lib.Q5_K, 8208, 1024),
    (_lib.Q2_K, 8200, 1280),
    # the matrix-core form from two, three, five or six tokens on
    (_lib.Q8_0, 4097, 64), (_lib.Q8_0, 16385, 32), (_lib.Q8_0, 2570, 2080), (_lib.Q8_0, 1031, 2336), (_lib.Q5_K, 2050, 512),
    (_lib.Q5_K, 2065, 2304), (_lib.Q2_K, 16390, 256), (_lib.Q2_K, 2561, 2560)])
def test_matvec_within_the_bar(ctx, dtype, rows, cols, n_tok):
    rng = np.random.default_rng(rows + cols + n_tok)
    raw = blocks(dtype, rows, cols, rng)
    x = rng.normal(size=(n_tok, cols)).astype(np.float32)
    y0 = rng.normal(size=(n_tok, rows)).astype(np.float32)
    got = streamed(ctx, QuantMatrix(ctx, dtype, rows, cols, raw), (x, n_tok), accumulate_into=y0).reshape(n_tok, rows)
    w = weights(dtype, raw, rows, cols)
    bound = 1e-5 * (np.abs(x).astype(np.float64) @ np.abs(w).T) + 1e-6 * np.abs(y0) + 1e-30
    assert np.all(np.abs(got - (y0 + x.astype(np.float64) @ w.T)) <= bound)


@pytest.mark.parametrize("gain", [False, True])
@pytest.mark.parametrize("n_tok", [3, 8])
@pytest.mark.parametrize("dtype,rows,cols", [(_lib.Q8_0, 100, 544), (_lib.Q8_0, 1111, 544), (_lib.Q5_K, 1100, 1024), (_lib.Q2_K, 70, 768)])
def test_gate_up_pair_within_the_bar(ctx, dtype, rows, cols, n_tok, gain):
    rng = np.random.default_rng(rows * 3 + n_tok)
    raws = [blocks(dtype, rows, cols, rng) for _ in range(2)]
    x = rng.normal(size=(n_tok, cols)).astype(np.float32)
    g = rng.uniform(0.5, 1.5, cols).astype(np.float32)
    bw, bu = (ctx.upload(r) for r in raws)
    bx, bg, by = ctx.upload(x), ctx.upload(g), ctx.alloc(4 * n_tok * rows)
    ctx.check(ctx.lib.emu_qmatvec_fused(ctx.h, dtype, bw.ptr, bu.ptr, rows, cols, bx.ptr, n_tok, bg.ptr if gain else None,
                                        1e-6, by.ptr, 0), "fused")
    xn = x.astype(np.float64)
    if gain:
        xn = xn / np.sqrt((xn * xn).mean(1, keepdims=True) + 1e-6) * g
    w, u = (weights(dtype, r, rows, cols) for r in raws)
    a, b = xn @ w.T, xn @ u.T
    sig = 1.0 / (1.0 + np.exp(-np.clip(a, -700, 700)))
    # silu's slope is at most 1.1: the pair's bound from the two dots' bounds
    ea, eb = (1e-5 * (np.abs(xn) @ np.abs(m).T) for m in (w, u))
    bound = 1.1 * ea * (np.abs(b) + eb) + np.abs(a * sig) * eb + 1e-6 * np.abs(a * sig * b) + 1e-30
    assert np.all(np.abs(by.read(np.float32).reshape(n_tok, rows) - a * sig * b) <= bound)


@pytest.mark.parametrize("dtype", FORMATS)
def test_a_token_with_an_infinity_touches_no_other(ctx, dtype):
    rng = np.random.default_rng(9)
    rows, cols, n = 40, 512, 6
    raw = blocks(dtype, rows, cols, rng)
    m = QuantMatrix(ctx, dtype, rows, cols, raw)
    x = rng.normal(size=(n, cols)).astype(np.float32)
    clean = streamed(ctx, m, (x, n)).reshape(n, rows)
    x[2, 300] = np.inf
    x[4, 7] = np.nan
    got = streamed(ctx, m, (x, n)).reshape(n, rows)
    keep = [0, 1, 3, 5]
    assert np.array_equal(got[keep], clean[keep])
    assert not np.any(np.isfinite(got[[2, 4]]))


@pytest.mark.parametrize("dtype", FORMATS)
def test_an_infinity_takes_the_signs_of_the_weights(ctx, dtype):
    """inf * w: infinite by w's sign, NaN where w is 0 or two infinities meet
    with opposite signs, as in the f32 sums of the vector form."""
    rng = np.random.default_rng(10)
    rows, cols, n = 1100, 512, 8
    raw = blocks(dtype, rows, cols, rng)
    x = rng.normal(size=(n, cols)).astype(np.float32)
    x[1, 300] = np.inf
    x[3, 511] = -np.inf
    x[6, 0], x[6, 40] = np.inf, np.inf
    got = streamed(ctx, QuantMatrix(ctx, dtype, rows, cols, raw), (x, n)).reshape(n, rows)
    w = weights(dtype, raw, rows, cols)
    for t, at in ((1, [300]), (3, [511]), (6, [0, 40])):
        with np.errstate(invalid="ignore"):
            want = sum(x[t, c].astype(np.float64) * w[:, c] for c in at)
        # w = d sc q - dmin m rounds in f32: its sign is sure away from zero
        ok = np.all([(np.abs(w[:, c]) > 1e-5 * np.abs(w).max(1)) | (w[:, c] == 0) for c in at], axis=0)
        assert ok.sum() > rows // 2
        assert np.array_equal(got[t][ok], want[ok].astype(np.float32), equal_nan=True), (t, at)
        assert not np.any(np.isfinite(got[t]))


@pytest.mark.parametrize("dtype", FORMATS)
def test_a_column_far_above_the_others(ctx, dtype):
    """Activations 2^24 times the others over zero weights: the result comes
    from the others, which keep 23 bits (a low half under the span's largest
    value alone would leave them 2e-5).  Bar 3e-7 of the norm: the forms' sums
    are off by 1.0e-7 to 2.6e-7 of it."""
    rng = np.random.default_rng(12)
    rows, cols, n = 4096, 4096, 8
    raw = blocks(dtype, rows, cols, rng)
    per = raw.reshape(rows, -1, npref.BLOCK_BYTES[dtype])
    if dtype == _lib.Q8_0:
        per[:, 100 // 32, 2 + 100 % 32] = 0
    elif dtype == _lib.Q5_K:  # scale and minimum of columns 96..127
        per[:, 0, [7, 11]] &= 0xC0
    else:  # of columns 96..111
        per[:, 0, 6] = 0
    x = rng.normal(size=(n, cols)).astype(np.float32)
    x[:, 100] = 3 * 2.0 ** 24
    got = streamed(ctx, QuantMatrix(ctx, dtype, rows, cols, raw), (x, n)).reshape(n, rows)
    want = x.astype(np.float64) @ weights(dtype, raw, rows, cols).T
    for t in range(n):
        assert np.linalg.norm(got[t] - want[t]) <= 3e-7 * np.linalg.norm(want[t]), t


def test_a_quantised_tail_past_the_matrix_is_not_used(ctx):
    """The last row's last span is read in 16-byte pieces that end with the
    matrix: bytes behind it (here NaN scales) must not reach the result."""
    rng = np.random.default_rng(3)
    rows, cols, n = 3, 288, 5
    raw = blocks(_lib.Q8_0, rows, cols, rng)
    x = rng.normal(size=(n, cols)).astype(np.float32)
    buf = ctx.upload(np.concatenate([raw, np.full(4096, 0xff, np.uint8)]))
    bx, by = ctx.upload(x), ctx.alloc(4 * n * rows)
    ctx.check(ctx.lib.emu_qmatvec(ctx.h, _lib.Q8_0, buf.ptr, raw.size, rows, cols, bx.ptr, x.size, n, by.ptr, 0), "mv")
    ref = oracle.qmatvec(_lib.Q8_0, raw, rows, cols, x, n, mode=1)
    w = weights(_lib.Q8_0, raw, rows, cols)
    bound = 1e-5 * (np.abs(x).astype(np.float64) @ np.abs(w).T) + 1e-30
    assert np.all(np.abs(by.read(np.float32).reshape(n, rows) - ref.reshape(n, rows)) <= bound)


@pytest.mark.parametrize("form", [
    replace(SMALL_SMOL, vocab=4096), replace(SMALL_QWEN3, encoding=_lib.Q5_K, ffn=1280, vocab=3000),
    replace(SMALL_QWEN3, encoding=_lib.Q2_K, ffn=4096), replace(SMALL_SMOL, layers=2, ffn=8224)],
    ids=["q8_0", "q5_k", "q2_k", "q8_0_tall"])
def test_a_client_in_any_company(ctx, form):
    """A session's step takes one form of each matvec for two to eight clients:
    a client's prompt and steps give the same bits whatever their number.  One client alone runs the batch-1 kernels: the
    decoder's bar, 1e-3 of the largest logit, and the same tokens."""
    model = Model(ctx, form)
    model.synth(31)
    rng = np.random.default_rng(5)
    prompts = rng.integers(0, form.vocab, size=(8, 9)).astype(np.uint32)
    feed = rng.integers(0, form.vocab, size=(4, 8)).astype(np.uint32)

    def run(n):
        s = Session(model, n, 32)
        first = s.generate(prompts[:n], 1)[:, 0]
        steps = [s.decode_step(f[:n], want_logits=True) for f in feed]
        return first, [nxt for nxt, _ in steps], [logits for _, logits in steps]

    whole = run(8)
    for n in (2, 3, 4, 5, 7):
        first, nxt, logits = run(n)
        assert np.array_equal(first, whole[0][:n]), n
        for i in range(len(feed)):
            assert np.array_equal(logits[i], whole[2][i][:n]), (n, i)
            assert np.array_equal(nxt[i], whole[1][i][:n]), (n, i)
    first, nxt, logits = run(1)
    assert first[0] == whole[0][0]
    for i in range(len(feed)):
        assert np.max(np.abs(logits[i][0] - whole[2][i][0])) <= 1e-3 * np.max(np.abs(whole[2][i][0]))
        assert nxt[i][0] == whole[1][i][0]
