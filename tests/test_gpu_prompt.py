"""emu_generate's prompt pass (csrc/prefill.hip) against the decode step fed
one prompt token at a time, which the oracle checks hold.

Both round keys and values to f16 once, so an entry whose 32-bit values differ
by rounding may land on the neighbouring half: one part in 2^10 of it at most,
and the next layers' differences follow from those.  Bar: 2^-10 of the tensor's
norm for the cache, the decoder's 1e-3 of the largest logit for the logits.
An f32 cache rounds nothing: 1e-5 in every layer (4e-6 at most were seen, from
the steps' limbs; a product without one operand's low half is off by 2^-12).
What the pass adds to the error is held against 64 bits.
Prompt lengths sit at the edges of the pass's tiles (32, 64, 128 tokens) and
of its range (4 tokens; more than 2048 over all clients take several passes).
"""
import ctypes as C
from dataclasses import replace

import numpy as np
import pytest

from emufpga_amd import _lib, gguf
from emufpga_amd.serve import QWEN3_8B_Q6K, Model, Session
from tests import npref
from tests.test_gpu_model import SMALL_QWEN3, SMALL_SMOL
from tests.test_gpu_moe_model import gemma_layer_scales, small_gemma, small_granite, small_olmoe

pytestmark = pytest.mark.gpu

FORMS = {
    "q6_k": SMALL_QWEN3,
    "q6_k_wide": replace(QWEN3_8B_Q6K, layers=2, vocab=1000),
    "q5_k_no_groups": replace(SMALL_QWEN3, encoding=_lib.Q5_K, heads=8, kv_heads=8, head_dim=64),
    "q2_k_head256": replace(SMALL_QWEN3, encoding=_lib.Q2_K, heads=4, kv_heads=1, head_dim=256),
    "q8_0_smol": SMALL_SMOL,
    "q8_0_half_stage": replace(SMALL_SMOL, hidden=480, heads=5, kv_heads=5, ffn=544),
    "granite": small_granite(),
    "olmoe": small_olmoe(),
    "gemma_window": small_gemma(),
    "granite_deep": replace(small_granite(), layers=4),
    "olmoe_deep": replace(small_olmoe(), layers=4),
    "gemma_deep": replace(small_gemma(), layers=4),  # layers 0 and 2 windowed, 1 and 3 global
}


def step_by_step(sess, prompts):
    for t in range(prompts.shape[1]):
        nxt = sess.decode_step(prompts[:, t])
    return nxt


def compare(model, a, b, n, feed, bar=2.0 ** -10):
    """Every client's cached rows, those of one more step among them.  With
    experts and an f16 cache, a router logit within its entries' rounding (some
    1e-4) of another's may give a token other experts: one in fifty at most."""
    assert np.array_equal(a.positions(), b.positions())
    ties = model.cfg.n_experts and bar > 1e-4
    steady = True
    (na, la), (nb, lb) = (s.decode_step(feed, want_logits=True) for s in (a, b))
    for layer in range(model.cfg.layers):
        for values in (False, True):
            for c, positions in enumerate(a.positions()):
                x, y = (s.read_kv(c, layer, values, int(positions)) for s in (a, b))
                same = np.linalg.norm(x - y, axis=1) <= 2.0 ** -8 * np.linalg.norm(y, axis=1)
                steady &= same[-1]
                assert np.all(same) or ties and np.mean(~same) <= 0.02, (layer, values, c)
                assert np.linalg.norm(x[same] - y[same]) <= bar * np.linalg.norm(y), (layer, values, c)
    if steady:
        assert np.max(np.abs(la - lb)) <= 1e-3 * np.max(np.abs(lb))
        assert np.array_equal(na, nb)


@pytest.mark.parametrize("n,plen", [(1, 4), (3, 23), (1, 33), (2, 66), (1, 130), (5, 61)])
@pytest.mark.parametrize("form", FORMS)
def test_prompt_pass_leaves_what_the_steps_leave(ctx, form, n, plen):
    model = Model(ctx, FORMS[form])
    model.synth(11)
    if form == "gemma_window":
        gemma_layer_scales(model)
    rng = np.random.default_rng(plen)
    prompts = rng.integers(0, model.cfg.vocab, size=(n, plen)).astype(np.uint32)
    a, b = (Session(model, n, plen + 2) for _ in range(2))
    first = a.generate(prompts, 1)[:, 0]
    assert np.array_equal(first, step_by_step(b, prompts))
    compare(model, a, b, n, rng.integers(0, model.cfg.vocab, size=n))


@pytest.mark.parametrize("form", FORMS)
def test_prompt_pass_over_an_f32_cache(ctx, form):
    model = Model(ctx, FORMS[form])
    model.synth(12)
    if form.startswith("gemma"):
        gemma_layer_scales(model)
    rng = np.random.default_rng(7)
    n, plen = 2, 75
    prompts = rng.integers(0, model.cfg.vocab, size=(n, plen)).astype(np.uint32)
    a, b = (Session(model, n, plen + 2, kv_f16=False) for _ in range(2))
    first = a.generate(prompts, 1)[:, 0]
    assert np.array_equal(first, step_by_step(b, prompts))
    compare(model, a, b, n, rng.integers(0, model.cfg.vocab, size=n), 1e-5)


@pytest.mark.parametrize("kv_f16", [True, False])
@pytest.mark.parametrize("form,n,plen", [("gemma_deep", 2, 300), ("gemma_deep", 8, 290), ("granite_deep", 8, 290),
                                         ("olmoe_deep", 7, 300), ("q6_k", 8, 290)])
def test_windows_and_experts_over_long_prompts(ctx, form, n, plen, kv_f16):
    """Prompts past the window's first tile (its earlier tiles are skipped), of
    more than 2048 tokens over the clients where there are eight, and a second
    prompt behind the first."""
    model = Model(ctx, FORMS[form])
    model.synth(21)
    if form.startswith("gemma"):
        gemma_layer_scales(model)
    rng = np.random.default_rng(plen + n)
    a, b = (Session(model, n, plen + 60, kv_f16) for _ in range(2))
    for length in (plen, 45):
        prompts = rng.integers(0, model.cfg.vocab, size=(n, length)).astype(np.uint32)
        first = a.generate(prompts, 1)[:, 0]
        assert np.array_equal(first, step_by_step(b, prompts))
        compare(model, a, b, n, rng.integers(0, model.cfg.vocab, size=n), 2.0 ** -10 if kv_f16 else 1e-5)


@pytest.mark.parametrize("form", ["q6_k", "q5_k_no_groups", "q8_0_smol", "granite"])
def test_a_token_that_is_not_finite(ctx, form):
    """An embedding row of NaN, and one of infinities: rows that are not finite
    become NaN under a NaN scale in the pass.  The caches hold finite entries
    where the steps' do: before the token, and in other clients."""
    cfg = FORMS[form]
    model = Model(ctx, cfg)
    model.synth(3)
    be, bb = gguf.LAYOUT[cfg.encoding]
    embed = model.read_tensor(_lib.EMU_T_EMBED)
    rows = embed.reshape(cfg.vocab, -1, bb)
    for token, value in ((7, np.nan), (9, np.inf)):
        for at in D_AT[cfg.encoding][:1]:
            rows[token, 0, at:at + 2] = np.array([value], np.float16).view(np.uint8)
    model.write_tensor(_lib.EMU_T_EMBED, embed)
    prompts = np.random.default_rng(4).integers(10, cfg.vocab, size=(3, 90)).astype(np.uint32)
    prompts[0, 40], prompts[1, 70] = 7, 9
    a, b = (Session(model, 3, 92) for _ in range(2))
    a.generate(prompts, 1)
    step_by_step(b, prompts)
    for layer in range(cfg.layers):
        for values in (False, True):
            for c, bad in enumerate((40, 70, 90)):
                x, y = (s.read_kv(c, layer, values, 90) for s in (a, b))
                assert np.array_equal(np.isfinite(x), np.isfinite(y)), (layer, values, c)
                assert np.all(np.isfinite(y[:bad])) and not np.any(np.isfinite(y[bad:bad + 1]))
                assert np.linalg.norm(x[:bad] - y[:bad]) <= 2.0 ** -10 * np.linalg.norm(y[:bad])


def layer_in_64_bits(ctx, model, tokens, keys, values):
    """Layer 1's values of a Qwen3-style model: layer 0 over the keys and values
    that its cache holds, in 64 bits but for the f32 rotation table."""
    cfg = model.cfg
    H, hd, QW, KW = cfg.hidden, cfg.head_dim, cfg.q_width, cfg.kv_width
    blobs = [model.read_tensor(_lib.EMU_T_LAYER, layer) for layer in range(2)]
    at = 0

    def take(blob, rows, cols):
        nonlocal at
        size = rows * gguf.row_bytes(cfg.encoding, cols)
        raw, at = blob[at:at + size], at + size
        return npref.DECODERS[cfg.encoding](raw).reshape(rows, cols).astype(np.float64)

    def rms(x):
        return x / np.sqrt((x * x).mean(-1, keepdims=True) + cfg.eps)

    wq, wk, wv, wo = (take(blobs[0], r, c) for r, c in ((QW, H), (KW, H), (KW, H), (H, QW)))
    gate, up, down = (take(blobs[0], r, c) for r, c in ((cfg.ffn, H), (cfg.ffn, H), (H, cfg.ffn)))
    at = 0
    next_values = [take(blobs[1], r, H) for r in (QW, KW, KW)][2]
    h = npref.DECODERS[cfg.encoding](model.read_tensor(_lib.EMU_T_EMBED)).reshape(-1, H).astype(np.float64)[tokens]
    n = len(tokens)
    table = ctx.alloc(n * hd * 4)
    ctx.check(ctx.lib.emu_rope_table(ctx.h, n, hd, cfg.rope_theta, table.ptr), "rope")
    cos, sin = np.moveaxis(table.read(np.float32).reshape(n, 1, hd // 2, 2).astype(np.float64), 3, 0)
    q = rms((rms(h) @ wq.T).reshape(n, cfg.heads, hd))
    x, y = q[..., :hd // 2], q[..., hd // 2:]
    q = np.concatenate([x * cos - y * sin, y * cos + x * sin], -1)
    k, v = (np.repeat(m.reshape(n, cfg.kv_heads, hd).astype(np.float64), cfg.heads // cfg.kv_heads, 1) for m in (keys, values))
    s = np.einsum("thd,phd->htp", q, k) / np.sqrt(hd)
    s[:, np.triu(np.ones((n, n), bool), 1)] = -np.inf
    p = np.exp(s - s.max(-1, keepdims=True))
    out = np.einsum("htp,phd->thd", p / p.sum(-1, keepdims=True), v).reshape(n, QW)
    h = h + out @ wo.T
    x = rms(h)
    a = x @ gate.T
    h = h + (a / (1 + np.exp(-a)) * (x @ up.T)) @ down.T
    return rms(h) @ next_values.T


@pytest.mark.parametrize("kv_f16", [True, False])
@pytest.mark.parametrize("form", ["q6_k", "q5_k_no_groups", "q2_k_head256"])
def test_a_layer_against_64_bits(ctx, form, kv_f16):
    """Projections, attention and FFN of layer 0 together.  They were seen off
    by 3.5e-7 of the values; a low half dropped anywhere adds 1.6e-4 to
    2.4e-4 (the same layer in 64 bits with one operand rounded to a half).  Over an f16 cache that moves an
    entry to the neighbouring half with a chance of twice its error over a
    half's spacing, 2^-10 to 2^-11 of it: 0.4% of the entries at most, 35% and
    more with a low half dropped."""
    model = Model(ctx, replace(FORMS[form], layers=2))
    model.synth(12)
    tokens = np.random.default_rng(7).integers(0, model.cfg.vocab, size=75).astype(np.uint32)
    a = Session(model, 1, 76, kv_f16)
    a.generate(tokens[None], 1)
    n = 74  # the last token is a decode step
    want = layer_in_64_bits(ctx, model, tokens[:n], *(a.read_kv(0, 0, values, n) for values in (False, True)))
    got = a.read_kv(0, 1, True, n)
    if kv_f16:
        assert np.mean(got != want.astype(np.float16).astype(np.float32)) <= 0.01
    else:
        assert np.linalg.norm(got - want) <= 1e-6 * np.linalg.norm(want)


@pytest.mark.parametrize("form", ["q6_k", "q5_k_no_groups", "q2_k_head256", "q8_0_smol", "q8_0_half_stage"])
def test_products_against_64_bits(ctx, form):
    """Layer 0's values over an f32 cache are the v rows' product with the
    normalised embeddings, unrounded.  Bar: 1.7e-7 of the norm.  The halves
    leave about 6e-8; a 64-column stage's sum takes 12 matrix instructions of
    two roundings each (2.4e-8 sqrt(12) = 8e-8), and the 4 to 9 stages' sums
    5e-8: 1.1e-7 to 1.4e-7 together.  256 columns in one chain leave 1.9e-7."""
    cfg = FORMS[form]
    model = Model(ctx, cfg)
    model.synth(12)
    prompts = np.random.default_rng(7).integers(0, cfg.vocab, size=(2, 75)).astype(np.uint32)
    a = Session(model, 2, 77, kv_f16=False)
    a.generate(prompts, 1)
    rb = gguf.row_bytes(cfg.encoding, cfg.hidden)
    blob = model.read_tensor(_lib.EMU_T_LAYER, 0)[(cfg.q_width + cfg.kv_width) * rb:][:cfg.kv_width * rb]
    w, embed = (npref.DECODERS[cfg.encoding](raw).reshape(-1, cfg.hidden).astype(np.float64)
                for raw in (blob, model.read_tensor(_lib.EMU_T_EMBED)))
    for c in range(2):
        x = embed[prompts[c, :74]]  # the last token is a decode step
        want = x / np.sqrt((x * x).mean(1, keepdims=True) + cfg.eps) @ w.T
        got = a.read_kv(c, 0, True, 74).astype(np.float64)
        assert np.linalg.norm(got - want) <= 1.7e-7 * np.linalg.norm(want)


def test_products_of_a_row_with_one_large_value(ctx):
    """A normalised row with one column 2^20 times the others over zero
    weights.  The others keep what test_products_against_64_bits holds, down to
    2^-25 under the power of two that puts the largest into [2^14, 2^15): 2^-39
    of it in each, times the weights' norm."""
    cfg = FORMS["q8_0_smol"]
    model = Model(ctx, cfg)
    model.synth(12)
    rb = gguf.row_bytes(cfg.encoding, cfg.hidden)
    at = (cfg.q_width + cfg.kv_width) * rb
    layer = model.read_tensor(_lib.EMU_T_LAYER, 0)
    layer[at:at + cfg.kv_width * rb].reshape(cfg.kv_width, -1, 34)[:, 100 // 32, 2 + 100 % 32] = 0
    model.write_tensor(_lib.EMU_T_LAYER, layer, 0)
    gain = np.ones((cfg.layers, cfg.hidden), np.float32)
    gain[0, 100] = 2.0 ** 20
    model.write_tensor(_lib.EMU_T_ATTN_NORM, gain)
    prompts = np.random.default_rng(7).integers(0, cfg.vocab, size=(1, 75)).astype(np.uint32)
    a = Session(model, 1, 77, kv_f16=False)
    a.generate(prompts, 1)
    w = npref.DECODERS[cfg.encoding](layer[at:at + cfg.kv_width * rb]).reshape(-1, cfg.hidden).astype(np.float64)
    embed = npref.DECODERS[cfg.encoding](model.read_tensor(_lib.EMU_T_EMBED)).reshape(-1, cfg.hidden).astype(np.float64)
    x = embed[prompts[0, :74]]
    x = x / np.sqrt((x * x).mean(1, keepdims=True) + cfg.eps) * gain[0]
    want, got = x @ w.T, a.read_kv(0, 0, True, 74).astype(np.float64)
    for t in range(74):
        bar = 1.7e-7 * np.linalg.norm(want[t]) + 2.0 ** -39 * np.abs(x[t]).max() * np.linalg.norm(w)
        assert np.linalg.norm(got[t] - want[t]) <= bar, t


@pytest.mark.parametrize("ratio", [2.0 ** 10, 2.0 ** 20])
@pytest.mark.parametrize("form", ["q6_k", "q5_k_no_groups", "q2_k_head256", "q8_0_smol"])
def test_products_of_rows_with_one_large_block(ctx, form, ratio):
    """Value rows whose first block's d is 2^10 or 2^20 times the others', over
    activations that are zero there.  The others keep what
    test_products_against_64_bits holds, down to 2^-25 under the power of two
    that puts the row's bound (the block's d times the largest code) into [2^14,
    2^15): 2^-39 of the bound in each weight, times the code (32; Q8_0 128) where
    the block's multiplier carries it."""
    cfg = FORMS[form]
    be, bb = gguf.LAYOUT[cfg.encoding]
    model = Model(ctx, cfg)
    model.synth(12)
    rb = gguf.row_bytes(cfg.encoding, cfg.hidden)
    at = (cfg.q_width + cfg.kv_width) * rb
    layer = model.read_tensor(_lib.EMU_T_LAYER, 0)
    raw = layer[at:at + cfg.kv_width * rb]
    per = raw.reshape(cfg.kv_width, -1, bb)
    bound = np.zeros(cfg.kv_width)
    largest = {_lib.Q6_K: [4096], _lib.Q5_K: [1953, 63], _lib.Q2_K: [45, 15], _lib.Q8_0: [128]}[cfg.encoding]
    for d_at, code in zip(D_AT[cfg.encoding], largest):
        per[:, 1:, d_at:d_at + 2] = np.array([2.0 ** -12], np.float16).view(np.uint8)
        per[:, 0, d_at:d_at + 2] = np.array([2.0 ** -12 * ratio], np.float16).view(np.uint8)
        bound += code * 2.0 ** -12 * ratio
    model.write_tensor(_lib.EMU_T_LAYER, layer, 0)
    gain = np.ones((cfg.layers, cfg.hidden), np.float32)
    gain[0, :be] = 0.0
    model.write_tensor(_lib.EMU_T_ATTN_NORM, gain)
    prompts = np.random.default_rng(7).integers(0, model.cfg.vocab, size=(1, 75)).astype(np.uint32)
    a = Session(model, 1, 77, kv_f16=False)
    a.generate(prompts, 1)
    w = npref.DECODERS[cfg.encoding](raw).reshape(-1, cfg.hidden).astype(np.float64)
    embed = npref.DECODERS[cfg.encoding](model.read_tensor(_lib.EMU_T_EMBED)).reshape(-1, cfg.hidden).astype(np.float64)
    x = embed[prompts[0, :74]]
    x = x / np.sqrt((x * x).mean(1, keepdims=True) + cfg.eps) * gain[0]
    want, got = x @ w.T, a.read_kv(0, 0, True, 74).astype(np.float64)
    code = {_lib.Q6_K: 32, _lib.Q8_0: 128}.get(cfg.encoding, 1)
    floor = 2.0 ** -39 * code * bound * np.abs(x).sum(1, keepdims=True)
    assert np.linalg.norm(got - want) <= 1.7e-7 * np.linalg.norm(want) + np.linalg.norm(floor)


@pytest.mark.parametrize("form", ["q5_k_no_groups", "q2_k_head256"])
def test_queries_over_an_f32_cache_are_f32(ctx, form):
    """Two query dimensions 2^24 times the others, over keys that hold zeros
    there: the scores come from the others alone, and need all their bits.
    Layer 1's entries carry layer 0's products' rounding (7e-7 of them; a pair
    of halves under the head's largest would leave 6e-5)."""
    model = Model(ctx, FORMS[form])
    model.synth(12)
    hd, layers = model.cfg.head_dim, model.cfg.layers
    q_gain, k_gain = (np.ones((layers, hd), np.float32) for _ in range(2))
    q_gain[:, [5, 5 + hd // 2]] = 2.0 ** 24
    k_gain[:, [5, 5 + hd // 2]] = 0.0
    model.write_tensor(_lib.EMU_T_Q_NORM, q_gain)
    model.write_tensor(_lib.EMU_T_K_NORM, k_gain)
    prompts = np.random.default_rng(7).integers(0, model.cfg.vocab, size=(2, 75)).astype(np.uint32)
    a, b = (Session(model, 2, 77, kv_f16=False) for _ in range(2))
    a.generate(prompts, 1)
    step_by_step(b, prompts)
    for layer in range(layers):
        x, y = (s.read_kv(1, layer, True, 75) for s in (a, b))
        assert np.linalg.norm(x - y) <= 3e-6 * np.linalg.norm(y), layer


def test_prompts_longer_than_a_pass_after_a_replaced_client(ctx):
    """Eight clients of 300 tokens (two passes), one of them fresh while the
    others sit at position 40."""
    model = Model(ctx, replace(SMALL_SMOL, layers=2))
    model.synth(5)
    rng = np.random.default_rng(1)
    n, plen = 8, 300
    warm = rng.integers(0, model.cfg.vocab, size=(n, 40)).astype(np.uint32)
    prompts = rng.integers(0, model.cfg.vocab, size=(n, plen)).astype(np.uint32)
    a, b = (Session(model, n, 400) for _ in range(2))
    a.generate(warm, 1)
    step_by_step(b, warm)
    for s in (a, b):
        s.reset_client(3)
    a.generate(prompts, 1)
    step_by_step(b, prompts)
    assert list(a.positions()) == [340, 340, 340, 300, 340, 340, 340, 340]
    compare(model, a, b, n, prompts[:, 0])


def test_weights_written_after_a_prompt_are_the_ones_used(ctx):
    """The pass keeps a scale per weight row: rewriting a tensor with rows a
    thousand times larger must renew it."""
    model = Model(ctx, SMALL_SMOL)
    model.synth(5)
    prompts = np.random.default_rng(2).integers(0, model.cfg.vocab, size=(1, 40)).astype(np.uint32)
    Session(model, 1, 64).generate(prompts, 1)
    blob = model.read_tensor(_lib.EMU_T_LAYER, 0).reshape(-1, 34)
    d = blob[:, :2].copy().view(np.float16) * np.float16(1000.0)
    blob[:, :2] = d.view(np.uint8)
    model.write_tensor(_lib.EMU_T_LAYER, blob, 0)
    a, b = Session(model, 1, 64), Session(model, 1, 64)
    a.generate(prompts, 1)
    step_by_step(b, prompts)
    x, y = a.read_kv(0, 0, True, 40), b.read_kv(0, 0, True, 40)
    assert np.all(np.isfinite(y)) and np.linalg.norm(x - y) <= 2.0 ** -10 * np.linalg.norm(y)


D_AT = {_lib.Q6_K: [208], _lib.Q5_K: [0, 2], _lib.Q2_K: [80, 82], _lib.Q8_0: [0]}  # a block's f16 factors


def scale_rows(model, first, rows, factor):
    """Rows first .. first + rows - 1 of layer 0's q, k, v times `factor`."""
    enc = model.cfg.encoding
    be, bb = gguf.LAYOUT[enc]
    blob = model.read_tensor(_lib.EMU_T_LAYER, 0)
    rb = model.cfg.hidden // be * bb
    part = blob[first * rb:(first + rows) * rb].reshape(-1, bb)
    for at in D_AT[enc]:
        d = (part[:, at:at + 2].copy().view(np.float16).astype(np.float64) * factor).astype(np.float16)
        assert np.all(np.isfinite(d))
        part[:, at:at + 2] = d.view(np.uint8)
    model.write_tensor(_lib.EMU_T_LAYER, blob, 0)


@pytest.mark.parametrize("what", ["keys", "values"])
@pytest.mark.parametrize("form", ["q6_k", "q5_k_no_groups", "q2_k_head256"])
def test_cache_entries_that_overflow_f16(ctx, form, what):
    """A key or value past f16's range is infinite in the cache.  A query whose
    score with such a key is -inf passes over it; where the steps give a
    finite row the pass does, and the same one, and nowhere else."""
    cfg = replace(FORMS[form], layers=2, heads=FORMS[form].kv_heads)
    model = Model(ctx, cfg)
    model.synth(3)
    n, plen, hd = 2, 150, cfg.head_dim
    prompts = np.random.default_rng(8).integers(0, cfg.vocab, size=(n, plen)).astype(np.uint32)
    a, b = (Session(model, n, plen + 2) for _ in range(2))
    if what == "keys":  # one normalised dimension of layer 0's keys, small in its queries
        q_gain, k_gain = (np.ones((cfg.layers, hd), np.float32) for _ in range(2))
        k_gain[0, 5] = 65504 / (1.6 if cfg.kv_heads == 1 else 2.3)
        q_gain[0, [5, 5 + hd // 2]] = 1e-5
        model.write_tensor(_lib.EMU_T_K_NORM, k_gain)
        model.write_tensor(_lib.EMU_T_Q_NORM, q_gain)
    else:  # one value row, past the range for its largest token alone
        step_by_step(b, prompts)
        v = b.read_kv(0, 0, True, plen)[:, 3]
        b.reset()
        top = int(np.argmax(np.abs(v)))
        prompts[0, [top, 80]] = prompts[0, [80, top]]
        scale_rows(model, cfg.q_width + cfg.kv_width + 3, 1, 65504 * 1.02 / np.abs(v).max())
    a.generate(prompts, 1)
    step_by_step(b, prompts)
    after = 0  # rows of layer 1 that stay finite behind layer 0's first infinity
    for c in range(n):
        first = plen
        for layer in range(2):
            for values in (False, True):
                x, y = (s.read_kv(c, layer, values, plen) for s in (a, b))
                assert np.array_equal(np.isfinite(x), np.isfinite(y)), (layer, values, c)
                fine = np.all(np.isfinite(y), axis=1)
                assert np.linalg.norm(x[fine] - y[fine]) <= 2.0 ** -10 * np.linalg.norm(y[fine])
                if layer == 0 and values == (what == "values"):
                    first = plen if fine.all() else int(np.argmin(fine))
                if layer == 1 and first < plen:
                    after += int(np.sum(fine[first:]))
        assert first > 0 and (c or first < plen)
    assert (after > 0) == (what == "keys")


def test_the_workspace_goes_with_the_model(ctx):
    """A long prompt's workspace (about 100 MB here) is held while the model lives,
    not until the context ends."""
    free, total = C.c_size_t(), C.c_size_t()
    hip = C.CDLL(ctx.lib._name)  # the HIP runtime it is linked to

    def left():
        ctx.sync()
        assert hip.hipMemGetInfo(C.byref(free), C.byref(total)) == 0
        return free.value

    def run(plen):
        model = Model(ctx, replace(SMALL_SMOL, layers=1))
        model.synth(5)
        sess = Session(model, 8, 264)
        sess.generate(np.ones((8, plen), np.uint32), 1)
        held = left()
        sess.close()
        model.close()
        return held

    run(4)  # whatever the runtime keeps from a first run
    before = left()
    held = run(257)
    assert before - held > 64 << 20
    assert left() >= before - (16 << 20)


@pytest.mark.parametrize("form", ["q8_0_smol", "granite", "gemma_window"])
def test_resident_bytes_count_the_row_scales(ctx, form):
    cfg = FORMS[form]
    model = Model(ctx, cfg)
    model.synth(5)
    sess = Session(model, 1, 16)
    sess.decode_step([1])
    before = model.resident_bytes()
    sess.generate(np.ones((1, 8), np.uint32), 1)
    rows = cfg.q_width + 2 * cfg.kv_width + cfg.hidden
    ff = cfg.shared_ff if cfg.n_experts else cfg.ffn
    rows += (2 * ff + cfg.hidden) if ff else 0
    rows += cfg.n_experts * (1 + 2 * cfg.expert_ff + cfg.hidden)
    assert model.resident_bytes() - before == 4 * rows * cfg.layers


@pytest.mark.parametrize("kv_f16", [True, False])
@pytest.mark.parametrize("form", ["q6_k", "q8_0_smol", "granite_deep", "olmoe_deep", "gemma_deep"])
def test_a_prompt_in_any_company(ctx, form, kv_f16):
    """A client's cached rows are the same bits alone (one pass of 299 tokens)
    and among eight (two passes, of 256 and 43)."""
    model = Model(ctx, FORMS[form])
    model.synth(9)
    if form.startswith("gemma"):
        gemma_layer_scales(model)
    prompts = np.random.default_rng(6).integers(0, model.cfg.vocab, size=(8, 300)).astype(np.uint32)
    a, b = Session(model, 8, 304, kv_f16), Session(model, 1, 304, kv_f16)
    a.generate(prompts, 1)
    for c in (0, 5):
        b.reset()
        b.generate(prompts[c:c + 1], 1)
        for layer in range(model.cfg.layers):
            for values in (False, True):
                x, y = a.read_kv(c, layer, values, 299), b.read_kv(0, layer, values, 299)
                assert np.array_equal(x.view(np.uint32), y.view(np.uint32)), (c, layer, values)
