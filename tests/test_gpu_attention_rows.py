"""The batched attention on the matrix cores (attention.hip, attention_rows): 16 query rows a
wave, so a group's tokens straddle splits and end inside a group.  Against attention in 64 bits
over the same cache entries, with non-finite value rows, which only tokens at or past their
position may see, with 8-bit scales too far apart for one shift, and against the f32 form's
(tactic attn_rows=0) partials, whose bits it keeps."""
import numpy as np
import pytest

from helpers import tactics
from test_gpu_decode import P, Bench, _cache, _cfg

pytestmark = pytest.mark.gpu


def _attention64(q, K, V, pos0, n_head, n_kv):
    out, rep = np.zeros(q.shape), n_head // n_kv
    K, V = K.astype(np.float64).reshape(len(K), n_kv, 128), V.astype(np.float64).reshape(len(V), n_kv, 128)
    for t in range(len(q)):
        m = pos0 + t + 1
        for h in range(n_head):
            s = K[:m, h // rep] @ q[t, 128 * h: 128 * (h + 1)].astype(np.float64) / np.sqrt(128.0)
            e = np.exp(s - s.max())
            out[t, 128 * h: 128 * (h + 1)] = e @ V[:m, h // rep] / e.sum()
    return out


def _run(ctx, precision, heads, pos0, n_tok, spoil=None, tower=None):
    c = _cfg(512, *heads)
    g = np.random.default_rng(100 * n_tok + pos0)
    n_pos = pos0 + n_tok
    b = Bench(ctx, c, precision, {"one": np.ones(128, np.float32)}, max_ctx=max(256, n_pos))
    try:
        a, kvl, kv_dim = b.a, b.a.kv_layout, c.n_head_kv * 128
        h = a.kv.host()
        for off, scales, q8 in ((kvl.keys(0), kvl.key_scales(0), precision.keys_q8),
                                (kvl.values(0), kvl.value_scales(0), precision.values_q8)):
            n = n_pos * kv_dim
            if q8:
                h.view(np.int8)[off: off + n] = g.integers(-127, 128, n)
                h.view("<f2")[scales: scales + n // 32] = np.exp(g.uniform(-9, -3, n // 32)).astype(np.float16)
            else:
                h.view("<f2")[off: off + n] = g.standard_normal(n).astype(np.float16)
        if spoil is not None:  # one value (8-bit: its block's scale) of the first head is infinite
            if precision.values_q8:
                h.view("<f2")[kvl.value_scales(0) + spoil * kv_dim // 32] = np.inf
                h.view(np.int8)[kvl.values(0) + spoil * kv_dim: kvl.values(0) + spoil * kv_dim + 32] = 5
            else:
                h.view("<f2")[kvl.values(0) + spoil * kv_dim] = np.inf
        if tower is not None:  # one position's values, of every head, tower over the others
            if precision.values_q8:
                h.view("<f2")[kvl.value_scales(0): kvl.value_scales(0) + n_pos * kv_dim // 32] *= np.float16(2.0 ** -6)
                h.view("<f2")[kvl.value_scales(0) + tower * kv_dim // 32:][: kv_dim // 32] = 30000.0
            else:
                h.view("<f2")[kvl.values(0) + tower * kv_dim:][: kv_dim] = 60000.0
        a.kv.upload()
        q = (g.standard_normal((n_tok, c.n_head * 128)) * 0.3).astype(np.float32)
        b.put_rows(a.q, a.s_q, q)
        a.set_ctl(0, pos0, n_tok)
        a.buffer.upload()
        b.run(lambda gr: gr.attend(0))
        a.buffer.download()
        got = b.rows(a.attn, a.s_attn, n_tok, c.n_head * 128).copy()
        Kd, Vd = _cache(b, 0, n_pos)
        with np.errstate(invalid="ignore"):
            return got, _attention64(q, Kd, Vd, pos0, c.n_head, c.n_head_kv)
    finally:
        b.free()


# f32 sums of m <= 300 terms with products exact to 2^-22: a relative 2e-6, as the decode form
@pytest.mark.parametrize("precision", list(P))
@pytest.mark.parametrize("pos0,n_tok", [(0, 2), (0, 17), (3, 128), (63, 16), (190, 45)])
@pytest.mark.parametrize("heads", [(4, 4), (4, 2), (8, 2), (8, 1)])
def test_attention_rows_against_64_bits(ctx, precision, pos0, n_tok, heads):
    got, want = _run(ctx, precision, heads, pos0, n_tok)
    for t in range(n_tok):
        assert np.linalg.norm(got[t] - want[t]) < 2e-6 * np.linalg.norm(want[t]), t


@pytest.mark.parametrize("precision", list(P))
def test_attention_rows_infinite_value(ctx, precision):
    """Position 20 of 30 holds an infinite value: tokens before it stay finite and right, tokens
    from it on are infinite there and right elsewhere."""
    got, want = _run(ctx, precision, (8, 2), 10, 20, spoil=20)
    fin = np.isfinite(want)
    assert fin[:10].all() and not fin[10:].all(axis=1).any()
    assert np.array_equal(np.isposinf(got), np.isposinf(want)) and np.array_equal(np.isnan(got), np.isnan(want))
    for t in range(20):
        d = np.where(fin[t], got[t] - np.where(fin[t], want[t], 0), 0)
        assert np.linalg.norm(d) < 2e-6 * np.linalg.norm(want[t][fin[t]]), t


@pytest.mark.parametrize("precision", list(P))
@pytest.mark.parametrize("heads", [(4, 4), (8, 2), (8, 1)])
def test_attention_rows_scales_far_apart(ctx, precision, heads):
    """Position 41 of 50 holds values some 2^24 above every other: the tokens before it, in the
    same groups and split, keep their own values' precision."""
    got, want = _run(ctx, precision, heads, 20, 30, tower=41)
    for t in range(30):
        assert np.linalg.norm(got[t] - want[t]) < 2e-6 * np.linalg.norm(want[t]), t


def _few_bits():
    """Query values that the score's scale 1/sqrt(128) takes to numbers of 8 bits exactly as f32
    rounds (among three neighbours one does while their steps are finer than the product's)."""
    scale = np.float32(1.0) / np.sqrt(np.float32(128.0))
    out = []
    for t in np.arange(129, 181, dtype=np.float32) / 256:
        q = np.float32(t / scale)
        near = [v for v in (q, np.nextafter(q, np.float32(0)), np.nextafter(q, np.float32(99))) if v * scale == t]
        assert near
        out.append(near[0])
    return np.array(out, np.float32)


def _partials(ctx, precision, heads, pos0, n_tok, form):
    """The (m, l, sum e v) partials of one attention whose scores are single exact products
    (one-hot queries of few bits, 8-bit key scales of powers of two) and whose value columns hold one nonzero
    position a split, so that a form's sums show its e and its e v alone."""
    c = _cfg(512, *heads)
    g = np.random.default_rng(n_tok)
    n_pos, d = pos0 + n_tok, c.n_head_kv * 128
    b = None
    with tactics(attn_rows=form):
        b = Bench(ctx, c, precision, {"one": np.ones(128, np.float32)}, max_ctx=max(256, n_pos))
    try:
        a, kvl = b.a, b.a.kv_layout
        h, n = a.kv.host(), n_pos * d
        if precision.keys_q8:
            h.view(np.int8)[kvl.keys(0): kvl.keys(0) + n] = g.integers(-100, 101, n)
            h.view("<f2")[kvl.key_scales(0): kvl.key_scales(0) + n // 32] = 2.0 ** -4
        else:
            h.view("<f2")[kvl.keys(0): kvl.keys(0) + n] = g.uniform(-6, 6, n).astype(np.float16)
        on = np.arange(n_pos)[:, None] % 64 == np.arange(d)[None, :] % 64
        if precision.values_q8:
            h.view(np.int8)[kvl.values(0): kvl.values(0) + n] = (g.integers(1, 128, on.shape) * on).ravel()
            h.view("<f2")[kvl.value_scales(0): kvl.value_scales(0) + n // 32] = g.uniform(1e-3, 1e-2, n // 32)
        else:
            h.view("<f2")[kvl.values(0): kvl.values(0) + n] = (g.uniform(0.5, 4, on.shape) * on).ravel()
        a.kv.upload()
        # (8 bits by at most 11 of a key: every score is one exact product)
        q = np.zeros((n_tok, c.n_head, 128), np.float32)
        q[..., 7] = g.choice(_few_bits(), q.shape[:2])
        b.put_rows(a.q, a.s_q, q.reshape(n_tok, -1))
        a.set_ctl(0, pos0, n_tok)
        a.buffer.upload()
        b.run(lambda gr: gr.attend(0))
        a.buffer.download()
        splits = -(-n_pos // 64)
        n_split = a.s_part // (c.n_head * 130)
        p = b.rows(a.part, a.s_part, n_tok, c.n_head * n_split * 130).reshape(n_tok, c.n_head, n_split, 130)
        return [p[t, :, s].copy() for t in range(n_tok) for s in range(splits) if 64 * s <= pos0 + t]
    finally:
        b.free()


@pytest.mark.parametrize("precision", list(P))
@pytest.mark.parametrize("heads", [(4, 4), (4, 2), (8, 2), (8, 1)])
def test_attention_rows_keeps_the_bits_of_e(ctx, precision, heads):
    """Each sum is one e v: the f32 form rounds it once (2^-24), the matrix cores' sums of its
    parts twice more in their last two products (2^-23): 1.5 * 2^-23 between them.  An e of 22
    bits, or products short of their low parts, pass that bar."""
    rows, plain = (_partials(ctx, precision, heads, 70, 21, form) for form in ("1", "0"))
    worst = 0.0
    for got, want in zip(rows, plain):
        assert np.array_equal(got[:, 0], want[:, 0])  # m: the same score
        assert np.allclose(got[:, 1], want[:, 1], rtol=64 * 2.0 ** -24, atol=0)
        g, w = got[:, 2:].astype(np.float64), want[:, 2:].astype(np.float64)
        assert np.array_equal(g == 0, w == 0)
        worst = max(worst, float(np.max(np.abs(g - w)[w != 0] / np.abs(w[w != 0]), initial=0.0)))
    print(f"worst {worst * 2 ** 24:.2f} * 2^-24")
    assert worst <= 1.5 * 2.0 ** -23
