"""The batched attention on the matrix cores (attention.hip, attention_rows): 16 query rows a
wave, so a group's tokens straddle splits and end inside a group.  Against attention in 64 bits
over the same cache entries, and with non-finite value rows, which only tokens at or past
their position may see."""
import numpy as np
import pytest

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


def _run(ctx, precision, heads, pos0, n_tok, spoil=None):
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
