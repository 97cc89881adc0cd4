"""The Q8_0 matvec without staging (matvec_q8_0_ks): every compiled shape (one to four waves a
row, 2, 4 or 8 rows a wave) at the edges of its rows and columns, plain, accumulating, with the
RMSNorm and with the SiLU folded in, against the oracle and in float64; and the LDS-staged
form that longer rows take (and, with q8_ks=0, these).

Bar: twice the distance of a plain f32 reordering of the same product (helpers.f32_reorder_bar);
the folded forms add the vector's own f32 roundings (a sum of squares, a division, an
exponential, two products: at most 8 ulp, 8 * 2^-24) to it."""
import numpy as np
import pytest

from helpers import Setup, f32_reorder_bar, rel_l2, tactics
from oracle import skyla_oracle as so
from skyla_hip import engine as E
from skyla_hip import synth

pytestmark = pytest.mark.gpu

SIZES = [(32, 1), (1024, 70), (1056, 33), (2048, 255), (2976, 13), (3072, 301), (4096, 64), (4128, 20)]


@pytest.mark.parametrize("rows", ["0", "1", "2", "4", "8"])
@pytest.mark.parametrize("form", [None, "accum", "norm", "silu"])
@pytest.mark.parametrize("n_in,n_out", SIZES)
def test_q8_ks_forms(ctx, n_in, n_out, form, rows):
    _form(ctx, n_in, n_out, form, rows)


# one and two staging passes of 8192 values, either side of the lines at 2048 rows and, with
# q8_small's variant, of its four rows a workgroup
@pytest.mark.parametrize("form", [None, "accum", "norm", "silu"])
@pytest.mark.parametrize("n_in,n_out", [(4608, 33), (8192, 2047), (8224, 301), (12288, 1025), (4608, 2049),
                                        (12288, 2101)])
def test_q8_staged_rows(ctx, n_in, n_out, form):
    _form(ctx, n_in, n_out, form, None)


def _form(ctx, n_in, n_out, form, rows):
    g = synth.rng("q8-ks", f"{n_in}-{n_out}-{form}")
    data = synth.matrix("q8-ks", f"{n_in}-{n_out}", E.DType.Q8_0, n_in, n_out)
    x, aux = (g.standard_normal(n_in).astype(np.float32) for _ in range(2))
    y0 = g.standard_normal(n_out).astype(np.float32) if form in ("accum", "silu") else np.zeros(n_out, np.float32)
    c = E.Config(n_embd=n_in, eps=1e-6)
    with tactics(q8_ks=rows):
        s = Setup(ctx, [(E.DType.Q8_0, n_in, n_out, data)], n_in, n_out, extra_f32=n_in)
        k = E.Kernels(ctx, s.weights, s.arena, fuse="all")
    try:
        s.arena.as_f32()[s.extra_off: s.extra_off + n_in] = aux
        s.set_x(x)
        s.set_y(y0)
        fused = form if form in ("norm", "silu") else None
        s.run(lambda r: E.Graph(r, k, None, c, False).matvec(
            s.q[0], (s.x_off, 0), (s.y_off, 0), form in ("accum", "silu"), False, form=fused,
            aux=s.extra_off if fused else 0))
        got = s.y(1, n_out)[0].astype(np.float64) - y0
    finally:
        s.free()
    v = x.astype(np.float64)
    if form == "norm":
        v = v / np.sqrt((v * v).mean() + 1e-6) * aux
    elif form == "silu":
        v = v / (1 + np.exp(-v)) * aux
    w = so.dequantize(int(E.DType.Q8_0), data, n_in * n_out).reshape(n_out, n_in).astype(np.float64)
    xf = v.astype(np.float32)
    bar = f32_reorder_bar(E.DType.Q8_0, data, n_in, n_out, xf, so.matvec(int(E.DType.Q8_0), data, n_in, n_out, xf))
    # (y0 + product rounds once more to y0's magnitude)
    bar += 8 * 2.0 ** -24 + 2.0 ** -24 * np.linalg.norm(y0) / max(np.linalg.norm(w @ v), 1e-30)
    assert rel_l2(got, w @ v) <= bar


def _plain(ctx, n_in, n_out, **tac):
    data = synth.matrix("q8-ks-tactics", f"{n_in}-{n_out}", E.DType.Q8_0, n_in, n_out)
    x = synth.activations("q8-ks-tactics", f"x-{n_in}", n_in)
    with tactics(**tac):
        s = Setup(ctx, [(E.DType.Q8_0, n_in, n_out, data)], n_in, n_out)
        try:
            s.set_x(x)
            s.matvec(0)
            return s.y(1, n_out)[0].view(np.uint32).copy()
        finally:
            s.free()


def test_ks_off_keeps_q8_ks(ctx):
    """Tactic ks is the K-quants': ks=0 leaves a Q8_0 launch on the form without staging."""
    default = _plain(ctx, 3072, 500)
    assert np.array_equal(_plain(ctx, 3072, 500, ks=0), default)
    assert not np.array_equal(_plain(ctx, 3072, 500, q8_ks=0), default)


@pytest.mark.parametrize("entry,n_out,taken", [({"variant": "4_1_64"}, 500, True), ({"variant": "4_1_64"}, 3000, True),
                                               ({"q8_small": "4_1_64"}, 500, True), ({"q8_small": ""}, 500, True),
                                               ({"q8_small": "4_1_64"}, 2048, False)])
def test_given_variants_act(ctx, entry, n_out, taken):
    """A variant or q8_small entry takes the Q8_0 launches that it names from the form without
    staging (the bits with q8_ks=0), and no others."""
    got, staged = _plain(ctx, 3072, n_out, **entry), _plain(ctx, 3072, n_out, q8_ks=0, **entry)
    assert np.array_equal(got, staged) == taken
    assert np.array_equal(got, _plain(ctx, 3072, n_out)) == (not taken)
