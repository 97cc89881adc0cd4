"""The ring tiles of the dense matmul (matmul_ring.hip): every compiled shape, forced by the
ring tactic, against the oracle and against the 128 x 128 tiles (tactic ring=0) on the same f16
rows, at the edges of their tiles.

Bars: 3e-3 relative L2 against the oracle's f32 product (f16 operands, as the matmul tests); the
same operands summed in another f32 order differ by at most sqrt(n_in) roundings of 2^-24 each
way, 2 * sqrt(n_in) * 2^-24 of the result's norm.  Q8_0 without the ring converts its rows in
the tile, in the same f16 values: past f16's range, both hold each run of 128 values of a row on
an exponent of its own."""
import numpy as np
import pytest

from helpers import Setup, rel_l2, tactics
from oracle import skyla_oracle as so
from skyla_hip import engine as E
from skyla_hip import synth
from test_gpu_matmul import GUARD, _run

pytestmark = pytest.mark.gpu

SHAPES = ["4_1_4_4", "4_1_4_3", "4_2_2_4", "1_4_2_3"]


def _both(ctx, dtype, n_in, n_out, n_tok, accum, form):
    with tactics(ring=form):
        got, want = _run(ctx, dtype, n_in, n_out, n_tok, accum=accum, tag="mm-ring")
    with tactics(ring=0):
        plain, _ = _run(ctx, dtype, n_in, n_out, n_tok, accum=accum, tag="mm-ring")
    assert rel_l2(got, want) <= GUARD
    assert rel_l2(got, plain) <= 2 * np.sqrt(n_in) * 2.0 ** -24


@pytest.mark.parametrize("shape", SHAPES)
@pytest.mark.parametrize("dtype,n_in,n_out,n_tok,accum,split", [
    (E.DType.Q4K, 256, 130, 1, False, 1), (E.DType.Q4K, 1280, 200, 37, True, 2), (E.DType.Q4K, 2048, 384, 129, True, 4),
    (E.DType.Q6K, 256, 31, 33, True, 1), (E.DType.Q6K, 768, 130, 100, False, 3), (E.DType.Q6K, 2304, 256, 70, True, 2),
    (E.DType.Q8_0, 32, 64, 5, False, 1), (E.DType.Q8_0, 1056, 140, 70, True, 2), (E.DType.Q8_0, 1504, 33, 200, True, 1),
])
def test_ring_shapes(ctx, dtype, n_in, n_out, n_tok, accum, split, shape):
    """Ragged rows, tokens and (Q8_0) columns; one, two and four live token blocks; K groups of
    unequal length and empty ones; K splits; ACCUM."""
    _both(ctx, dtype, n_in, n_out, n_tok, accum, f"{shape}_{split}")


@pytest.mark.parametrize("dtype,n_in,n_out,n_tok", [
    (E.DType.Q4K, 4096, 12288, 384), (E.DType.Q4K, 4096, 12288, 128), (E.DType.Q6K, 4096, 4096, 512),
    (E.DType.Q4K, 4096, 6144, 128), (E.DType.Q4K, 4096, 4096, 100), (E.DType.Q8_0, 3072, 1024, 60),
    (E.DType.Q8_0, 2080, 20000, 200), (E.DType.Q6K, 256, 500, 9), (E.DType.Q6K, 8192, 1000, 60),
    (E.DType.Q4K, 12288, 5504, 128), (E.DType.Q6K, 6400, 8200, 100), (E.DType.Q8_0, 5120, 9000, 128),
    (E.DType.Q8_0, 1024, 8192, 128),
])
def test_ring_rule(ctx, dtype, n_in, n_out, n_tok):
    """The shapes the runtime's rule picks, one launch size of each of its lines."""
    _both(ctx, dtype, n_in, n_out, n_tok, True, 1)


@pytest.mark.parametrize("shape", SHAPES)
@pytest.mark.parametrize("n_in,n_out,n_tok,split", [(1056, 140, 70, 1), (1504, 33, 200, 2), (2048, 130, 129, 4),
                                                    (96, 64, 5, 1)])
def test_ring_q8_range_per_run(ctx, n_in, n_out, n_tok, split, shape):
    """A third of the tokens hold one value of 1e12 alone in its run of 128, where every weight
    is zero (their other runs must keep their bits), a third a run of values near 1e6 or all of
    them near 4e4, the rest none past 2^15."""
    tag = f"{n_in}-{n_out}"
    data = synth.matrix("mm-ring-range", tag, E.DType.Q8_0, n_in, n_out)
    runs = -(-n_in // 128)
    q = data.reshape(n_out, n_in // 32, 34)[:, :, 2:]
    q[:, ::4, 5] = 0  # column 5 of every run
    g = synth.rng("mm-ring-range", f"x-{tag}-{n_tok}")
    x = g.standard_normal((n_tok, n_in)).astype(np.float32)
    for t in range(n_tok):
        r = 128 * int(g.integers(runs))
        if t % 3 == 0:
            x[t, r: r + 128] = 0
            x[t, r + 5] = 1e12
        elif t % 6 == 1:
            x[t, r: r + 128] *= 1e6
        elif t % 6 == 4:
            x[t] *= 4e4
    got = {}
    for form in (f"{shape}_{split}", "0"):
        with tactics(ring=form):
            s = Setup(ctx, [(E.DType.Q8_0, n_in, n_out, data)], n_in, n_out, rows=n_tok)
            try:
                s.set_x(x)
                s.matmul(0, n_tok)
                got[form] = s.y(n_tok, n_out)
            finally:
                s.free()
    want = so.matmul(int(E.DType.Q8_0), data, n_in, n_out, x)
    for t in range(n_tok):
        if not want[t].any():  # (a row of one run, all of it zero weights)
            assert not got[f"{shape}_{split}"][t].any()
            continue
        assert rel_l2(got[f"{shape}_{split}"][t], want[t]) <= GUARD, t
        assert rel_l2(got[f"{shape}_{split}"][t], got["0"][t]) <= 2 * np.sqrt(n_in) * 2.0 ** -24, t


@pytest.mark.parametrize("dtype,n_in,n_out,n_tok", [(E.DType.Q8_0, 1024, 256, 60), (E.DType.Q4K, 2048, 256, 60),
                                                    (E.DType.Q8_0, 3072, 2048, 128), (E.DType.Q6K, 4096, 4096, 128)])
def test_ring_splitk_off_sums_whole(ctx, dtype, n_in, n_out, n_tok):
    """Tactic splitk=0: every row in one sum, whatever the type (the bits of the unsplit wide
    shape); by default these launches split K inside the workgroup or over several."""
    got = {}
    for tac in ({}, {"splitk": 0}, {"ring": "4_1_4_4_1"}):
        with tactics(**tac):
            got[tuple(tac)] = _run(ctx, dtype, n_in, n_out, n_tok, tag="mm-ring")[0].view(np.uint32)
    assert np.array_equal(got["splitk",], got["ring",])
    assert not np.array_equal(got[()], got["ring",])
