"""The ring tiles of the dense matmul (matmul_ring.hip): every compiled shape, forced by the
ring tactic, against the oracle and against the 128 x 128 tiles (tactic ring=0) on the same f16
rows, at the edges of their tiles.

Bars: 3e-3 relative L2 against the oracle's f32 product (f16 operands, as the matmul tests); the
same operands summed in another f32 order differ by at most sqrt(n_in) roundings of 2^-24 each
way, 2 * sqrt(n_in) * 2^-24 of the result's norm.  Q8_0 without the ring converts its rows in
the tile, in the same f16 values."""
import numpy as np
import pytest

from helpers import rel_l2, tactics
from skyla_hip import engine as E
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
    (E.DType.Q8_0, 2080, 20000, 200), (E.DType.Q6K, 256, 500, 9),
])
def test_ring_rule(ctx, dtype, n_in, n_out, n_tok):
    """The shapes the runtime's rule picks, one launch size of each of its lines."""
    _both(ctx, dtype, n_in, n_out, n_tok, True, 1)
