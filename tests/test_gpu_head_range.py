"""GPU: the heads over the whole range of fp32 hidden values and bf16 weights. Hidden rows from 1 down to
the smallest subnormals, weights of both extremes, in every form the rule picks: each output within the
bound of any fp32 evaluation, gamma_K sum |x w| and half a unit of the smallest subnormal (2^-150) per
operation."""
import numpy as np
import pytest

from oracle.head_np import head_bound, head_exact, head_int8_bound, head_int8_exact, pack_int8
from test_gpu_head import _bf16, _run, _run_int8

pytestmark = pytest.mark.gpu

# the VALU form, split-K 16 x 16, 16 x 48 and 32 x 96, tiled 32 x 64 and 64 x 128
SHAPES = [(2, 1024, 600), (5, 1024, 600), (64, 1024, 3072), (256, 512, 3072), (400, 72, 2050), (1100, 264, 3001)]
UNDERFLOW = 2.0**-150


def _hidden(rng, rows, k):
    """Normal values, row r scaled by 2^-(5 r mod 150): exact down to the subnormals they are rounded to."""
    e = -(5 * np.arange(rows) % 150)
    return np.ldexp(rng.standard_normal((rows, k)), e[:, None]).astype(np.float32)


@pytest.mark.parametrize("wexp", [100, 0, -60, -132])
@pytest.mark.parametrize("rows,k,n", SHAPES)
def test_head_over_the_range_of_values(ctx, rows, k, n, wexp):
    rng = np.random.default_rng(rows + k + n)
    x = _hidden(rng, rows, k)
    w = _bf16(np.ldexp(rng.standard_normal((n, k)), wexp))
    if wexp < 0:  # hidden values that bring the products of small weights back into range
        x = np.ldexp(x.astype(np.float64), min(-wexp, 85)).astype(np.float32)
    got = _run(ctx, x, w)
    err, bound = np.abs(got - head_exact(x, w)), head_bound(x, w) + 2 * k * UNDERFLOW
    assert np.all(err <= bound), f"max err/bound {np.max(err / bound):.3f}, rows {np.nonzero((err > bound).any(1))[0][:8]}"


@pytest.mark.parametrize("rows,k,n", SHAPES)
def test_head_int8_over_the_range_of_values(ctx, rows, k, n):
    rng = np.random.default_rng(rows + k + n)
    x = _hidden(rng, rows, k)
    q, scale = pack_int8(_bf16(np.ldexp(rng.standard_normal((n, k)), 100)))
    got = _run_int8(ctx, x, q, scale)
    # the dot's own underflow, scaled
    err = np.abs(got - head_int8_exact(x, q, scale))
    bound = head_int8_bound(x, q, scale) + 2 * (k + 1) * UNDERFLOW * np.maximum(scale, 1).astype(np.float64)[None, :]
    assert np.all(err <= bound), f"max err/bound {np.max(err / bound):.3f}, rows {np.nonzero((err > bound).any(1))[0][:8]}"
