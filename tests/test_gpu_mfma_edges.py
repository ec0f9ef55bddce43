"""The matrix-core propagation where a column of its products has no source in a tile, on
grids of small voxels: the path-table entries read there (up to 1/pitch^2) belong to other
sources than the exponents that scale them, which are 0 beyond the coupling threshold and
where the path integral across the grid underflows.  And the bits that its operands keep.

Tolerances: max |difference| / max |reference|, the mixed operators' 1e-5; a pencil beam's
first term, whose sums are short, root mean square 4 x 2^-24 (a rounding to 24 bits of the
table, the harmonics, the coefficients and the weighted projections).
"""
import numpy as np
import pytest

from doi_amd import rte
from tests.helpers import bounds_for, hetero_maps, rel_max

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("shape,thr,mus", [((32, 32, 32), 0.04, 1.0), ((4, 40, 105), 0.0, 95.0)])
@pytest.mark.parametrize("L", [4, 5])
def test_columns_without_a_source(ctx, L, shape, thr, mus):
    bounds = bounds_for(shape, d=(0.01, 0.01, 0.01))
    ma, ms = hetero_maps(shape, seed=31, mua=0.05, mus=mus, sigma=0.02)
    W = np.random.default_rng(L).standard_normal(((L + 1) ** 2, int(np.prod(shape))))
    print("columns without a source", L, shape, thr, flush=True)
    ref, got, got32 = (ctx.propagate(shape, bounds, ma, ms, 0.9, W, L, prop_thresh=thr, precision=p)
                       for p in (rte.PREC_FP64, rte.PREC_MIXED, rte.PREC_FP32))
    assert np.isfinite(got).all() and np.isfinite(got32).all()
    assert rel_max(got, ref) < 1e-5
    assert rel_max(got32, ref) < 1e-5


def test_short_sums_keep_24_bits(ctx):
    shape, L, g = (32, 32, 32), 5, 0.8
    bounds, N = bounds_for(shape), 32 ** 3
    ma, ms = np.full(N, 0.25), np.full(N, 4.75)
    W = ctx.source(shape, bounds, ma, ms, g, (0.05, 0.05, 0.1, 1.0), L)[0]
    print("short sums", flush=True)
    ref, got = (ctx.propagate(shape, bounds, ma, ms, g, W, L, precision=p) for p in (rte.PREC_FP64, rte.PREC_MIXED))
    assert np.sqrt(np.mean((got - ref) ** 2) / np.mean(ref ** 2)) < 4 * 2.0 ** -24
