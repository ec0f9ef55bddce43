"""The matrix-core propagation (FP32, L = 4 and 5, large grids) against the FP64 path, at
the edges of its tiles: grids that are not whole bricks on each axis, flat and long ones
(few translations in z or x), a coupling threshold that leaves brick columns out, and
inputs over a wide range of magnitudes (its scales); and a solve's bits in groups of every
size class (1-16 columns of a product, one group and several).

Tolerance (max |difference| / max |reference|): the mixed operators' 1e-5; a solve's bits
are equal.
"""
import numpy as np
import pytest

from doi_amd import rte
from tests.helpers import bounds_for, hetero_maps, rel_max

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("shape,thr,spread", [((32, 32, 32), 0.0, 0.0), ((32, 32, 32), 0.0, 4.0), ((32, 32, 32), 0.47, 0.0),
                                              ((31, 30, 32), 0.0, 0.0), ((32, 31, 31), 0.95, 2.0), ((64, 64, 8), 0.0, 0.0),
                                              ((62, 32, 16), 0.0, 1.0)])
@pytest.mark.parametrize("L", [4, 5])
def test_operator_against_fp64(ctx, L, shape, thr, spread):
    N, K = int(np.prod(shape)), (L + 1) ** 2
    bounds = bounds_for(shape)
    ma, ms = hetero_maps(shape, seed=29)
    rng = np.random.default_rng(L)
    W = rng.standard_normal((K, N)) * np.exp(spread * rng.standard_normal((1, N)))
    out = []
    for prec in (rte.PREC_FP64, rte.PREC_MIXED, rte.PREC_FP32):
        print("operator", L, shape, thr, spread, prec, flush=True)
        out.append(ctx.propagate(shape, bounds, ma, ms, 0.9, W, L, prop_thresh=thr, precision=prec))
    assert rel_max(out[1], out[0]) < 1e-5
    assert rel_max(out[2], out[0]) < 1e-5


@pytest.mark.parametrize("L", [4, 5])
def test_bits_do_not_depend_on_the_group(ctx, L):
    shape = (32, 32, 32)
    media = [ctx.medium(shape, bounds_for(shape), *hetero_maps(shape, seed=70 + k), 0.9) for k in range(2)]
    beams = [(0.05 + 0.1 * (k % 5), -0.35 + 0.1 * k, 0.1, 1.0) for k in range(17)]
    p = rte.make_params(L, precision=rte.PREC_MIXED, stop_rule=rte.STOP_DELTA, tol=0.0, max_terms=4)
    pairs = [(media[(k // 3) % 2], b) for k, b in enumerate(beams)]
    alone = [ctx.solve_images([m], [b], p)[:2] for m, b in pairs]
    for n in (2, 3, 4, 5, 8, 15, 16, 17):
        print("group of", n, flush=True)
        img, refl, _ = ctx.solve_images([m for m, _ in pairs[:n]], [b for _, b in pairs[:n]], p)
        for k in range(n):
            assert np.array_equal(img[k], alone[k][0][0]), (n, k)
            assert np.array_equal(refl[k], alone[k][1][0]), (n, k)
    for m in media:
        m.close()
