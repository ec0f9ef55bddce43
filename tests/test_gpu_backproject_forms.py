"""The gradient's back-projection over the forms that its launch distinguishes: 1, 4 and 16
translations per wave (small, thin, cut-off and large grids), z planes that fill bricks and
that do not (units moved on from run to run), threads and blocks by the accumulator's
size.  The derivative of a weighted exitance along a random direction of all voxels against
central differences of FP64 solves with the same number of terms, and the mixed path's
gradient against FP64's.

Tolerances: 1e-5 of sum |gradient x direction|, the finite differences' own bound elsewhere;
mixed 2e-5 of the largest entry (the operators' 1e-5, forward and adjoint).
"""
import numpy as np
import pytest

from doi_amd import rte
from tests.helpers import bounds_for, hetero_maps, rel_max

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("shape,thr", [((1, 1, 1), 0.0), ((1, 1, 61), 0.0), ((5, 61, 5), 0.0), ((13, 14, 6), 0.0),
                                       ((13, 14, 6), 0.47), ((22, 21, 23), 0.0), ((22, 21, 23), 0.47), ((22, 21, 23), 1.09),
                                       ((24, 24, 20), 0.0), ((64, 63, 2), 0.0), ((64, 63, 2), 0.47), ((20, 20, 20), 0.0)])
def test_directional_derivative(ctx, shape, thr):
    bounds, L, g = bounds_for(shape), 1, 0.7
    ma, ms = hetero_maps(shape, seed=87)
    rng = np.random.default_rng(3)
    cot = 0.5 + rng.random(shape[0] * shape[1])
    da, ds = ma * rng.random(ma.size), ms * rng.random(ms.size)
    beam = (0.05 if shape[0] % 2 == 0 else 0.0, 0.05 if shape[1] % 2 == 0 else 0.0, 0.1, 1.0)
    print("back-projection", shape, thr, flush=True)
    m, out = ctx.medium(shape, bounds, ma, ms, g), []
    for prec in (rte.PREC_FP64, rte.PREC_MIXED):
        p = rte.make_params(L, precision=prec, stop_rule=rte.STOP_DELTA, tol=0.0, max_terms=4, prop_thresh=thr)
        out.append(ctx.exitance_vjp(m, beam, p, cot))
    m.close()
    (_, ga, gs, st), (_, ga32, gs32, _) = out
    assert rel_max(ga32, ga) < 2e-5 and rel_max(gs32, gs) < 2e-5
    p = rte.make_params(L, precision=rte.PREC_FP64, stop_rule=rte.STOP_DELTA, tol=0.0, max_terms=st["terms"], prop_thresh=thr)
    h, loss = 1e-4, []
    for s in (1.0, -1.0):
        img, _ = ctx.solve(shape, bounds, ma + s * h * da, ms + s * h * ds, g, beam, p)
        loss.append(float(np.dot(cot, img.ravel())))
    size = float(np.abs(ga * da).sum() + np.abs(gs * ds).sum())
    assert abs(float(ga @ da + gs @ ds) - (loss[0] - loss[1]) / (2 * h)) <= 1e-5 * size
