"""The gradient's back-projection at the edges of its kernel's choices: the derivative of a
weighted exitance along a random direction of all voxels, from the reverse pass, against
central differences of FP64 solves with the same number of terms.

Grids: 4 and 16 translations per wave (below and from 64 bricks, padded bricks), sums that fit
the LDS padded, only just (32x32x20, no room for the counter), in two slabs (28^3) and not at
all (150x140x1, atomics in memory); a coupling threshold.

Tolerance: 1e-5 of sum |gradient x direction|, the finite differences' own bound elsewhere.
"""
import numpy as np
import pytest

from doi_amd import rte
from tests.helpers import bounds_for, hetero_maps

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("shape,thr", [((5, 3, 4), 0.0), ((12, 12, 12), 0.0), ((12, 12, 12), 0.47), ((17, 18, 19), 0.0),
                                       ((32, 32, 20), 0.0), ((28, 28, 28), 0.0), ((150, 140, 1), 0.0)])
def test_directional_derivative(ctx, shape, thr):
    bounds, L, g = bounds_for(shape), 1, 0.7
    ma, ms = hetero_maps(shape, seed=83)
    rng = np.random.default_rng(9)
    cot = 0.5 + rng.random(shape[0] * shape[1])
    da, ds = ma * rng.random(ma.size), ms * rng.random(ms.size)
    beam = (0.05 if shape[0] % 2 == 0 else 0.0, 0.05 if shape[1] % 2 == 0 else 0.0, 0.1, 1.0)
    p = rte.make_params(L, precision=rte.PREC_FP64, stop_rule=rte.STOP_DELTA, tol=0.0, max_terms=4, prop_thresh=thr)
    print("gradient", shape, thr, flush=True)
    med = ctx.medium(shape, bounds, ma, ms, g)
    _, ga, gs, st = ctx.exitance_vjp(med, beam, p, cot)
    med.close()
    h, loss = 1e-4, []
    for s in (1.0, -1.0):
        img, stf = ctx.solve(shape, bounds, ma + s * h * da, ms + s * h * ds, g, beam, p)
        assert stf["terms"] == st["terms"]
        loss.append(float(np.dot(cot, img.ravel())))
    fd = (loss[0] - loss[1]) / (2 * h)
    size = float(np.abs(ga * da).sum() + np.abs(gs * ds).sum())
    assert abs(float(ga @ da + gs @ ds) - fd) <= 1e-5 * size
