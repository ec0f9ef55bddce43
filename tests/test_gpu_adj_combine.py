"""The adjoint combine at the edges of its blocks of VB = 2 min(64, 256 // K) voxels, every
order: the derivative of a weighted exitance along a random direction against central
differences of FP64 solves, and the mixed path's gradient against FP64's.

Tolerance: finite differences 1e-5 of sum |gradient x direction|; mixed 2e-5 of the largest
entry (the operators' 1e-5, forward and adjoint).
"""
import numpy as np
import pytest

from doi_amd import rte
from tests.helpers import bounds_for, hetero_maps, rel_max

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("kind", ["less", "more", "deep"])
@pytest.mark.parametrize("L", range(8))
def test_block_edges(ctx, L, kind):
    VB = 2 * min(64, 256 // (L + 1) ** 2)
    shape = {"less": (VB - 1, 1, 1), "more": (1, VB + 1, 1), "deep": (3, 2, VB // 5 + 2)}[kind]
    bounds, g = bounds_for(shape), 0.8
    ma, ms = hetero_maps(shape, seed=91 + L)
    rng = np.random.default_rng(L)
    cot = 0.5 + rng.random(shape[0] * shape[1])
    da, ds = ma * rng.random(ma.size), ms * rng.random(ms.size)
    beam = (0.0, 0.0, 0.26, 1.0)
    print("adjoint combine", L, kind, flush=True)
    med, out = ctx.medium(shape, bounds, ma, ms, g), []
    for prec in (rte.PREC_FP64, rte.PREC_MIXED):
        p = rte.make_params(L, precision=prec, stop_rule=rte.STOP_DELTA, tol=0.0, max_terms=4)
        out.append(ctx.exitance_vjp(med, beam, p, cot))
    med.close()
    (_, ga, gs, st), (_, ga32, gs32, _) = out
    assert rel_max(ga32, ga) < 2e-5 and rel_max(gs32, gs) < 2e-5
    p = rte.make_params(L, precision=rte.PREC_FP64, stop_rule=rte.STOP_DELTA, tol=0.0, max_terms=st["terms"])
    h, loss = 1e-4, []
    for s in (1.0, -1.0):
        img, _ = ctx.solve(shape, bounds, ma + s * h * da, ms + s * h * ds, g, beam, p)
        loss.append(float(np.dot(cot, img.ravel())))
    size = float(np.abs(ga * da).sum() + np.abs(gs * ds).sum())
    assert abs(float(ga @ da + gs @ ds) - (loss[0] - loss[1]) / (2 * h)) <= 1e-5 * size
