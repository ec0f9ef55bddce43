"""The combine kernel at the edges of its blocks, against the FP64 oracle.

A block holds VB = 2 min(64, 256 // K) voxels (K = (L + 1)^2): one voxel, one less and
one more than a block (flat grids, where every voxel is both top and bottom face), and a
grid whose faces fall inside blocks, for every order; A W alone and the frequency-domain
solve (both halves of a voxel in one block, the field, both images).

Tolerances (max |gpu - ref| / max |ref|), those of the operators and solves elsewhere:
FP64 1e-10 (operator), 1e-9 (solve); mixed 1e-5.
"""
import numpy as np
import pytest

from doi_amd import rte
from oracle import oracle as O
from tests.helpers import bounds_for, hetero_maps, rel_max

pytestmark = pytest.mark.gpu


def crel(a, b):
    a, b = np.asarray(a), np.asarray(b)
    return float(np.max(np.abs(a - b)) / np.max(np.abs(b)))


@pytest.mark.parametrize("kind", ["one", "less", "more", "deep"])
@pytest.mark.parametrize("L", range(8))
def test_block_edges(ctx, L, kind):
    K = (L + 1) ** 2
    VB = 2 * min(64, 256 // K)
    shape = {"one": (1, 1, 1), "less": (VB - 1, 1, 1), "more": (1, VB + 1, 1), "deep": (3, 2, VB // 5 + 2)}[kind]
    bounds = bounds_for(shape, d=(0.1, 0.12, 0.09))
    ma, ms = hetero_maps(shape, seed=61 + L, mua=0.04, mus=1.3)
    P = O.Problem(shape, bounds, ma, ms, 0.8, n=1.3)
    W = np.random.default_rng(L).standard_normal((K, int(np.prod(shape))))
    ref = P.propagate(W, L)
    beam, om = (0.05 if shape[0] % 2 == 0 else 0.0, 0.0, 0.26, 1.0), 3.0e10
    fd = P.solve_fd(beam, L, om, stop_rule=O.STOP_DELTA, tol=1e-9, max_terms=4, field=True)
    m = ctx.medium(shape, bounds, ma, ms, 0.8, n=1.3)
    for prec, tol_op, tol in ((rte.PREC_FP64, 1e-10, 1e-9), (rte.PREC_MIXED, 1e-5, 1e-5)):
        print("combine", L, kind, prec, flush=True)
        got = ctx.propagate(shape, bounds, ma, ms, 0.8, W, L, precision=prec, n=1.3)
        assert rel_max(got, ref) < tol_op
        p = rte.make_params(L, precision=prec, stop_rule=rte.STOP_DELTA, tol=1e-9, max_terms=4)
        img, refl, st, fld = ctx.solve_fd([m], [beam], [om], p, field=True)
        assert st[0]["terms"] == fd["terms"]
        assert crel(img[0], fd["exitance"]) < tol
        if prec == rte.PREC_FP64:  # its order sum cancels: FP32 fields of one thin layer leave ~2e-5 of it
            assert crel(refl[0], fd["reflectance"]) < tol
        assert crel(fld, fd["w"]) < tol
    m.close()
