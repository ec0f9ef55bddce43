"""The matrix-core propagation on grids of more than 8 bricks along y and z, ragged on every
axis, with a pitch of its own on each: the operator against FP64, a solve's bits alone and
in groups, and the reverse pass, whose forward series and recomputed terms run on the
matrix cores beside the adjoint's FP32 products.

Tolerances: the mixed operators' 1e-5 (max |difference| / max |reference|), twice that for
gradients (forward and adjoint); recomputed terms leave gradients equal to the rounding of
their atomic FP64 sums, 1e-12 of the largest entry; bits are equal.
"""
import numpy as np
import pytest

from doi_amd import rte
from tests.helpers import bounds_for, hetero_maps, rel_max

pytestmark = pytest.mark.gpu

PITCH = (0.1, 0.12, 0.09)


@pytest.mark.parametrize("L,shape", [(4, (12, 36, 63))])
def test_operator(ctx, L, shape):
    N, K = int(np.prod(shape)), (L + 1) ** 2
    bounds = bounds_for(shape, d=PITCH)
    ma, ms = hetero_maps(shape, seed=40)
    W = np.random.default_rng(L).standard_normal((K, N))
    print("operator", L, shape, flush=True)
    ref, got = (ctx.propagate(shape, bounds, ma, ms, 0.9, W, L, precision=p) for p in (rte.PREC_FP64, rte.PREC_MIXED))
    assert rel_max(got, ref) < 1e-5


@pytest.mark.parametrize("L,shape", [(4, (12, 36, 63)), (5, (29, 34, 45)), (5, (30, 39, 38))])
def test_groups(ctx, L, shape):
    bounds = bounds_for(shape, d=PITCH)
    maps = [hetero_maps(shape, seed=40 + k) for k in range(2)]
    media = [ctx.medium(shape, bounds, *mm, 0.9) for mm in maps]
    p = rte.make_params(L, stop_rule=rte.STOP_DELTA, tol=0.0, max_terms=3)
    assert all(m.on_matrix_cores(p) for m in media)
    x0, y0 = (0.5 - shape[0] / 2) * PITCH[0], (0.5 - shape[1] / 2) * PITCH[1]
    pairs = [(media[(k // 2) % 2], (x0 + k % 5 * 2 * PITCH[0], y0 + k * PITCH[1], 0.09, 1.0)) for k in range(17)]
    alone = [ctx.solve_images([m], [b], p)[:2] for m, b in pairs]
    for n in (2, 5, 16, 17):
        print("group of", n, flush=True)
        img, refl, _ = ctx.solve_images([m for m, _ in pairs[:n]], [b for _, b in pairs[:n]], p)
        for k in range(n):
            assert np.array_equal(img[k], alone[k][0][0]) and np.array_equal(refl[k], alone[k][1][0]), (n, k)
    for m in media:
        m.close()


@pytest.mark.parametrize("L,shape", [(4, (32, 32, 32)), (5, (32, 32, 32)), (5, (29, 34, 45))])
def test_gradient(ctx, L, shape):
    bounds = bounds_for(shape, d=PITCH)
    ma, ms = hetero_maps(shape, seed=51)
    cot = 0.5 + np.random.default_rng(L).random(shape[0] * shape[1])
    beam = (0.05 if shape[0] % 2 == 0 else 0.0, 0.06 if shape[1] % 2 == 0 else 0.0, 0.09, 1.0)
    m, out = ctx.medium(shape, bounds, ma, ms, 0.8), []
    for prec, stride in ((rte.PREC_FP64, 1), (rte.PREC_MIXED, 1), (rte.PREC_MIXED, 3)):
        print("gradient", L, shape, prec, stride, flush=True)
        p = rte.make_params(L, precision=prec, stop_rule=rte.STOP_DELTA, tol=0.0, max_terms=5)
        assert m.on_matrix_cores(p) == (prec == rte.PREC_MIXED)
        out.append(ctx.exitance_vjp(m, beam, p, cot, checkpoint_stride=stride)[:3])
    p = rte.make_params(L, stop_rule=rte.STOP_DELTA, tol=0.0, max_terms=5)
    assert rel_max(out[1][0].ravel(), ctx.solve_media([m], [beam], p)[0][0].ravel()) < 1e-12
    m.close()
    for a, b, c in zip(*out):
        assert rel_max(b, a) < 2e-5
        assert rel_max(c, b) < 1e-12
