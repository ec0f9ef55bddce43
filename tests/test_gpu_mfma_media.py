"""Which media propagate on the matrix cores, and that the others lose nothing: A W of a
pencil beam's first two terms in every voxel, relative to the voxel's own value, in media
whose sources differ too much for the products' shared scales (thick voxels, one thick
sheet, a short coupling threshold with hollows); a batch and a server that hold media of
both kinds give each solve the bits it has alone.

Tolerance, voxel by voxel: 1e-3 = 16 x 36 coefficients that may cancel x 30 (path integral)
x 2^-24.  Bits are equal.
"""
import numpy as np
import pytest

from doi_amd import rte
from tests.helpers import bounds_for, hetero_maps

pytestmark = pytest.mark.gpu

SHAPE = (32, 32, 32)
BOUNDS = bounds_for(SHAPE)
N = 32 ** 3


def _maps(kind):
    ma, ms = np.full(N, 0.1), np.full(N, 1.0)
    x = np.arange(N) % 32
    if kind == "thick":
        ma, ms = ma * 15, ms * 28.5
    if kind == "sheet":
        ms[x == 13] = 100.0
    if kind == "hollows":
        r = np.random.default_rng(3).random(N)
        ms[r < 0.3] = 1e-4
        ms[r < 0.05] = 1e-7
    return ma, ms


@pytest.mark.parametrize("L", [4, 5])
@pytest.mark.parametrize("kind,thr,on", [("even", 0.0, True), ("even", 0.81, True), ("even", 0.31, False),
                                         ("hollows", 0.0, True), ("hollows", 0.81, False), ("hollows", 0.26, False),
                                         ("thick", 0.0, False), ("sheet", 0.0, False)])
def test_every_voxel(ctx, L, kind, thr, on):
    ma, ms = _maps(kind)
    K = (L + 1) ** 2
    m = ctx.medium(SHAPE, BOUNDS, ma, ms, 0.8)
    for prec in (rte.PREC_MIXED, rte.PREC_FP32):
        assert m.on_matrix_cores(rte.make_params(L, precision=prec, prop_thresh=thr)) == on
    assert not m.on_matrix_cores(rte.make_params(L, precision=rte.PREC_FP64, prop_thresh=thr))
    assert not m.on_matrix_cores(rte.make_params(L, prop_thresh=thr, path_mode=rte.PATH_MARCH))
    assert not m.on_matrix_cores(rte.make_params(3, prop_thresh=thr))
    m.close()
    W = ctx.source(SHAPE, BOUNDS, ma, ms, 0.8, (0.05, 0.05, 0.1, 1.0), L)[0].reshape(K, N)
    for term in range(2):
        print("voxels", L, kind, thr, term, flush=True)
        ref, got = (ctx.propagate(SHAPE, BOUNDS, ma, ms, 0.8, W, L, prop_thresh=thr, precision=p)
                    for p in (rte.PREC_FP64, rte.PREC_MIXED))
        size = np.abs(ref).max(axis=0)
        seen = size > 1e-20 * size.max()
        assert (np.abs(got - ref).max(axis=0)[seen] / size[seen]).max() < 1e-3
        W = ctx.scatter(SHAPE, BOUNDS, ma, ms, 0.8, ref, L)


@pytest.mark.parametrize("L", [4, 5])
def test_bits_in_a_mixed_batch(ctx, L):
    p = rte.make_params(L, stop_rule=rte.STOP_DELTA, tol=1e-3, max_terms=6)
    maps = [hetero_maps(SHAPE, seed=1), _maps("thick"), _maps("sheet"), hetero_maps(SHAPE, seed=2)]
    media = [ctx.medium(SHAPE, BOUNDS, *mm, 0.8) for mm in maps]
    assert [m.on_matrix_cores(p) for m in media] == [True, False, False, True]
    beams = [(0.05 + 0.1 * k, -0.25, 0.1, 1.0) for k in range(6)]
    pairs = [(k % 4, b) for k, b in enumerate(beams)]
    alone = [ctx.solve_images([media[k]], [b], p) for k, b in pairs]
    img, refl, st = ctx.solve_images([media[k] for k, _ in pairs], beams, p)
    for i in range(6):
        assert np.array_equal(img[i], alone[i][0][0]) and np.array_equal(refl[i], alone[i][1][0])
        assert st[i]["terms"] == alone[i][2][0]["terms"] and st[i]["gpu_ms"] > 0 and st[i]["latency_ms"] > 0
    with rte.Context() as own:
        srv = rte.Server(own)
        ids = [srv.submit(SHAPE, BOUNDS, *maps[k], 0.8, b, p) for k, b in pairs]
        for i, r in enumerate(ids):
            assert np.array_equal(srv.wait(r)[1], alone[i][0][0])
        srv.close()
    for m in media:
        m.close()
