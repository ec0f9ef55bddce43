"""The path table at the edges of its kernel's choices: A W from the table against the
oracle (small grids) and against the marched path integrals (every grid), L = 0.

Grids: one voxel; padded bricks on each axis; few translations of a brick pair (flat, long);
4 and 8 translations per wave (17x18x19, 20^3); the map in LDS with padded pitches (24^3),
without (33^3), clamped (34^3), filling the LDS (32x32x40), and in memory (36^3).

Tolerances (max |difference| / max |reference|): those of the operators against the oracle,
FP64 1e-10 and mixed 1e-5, and twice that between the two paths.
"""
import numpy as np
import pytest

from doi_amd import rte
from oracle import oracle as O
from tests.helpers import bounds_for, hetero_maps, rel_max

pytestmark = pytest.mark.gpu

TOL = {rte.PREC_FP64: 1e-10, rte.PREC_MIXED: 1e-5}


@pytest.mark.parametrize("thr", [0.0, 0.31])
@pytest.mark.parametrize("shape", [(1, 1, 1), (4, 4, 4), (5, 3, 4), (4, 40, 3), (41, 5, 2), (17, 18, 19), (20, 20, 20),
                                   (24, 24, 24), (33, 33, 33), (34, 34, 34), (32, 32, 40), (36, 36, 36)])
def test_table_against_march_and_oracle(ctx, shape, thr):
    N = int(np.prod(shape))
    bounds = bounds_for(shape, d=(0.1, 0.12, 0.09))
    ma, ms = hetero_maps(shape, seed=17)
    W = np.random.default_rng(N).standard_normal((1, N))
    for prec in (rte.PREC_MIXED, rte.PREC_FP64):
        if prec == rte.PREC_FP64 and N > 14000:
            continue
        print("table", shape, thr, prec, flush=True)
        got, march = (ctx.propagate(shape, bounds, ma, ms, 0.8, W, 0, prop_thresh=thr, precision=prec, path_mode=path,
                                    n=1.3) for path in (rte.PATH_CACHED, rte.PATH_MARCH))
        assert rel_max(got, march) < 2 * TOL[prec]
        if N <= 500:
            P = O.Problem(shape, bounds, ma, ms, 0.8, n=1.3)
            ref = P.propagate(W, 0, prop_thresh=thr) if thr else P.propagate(W, 0)
            assert rel_max(got, ref) < TOL[prec]
