"""The path table on flat and thin grids (sources beyond the grid left out) and with coupling
thresholds (rows without a coupled pair; brick pairs left out of a table of zeros): A W
from the table against the marched path integrals, L = 0, on media one after another, so
that a table's memory holds another's entries before.

Tolerances (max |difference| / max |reference|): twice those of the operators, FP64 1e-10
and mixed 1e-5.
"""
import numpy as np
import pytest

from doi_amd import rte
from tests.helpers import bounds_for, hetero_maps, rel_max

pytestmark = pytest.mark.gpu

TOL = {rte.PREC_FP64: 1e-10, rte.PREC_MIXED: 1e-5}


@pytest.mark.parametrize("thr", [0.0, 0.317, 1.013, 2.471])
@pytest.mark.parametrize("shape", [(1, 1, 70), (70, 1, 1), (1, 70, 1), (1, 60, 61), (61, 1, 60), (61, 60, 1), (64, 63, 2),
                                   (5, 6, 90), (16, 16, 16), (22, 21, 23), (26, 25, 24)])
def test_table_against_march(ctx, shape, thr):
    N = int(np.prod(shape))
    bounds = bounds_for(shape, d=(0.1, 0.12, 0.09))
    W = np.random.default_rng(N).standard_normal((1, N))
    for prec in (rte.PREC_MIXED, rte.PREC_FP64):
        for seed, scale in ((17, 1.0), (18, 3.0)):
            ma, ms = hetero_maps(shape, seed=seed, mus=scale)
            print("table", shape, thr, prec, seed, flush=True)
            got, march = (ctx.propagate(shape, bounds, ma, ms, 0.8, W, 0, prop_thresh=thr, precision=prec, path_mode=path)
                          for path in (rte.PATH_CACHED, rte.PATH_MARCH))
            assert rel_max(got, march) < 2 * TOL[prec]
