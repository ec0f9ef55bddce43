"""Path tables of gone media that a context keeps for media of the same size: a medium whose
table was another's gives the bits that a context without any kept table gives.

Orders 3 (the table alone) and 5 (the table and its exponents, where the matrix cores
propagate), both precisions, media destroyed and media reset.
"""
import numpy as np
import pytest

from doi_amd import rte
from tests.helpers import bounds_for, hetero_maps

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("shape,L,prec", [((5, 3, 4), 3, rte.PREC_FP64), ((9, 8, 7), 3, rte.PREC_MIXED),
                                          ((24, 24, 24), 5, rte.PREC_MIXED)])
def test_a_kept_table_is_filled_again(shape, L, prec):
    bounds = bounds_for(shape, d=(0.1, 0.12, 0.09))
    params = rte.make_params(L, precision=prec, max_terms=3)
    rng = np.random.default_rng(5)
    W = rng.standard_normal(((L + 1) ** 2, int(np.prod(shape))))
    maps = [hetero_maps(shape, seed=s) for s in (1, 2)]

    def run(ctx, ma, ms, reset=False):
        print("tables", shape, L, prec, reset, flush=True)
        m = ctx.medium(shape, bounds, ma, ms, 0.8)
        out = [np.array(ctx.neumann(m, W, params)[0])]
        if reset:
            m.reset_cache()
            out.append(np.array(ctx.neumann(m, W, params)[0]))
        m.close()
        return out

    fresh = []
    for ma, ms in maps:
        with rte.Context() as ctx:
            fresh.append(run(ctx, ma, ms)[0])
    assert not np.array_equal(fresh[0], fresh[1])
    with rte.Context() as ctx:
        for i in (0, 1, 0):
            for got in run(ctx, *maps[i], reset=i == 1):
                assert np.array_equal(got, fresh[i])
