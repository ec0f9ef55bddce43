"""What a server counts for a solve: rte_solve_footprint of a marched solve is its buffers'
size whatever a cached one would take, and the slots of solves on the matrix cores hold
their exponents (1/64 of the path table) as well.
"""
import pytest

from doi_amd import rte
from tests.helpers import bounds_for, hetero_maps

SHAPE = (32, 32, 30)
BOUNDS = bounds_for(SHAPE)
N = 32 * 32 * 30


@pytest.mark.parametrize("L", [3, 4, 5])
def test_marched(L):
    K = (L + 1) ** 2
    chunks = 8  # 512 bricks, 4096 waves
    want = N * (3 * 8 + 2 * 4) + N * K * 4 * (2 + chunks) + 32 * 32 * 5 * 8 + 64
    assert rte.footprint(SHAPE, BOUNDS, rte.make_params(L), rte.PATH_MARCH) == want


@pytest.mark.gpu
def test_slots_on_the_matrix_cores():
    p = rte.make_params(5, max_terms=3)
    ma, ms = hetero_maps(SHAPE, seed=1)
    with rte.Context() as ctx:
        m = ctx.medium(SHAPE, BOUNDS, ma, ms, 0.8)
        assert m.on_matrix_cores(p)
        m.close()
        srv = rte.Server(ctx, hbm_budget=16 << 30)
        for k, thick in enumerate((1.0, 40.0)):
            srv.wait(srv.submit(SHAPE, BOUNDS, ma, ms * thick, 0.8, (0.05, 0.05, 0.1, 1.0), p))
            used = srv.info()["hbm_used"]
            plain = rte.footprint(SHAPE, BOUNDS, p)
            exponents = (8 * 8 * 30 + 1) * 8 * 8 * 8 * 64
            if k == 0:
                assert plain + exponents <= used <= plain + 2 * exponents
                first = used
        assert used - first == plain  # a bucket of its own, k_prop's buffers
        srv.close()
