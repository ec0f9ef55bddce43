"""The device memory that a context keeps of gone media: the newest sizes stay and the oldest
go once 8 GiB are kept, rte_ctx_trim and the context's end give it back; and a kept table
and its kept exponents are filled again for a medium on the matrix cores (the bits of a
context that keeps nothing), after a destroyed and after a reset medium.

Memory is read from the device, to 512 MB (workspaces, the runtime's own).
"""
import numpy as np
import pytest
import torch

from doi_amd import rte
from tests.helpers import bounds_for, hetero_maps

pytestmark = pytest.mark.gpu

SLACK = 512e6


def _used():
    free, total = torch.cuda.mem_get_info(0)
    return total - free


def _table(shape):
    bricks = int(np.prod([(e + 3) // 4 for e in shape]))
    return float(np.prod(shape)) * bricks * 64 * 4


def _solves(ctx, shape, n):
    media = [ctx.medium(shape, bounds_for(shape), *hetero_maps(shape, seed=i), 0.8) for i in range(n)]
    ctx.solve_media(media, [(0.05, 0.05, 0.1, 1.0)] * n, rte.make_params(0, max_terms=1))
    for m in media:
        m.close()


def test_the_oldest_tables_go_first_and_trim_gives_back():
    with rte.Context() as ctx:
        _solves(ctx, (8, 8, 8), 1)
        base = _used()
        print("kept tables", flush=True)
        _solves(ctx, (34, 34, 34), 1)
        assert abs(_used() - base - _table((34, 34, 34))) < SLACK
        _solves(ctx, (26, 26, 26), 2)  # 7.3 + 2 x 1.5 GB: more than is kept
        assert abs(_used() - base - 2 * _table((26, 26, 26))) < SLACK
        ctx.trim()
        assert abs(_used() - base) < SLACK
        _solves(ctx, (26, 26, 26), 2)
        assert abs(_used() - base - 2 * _table((26, 26, 26))) < SLACK
    assert abs(_used() - base) < SLACK


@pytest.mark.parametrize("L", [4, 5])
def test_kept_exponents_are_filled_again(L):
    shape = (32, 32, 32)
    bounds = bounds_for(shape)
    params = rte.make_params(L, max_terms=2)
    W = np.random.default_rng(5).standard_normal(((L + 1) ** 2, 32 ** 3))
    maps = [hetero_maps(shape, seed=1), hetero_maps(shape, seed=2, mua=0.3, mus=4.0, sigma=0.2)]

    def run(ctx, ma, ms, reset=False):
        print("kept exponents", L, reset, flush=True)
        m = ctx.medium(shape, bounds, ma, ms, 0.8)
        assert m.on_matrix_cores(params)
        out = [ctx.neumann(m, W, params)[0]]
        if reset:
            m.reset_cache()
            out.append(ctx.neumann(m, W, params)[0])
        m.close()
        return out

    fresh = []
    for mm in maps:
        with rte.Context() as ctx:
            fresh.append(run(ctx, *mm)[0])
    assert not np.array_equal(fresh[0], fresh[1])
    with rte.Context() as ctx:
        for i in (0, 1, 0):
            for got in run(ctx, *maps[i], reset=i == 1):
                assert np.array_equal(got, fresh[i])
        ctx.trim()
        assert np.array_equal(run(ctx, *maps[1])[0], fresh[1])
