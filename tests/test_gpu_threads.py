"""Contexts in several host threads of one process: solves and gradients made at the same
time have the bits of those made alone (gradients, whose sums are atomic, to 1e-9 of the
largest entry, their own spread).
"""
import threading

import numpy as np
import pytest

from doi_amd import rte
from tests.helpers import bounds_for, hetero_maps, rel_max

pytestmark = pytest.mark.gpu


def test_contexts_in_threads():
    shapes = [(9, 8, 7), (16, 16, 16), (12, 20, 5), (5, 5, 5)]
    p = rte.make_params(3, precision=rte.PREC_FP64, stop_rule=rte.STOP_DELTA, tol=0.0, max_terms=4)

    def work(k):
        s = shapes[k]
        ma, ms = hetero_maps(s, seed=k)
        beam = (0.05 if s[0] % 2 == 0 else 0.0, 0.05 if s[1] % 2 == 0 else 0.0, 0.1, 1.0)
        with rte.Context() as c:
            m = c.medium(s, bounds_for(s), ma, ms, 0.8)
            img = c.solve_images([m], [beam], p)[:2]
            grad = c.exitance_vjp(m, beam, p, np.ones(s[0] * s[1]))[1:3]
            m.close()
        return img, grad

    out, bad = [None] * 8, []

    def run(i):
        try:
            out[i] = work(i % 4)
        except Exception as e:  # shown by the main thread
            bad.append(e)

    print("threads", flush=True)
    threads = [threading.Thread(target=run, args=(i,)) for i in range(8)]
    for t in threads:
        t.start()
    for t in threads:
        t.join()
    assert not bad
    for i in range(8):
        img, grad = work(i % 4)
        assert all(np.array_equal(a, b) for a, b in zip(out[i][0], img))
        assert all(rel_max(a, b) < 1e-9 for a, b in zip(out[i][1], grad))
