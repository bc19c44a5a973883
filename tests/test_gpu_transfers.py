"""set_q and get_q give back what they were given, bit for bit: arrays below
the size that threads copy, with one chunk, with several and a remainder, and
longer than two bounce chunks; from two threads at once on contexts of their
own; and again after every context was closed.
"""
import threading

import numpy as np
import pytest

from tests.helpers import perturbed

pytestmark = pytest.mark.gpu

DIMS = [(7, 6, 5), (24, 21, 33), (61, 53, 67), (131, 97, 121)]


@pytest.mark.parametrize("dims", DIMS)
def test_round_trip(dims):
    from magic_master_amd.hip import MagicHIP
    for meqn in (5, 7):
        c, p, g, aux, q = perturbed(*dims, [1] * 6, seed=meqn, meqn=meqn)
        d = MagicHIP(g, p, aux, q)
        try:
            for n in range(3):
                a = np.random.default_rng(n).standard_normal(g.shape_q)
                d.set_q(a)
                np.testing.assert_array_equal(d.get_q(), a)
        finally:
            d.close()


def test_two_threads():
    from magic_master_amd.hip import MagicHIP
    bad = []

    def run(k):
        c, p, g, aux, q = perturbed(*DIMS[k], [1] * 6, seed=k)
        d = MagicHIP(g, p, aux, q)
        try:
            for n in range(10):
                a = np.random.default_rng(10 * k + n).standard_normal(g.shape_q)
                d.set_q(a)
                if not np.array_equal(d.get_q(), a):
                    bad.append((k, n))
        finally:
            d.close()
    th = [threading.Thread(target=run, args=(k,)) for k in (1, 2)]
    for t in th:
        t.start()
    for t in th:
        t.join()
    assert not bad
