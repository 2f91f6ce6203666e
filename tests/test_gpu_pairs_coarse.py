"""The pair set on coarse grids: many particles per cell, up to all of them in
one.  The same pairs as a brute-force search, in a time that the search over
pairs sets and not the ordering of a cell's members."""
import time

import numpy as np
import pytest

from mtcode_amd import mdx

pytestmark = pytest.mark.gpu


def _brute(x, L, cut, periodic):
    out = []
    for i in range(len(x)):
        d = x[i + 1:] - x[i]
        if periodic:
            d -= np.where(np.abs(d) > 0.5 * L, np.where(d >= 0, L, -L), 0.0)
        j = np.flatnonzero((d * d).sum(1) < cut * cut)
        out.append(np.stack([np.full(len(j), i), i + 1 + j], 1))
    return np.concatenate(out)


@pytest.mark.parametrize("periodic", [True, False])
@pytest.mark.parametrize("n,cells,cut", [(1, 1, 1.0), (255, 1, 9.0), (1025, 1, 2.0),
                                         (1025, 2, 5.0), (1500, 3, 3.0), (900, (1, 2, 7), 2.5)])
def test_pairs(n, cells, cut, periodic):
    L = 20.0
    x = np.random.default_rng(n).uniform(0, L, (n, 3))
    with mdx.Engine(n, L, 1.0, 0.005, periodic=periodic) as e:
        e.upload(x)
        assert np.array_equal(e.neighbor_pairs(cells, cut), _brute(x, L, cut, periodic))


def test_one_cell_in_linear_time_per_particle():
    """3,000 particles in one cell: 5 ms for the count, the pairs and their
    copies; 0.8 s with the cell's members ordered one by one in a single lane"""
    n, L = 3000, 20.0
    x = np.random.default_rng(2).uniform(0, L, (n, 3))
    with mdx.Engine(n, L, 1.0, 0.005) as e:
        e.upload(x)
        e.neighbor_pairs(1, 1.0)
        t = []
        for _ in range(3):
            t0 = time.perf_counter()
            e.neighbor_pairs(1, 1.0)
            t.append(time.perf_counter() - t0)
    assert min(t) < 0.15, t
