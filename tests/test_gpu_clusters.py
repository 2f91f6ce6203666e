"""Cluster labels from one pass over the cells against scipy's components of
the pair list of the same call's stencil: grids of 1, 2, 3 and many cells a
side, one particle, crowded cells, long chains (deep forests), walls, ranges
left out; the same pairs and histogram from the device's cell lists."""
import numpy as np
import pytest
from scipy.sparse import coo_matrix
from scipy.sparse.csgraph import connected_components

from mtcode_amd import mdx

pytestmark = pytest.mark.gpu


def _brute_labels(n, pairs, exclude):
    if exclude is not None and exclude[0] <= exclude[1]:
        out = (pairs >= exclude[0]) & (pairs <= exclude[1])
        pairs = pairs[~out.any(1)]
    g = coo_matrix((np.ones(len(pairs)), (pairs[:, 0], pairs[:, 1])), shape=(n, n))
    _, comp = connected_components(g, directed=False)
    first = np.full(comp.max() + 1, n)
    np.minimum.at(first, comp, np.arange(n))
    return first[comp]


def _pairs(x, L, cut, periodic):
    d = x[:, None] - x[None]
    if periodic:
        d -= np.where(np.abs(d) > 0.5 * L, np.sign(d) * L, 0.0)
    i, j = np.nonzero(np.triu((d * d).sum(-1) < cut * cut, 1))
    return np.stack([i, j], 1)


@pytest.mark.parametrize("periodic", [True, False])
@pytest.mark.parametrize("n,L,cells,cut", [(1, 5.0, 1, 1.0), (40, 4.0, 1, 1.2), (60, 5.0, 2, 1.0),
                                           (257, 9.0, 3, 1.3), (1500, 30.0, 12, 2.4),
                                           (1024, 12.0, 4, 0.9)])
def test_labels(n, L, cells, cut, periodic):
    rng = np.random.default_rng(n)
    x = rng.uniform(0, L, (n, 3))
    pairs = _pairs(x, L, cut, periodic)
    with mdx.Engine(n, L, 1.0, 0.005, periodic=periodic) as e:
        e.upload(x)
        for exclude in (None, (n // 3, n // 2), (5, 4)):
            lab, count = e.clusters(cells, cut, exclude)
            ref = _brute_labels(n, pairs, exclude)
            assert np.array_equal(lab, ref) and count == len(np.unique(ref))
        got = e.neighbor_pairs(cells, cut)
        assert np.array_equal(got, pairs)


def test_long_chain_and_crowded_cell():
    """one component threaded through every cell in scattered index order, and
    2,000 particles in one cell"""
    rng = np.random.default_rng(1)
    n = 5000
    t = np.arange(n)
    side = 20.0
    x = np.stack([(t * 0.5) % side, (t // 40 * 0.5) % side, t // 1600 * 0.9 + 0.1], 1)
    x = np.mod(x, side)[rng.permutation(n)]
    pairs = _pairs(x, side, 0.6, True)
    ref = _brute_labels(n, pairs, None)
    with mdx.Engine(n, side, 1.0, 0.005) as e:
        e.upload(x)
        for _ in range(3):
            lab, count = e.clusters(20, 0.6)
            assert np.array_equal(lab, ref) and count == len(np.unique(ref))
    y = rng.uniform(0, 0.9, (2000, 3))
    with mdx.Engine(2000, side, 1.0, 0.005) as e:
        e.upload(y)
        lab, count = e.clusters(20, 0.95)
        assert np.array_equal(lab, _brute_labels(2000, _pairs(y, side, 0.95, True), None))
