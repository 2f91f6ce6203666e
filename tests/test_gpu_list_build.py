"""The neighbour list that the step's kernels build against the pair search of
the parity entry point: one and four lanes per position (100,000 particles),
block edges, the smallest grids, two list radii, walls, dense rows; and the
same forces whatever the lanes."""
import numpy as np
import pytest

from mtcode_amd import mdx
from mtcode_amd import workloads as wl

pytestmark = pytest.mark.gpu


def _system(n, kind, density, seed, periodic=True):
    rng = np.random.default_rng(seed)
    L = max((n / density) ** (1 / 3), 6.2)
    s = wl._base(kind, n, L, 0.005, 1.0, 1.0, 1.0 / 3.0, "rotor")
    s["x"] = rng.uniform(0, L, (n, 3))
    s["Q"] = wl.arvo_rotations(n, rng)
    s["periodic"] = periodic
    ps = wl.tetra_patchset(6.0) if kind == "tetra" else wl.two_species_patchset(8.0)
    types = np.zeros(n, dtype=np.int32)
    if kind != "tetra":
        types[n // 2:] = 1
    ps["types"], ps["maxd2"] = types, 2.4
    s["patches"] = ps
    return s


@pytest.mark.parametrize("kind", ["tetra", "condensate"])
@pytest.mark.parametrize("n,density,periodic", [(1, 0.2, True), (63, 0.2, True), (64, 0.2, False),
                                                (257, 0.9, True), (5000, 0.1, False),
                                                (20000, 0.8, True), (100000, 0.1, True),
                                                (100001, 0.1, True), (130000, 0.5, True)])
def test_list_is_the_pair_set(n, density, periodic, kind):
    s = _system(n, kind, density, n, periodic)
    with mdx.engine_from_system(s, precision=mdx.PREC_MIXED) as e:
        e.set_neighbor_list(kmax=96)
        got, (rl, rw) = e.list_pairs()
        cells = np.maximum((s["box"] // rl).astype(int), 1)
        near = e.neighbor_pairs(cells, rl)
        if rw < rl:
            same = s["patches"]["types"][near[:, 0]] == s["patches"]["types"][near[:, 1]]
            inner = e.neighbor_pairs(cells, rw)
            types = s["patches"]["types"]
            inner = inner[types[inner[:, 0]] == types[inner[:, 1]]]
            near = np.concatenate([near[~same], inner])
            near = near[np.lexsort((near[:, 1], near[:, 0]))]
        assert np.array_equal(got, near)
