"""The neighbour list is the set of pairs within its radii in FP64, whatever the
coordinates: particles far outside the box (an upload takes any finite
position), boxes whose edge makes an FP32 coordinate coarse, the periodic seam,
two list radii.  Against a brute-force search."""
import numpy as np
import pytest
from scipy.spatial import cKDTree

from mtcode_amd import mdx
from mtcode_amd import workloads as wl

pytestmark = pytest.mark.gpu


def _system(n, box, x, kind, periodic):
    rng = np.random.default_rng(n)
    s = wl._base(kind, n, box, 0.005, 1.0, 1.0, 1.0 / 3.0, "rotor")
    s["periodic"] = periodic
    s["x"] = x
    s["Q"] = wl.arvo_rotations(n, rng)
    ps = wl.tetra_patchset(6.0) if kind == "tetra" else wl.two_species_patchset(8.0)
    types = np.zeros(n, dtype=np.int32)
    if kind != "tetra":
        types[n // 2:] = 1
    ps["types"], ps["maxd2"] = types, 2.4
    s["patches"] = ps
    return s


def _list(s, kmax=200):
    with mdx.engine_from_system(s, precision=mdx.PREC_MIXED) as e:
        e.set_neighbor_list(kmax=kmax)
        got, (rl, rw) = e.list_pairs()
    return got, rl, rw


def _within(s, pairs, rl, rw):
    """of the candidate pairs, those that the list holds"""
    d = s["x"][pairs[:, 0]] - s["x"][pairs[:, 1]]
    box = np.broadcast_to(np.asarray(s["box"], dtype=float), (3,))
    if s["periodic"]:
        d -= np.where(np.abs(d) > 0.5 * box, np.where(d >= 0, box, -box), 0.0)
    r2 = (d[:, 0] * d[:, 0] + d[:, 1] * d[:, 1]) + d[:, 2] * d[:, 2]
    types = s["patches"]["types"]
    same = types[pairs[:, 0]] == types[pairs[:, 1]]
    return pairs[np.where(same & (rw < rl), r2 < rw * rw, r2 < rl * rl)]


def _sorted(p):
    p = np.sort(p, 1)
    return p[np.lexsort((p[:, 1], p[:, 0]))]


@pytest.mark.parametrize("kind", ["tetra", "condensate"])
@pytest.mark.parametrize("periodic", [True, False])
@pytest.mark.parametrize("shift", [0.0, 13.0, 30.0, 3.0e4, 1.0e8])
def test_particles_outside_the_box(shift, periodic, kind):
    n, L = 600, 20.0
    rng = np.random.default_rng(3)
    x = rng.uniform(0, L, (n, 3))
    # a dense droplet beyond one face, one beyond another
    x[:200] = rng.uniform(0, 4, (200, 3)) + [shift, 7.0, 7.0]
    x[200:300] = rng.uniform(0, 3, (100, 3)) + [5.0, -shift, 9.0]
    x = x[rng.permutation(n)]
    s = _system(n, L, x, kind, periodic)
    got, rl, rw = _list(s)
    i, j = np.triu_indices(n, 1)
    want = _within(s, np.stack([i, j], 1), rl, rw)
    if periodic:
        # (a pair through the seam of which one lies outside the box is in no
        # neighbouring cells: not the list's to hold)
        d = np.abs(x[want[:, 0]] - x[want[:, 1]])
        inside = ((x >= 0) & (x < L)).all(1)
        want = want[(d <= 0.5 * L).all(1) | (inside[want[:, 0]] & inside[want[:, 1]])]
        d = np.abs(x[got[:, 0]] - x[got[:, 1]])
        got = got[(d <= 0.5 * L).all(1) | (inside[got[:, 0]] & inside[got[:, 1]])]
    assert np.array_equal(got, _sorted(want))


@pytest.mark.parametrize("kind", ["tetra", "condensate"])
@pytest.mark.parametrize("n,box,periodic", [(4000, (4000.0, 12.0, 12.0), True),
                                            (4000, (12.0, 12.0, 9000.0), True),
                                            (1000, (1.0e6, 9.0, 9.0), True),
                                            (1000, (1.0e7, 9.0, 9.0), True),
                                            (4000, (4000.0, 12.0, 12.0), False),
                                            (120000, (2000.0, 40.0, 12.0), True)])
def test_long_boxes(n, box, periodic, kind):
    rng = np.random.default_rng(n)
    box = np.array(box)
    x = rng.uniform(0, 1, (n, 3)) * box
    if box.max() > 1e5:
        # crowded ends on both sides of the seam
        x[:, 0] = np.mod(rng.uniform(-40, 40, n), box[0])
    x = np.minimum(x, np.nextafter(box, 0))
    # a share of the pairs lies right at the list radius
    far = rng.integers(0, n // 2, n // 8)
    u = rng.normal(size=(n // 8, 3))
    u /= np.linalg.norm(u, axis=1)[:, None]
    s = _system(n, box, x, kind, periodic)
    _, rl, rw = _list(s)
    step = np.where(rng.random(n // 8) < 0.5, rl, rw) * (1 + rng.uniform(-3e-7, 3e-7, n // 8))
    y = x[far] + u * step[:, None]
    ok = ((y >= 0) & (y < box)).all(1)
    x[n - n // 8:][ok] = y[ok]
    s["x"] = x
    got, rl, rw = _list(s)
    tree = cKDTree(x, boxsize=box if periodic else None)
    want = _within(s, tree.query_pairs(rl * (1 + 1e-6), output_type="ndarray"), rl, rw)
    assert len(want) > 300
    assert np.array_equal(got, _sorted(want))


@pytest.mark.parametrize("kind", ["tetra", "condensate"])
@pytest.mark.parametrize("forced", ["", "0", "1"])
@pytest.mark.parametrize("n,box", [(63, (9.0, 9.0, 9.0)), (65, (30.0, 7.0, 7.0)),
                                   (6000, (300.0, 11.0, 11.0)),  # 240 particles in a row of cells
                                   (8750, (400.0, 11.0, 11.0)),  # 350
                                   (5000, (24.0, 24.0, 24.0))])
def test_forms_of_the_build(n, box, forced, kind, monkeypatch):
    """both stagings, by size and forced, and rows that neither holds"""
    if forced:
        monkeypatch.setenv("MDX_NBDENSE", forced)
    box = np.array(box)
    s = _system(n, box, np.random.default_rng(n).uniform(0, 1, (n, 3)) * box, kind, True)
    got, rl, rw = _list(s)
    tree = cKDTree(s["x"], boxsize=box)
    want = _within(s, tree.query_pairs(rl * (1 + 1e-6), output_type="ndarray"), rl, rw)
    assert np.array_equal(got, _sorted(want))
