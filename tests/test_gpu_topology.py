"""Bonds, angles and active forces of list steps (slot tables) against steps
that bin and walk the cells every time (tables by original index): uniform and
per-bond parameters, both bond and angle forms, more partners than the tables
hold, topology changed or switched off between calls, several re-sorts."""
import numpy as np
import pytest

from mtcode_amd import mdx
from mtcode_amd import workloads as wl

pytestmark = pytest.mark.gpu


def _chains(nc, nb, seed, integrator="rotor"):
    rng = np.random.default_rng(seed)
    n = nc * nb
    side = int(np.ceil(np.sqrt(nc)))
    box = np.array([max(7.0, 1.6 * side)] * 2 + [nb + 2.0])
    s = wl._base("chains", n, box, 0.004, 1.0, 1.0, 1.0 / 3.0, integrator)
    lane = rng.permutation(side * side)[:nc]
    x = np.empty((nc, nb, 3))
    x[..., 0] = (0.8 + 1.6 * (lane % side))[:, None]
    x[..., 1] = (0.8 + 1.6 * (lane // side))[:, None]
    x[..., 2] = np.arange(nb) + 0.5
    s["x"] = np.mod(x.reshape(n, 3) + rng.normal(0, 0.03, (n, 3)), box)
    s["Q"] = wl.arvo_rotations(n, rng)
    s["p"] = rng.normal(0, 1, (n, 3))
    idx = np.arange(n).reshape(nc, nb)
    s["bonds"] = np.stack([idx[:, :-1].ravel(), idx[:, 1:].ravel()], 1).astype(np.int32)
    s["bond_k"] = np.full(len(s["bonds"]), 100.0)
    s["bond_r0"] = np.ones(len(s["bonds"]))
    s["angles"] = np.stack([idx[:, :-2].ravel(), idx[:, 1:-1].ravel(), idx[:, 2:].ravel()],
                           1).astype(np.int32)
    s["angle_k"] = np.full(len(s["angles"]), 15.0)
    s["angle_theta0"] = np.zeros(len(s["angles"]))
    s["angle_form"] = 1
    s["exclusions"] = s["bonds"].copy()
    prev = np.full((nc, nb), -1, dtype=np.int32)
    nxt = np.full((nc, nb), -1, dtype=np.int32)
    prev[:, 1:], nxt[:, :-1] = idx[:, :-1], idx[:, 1:]
    s["active"] = {"fa": 1.5, "prev": prev.ravel(), "next": nxt.ravel()}
    return s


def _run(s, skin, split, monkeypatch, calls, precision=mdx.PREC_FP64):
    monkeypatch.setenv("MDX_SPLIT", str(split))
    with mdx.engine_from_system(s, precision=precision, seed=7) as e:
        e.set_neighbor_list(skin=skin, resort_every=11)
        for change in calls:
            if change:
                change(e)
            if s["integrator"] == "rotor":
                e.prime()
            e.step(15)
        return e.download()


def _same(s, monkeypatch, split, calls=(None, None)):
    a = _run(s, 0.4, split, monkeypatch, calls)
    b = _run(s, 0.0, split, monkeypatch, calls)
    for k in a:
        # the pair sums run in another cell order: FP64 rounding over the steps
        assert np.abs(a[k] - b[k]).max() < 1e-9, k


@pytest.mark.parametrize("split", [0, 1])
@pytest.mark.parametrize("integrator", ["rotor", "bead"])
@pytest.mark.parametrize("form", ["uniform", "per_bond", "fene_harmonic"])
def test_tables(form, integrator, split, monkeypatch):
    s = _chains(37, 25, 3, integrator)
    rng = np.random.default_rng(4)
    if form != "uniform":
        s["bond_k"] = rng.uniform(50, 150, len(s["bonds"]))
        s["bond_r0"] = rng.uniform(0.95, 1.05, len(s["bonds"]))
        s["angle_k"] = rng.uniform(5, 20, len(s["angles"]))
    if form == "fene_harmonic":
        s["bond_kind"], s["bond_r0"] = 2, rng.uniform(1.8, 2.2, len(s["bonds"]))
        s["bond_k"] = np.full(len(s["bonds"]), 5.0)
        s["angle_form"], s["angle_theta0"] = 0, rng.uniform(0.1, 0.3, len(s["angles"]))
    _same(s, monkeypatch, split)


@pytest.mark.parametrize("extra", ["bonds", "angles"])
def test_more_partners_than_the_tables_hold(extra, monkeypatch):
    """particle 0 bonded to six others, or in five angles"""
    s = _chains(20, 20, 5)
    if extra == "bonds":
        add = np.array([[0, 40 + 20 * k] for k in range(5)], dtype=np.int32)
        s["bonds"] = np.concatenate([s["bonds"], add])
        s["bond_k"] = np.concatenate([s["bond_k"], np.full(5, 0.01)])
        s["bond_r0"] = np.concatenate([s["bond_r0"], np.full(5, 3.0)])
    else:
        add = np.array([[k, 0, k + 1] for k in range(3, 8)], dtype=np.int32)
        s["angles"] = np.concatenate([s["angles"], add])
        s["angle_k"] = np.concatenate([s["angle_k"], np.full(5, 0.01)])
        s["angle_theta0"] = np.zeros(len(s["angles"]))
    _same(s, monkeypatch, 0)


def test_topology_changed_between_calls(monkeypatch):
    s = _chains(20, 20, 6)
    keep = len(s["bonds"]) - 50

    def fewer(e):
        e.set_bonds(s["bonds"][:keep], s["bond_k"][:keep] * 0.5, s["bond_r0"][:keep])

    def off(e):
        mdx._check(mdx.lib().mdx_clear_interactions(e.h, 8 | 32))

    def on(e):
        e.set_angles(s["angles"][::2], s["angle_k"][::2], s["angle_theta0"][::2], 1)
        e.set_active(0.5, s["active"]["prev"], s["active"]["next"])

    _same(s, monkeypatch, 0, (None, fewer, off, on))
