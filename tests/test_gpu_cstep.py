"""The one-kernel list step of small systems against the split kernels (same
sums in the same order: the same bits) and, where a particle pair binds
through several patch pairs, against the one-lane kernel: sizes around its
blocks (16 and 32 positions, 4,096 particles), both precisions, rotors and
beads, lists that overflow into the cells, more patch candidates than one
pass takes."""
import numpy as np
import pytest

from mtcode_amd import mdx
from mtcode_amd import workloads as wl

pytestmark = pytest.mark.gpu


def _fluid(n, theta=wl.THETAM_095, eps=6.0, pitch=1.12):
    side = max(3, int(np.ceil(n ** (1 / 3))))
    rng = np.random.default_rng(n)
    site = rng.permutation(side ** 3)[:n]
    ijk = np.stack([site % side, site // side % side, site // side ** 2], 1)
    s = wl._base("lattice", n, side * pitch, 0.005, 1.0, 1.0, 1.0 / 3.0, "rotor")
    s["x"] = (ijk + 0.5) * pitch + rng.uniform(-0.03, 0.03, (n, 3))
    s["Q"] = wl.arvo_rotations(n, rng)
    ps = wl.tetra_patchset(eps, thetam=theta)
    ps["types"] = np.zeros(n, dtype=np.int32)
    ps["maxd2"] = 2.4
    s["patches"] = ps
    return wl.thermal_momenta(s, n)


def _run(s, precision, monkeypatch, env, kmax=64, steps=30):
    for k in ("MDX_SPLIT", "MDX_WALKC"):
        monkeypatch.delenv(k, raising=False)
    for k, v in env.items():
        monkeypatch.setenv(k, v)
    with mdx.engine_from_system(s, precision=precision, seed=5) as e:
        e.set_neighbor_list(kmax=kmax)
        if s["integrator"] == "rotor":
            e.prime()
        e.step(steps)
        out = e.download()
        if s["integrator"] == "rotor":
            out["F"], out["T"] = e.carried_forces()
        return out


@pytest.mark.parametrize("precision", [mdx.PREC_FP64, mdx.PREC_MIXED])
@pytest.mark.parametrize("n", [1, 15, 16, 17, 33, 1000, 4096, 4097, 4129])
def test_same_bits_as_split(n, precision, monkeypatch):
    s = _fluid(n)
    a = _run(s, precision, monkeypatch, {"MDX_SPLIT": "0"})
    b = _run(s, precision, monkeypatch, {"MDX_SPLIT": "1"})
    for k in a:
        assert np.array_equal(a[k], b[k]), k


@pytest.mark.parametrize("precision", [mdx.PREC_FP64, mdx.PREC_MIXED])
def test_list_overflow(precision, monkeypatch):
    """kmax 4: most particles walk the cells of the build"""
    s = _fluid(1500)
    a = _run(s, precision, monkeypatch, {"MDX_SPLIT": "0"}, kmax=4)
    b = _run(s, precision, monkeypatch, {"MDX_SPLIT": "1"}, kmax=4)
    for k in a:
        assert np.array_equal(a[k], b[k]), k


def test_many_candidates(monkeypatch):
    """cones of 86 degrees on a dense lattice: about 13 candidates each (two
    passes), several patch pairs per particle pair"""
    s = _fluid(1331, theta=1.5, eps=0.05)
    a = _run(s, mdx.PREC_FP64, monkeypatch, {"MDX_SPLIT": "0"}, steps=10)
    b = _run(s, mdx.PREC_FP64, monkeypatch, {"MDX_SPLIT": "0", "MDX_WALKC": "0"}, steps=10)
    for k in a:
        # a pair's terms are summed before they are added: FP64 rounding
        assert np.abs(a[k] - b[k]).max() <= 1e-11 * max(1.0, np.abs(b[k]).max()), k


@pytest.mark.parametrize("precision", [mdx.PREC_FP64, mdx.PREC_MIXED])
@pytest.mark.parametrize("integrator", ["bead", "rotor"])
def test_chains(integrator, precision, monkeypatch):
    """bonds, angles, exclusions: 3 chains of 40 in a box with walls"""
    s = wl.mt_bundle(1, 13, 40, 25.0, (25.0, 25.0, 60.0))
    rng = np.random.default_rng(2)
    s["x"] = s["x"] + rng.normal(0, 0.02, s["x"].shape)
    s["p"] = rng.normal(0, 1, s["x"].shape)
    s["periodic"] = False
    s["integrator"] = integrator
    a = _run(s, precision, monkeypatch, {"MDX_SPLIT": "0"})
    b = _run(s, precision, monkeypatch, {"MDX_SPLIT": "0", "MDX_WALKC": "0"})
    for k in a:
        assert np.array_equal(a[k], b[k]), k
