"""Forces from the cells with several lanes per position against the one-lane
kernel: the same terms in the same order, so the same bits.  Sizes around its
blocks (16 positions), boxes of few cells, more neighbours in reach than a
block's buffer holds, several bound patch pairs per particle pair, chains with
walls, both precisions."""
import numpy as np
import pytest

from mtcode_amd import mdx
from mtcode_amd import workloads as wl

pytestmark = pytest.mark.gpu


def _fluid(n, pitch=1.12, box=None, theta=wl.THETAM_095, eps=6.0, maxd2=2.4):
    side = max(2, int(np.ceil(n ** (1 / 3))))
    rng = np.random.default_rng(n)
    site = rng.permutation(side ** 3)[:n]
    ijk = np.stack([site % side, site // side % side, site // side ** 2], 1)
    s = wl._base("lattice", n, box or max(side * pitch, 3.4), 0.005, 1.0, 1.0, 1.0 / 3.0, "rotor")
    s["x"] = (ijk + 0.5) * pitch + rng.uniform(-0.03, 0.03, (n, 3))
    s["Q"] = wl.arvo_rotations(n, rng)
    ps = wl.tetra_patchset(eps, thetam=theta)
    ps["types"] = np.zeros(n, dtype=np.int32)
    ps["maxd2"] = maxd2
    s["patches"] = ps
    return wl.thermal_momenta(s, n)


def _run(s, precision, monkeypatch, env):
    for k in ("MDX_SPLIT", "MDX_WALKC"):
        monkeypatch.delenv(k, raising=False)
    for k, v in env.items():
        monkeypatch.setenv(k, v)
    with mdx.engine_from_system(s, precision=precision, seed=5) as e:
        rotor = s["integrator"] == "rotor"
        out = {}
        if rotor:
            out["F0"], out["T0"] = e.compute_forces()
            e.prime()
        for _ in range(3):
            e.step(1)
        out.update(e.download())
        if rotor:
            out["F"], out["T"] = e.carried_forces()
        return out


def _same(s, precision, monkeypatch):
    a = _run(s, precision, monkeypatch, {"MDX_SPLIT": "0"})
    b = _run(s, precision, monkeypatch, {"MDX_SPLIT": "0", "MDX_WALKC": "0"})
    for k in a:
        assert np.isfinite(b[k]).all(), k
        assert np.array_equal(a[k], b[k]), k


BOTH = pytest.mark.parametrize("precision", [mdx.PREC_FP64, mdx.PREC_MIXED])


@BOTH
@pytest.mark.parametrize("n", [1, 2, 15, 16, 17, 64, 1000, 4097])
def test_sizes(n, precision, monkeypatch):
    _same(_fluid(n), precision, monkeypatch)


@BOTH
@pytest.mark.parametrize("reach", [2.4, 5.8, 8.9])
def test_many_in_reach(reach, precision, monkeypatch):
    """up to 80 neighbours within reach of each position (1,300 a block), in
    boxes of 5 to 3 and fewer cells a side"""
    _same(_fluid(729, maxd2=reach), precision, monkeypatch)


@BOTH
def test_several_bonds_per_pair(precision, monkeypatch):
    """cones of 86 degrees: more candidates than a pass takes, and pairs that
    bind through several patch pairs"""
    _same(_fluid(1331, theta=1.5, eps=0.05), precision, monkeypatch)


@BOTH
def test_chains(precision, monkeypatch):
    s = wl.mt_bundle(1, 13, 40, 25.0, (25.0, 25.0, 60.0))
    rng = np.random.default_rng(2)
    s["x"] = s["x"] + rng.normal(0, 0.02, s["x"].shape)
    s["p"] = rng.normal(0, 1, s["x"].shape)
    s["periodic"] = False
    s["integrator"] = "rotor"
    _same(s, precision, monkeypatch)
