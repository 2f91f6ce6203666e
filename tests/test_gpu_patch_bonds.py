"""Patch bonds per particle against every patch pair in FP64 numpy: types with 0
to 6 patches, a row of its own for each patch pair (depths of zero among them,
narrow and wide cones), both precisions, periodic and walls.  Particles with a
decision closer to its threshold than the stored orientations' rounding are
left out of the comparison."""
import numpy as np
import pytest

from mtcode_amd import mdx
from mtcode_amd import workloads as wl

pytestmark = pytest.mark.gpu

NP = [6, 0, 3, 1]


def _system(n, L, periodic, seed):
    rng = np.random.default_rng(seed)
    s = wl._base("mix", n, L, 0.005, 1.0, 1.0, 1.0 / 3.0, "rotor")
    s["periodic"] = periodic
    s["x"] = rng.uniform(0, L, (n, 3))
    s["Q"] = wl.arvo_rotations(n, rng)
    dirs = rng.normal(size=(sum(NP), 3))
    dirs /= np.linalg.norm(dirs, axis=1)[:, None]
    rows = sum(NP[i] * NP[j] for i in range(4) for j in range(i, 4))
    params = np.stack([rng.choice([0.0, 3.0, 6.0], rows), rng.uniform(0.9, 1.3, rows),
                       rng.uniform(0.2, 1.3, rows)], 1)
    s["patches"] = {"npatch": NP, "dirs": dirs, "params": params, "maxd2": 2.9,
                    "types": rng.integers(0, 4, n).astype(np.int32)}
    return s


def _brute(s, Q, near):
    """bonds per particle, and the particles with a decision nearer than near"""
    x, L, ps = s["x"], s["box"], s["patches"]
    n, types = len(x), ps["types"]
    first = np.concatenate([[0], np.cumsum(NP)])
    row0, r = {}, 0
    for i in range(4):
        for j in range(i, 4):
            row0[i, j] = r
            r += NP[i] * NP[j]
    bonds, close = np.zeros(n, dtype=int), np.zeros(n, dtype=bool)
    for i in range(n):
        for j in range(i + 1, n):
            d = x[i] - x[j]
            if s["periodic"]:
                d = np.where(np.abs(d) > 0.5 * L, d - np.sign(d) * L, d)
            r2 = d @ d
            if r2 >= ps["maxd2"]:
                continue
            rij = np.sqrt(r2)
            # role a: the lower type (of equal ones the lower index)
            a, c, u = (i, j, d / rij) if types[i] <= types[j] else (j, i, -d / rij)
            ta, tc = types[a], types[c]
            na = ps["dirs"][first[ta]:first[ta + 1]] @ Q[a].reshape(3, 3)
            nc = ps["dirs"][first[tc]:first[tc + 1]] @ Q[c].reshape(3, 3)
            bonded = False
            for p, u1 in enumerate(na):
                for q, u2 in enumerate(nc):
                    eps, dd, th = ps["params"][row0[ta, tc] + p * NP[tc] + q]
                    if eps == 0.0:
                        continue
                    m = [1.4 * dd - rij, -(u1 @ u) - np.cos(th), u2 @ u - np.cos(th)]
                    bonded |= min(m) > 0
                    if min(m) > -near and min(np.abs(m)) < near:
                        close[[i, j]] = True
            bonds[i] += bonded
            bonds[j] += bonded
    return bonds, close


@pytest.mark.parametrize("periodic", [True, False])
@pytest.mark.parametrize("precision", [mdx.PREC_FP64, mdx.PREC_MIXED])
@pytest.mark.parametrize("n,L", [(1, 6.0), (2, 1.7), (257, 7.0), (500, 12.0)])
def test_bonds(n, L, precision, periodic):
    s = _system(n, L, periodic, n)
    fp64 = precision == mdx.PREC_FP64
    Q = s["Q"] if fp64 else wl.mixed_orientations(s["Q"])
    want, close = _brute(s, Q, 1e-12 if fp64 else 1e-6)
    with mdx.engine_from_system(s, precision=precision) as e:
        got = e.patch_bonds()
    assert close.sum() <= n // 20
    assert n < 3 or want.max() >= 3
    assert np.array_equal(got[~close], want[~close])
