"""Empty interaction sets through the setters: no exclusions after some, no
bonds, no angles, patch types without any patch.  The engine then computes what
one computes that was never given them."""
import numpy as np
import pytest

from mtcode_amd import mdx
from mtcode_amd import workloads as wl

pytestmark = pytest.mark.gpu

PRECISION = pytest.mark.parametrize("precision", [mdx.PREC_FP64, mdx.PREC_MIXED])


def _gas(n, integrator):
    rng = np.random.default_rng(n)
    side = int(np.ceil(n ** (1 / 3)))
    ijk = np.stack([np.arange(n) % side, np.arange(n) // side % side, np.arange(n) // side ** 2], 1)
    s = wl._base("gas", n, side * 1.1 + 3.0, 0.002, 1.0, 1.0, 1.0 / 3.0, integrator)
    s["x"] = (ijk + 0.5) * 1.1 + rng.uniform(-0.02, 0.02, (n, 3))
    s["Q"] = wl.arvo_rotations(n, rng)
    return wl.thermal_momenta(s, 3)


def _frame(e, rotor):
    out = {}
    out["F"], out["T"] = e.compute_forces()
    if rotor:
        e.prime()
    e.step(5)
    out.update(e.download())
    return out


@PRECISION
@pytest.mark.parametrize("integrator", ["bead", "rotor"])
def test_topology_taken_back(integrator, precision):
    s = _gas(300, integrator)
    pairs = np.array([[0, 1], [1, 2]], dtype=np.int32)
    none2, none3 = np.zeros((0, 2), dtype=np.int32), np.zeros((0, 3), dtype=np.int32)
    with mdx.engine_from_system(s, precision=precision, seed=4) as e:
        ref = _frame(e, integrator == "rotor")
    with mdx.engine_from_system(s, precision=precision, seed=4) as e:
        e.set_exclusions(pairs)
        e.set_bonds(pairs, [1.0, 1.0], [1.0, 1.0])
        e.set_angles([[0, 1, 2]], [2.0], [0.0])
        e.set_exclusions(none2)
        e.set_bonds(none2, [], [])
        e.set_angles(none3, [], [])
        got = _frame(e, integrator == "rotor")
    for k in ref:
        assert np.array_equal(got[k], ref[k]), k


@PRECISION
@pytest.mark.parametrize("types", [1, 3])
def test_types_without_patches(types, precision):
    s = _gas(300, "rotor")
    with mdx.engine_from_system(s, precision=precision, seed=4) as e:
        ref = _frame(e, True)
    with mdx.engine_from_system(s, precision=precision, seed=4) as e:
        e.set_patches(np.arange(300) % types, [0] * types, [], np.zeros((0, 3)))
        got = _frame(e, True)
    for k in ref:
        assert np.array_equal(got[k], ref[k]), k
