"""Exclusions replaced between two calls of an engine whose neighbour list is
live: the steps that follow use the new ones at once.  A list is built without
the pairs that were excluded then, and its walk does not look at exclusions
where it holds none, so it must not outlive them.  Against engines without a
list; a few steps, so that neither a rebuild nor a re-sort comes in between."""
import numpy as np
import pytest
from scipy.spatial import cKDTree

from mtcode_amd import mdx
from mtcode_amd import workloads as wl

pytestmark = pytest.mark.gpu


def _system(kind, n=700):
    rng = np.random.default_rng(7)
    side = int(np.ceil(n ** (1 / 3)))
    pitch = 1.1
    site = rng.permutation(side ** 3)[:n]
    ijk = np.stack([site % side, site // side % side, site // side ** 2], 1)
    s = wl._base("gas", n, side * pitch + 2.0, 0.002, 1.0, 1.0, 1.0 / 3.0, kind)
    s["x"] = (ijk + 0.5) * pitch + rng.uniform(-0.02, 0.02, (n, 3))
    s["Q"] = wl.arvo_rotations(n, rng)
    if kind == "rotor":
        ps = wl.two_species_patchset(6.0)
        types = np.zeros(n, dtype=np.int32)
        types[n // 2:] = 1
        ps["types"], ps["maxd2"] = types, 2.4
        s["patches"] = ps
    near = cKDTree(s["x"]).query_pairs(1.12, output_type="ndarray")
    near = near[np.lexsort((near[:, 1], near[:, 0]))]
    # (at most two exclusions per particle in either half)
    return wl.thermal_momenta(s, 3), near[0::3].astype(np.int32), near[1::3].astype(np.int32)


def _run(kind, skin, form):
    s, first, second = _system(kind)
    out = []
    with mdx.engine_from_system(s, precision=mdx.PREC_FP64, seed=5) as e:
        if skin is not None:
            e.set_neighbor_list(skin=skin)
        e.set_exclusions(first)
        if kind == "rotor":
            e.prime()
        e.step(6)
        if form == "replace":
            e.set_exclusions(second)
        else:
            e.set_exclusions(np.zeros((0, 2), dtype=np.int32))
        builds = e.info()["list_builds"]
        e.step(6)
        out = e.download()
        return out, builds


@pytest.mark.parametrize("form", ["replace", "none"])
@pytest.mark.parametrize("kind", ["bead", "rotor"])
def test_new_exclusions_count_at_once(kind, form):
    got, builds = _run(kind, None, form)
    ref, none = _run(kind, 0.0, form)
    assert builds >= 1 and none == 0
    for k in ("x", "p"):
        # the sums run in another order: FP64 rounding over 12 steps
        assert np.abs(got[k] - ref[k]).max() < 1e-10, k
