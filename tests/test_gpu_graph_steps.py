"""List steps replayed as graphs of one and of eight steps against eager
launches, bit for bit: calls that end before, at and after a multiple of
eight, a re-sort inside the run, other eager work between the replays."""
import numpy as np
import pytest

from mtcode_amd import mdx
from mtcode_amd import workloads as wl

pytestmark = pytest.mark.gpu


def _states(s, precision, resort, graph, monkeypatch):
    monkeypatch.setenv("MDX_GRAPH", str(graph))
    out = []
    with mdx.engine_from_system(s, precision=precision, seed=9) as e:
        e.set_neighbor_list(resort_every=resort)
        if s["integrator"] == "rotor":
            e.prime()
        for n in (1, 9, 10, 11, 17, 8, 26, 7, 18, 33):
            e.step(n)
            out.append(e.download())
            out[-1]["count"] = np.array(e.noise_counter())
            out[-1]["epot"] = np.array(e.observables()["epot"])
        return out


@pytest.mark.parametrize("precision", [mdx.PREC_FP64, mdx.PREC_MIXED])
@pytest.mark.parametrize("kind,resort", [("rotor", 200), ("rotor", 13), ("bead", 200), ("bead", 13),
                                         ("bind", 200)])
def test_replays_equal_eager(kind, resort, precision, monkeypatch):
    if kind == "bead":
        s = wl.mt_bundle(1, 13, 60, 25.0, (25.0, 25.0, 80.0))
        s = wl.thermal_momenta(s, 3)
    else:
        s = wl.thermal_momenta(wl.patchy_tetra(600), 3)
        if kind == "bind":
            s["binding"] = (0.6, 0.4)
    a = _states(s, precision, resort, 1, monkeypatch)
    b = _states(s, precision, resort, 0, monkeypatch)
    for x, y in zip(a, b):
        for k in x:
            assert np.array_equal(x[k], y[k]), k
