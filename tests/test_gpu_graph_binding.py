"""List steps of a system under binding whose patch numbering changes between
calls: the steps replayed from graphs against eager launches, bit for bit.
The same patch definitions with another type of each particle leave the pair
kernels' arguments as they were; the number of patches, and with it the grids
and arrays of the binding kernels, differs (larger, smaller, as at first)."""
import numpy as np
import pytest

from mtcode_amd import mdx
from mtcode_amd import workloads as wl

pytestmark = pytest.mark.gpu

N = 1500


def _run(graph, precision, monkeypatch):
    monkeypatch.setenv("MDX_GRAPH", str(graph))
    s = wl.thermal_momenta(wl.condensate_ab(N), 3)
    s["binding"] = (0.6, 0.4)
    ps = s["patches"]
    order = np.random.default_rng(4).permutation(N)
    out = []
    with mdx.engine_from_system(s, precision=precision, seed=9) as e:
        for with_three in (N // 5, 4 * N // 5, N // 3, N // 5):
            types = np.ones(N, dtype=np.int32)
            types[order[:with_three]] = 0
            e.set_patches(types, ps["npatch"], ps["dirs"], ps["params"], ps["maxd2"])
            assert e.set_binding(0.6, 0.4) == 2 * N + with_three
            e.prime()
            for n in (12, 31):
                e.step(n)
                out.append(e.download())
                out[-1]["bound"], out[-1]["to"] = e.get_bindings()
    return out


@pytest.mark.parametrize("precision", [mdx.PREC_FP64, mdx.PREC_MIXED])
def test_patch_numbering_changes_between_replays(precision, monkeypatch):
    a = _run(1, precision, monkeypatch)
    b = _run(0, precision, monkeypatch)
    assert any(x["bound"].any() for x in b)
    for x, y in zip(a, b):
        for k in x:
            assert np.array_equal(x[k], y[k]), k
