"""Forces from the cells with several lanes per position in boxes of three, two
and one cell a side (the seam's rows, the stencils with fewer rows), against the
one-lane kernel bit for bit, and against every pair's minimum image."""
import numpy as np
import pytest

from mtcode_amd import mdx
from mtcode_amd import workloads as wl
from test_gpu_cells import BOTH, _fluid, _same

pytestmark = pytest.mark.gpu

BOXES = pytest.mark.parametrize("n,box,cells", [
    (125, (6.0, 6.0, 6.0), (3, 3, 3)), (64, (4.5, 4.5, 4.5), (2, 2, 2)), (27, (3.5, 3.5, 3.5), (1, 1, 1)),
    (64, (6.0, 4.5, 12.0), (3, 2, 6)), (64, (4.5, 12.0, 6.0), (2, 6, 3)), (125, (12.0, 6.0, 6.0), (6, 3, 3))])


@BOTH
@BOXES
def test_few_cells_a_side(n, box, cells, precision, monkeypatch):
    s = _fluid(n, box=box)
    with mdx.engine_from_system(s, precision=precision) as e:
        assert e.info()["cells"] == cells[0] * cells[1] * cells[2]
    _same(s, precision, monkeypatch)


@BOXES
def test_wca_of_every_pair(n, box, cells):
    s = _fluid(n, box=box)
    s["wca"] = (1.0, 1.0, 0.0)
    s["patches"]["params"][:, 0] = 1e-300  # the patch path, without its forces
    with mdx.engine_from_system(s, precision=mdx.PREC_FP64) as e:
        F, _ = e.compute_forces()
    d = s["x"][:, None] - s["x"][None]
    b = np.array(box)
    d -= np.where(np.abs(d) > 0.5 * b, np.where(d >= 0, b, -b), 0.0)
    r2 = (d * d).sum(-1)
    np.fill_diagonal(r2, 1e9)
    i6 = 1.0 / r2 ** 3
    f = np.where(r2 < wl.WCA_CUT_LITERAL ** 2, 24.0 * (2.0 * i6 * i6 - i6) / r2, 0.0)
    ref = (f[..., None] * d).sum(1)
    assert np.abs(ref).max() > 1.0
    # sums in another order
    assert np.abs(F - ref).max() < 1e-11 * np.abs(ref).max()
