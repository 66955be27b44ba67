"""The cut-cell geometry of solids at and over the domain's edges, on grids that
do not fill or just overrun the kernels' tiles: a closed U or V cell there has
neighbours, or ghosts, on the other side of a tile's or the grid's edge, whose
faces it shuts.  Bit for bit against the host builder, as both write the same
expressions."""
import pytest

from simcoflow_amd import cases as C
from test_gpu_geometry import _compare, _fresh, _shape

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("ni,nj", [(4, 4), (31, 9), (33, 8), (65, 34)])
def test_solids_at_the_edges(ni, nj):
    from simcoflow_amd.projection import Projection, params_for
    g = C.uniform_grid(ni, nj, 1.0, nj / ni)
    ly = nj / ni
    pj = Projection(g, params_for(C.Fluids()))
    prev = _fresh(g)
    try:
        for kind, cx, cy, a, b in [("box", 0.0, 0.0, 0.4, 0.4 * ly), ("box", 1.0, ly, 0.33, 0.45 * ly),
                                   ("circle", 1.0, 0.0, 0.45 * min(1.0, ly), 0.0), ("box", 0.5, 0.5 * ly, 0.6, 0.2 * ly),
                                   ("box", 0.5, 0.5 * ly, 2.0, 2.0)]:
            print(f"[geometry edges] {ni}x{nj} {kind} at ({cx}, {cy}) sizes ({a}, {b})", flush=True)
            pj.geometry_rebuild(kind, cx, cy, a, b)
            errs, _, prev = _compare(pj, g, _shape(kind, cx, cy, a, b), prev)
            assert not errs, "\n".join(errs)
    finally:
        pj.close()
