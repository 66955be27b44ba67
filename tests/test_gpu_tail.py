"""The one-workgroup tail of the multigrid cycle on levels of every shape: one
to six levels, blocks of 2 x 2 cells that do and do not fit 256 threads, odd
sizes whose last blocks hang over the edge, levels below the second run by one
wavefront from registers, by one wavefront from LDS and by all of them, solid
points, and the constant of an all-Neumann system.  The preconditioned solve
has to reach the direct solution, with the inner iterations and without, the
inner ones costing no outer iterations."""
import numpy as np
import pytest

from simcoflow_amd import cases as C

pytestmark = pytest.mark.gpu

# fine grid -> the tail's first level
SHAPES = [
    (8, 8),      # 4 x 4: the coarsest level alone
    (16, 16),    # 8 x 8 above it
    (32, 32),    # three levels
    (64, 64),    # 32 x 32: the usual four, 256 blocks
    (63, 63),    # the same from an odd size
    (62, 66),    # 31 x 33: 272 blocks
    (34, 108),   # 17 x 54
    (104, 34),   # 52 x 17: third level of 65 points
    (2, 300),    # 1 x 150: five levels, third of 38 points
    (2, 600),    # 1 x 300: third of 75 points
    (18, 40),    # 9 x 20
    (129, 131),  # 65 x 66, 33 x 33, 17 x 17
]


def _case(ni, nj, solid=False):
    lx, ly = 1.0, nj / ni  # square cells: the coarsening is 2 x 2 everywhere
    g = C.uniform_grid(ni, nj, lx, ly)
    sol = (lambda X, Y: C.sdf_circle(X, Y, 0.5 * lx, 0.4 * ly, 0.2 * min(lx, ly))) if solid else None
    geo = C.build_geometry(g, sol)
    itf = C.interface_from_levelset(g, geo, lambda X, Y: (Y - 0.7 * ly, np.zeros(X.shape), np.ones(X.shape)))
    return C.Case("tank", g, C.Fluids(), geo, itf, dt=0.25 * g.dx[0], tol=1e-10, solid=sol)


def _solve(case, precision, krylov, tol=1e-10, bc=(1, 1, 1, 0)):
    from simcoflow_amd.projection import Projection, params_for
    u, v, DpU, DpV = C.predictor_fields(case)
    if bc[3]:
        v[case.grid.nj, :] = 0.0  # closed: the right-hand side sums to zero
    prm = params_for(case.fluids, tol=tol, precision=precision, max_iter=300, bc=bc, mg_coarse_krylov=krylov)
    with Projection(case.grid, prm) as pj:
        pj.set_geometry(case.geo)
        pj.set_interface(case.itf.vof, case.itf.phi)
        pj.set_predictor(u, v, DpU, DpV)
        pj.build(0.0)
        rows, rhs = pj.matrix(), pj.rhs()
        info = pj.solve()
        return pj.download("PP")[1:-1, 1:-1], info, rows, rhs


@pytest.mark.parametrize("precision", [0, 1], ids=["fp64", "mixed"])
@pytest.mark.parametrize("solid", [False, True], ids=["open", "solid"])
@pytest.mark.parametrize("ni,nj", SHAPES)
def test_tail_of_any_shape(oracle_lib, ni, nj, solid, precision):
    import scipy.sparse.linalg as spl
    if solid and min(ni, nj) < 18:
        pytest.skip("no room for a solid")
    print(f"[tail] {ni} x {nj} solid={solid} precision {precision}", flush=True)
    case = _case(ni, nj, solid)
    its = {}
    for krylov in (4, 0):
        p, info, M, b = _solve(case, precision, krylov)
        x = spl.spsolve(oracle_lib.matr_to_scipy(case.grid, case.geo, M).tocsc(), b.ravel()).reshape(case.grid.shape)
        assert info.relres <= 1e-10 * 1.01
        assert np.linalg.norm(p - x) <= 1e-8 * np.linalg.norm(x)
        its[krylov] = info.iterations
    print(f"[tail] iterations {its}", flush=True)
    assert its[4] <= its[0] + 1


@pytest.mark.parametrize("ni,nj,solid,precision", [
    (58, 70, True, 0), (58, 70, False, 1),    # 29 x 35: 270 blocks, of which the last hang over both edges
    (18, 216, True, 0), (18, 216, False, 1),  # 9 x 108: the largest LDS of FP64, third level of 81 points
    (2, 1400, False, 1),                      # 1 x 700: 350 blocks, third level of 175 points (FP32 only)
])
def test_tail_of_more_than_256_blocks(oracle_lib, ni, nj, solid, precision):
    """The levels that take 512 threads, whose weights to level 2, and in FP64
    between the first two levels, stand in LDS."""
    test_tail_of_any_shape(oracle_lib, ni, nj, solid, precision)


@pytest.mark.parametrize("precision", [0, 1], ids=["fp64", "mixed"])
@pytest.mark.parametrize("ni,nj", [(64, 64), (60, 34), (128, 96), (37, 75)])
def test_all_neumann(ni, nj, precision):
    """A closed box leaves the constant undetermined."""
    case = _case(ni, nj)
    p, info, _, _ = _solve(case, precision, 4, tol=1e-9, bc=(1, 1, 1, 1))
    q, _, _, _ = _solve(case, precision, 0, tol=1e-9, bc=(1, 1, 1, 1))
    assert info.relres <= 1e-9 * 1.01 and np.isfinite(p).all()
    p, q = p - p.mean(), q - q.mean()
    assert np.linalg.norm(p - q) <= 1e-7 * np.linalg.norm(q)
