"""The PCG scalars at the numbers of partial sums where the way they are added up
changes: a few, whole and broken groups of 64 of them added by the kernels that
use them, and the first number that takes a launch of its own.  The solution
has to satisfy the assembled rows to the solve's tolerance (in numpy, with 1%
for the rounding of that evaluation), and the first size that takes the launch
needs the iterations of the last one that does not, give or take the two that a
column of cells more may cost."""
import numpy as np
import pytest

from test_gpu_tail import _solve, _case

pytestmark = pytest.mark.gpu

# cells -> partials of the 64 x 16 tiles
SIZES = [(64, 64, 4), (256, 256, 64), (384, 192, 72), (500, 479, 240), (512, 512, 256), (513, 512, 288)]


@pytest.mark.parametrize("precision", [0, 1], ids=["fp64", "mixed"])
def test_sums_of_any_number_of_partials(oracle_lib, precision):
    tol, its = 1e-9, {}
    for ni, nj, partials in SIZES:
        assert -(-ni // 64) * -(-nj // 16) == partials
        print(f"[pcg sums] {ni}x{nj} {partials} partials precision {precision}", flush=True)
        case = _case(ni, nj)
        p, info, M, b = _solve(case, precision, 4, tol=tol)
        A = oracle_lib.matr_to_scipy(case.grid, case.geo, M)
        r = b.ravel() - A @ p.ravel()
        assert np.linalg.norm(r) <= 1.01 * tol * np.linalg.norm(b), partials
        its[partials] = info.iterations
    print(f"[pcg sums] iterations {its}", flush=True)
    assert abs(its[288] - its[256]) <= 2


@pytest.mark.parametrize("precision", [0, 1], ids=["fp64", "mixed"])
@pytest.mark.parametrize("ni,nj,partials", SIZES + [(7, 5, 1), (130, 16, 3), (448, 250, 112)])
def test_sums_are_those_of_a_finalize_launch(monkeypatch, ni, nj, partials, precision):
    """The same solve with the sums added up by the kernels that use them and by
    launches of their own: the same iterations and the same pressure in every bit,
    which any other order of a sum's terms would change."""
    assert -(-ni // 64) * -(-nj // 16) == partials
    print(f"[pcg sums] fused or not {ni}x{nj} {partials} partials precision {precision}", flush=True)
    case = _case(ni, nj)
    got = []
    for off in ("0", "1"):
        monkeypatch.setenv("SG_NO_FUSED_SUMS", off)
        p, info, _, _ = _solve(case, precision, 4, tol=1e-9)
        got.append((p, info.iterations, info.relres))
    assert got[0][1:] == got[1][1:]
    assert np.array_equal(got[0][0], got[1][0])
