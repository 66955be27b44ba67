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
