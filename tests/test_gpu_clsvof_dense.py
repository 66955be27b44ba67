"""The transport where most cells are interface cells: a reconstruction lists the
cells of 64 columns by some rows a workgroup, 4, 16 or 32 by the size of the
grid, with those on the west and east edges first, and gives each thread its
share of the list.

Random states (an interface cell in three or four, a run of them up the edges,
three-phase cells without a plane of their own) bit for bit against the CPU
oracle, which evaluates the same expressions in the same order; and the time of a
call on a grid of interface cells only, whose edge cells each take a walk as long
as the edge: done one after the other by one thread they make the call many
times longer."""
import time

import numpy as np
import pytest

from simcoflow_amd import cases as C
from test_gpu_clsvof import _ctx, _random_state, _run_both

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("ni,nj", [(64, 37), (131, 130), (511, 513), (512, 512), (521, 509), (2050, 1030)],
                         ids=lambda n: str(n))
def test_dense_interface_bit_exact(oracle_lib, ni, nj):
    g, geo, vof, phi = _random_state(ni, nj, ni + nj, nonuniform=nj % 2 == 1)
    rng = np.random.default_rng(nj)
    for i in (0, ni - 1):  # a run of interface cells up each edge
        geo.vofS[:, i] = 0.0
        vof[:, i] = rng.uniform(0.1, 0.9, nj)
    u, v = C.transport_velocity(g, "random", amp=0.5, seed=ni, walls=ni % 2 == 0)
    print(f"[clsvof] dense interface {ni}x{nj}", flush=True)
    _run_both(oracle_lib, g, geo, vof, phi, u, v, 0.2 * float(min(g.dx.min(), g.dy.min())), steps=1, nsub=2)


@pytest.mark.parametrize("nj", [30, 63, 64, 65, 66, 67, 68, 131, 200])
def test_run_of_cells_without_a_plane_bit_exact(oracle_lib, nj):
    """Columns of three-phase cells whose solid's line leaves less room than their
    volume: none has a plane constant of its own, and the whole column takes the
    one of the cell before its foot (above, or at the start of the loop, none)."""
    g, geo, vof, phi = _column(40, nj, (0, 1, 12, 13, 30))
    print(f"[clsvof] run of {nj} cells without a plane", flush=True)
    z = np.zeros((nj + 2, 42))
    _run_both(oracle_lib, g, geo, vof, phi, z, z, 1e-9, steps=1, nsub=1)


def _column(ni, nj, cols):
    """A liquid film between x = 0 and 0.4 and columns `cols` of such cells."""
    g, geo, vof, phi = _random_state(ni, nj, 3)
    for a in (geo.vofS, geo.nxS, geo.nyS, geo.phiS):
        a[:] = 0.0
    vof = np.where(g.xc[None, :] < 0.4, 1.0, 0.0) * np.ones((nj, 1))
    for i in cols:
        geo.vofS[:, i], geo.nxS[:, i], geo.phiS[:, i], vof[:, i] = 0.5, 1.0, -0.45 * g.dx[0], 0.3
    return g, geo, vof, np.ascontiguousarray(g.xc[None, :] - 0.4 + np.zeros((nj, 1)))


def _time(pj, dt):
    best = 1e9
    for _ in range(4):
        t = time.perf_counter()
        pj.clsvof_advect_resident(dt)
        pj.synchronize()
        best = min(best, time.perf_counter() - t)
    return best


def _compare(states, n):
    took = {}
    z = np.zeros((n + 2, n + 2))
    for name, (g, geo, vof, phi) in states.items():
        pj = _ctx(g, geo)
        try:
            for k, a in (("VOF", vof), ("PHI", phi), ("U", z), ("V", z)):
                pj.upload(k, np.ascontiguousarray(a))
            took[name] = _time(pj, 1e-9)
        finally:
            pj.close()
    print(f"[clsvof] {took}", flush=True)
    return took


def test_interface_everywhere_costs_no_serial_walks():
    """256 x 256: 2.8 ms against 0.3 ms with a line of interface cells; 50 ms with
    sixteen cells a thread, edge cells among them."""
    n = 256
    case = C.case_swarm(n, n, seed=3)
    g = case.grid
    X, Y = np.meshgrid(g.xc, g.yc)
    line = np.where(Y < 0.5, 1.0, 0.0) + np.where((Y > 0.5) & (Y < 0.5 + g.dy[0]), 1e-3, 0.0)
    wave = np.sin(40 * X) * np.sin(40 * Y)
    took = _compare({"line": (g, case.geo, line, Y - 0.5),
                     "everywhere": (g, case.geo, 0.5 + 0.2 * wave, g.dx[0] * wave)}, n)
    assert took["everywhere"] <= 40 * took["line"]


def test_run_without_a_plane_costs_no_serial_walk():
    """256 x 256: 0.6 ms against 0.2 ms without the column; 15 ms when every cell
    of the run walks back by itself."""
    n = 256
    took = _compare({"none": _column(n, n, ()), "run": _column(n, n, (100,))}, n)
    assert took["run"] <= 15 * took["none"]
