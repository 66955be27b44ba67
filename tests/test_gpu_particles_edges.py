"""The particle tracker where its look-up, its quotients and its count can go
wrong: an uneven grid (the column is not where an even spacing puts it), sets
that fill one workgroup, miss it or run over by one, failed particles in the
first, the last and no workgroup, and particles so small or light that the
quotients by their own constants leave the range of the quick ones.  Against
the CPU oracle, 1e-12 of the scale: pow and exp are two libraries'."""
import numpy as np
import pytest

from simcoflow_amd import cases as C
from test_gpu_clsvof import _random_state
from test_gpu_particles import _close, _device, _params, _particles

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n", [1, 64, 255, 256, 257, 1000])
@pytest.mark.parametrize("tiny", [False, True], ids=["usual", "tiny"])
def test_uneven_grid_and_counts(oracle_lib, n, tiny):
    g, geo, vof, phi = _random_state(48, 40, 5, nonuniform=True)
    case = C.Case("uneven", g, C.Fluids(), geo, C.Interface(vof, phi, np.zeros_like(vof), np.ones_like(vof)), dt=1e-3,
                  tol=1e-8)
    u, v = C.transport_velocity(g, "random", amp=0.3, seed=2)
    parts = [np.array(a) for a in _particles(g, n, n, with_edges=n >= 64)]
    if tiny:
        parts[4][::3] = 1e-30  # its Reynolds number and drag are far outside the usual
    if n >= 255:
        parts[2][[0, n - 1]] = np.nan  # fail in the first and the last workgroup
    P = _params(case)
    print(f"[particles] uneven 48x40, {n} particles tiny={tiny}", flush=True)
    (x, y, pu, pv), flagged = _device(case, u, v, parts, P, 1e-3, 2)
    o, flags = list(parts), []
    for _ in range(2):
        o[0], o[1], o[2], o[3], bad = oracle_lib.particle_track(g, vof, geo.vofS, u, v, o[0], o[1], o[2], o[3], o[4],
                                                                P, 1e-3)
        flags.append(bad)
    assert flagged == flags
    for a, b in ((x, o[0]), (y, o[1]), (pu, o[2]), (pv, o[3])):
        fin = np.isfinite(b)
        assert np.array_equal(np.isfinite(a), fin)
        _close("state", a[fin], b[fin], np.maximum(1.0, np.abs(b[fin])))
