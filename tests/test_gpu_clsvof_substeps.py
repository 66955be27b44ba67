"""The transport with many sub-steps a call: up to the most it takes, bit for bit
against the CPU oracle as elsewhere, and refused beyond; the sweep timer's pool of
event pairs runs out within one."""
import ctypes

import numpy as np
import pytest

from simcoflow_amd import cases as C
from test_gpu_clsvof import _ctx, _run_both

pytestmark = pytest.mark.gpu


def _case():
    case = C.case_bubble(16, 32)
    u, v = C.transport_velocity(case.grid, "vortex", amp=0.5, seed=1)
    return case, u, v


@pytest.mark.parametrize("nsub", [255, 256, 257, 600])
def test_sweep_timer_counts_every_sweep(nsub):
    """Two sweeps a sub-step, over two calls, with a pool of 512 pairs."""
    from simcoflow_amd import _lib
    case, u, v = _case()
    print(f"[clsvof] sweep timer, {nsub} sub-steps", flush=True)
    pj = _ctx(case.grid, case.geo)
    try:
        _lib.check(pj.lib.sg_sweep_timing(pj.ctx, 1, None, None))
        for _ in range(2):
            vof, phi, _, _ = pj.clsvof_advect(case.itf.vof, case.itf.phi, u, v, 1e-4, nsub=nsub)
        n, ms = ctypes.c_longlong(0), ctypes.c_double(0.0)
        _lib.check(pj.lib.sg_sweep_timing(pj.ctx, 0, ctypes.byref(n), ctypes.byref(ms)))
    finally:
        pj.close()
    assert n.value == 4 * nsub and ms.value > 0.0
    assert np.isfinite(vof).all() and np.isfinite(phi).all()


@pytest.mark.parametrize("nsub", [614, 615, 1024])
def test_most_sub_steps_bit_exact(oracle_lib, nsub):
    case, u, v = _case()
    print(f"[clsvof] {nsub} sub-steps", flush=True)
    _run_both(oracle_lib, case.grid, case.geo, case.itf.vof, case.itf.phi, u, v, case.dt, steps=1, nsub=nsub)


@pytest.mark.parametrize("nsub", [-1, 0, 1025])
def test_sub_steps_out_of_range_refused(nsub):
    from simcoflow_amd import _lib
    case, u, v = _case()
    pj = _ctx(case.grid, case.geo)
    try:
        with pytest.raises(_lib.SimcoError, match=r"nsub must be in \[1, 1024\]"):
            pj.clsvof_advect(case.itf.vof, case.itf.phi, u, v, case.dt, nsub=nsub)
    finally:
        pj.close()
