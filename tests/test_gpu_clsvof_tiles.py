"""The transport at the edges of its kernels' tiles, bit for bit against the
CPU oracle: a sweep's 32 x 8 cells (every thread works out an inner cell, so a
ring cell may be alone in its tile), the 64-cell words of the class bits, the
64 x 64 cells of a reconstruction, and the tiles found free of solid, which
exist from 2^21 cells up.

The oracle evaluates the same expressions in the same order without FP
contraction, so nothing may differ in any bit.
"""
import dataclasses

import numpy as np
import pytest

from simcoflow_amd import cases as C
from test_gpu_clsvof import _random_state, _run_both

pytestmark = pytest.mark.gpu

SHAPES = [(4, 4), (5, 4), (4, 9), (33, 9), (32, 8), (34, 17), (64, 64), (65, 65), (97, 66), (129, 10), (63, 128)]


@pytest.mark.parametrize("ni,nj", SHAPES, ids=[f"{a}x{b}" for a, b in SHAPES])
def test_tile_edges_bit_exact(oracle_lib, ni, nj):
    g, geo, vof, phi = _random_state(ni, nj, ni * 1000 + nj, nonuniform=nj % 2 == 1)
    u, v = C.transport_velocity(g, "random", amp=0.5, seed=ni, walls=ni % 2 == 0)
    print(f"[clsvof] tile edges {ni}x{nj}", flush=True)
    _run_both(oracle_lib, g, geo, vof, phi, u, v, 0.2 * float(min(g.dx.min(), g.dy.min())), steps=1, nsub=3)


@pytest.mark.parametrize("ni,nj", [(1472, 1427), (2049, 1025)])
def test_open_tiles_bit_exact(oracle_lib, ni, nj):
    """Solid, part-open faces and masked faces on single cells around the edges
    of tiles that are otherwise free of them, one kind of disturbance at a time."""
    case = C.case_swarm(ni, nj, seed=7)
    g, geo = case.grid, case.geo
    vofS, uflag, vflag = (np.array(a, order="C") for a in (geo.vofS, geo.uflag, geo.vflag))
    ap = {k: np.array(getattr(geo, k), order="C") for k in ("aE", "aW", "aN", "aS")}
    rng = np.random.default_rng(ni)
    # offsets within a tile: its corners, the cells just outside, one inside
    spots = [(-1, 3), (32, 4), (0, 0), (31, 7), (15, -1), (16, 8), (10, 4)]
    kinds = ["vofS", "aE", "aW", "aN", "aS", "uflag", "vflag"]
    for n, (kind, (dx, dy)) in enumerate((k, s) for k in kinds for s in spots):
        i = 32 * (2 + 2 * (n % 6)) + dx
        j = 8 * (3 + 3 * (n // 6)) + dy
        if kind == "vofS":
            vofS[j, i] = rng.uniform(0.05, 0.9)
        elif kind == "uflag":
            uflag[j, i] = 0
        elif kind == "vflag":
            vflag[j, i] = 0
        else:
            ap[kind][j + 1, i + 1] = rng.uniform(0.0, 0.99)
    geo = dataclasses.replace(geo, vofS=vofS, uflag=uflag, vflag=vflag, **ap)
    vof = np.ascontiguousarray(np.minimum(case.itf.vof, 1.0 - vofS))
    u, v = C.transport_velocity(g, "vortex", amp=1.0, seed=3)
    print(f"[clsvof] open tiles {ni}x{nj}", flush=True)
    _run_both(oracle_lib, g, geo, vof, case.itf.phi, u, v, case.dt, steps=1, nsub=2)
