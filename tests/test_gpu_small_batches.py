"""Batches of many small grids: each case equals itself alone, bit for bit.

A case's tiles are dealt out in runs per XCD, among the workgroups that the
batch's largest case needs.  The grids have 1 to 8 and more tiles of every kernel that deals them
out: 32x8 cells (viscous terms, SA right-hand side), 256 cells (SST blend and
right-hand side), 8 columns (line solves), FP32 operator tiles.
"""
import numpy as np
import pytest

from turns2d_urans_git_amd import abi, grid

pytestmark = pytest.mark.gpu

DECK = dict(fsmach=0.4, alfa=1.0, rey=1.0e6, invisc=0, lamin=0, vnuinf=3.0, irhsy=-3, ilim=1, ilhs=1, iconstant_cfl=1,
            dt=2.0, epse=0.01, iunst=0, ntac=1, itnmax=1, timeac=1.0)
SHAPES = [(33, 17), (17, 9), (33, 33), (65, 33), (41, 25), (17, 41), (67, 9), (97, 17), (35, 18), (33, 65), (49, 57)]


@pytest.mark.parametrize("iturb,fp32", [(1, 0), (1, 1), (2, 0), (2, 1)])
def test_batch_equals_alone(iturb, fp32):
    import turns2d_urans_git_amd as t2d
    print(f"[small batches] iturb {iturb} fp32 {fp32}", flush=True)
    gs = [grid.naca4_cgrid(j, k, ds_wall=1e-3) for j, k in SHAPES]
    ps = [t2d.default_params(**dict(DECK, iturb=iturb, alfa=0.1 * i), lu_fp32=fp32) for i in range(len(gs))]
    ms = [abi.mesh_desc(g.jmax, g.kmax, grid.cgrid_bc(g.jtail1)) for g in gs]
    b = t2d.Batch(ps, ms)
    for i, g in enumerate(gs):
        b.set_grid(i, g.xv, g.yv)
    rc, _, done = b.iterate(10)
    st, _ = b.batch_status()
    for i, g in enumerate(gs):
        one = t2d.Case(ps[i], [ms[i]])
        one.set_grid(0, g.xv, g.yv)
        rc1, _, _ = one.iterate(10)
        assert rc1 == st[i], (i, rc1, st[i])
        np.testing.assert_array_equal(b.get_state(i), one.get_state(0), err_msg=f"case {i}, {SHAPES[i]}")
        np.testing.assert_array_equal(b.get_field(i, abi.F_TURMU), one.get_field(0, abi.F_TURMU),
                                      err_msg=f"case {i}, {SHAPES[i]}")
        one.close()
    b.close()
