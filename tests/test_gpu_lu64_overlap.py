"""FP64 cases whose LU-SGS sweeps span several workgroups (k_lu_sweep64) on
streams of their own.

The workgroups of such a sweep wait for one another's mail, as those of the
FP32 sweeps do, so by default the library keeps the steps of different such
cases apart on a device, and overlapping them (ot2d_set_fp32_order(0)) must
not change a bit either.
"""
import numpy as np
import pytest

from turns2d_urans_git_amd import abi, grid

pytestmark = pytest.mark.gpu

SA_DECK = dict(fsmach=0.5, alfa=2.0, rey=4.0e6, invisc=0, lamin=0, iturb=1, vnuinf=3.0, irhsy=-3, ilim=1, ilhs=1,
               iconstant_cfl=1, dt=5.0, epse=0.01, iunst=0, ntac=1, itnmax=1, timeac=1.0)


def _batch(shapes, alfa0=0.0):
    import turns2d_urans_git_amd as t2d
    gs = [grid.naca4_cgrid(j, k, m=0.0, p=0.0, t=0.12, ds_wall=1e-5, wake_aspect=1000.0, te_cluster=False)
          for j, k in shapes]
    ps = [t2d.default_params(**dict(SA_DECK, alfa=alfa0 + 0.25 * i), lu_fp32=0) for i in range(len(gs))]
    b = t2d.Batch(ps, [abi.mesh_desc(g.jmax, g.kmax, grid.cgrid_bc(g.jtail1)) for g in gs])
    for i, g in enumerate(gs):
        b.set_grid(i, g.xv, g.yv)
    return b


def test_steps_of_multiblock_cases_are_ordered():
    """A case enqueued behind another's 400 steps ends after them: by the time
    its one step is done, the other is idle."""
    print("[lu64 order] 193x97 behind 257x129", flush=True)
    a, b = _batch([(257, 129)]), _batch([(193, 97)])
    for c in (a, b):   # capture both steps
        c.iterate_async(1)
        c.sync()
    a.iterate_async(400)
    b.iterate_async(1)
    b.sync()
    assert a.idle()
    for c in (a, b):
        st, ist = c.batch_status()
        assert list(st) == [0], st
        c.close()


@pytest.mark.parametrize("ordered", [True, False])
def test_overlapped_batches_equal_alone(ordered):
    """Three FP64 batches (2 to 6 blocks of 32 rows, one case of one block)
    enqueued on three streams at once against the same batches run with
    nothing beside them, bit for bit, checked every 100 steps."""
    import turns2d_urans_git_amd as t2d
    lib = t2d.load_library()
    shapes = [[(257, 97), (129, 193), (97, 33)], [(193, 129), (161, 65), (225, 66)], [(129, 161), (289, 98), (65, 34)]]
    over = [_batch(s, n) for n, s in enumerate(shapes)]
    alone = [_batch(s, n) for n, s in enumerate(shapes)]
    abi.set_fp32_order(lib, "ot2d_", ordered)
    try:
        for chunk in range(8):
            for b in over:
                b.iterate_async(100)
            for b in over:
                b.sync()
            for b in alone:
                b.iterate_async(100)
                b.sync()
            for n, (x, y) in enumerate(zip(over, alone)):
                sx, sy = x.batch_status(), y.batch_status()
                np.testing.assert_array_equal(sx[0], sy[0], err_msg=f"status, batch {n}, chunk {chunk}")
                np.testing.assert_array_equal(sx[1], sy[1], err_msg=f"steps, batch {n}, chunk {chunk}")
                for i in range(len(shapes[n])):
                    assert np.array_equal(x.get_state(i), y.get_state(i), equal_nan=True), \
                        f"batch {n} case {i} differs after {100 * (chunk + 1)} steps (ordered={ordered})"
            print(f"[lu64 overlap ordered={ordered}] {100 * (chunk + 1)} steps equal", flush=True)
    finally:
        abi.set_fp32_order(lib, "ot2d_", True)
    for b in over + alone:
        b.close()
