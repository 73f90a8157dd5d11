"""FP64 LU-SGS sweeps of several blocks (k_lu_sweep64) in the forms a single
steady case does not reach: grid velocities and several instances of one case
(time-spectral, against the oracle), and a batch slot taken over by a grid of
another number of blocks (against the grid alone, bit for bit).

Bound of the time-spectral runs: residual norms and state per cell to 1e-10,
that of the time-spectral trajectories of one block (FP64 throughout; the
instances' metrics come from the device's sine and cosine)."""
import numpy as np
import pytest

from tests import helpers as H
from turns2d_urans_git_amd import abi, grid

pytestmark = pytest.mark.gpu

BASE = dict(irhsy=-3, ilim=1, ilhs=1, iconstant_cfl=1, epse=0.01, iunst=0, ntac=1, itnmax=1, timeac=1.0)
EULER = dict(BASE, invisc=1, lamin=1)
SA = dict(BASE, invisc=0, lamin=0, iturb=1, vnuinf=3.0, rey=1.0e6)


@pytest.mark.parametrize("deck", [EULER, SA], ids=["euler", "sa"])
@pytest.mark.parametrize("jm,km", [(41, 34), (65, 65), (49, 98)])
def test_time_spectral_vs_oracle(jm, km, deck):
    print(f"[lu64 forms] time-spectral {jm}x{km}", flush=True)
    g = H.cgrid(jm, km, ds_wall=1e-3)
    d = dict(deck, fsmach=0.3, alfa=-1.0, angmax=2.0, rf=0.05, dt=5.0, timespectral=1, nspec=3, motiontype=1)
    o, c = H.oracle_case(g, d), H.gpu_case(g, d)
    ro, ho, no = o.iterate(6)
    rc, hc, nc = c.iterate(6)
    assert ro == rc == 0 and no == nc == 6
    assert np.abs(c.get_field(0, abi.F_UG)).max() > 0.0
    np.testing.assert_allclose(hc, ho, rtol=1e-10)
    H.assert_cellwise(c.get_state(0), o.get_state(0), 1e-10, "q (all instances)")
    c.close()


@pytest.mark.parametrize("first,second", [((65, 98), (65, 34)), ((49, 66), (41, 65)), ((49, 34), (49, 25))])
def test_slot_taken_over_with_other_blocks(first, second):
    import turns2d_urans_git_amd as t2d
    print(f"[lu64 forms] slot of {first} taken by {second}", flush=True)

    def case(shape, alfa):
        g = H.cgrid(*shape, ds_wall=1e-3)
        return g, t2d.default_params(**dict(SA, fsmach=0.4, alfa=alfa, dt=2.0)), \
            abi.mesh_desc(g.jmax, g.kmax, grid.cgrid_bc(g.jtail1))

    (ga, pa, ma), (gb, pb, mb), (gn, pn, mn) = case(first, 1.0), case((57, 66), 2.0), case(second, 0.5)
    b = t2d.Batch([pa, pb], [ma, mb])
    b.set_grid(0, ga.xv, ga.yv)
    b.set_grid(1, gb.xv, gb.yv)
    rc, _, _ = b.iterate(10)
    assert rc == 0
    b.batch_retire(0)
    b.batch_admit(0, pn, mn)
    b.set_grid(0, gn.xv, gn.yv)
    rc, _, _ = b.iterate(15)
    assert rc == 0
    for slot, g, p, m, n in ((0, gn, pn, mn, 15), (1, gb, pb, mb, 25)):
        one = t2d.Case(p, [m])
        one.set_grid(0, g.xv, g.yv)
        rc, _, _ = one.iterate(n)
        assert rc == 0
        np.testing.assert_array_equal(b.get_state(slot), one.get_state(0), err_msg=f"slot {slot}")
        one.close()
    b.close()
