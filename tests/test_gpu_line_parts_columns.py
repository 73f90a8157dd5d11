"""The SA k solve with 16 columns a workgroup (ot2d_set_launch, sa_lane 0, for
columns of up to 256 cells; otherwise 8): state and eddy viscosity equal those
of 8 columns, bit for bit, at column counts on both sides of a group."""
import numpy as np
import pytest

from tests import helpers as H
from turns2d_urans_git_amd import abi

pytestmark = pytest.mark.gpu

DECK = dict(fsmach=0.5, alfa=2.0, rey=1.0e6, invisc=0, lamin=0, iturb=1, vnuinf=3.0, irhsy=-3, ilim=1, ilhs=1,
            iconstant_cfl=1, dt=5.0, epse=0.01, iunst=0, ntac=1, itnmax=1, timeac=1.0)


@pytest.mark.parametrize("jm,km", [(17, 9), (19, 10), (33, 18), (35, 65), (49, 129), (131, 257)])
def test_sixteen_columns_equal_eight(jm, km):
    print(f"[line parts columns] {jm}x{km}", flush=True)
    g = H.cgrid(jm, km, ds_wall=1e-3)
    o, d = H.oracle_case(g, DECK), H.gpu_case(g, DECK)
    rc, _, _ = o.iterate(2)
    assert rc == 0
    r = np.random.default_rng(jm * km)
    q = o.get_state(0)
    q[..., 4] *= 1.0 + 0.5 * r.random(q[..., 4].shape)
    tm = o.get_field(0, abi.F_TURMU) * (1.0 + r.random(q.shape[:3]))
    got = []
    for sl in (1, 0):
        d.set_launch(0, sl)
        d.istep0 = 2
        d.set_state(0, q)
        d.set_field(0, abi.F_TURMU, tm)
        d.set_field(0, abi.F_S, np.zeros(o.get_field(0, abi.F_S).shape))
        d.time_step()
        d.turbulence()
        got.append((d.get_state(0), d.get_field(0, abi.F_TURMU)))
    assert not np.array_equal(got[0][0], q)
    for a, b, what in zip(got[0], got[1], ("state", "eddy viscosity")):
        np.testing.assert_array_equal(b, a, err_msg=what)
    d.close()
