"""Metrics of a grid that turns in every step (k_metrics for the interior, the
halo after it): after a time step they are, bit for bit, those of a fresh case
given the turned vertices, and the oracle's metfv (src/setup.f:440-724) of
them.  Sizes below, at and past one workgroup's 256 cells.  Bound against the
oracle: 1e-12 per cell, the same operations in the same order.
"""
import numpy as np
import pytest

from tests import helpers as H
from turns2d_urans_git_amd import abi

pytestmark = pytest.mark.gpu

DECK = dict(fsmach=0.3, alfa=1.0, rey=1.0e6, invisc=0, lamin=0, iturb=1, vnuinf=3.0, irhsy=-3, ilim=1, ilhs=1,
            iconstant_cfl=0, dt=0.05, epse=0.01, iunst=1, motiontype=1, rf=0.1, angmax=2.0, ntac=2, itnmax=2,
            idual=1, dualtime=5.0, timeac=1.0)


@pytest.mark.parametrize("jm,km", [(17, 9), (33, 9), (35, 10), (129, 33)])
def test_turned_metrics(jm, km):
    print(f"[turned metrics] {jm}x{km}", flush=True)
    g = H.cgrid(jm, km, ds_wall=1e-3)
    d = H.gpu_case(g, DECK)
    rc, _, _ = d.iterate(2)
    assert rc == 0
    xv, yv = d.get_field(0, abi.F_XV), d.get_field(0, abi.F_YV)
    f, o = H.gpu_case(g, DECK), H.oracle_case(g, DECK)
    assert not np.array_equal(xv, f.get_field(0, abi.F_XV)), "the grid did not turn"
    for c in (f, o):
        c.set_grid(0, xv[:, :, 0], yv[:, :, 0])
    for n in (abi.F_XX, abi.F_XY, abi.F_YX, abi.F_YY):
        np.testing.assert_array_equal(d.get_field(0, n), f.get_field(0, n), err_msg=f"field {n}")
        H.assert_cellwise(d.get_field(0, n), o.get_field(0, n), 1e-12, f"field {n}")
    np.testing.assert_array_equal(d.get_state(0)[..., -1], f.get_state(0)[..., -1])
    d.close()
    f.close()
