"""FP64 LU-SGS sweeps whose rows span several workgroups (k_lu_sweep64).

The sweep cuts the rows into blocks of 32 that pass each column's edge row to
the next block; the halo row k = ke+1 is a row of the last block where that
has room and a fill of its own otherwise, and k = ks-1 always is.  Every cell
takes the reference's operands in the reference's order (ilu2d,
src/lhs.f:470-814), with IEEE division and square root, so from the same
state, time step and residual the update equals the oracle's exactly.  The
row counts lie on both sides of one, two and three blocks; a random residual
(halo ring included) and eddy viscosity reach every operand, and several
sweeps in a row reach the tags of later sweeps.
"""
import numpy as np
import pytest

from tests import helpers as H
from turns2d_urans_git_amd import abi

pytestmark = pytest.mark.gpu

GRIDS = [(11, 5), (33, 17), (33, 32), (35, 33), (33, 34), (65, 64), (65, 65), (67, 66), (129, 97), (41, 193)]


@pytest.mark.parametrize("jm,km", GRIDS)
def test_lu_stage_equals_oracle(jm, km):
    print(f"[lu64 stage] {jm}x{km} rows {km - 1}", flush=True)
    g = H.cgrid(jm, km, ds_wall=1e-3)
    o, d = H.oracle_case(g, H.EULER), H.gpu_case(g, H.EULER)
    rc, _, _ = o.iterate(5)
    assert rc == 0
    r = np.random.default_rng(jm * 1000 + km)
    q = o.get_state(0)
    q[..., :4] *= 1.0 + 0.02 * r.standard_normal(q[..., :4].shape)
    tm = np.abs(r.standard_normal(o.get_field(0, abi.F_TURMU).shape)) * 100.0
    for c in (o, d):
        c.set_state(0, q)
        c.set_field(0, abi.F_TURMU, tm)
        c.time_step()
    np.testing.assert_array_equal(d.get_field(0, abi.F_TSCALE), o.get_field(0, abi.F_TSCALE))
    for n in range(4):
        s = r.standard_normal(o.get_field(0, abi.F_S).shape) * q[..., :4]
        for c in (o, d):
            c.set_state(0, q)
            c.set_field(0, abi.F_S, s)
            c.lhs()
        np.testing.assert_array_equal(d.get_field(0, abi.F_S), o.get_field(0, abi.F_S), err_msg=f"sweep {n}")
    d.close()
