"""The turbulence models' tridiagonal line solves in parts (part_line,
part_columns): one turbulence-model call from the same state against the
oracle's one-sided recurrence (src/samodel2d.f:1306-1385,
src/komegasst.f:1435-1518), at line lengths on both sides of one part (8
cells), of a whole number of parts, of the lengths where parts grow to 12 and
16 cells (j lines of more than 512 and 768 cells) and of the column counts of
one workgroup (k lines of more than 256 cells).  Bound: 1e-12 per cell, the
stage bound of the turbulence models; the solves of these diagonally dominant
lines differ in rounding only (about 1e-16 relative, times the few hundred
operations of a line at most).
"""
import numpy as np
import pytest

from tests import helpers as H
from turns2d_urans_git_amd import abi

pytestmark = pytest.mark.gpu

DECK = dict(fsmach=0.5, alfa=2.0, rey=1.0e6, invisc=0, lamin=0, vnuinf=3.0, irhsy=-3, ilim=1, ilhs=1,
            iconstant_cfl=1, dt=5.0, epse=0.01, iunst=0, ntac=1, itnmax=1, timeac=1.0)
# (jmax, kmax): lines of jmax-1 and kmax-1 cells
SIZES = [(13, 8), (17, 9), (19, 10), (33, 18), (131, 65), (513, 9), (515, 12), (771, 9), (1025, 6), (21, 258),
         (19, 300)]


@pytest.mark.parametrize("iturb", [1, 2])
@pytest.mark.parametrize("jm,km", SIZES)
def test_turbulence_stage_vs_oracle(jm, km, iturb):
    print(f"[line parts] {jm}x{km} iturb {iturb}", flush=True)
    g = H.cgrid(jm, km, ds_wall=1e-3)
    deck = dict(DECK, iturb=iturb)
    o, d = H.oracle_case(g, deck), H.gpu_case(g, deck)
    rc, _, _ = o.iterate(2)
    assert rc == 0
    r = np.random.default_rng(jm + km)
    q = o.get_state(0)
    n = q.shape[3] - 1
    q[..., 4:n] *= 1.0 + 0.5 * r.random(q[..., 4:n].shape)
    tm = o.get_field(0, abi.F_TURMU) * (1.0 + r.random(q.shape[:3]))
    s = np.zeros(o.get_field(0, abi.F_S).shape)
    for c in (o, d):
        c.istep0 = 2   # the SST wall condition ramps with it
        c.set_state(0, q)
        c.set_field(0, abi.F_TURMU, tm)
        c.set_field(0, abi.F_S, s)
        c.time_step()
        c.turbulence()
    qo, qd = o.get_state(0), d.get_state(0)
    for v in range(4, n):
        H.assert_cellwise(qd[..., v], qo[..., v], 1e-12, f"q{v + 1}")
    H.assert_cellwise(d.get_field(0, abi.F_TURMU), o.get_field(0, abi.F_TURMU), 1e-12, "turmu")
    if iturb == 1:   # every number of columns per workgroup gives the same bits
        for sl in (0, 1):
            d.set_launch(0, sl)
            d.set_state(0, q)
            d.set_field(0, abi.F_TURMU, tm)
            d.turbulence()
            np.testing.assert_array_equal(d.get_state(0), qd)
    d.close()
