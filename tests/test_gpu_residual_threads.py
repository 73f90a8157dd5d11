"""The residual kernel's two shapes (576 threads for few tiles, 256 for many):
every case of a batch whose tiles lie on either side of the line equals the
case alone (few tiles), bit for bit.  A 257x65 grid has 64 tiles of 32x8
cells; the line lies at 768 tiles (MUSCL) and 1280 (WENO5)."""
import numpy as np
import pytest

from tests import helpers as H
from turns2d_urans_git_amd import abi, grid

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("ilim,n", [(1, 12), (1, 13), (4, 20), (4, 21)])
def test_batch_equals_alone(ilim, n):
    import turns2d_urans_git_amd as t2d
    print(f"[residual threads] ilim {ilim}, {64 * n} tiles", flush=True)
    g = H.cgrid(257, 65, ds_wall=1e-3)
    ps = [t2d.default_params(**dict(H.EULER, ilim=ilim, alfa=0.1 * i)) for i in range(n)]
    m = abi.mesh_desc(g.jmax, g.kmax, grid.cgrid_bc(g.jtail1))
    b = t2d.Batch(ps, [m] * n)
    for i in range(n):
        b.set_grid(i, g.xv, g.yv)
    rc, hist, done = b.iterate(3)
    assert rc == 0 and done == 3
    for i in (0, n // 2, n - 1):
        one = t2d.Case(ps[i], [m])
        one.set_grid(0, g.xv, g.yv)
        rc, h1, done = one.iterate(3)
        assert rc == 0 and done == 3
        np.testing.assert_array_equal(hist[:, i], h1[:, 0], err_msg=f"case {i}")
        np.testing.assert_array_equal(b.get_state(i), one.get_state(0), err_msg=f"case {i}")
        one.close()
    b.close()
