"""Launch choices cached in a file by a library whose numbers stood for other
launches are not taken over: their class key names no set of choices, or
another one, and the search runs."""
import os
import re
import subprocess
import sys
import textwrap

import pytest

pytestmark = pytest.mark.gpu

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
CHILD = textwrap.dedent("""
    import sys
    sys.path.insert(0, {root!r})
    from tests import helpers as H
    deck = dict(fsmach=0.5, alfa=2.0, rey=1.0e6, invisc=0, lamin=0, iturb=1, vnuinf=3.0, irhsy=-3, ilim=1, ilhs=1,
                iconstant_cfl=1, dt=5.0, epse=0.01, iunst=0, ntac=1, itnmax=1, timeac=1.0, lu_fp32=1)
    c = H.gpu_case(H.cgrid(65, 33, ds_wall=1e-3), deck)
    print(c.autotune(steps=3), flush=True)
    c.close()
""")


def _autotune(cache):
    r = subprocess.run([sys.executable, "-c", CHILD.format(root=ROOT)], cwd=ROOT, capture_output=True, text=True,
                       env=dict(os.environ, OT2D_TUNE_CACHE=str(cache)), timeout=100)
    assert r.returncode == 0, r.stderr
    return eval(r.stdout.strip().splitlines()[-1])


def test_choices_of_another_set_are_searched_again(tmp_path):
    cache = tmp_path / "tune.txt"
    print("[tune cache version] first search", flush=True)
    assert _autotune(cache)[2] is True
    key = cache.read_text().split()[0]
    assert _autotune(cache)[2] is False
    # the same class as a library without sets wrote it, and as a later one might
    plain = re.sub(r"^set=\d+,", "", key)
    for old in (plain, "set=1," + plain, "set=999," + plain):
        print(f"[tune cache version] {old}", flush=True)
        cache.write_text(f"{old} 2 0\n")
        assert _autotune(cache)[2] is True, old
