"""Rules the kernels share with the host (csrc/ot2d_plain.h), compiled for the
CPU.  Each check program says what it holds the rule to."""
import os
import shutil
import subprocess

import pytest

HERE = os.path.dirname(os.path.abspath(__file__))
CSRC = os.path.join(os.path.dirname(HERE), "turns2d_urans_git_amd", "csrc")


@pytest.fixture(scope="module")
def run_check(tmp_path_factory):
    if not shutil.which("g++"):
        pytest.skip("g++ not available")
    out = tmp_path_factory.mktemp("plain")

    def run(name, *args):
        exe = str(out / name)
        subprocess.run(["g++", "-O2", "-std=gnu++17", "-ffp-contract=off", "-Wall", "-Wno-unknown-pragmas", "-I", CSRC,
                        "-o", exe, os.path.join(HERE, name + ".cpp")], check=True)
        r = subprocess.run([exe, *args], capture_output=True, text=True, timeout=300)
        print(r.stdout)
        assert r.returncode == 0, r.stdout + r.stderr

    return run


def test_sweep_waits_outlast_a_queue_put_aside(run_check):
    """A wait of the sweeps is not given up because the queue was put aside
    between two polls, and always ends when no answer comes."""
    run_check("wait_limit_check")


def test_tiles_go_round_the_xcds(run_check):
    """Every tile of a record goes to one workgroup, each XCD takes a run of
    neighbours, no workgroup of a record's own number of tiles is empty, and
    over equal records no XCD is left behind."""
    run_check("xcd_deal_check")


def test_search_keeps_the_default_unless_clearly_slower(run_check):
    """A launch choice is taken over the default only when it wins by more
    than the timings differ among themselves."""
    run_check("launch_pick_check")


def test_line_solves_in_parts_are_as_accurate_as_the_recurrence(run_check):
    """Lines in parts against 113-bit solutions, non-dominant rows among them,
    beside the one-sided recurrence."""
    run_check("line_parts_check")
