"""The FP64 LU-SGS sweeps' hand-offs, checked on a host model
(tests/lu64_protocol_model.cpp; CPU only).

The model runs the forward and backward sweeps of k_lu_sweep64 with real
threads (computing wave, producers and mail wave per workgroup, three streams
sharing few CU slots over several XCDs) and compares every result with a
sequential evaluation, bit for bit: row counts with the halo row inside the
last block and apart from it, one to four blocks, scarce slots.  Under
ThreadSanitizer the ring's hand-offs (records and fills, each with its own
tag) are free of data races.  Mistakes planted in the model are found: a slot
refilled one step early by ThreadSanitizer, an entry taken by the first of its
two words by the comparison.
"""
import os
import shutil
import subprocess

import pytest

HERE = os.path.dirname(os.path.abspath(__file__))
SRC = os.path.join(HERE, "lu64_protocol_model.cpp")
CSRC = os.path.join(os.path.dirname(HERE), "turns2d_urans_git_amd", "csrc")


def _build(tmp_path_factory, tsan):
    if not shutil.which("g++"):
        pytest.skip("g++ not available")
    out = str(tmp_path_factory.mktemp("lu64model") / ("model_tsan" if tsan else "model"))
    flags = ["-O1", "-g", "-fsanitize=thread"] if tsan else ["-O2"]
    subprocess.run(["g++", *flags, "-std=gnu++17", "-ffp-contract=off", "-Wno-unknown-pragmas", "-pthread", "-I", CSRC,
                    "-o", out, SRC], check=True)
    return out


@pytest.fixture(scope="module")
def model(tmp_path_factory):
    return _build(tmp_path_factory, False)


@pytest.fixture(scope="module")
def model_tsan(tmp_path_factory):
    return _build(tmp_path_factory, True)


def _run(exe, *args, env=None):
    r = subprocess.run([exe, *args], capture_output=True, text=True, timeout=300, env=env)
    return r.returncode, r.stdout + r.stderr


@pytest.mark.parametrize("nk", [3, 4, 5, 8, 9, 12, 13, 16])
def test_sweeps_equal_the_sequential_evaluation(model, nk):
    rc, out = _run(model, f"--nk={nk}", "--sweeps=25")
    assert rc == 0, out


@pytest.mark.parametrize("ni", [1, 3, 4, 5, 8, 33])
def test_windows_of_columns(model, ni):
    rc, out = _run(model, f"--ni={ni}", "--sweeps=25")
    assert rc == 0, out


def test_scarce_slots(model):
    rc, out = _run(model, "--xcds=3", "--slots=1", "--nk=15", "--sweeps=25")
    assert rc == 0, out


def test_half_entries_are_noticed(model):
    rc, out = _run(model, "--plant-half-entry", "--sweeps=40")
    assert rc == 1 and "wrong=0" not in out, out


@pytest.mark.parametrize("args", [["--nk=8"], ["--nk=11"], ["--xcds=3", "--slots=1", "--nk=15"]])
def test_race_free_under_tsan(model_tsan, args):
    env = dict(os.environ, TSAN_OPTIONS="halt_on_error=1 exitcode=66")
    rc, out = _run(model_tsan, "--sweeps=6", *args, env=env)
    assert rc == 0 and "ThreadSanitizer" not in out, out


def test_tsan_reports_a_ring_slot_refilled_early(model_tsan):
    env = dict(os.environ, TSAN_OPTIONS="halt_on_error=1 exitcode=66")
    rc, out = _run(model_tsan, "--plant-ring-bug", "--sweeps=5", env=env)
    assert rc == 66 and "data race" in out, out
