"""What calls leave in the state of a context (tests/cxx/ctx_state_check.cpp): each call off the straight path is followed
by ordinary ones on the same context, whose results are compared bit for bit with those of an untouched one."""
import json
import pathlib
import subprocess

import pytest

pytestmark = pytest.mark.gpu

CXX = pathlib.Path(__file__).resolve().parent / "cxx"


def run(check):
    exe = CXX / "ctx_state_check"
    if not exe.exists():
        subprocess.run(["make", "-s", "-C", str(CXX)], check=True)
    print("case", check, flush=True)
    p = subprocess.run([str(exe), check], capture_output=True, text=True, timeout=100)
    assert p.returncode == 0, p.stderr[-2000:]
    (out,) = [json.loads(s) for s in p.stdout.splitlines()]
    assert out.pop("check") == check
    return out


def test_after_a_wait_given_up():
    assert run("after_a_wait_given_up") == {"status": 1, "newer_words": 0, "same": 1}


def test_flag_is_read():
    """A resident launch is taken back by its flag, not by its count. The residual that the solve stopped on is updated, not
    recomputed: a true one of up to 1.05 times the tolerance, as in the tests of the solvers."""
    out = run("flag_is_read")
    assert out.pop("residual") <= 1.05
    assert out == {"status": 1, "up": 0}


def test_matrix_of_another_context():
    assert run("matrix_of_another_context") == {"moved": 0, "same": 1}


def test_captured_dot():
    assert run("captured_dot") == {"value": 9 * 5000, "eager": 9 * 5000}


def test_future_synchronises():
    assert run("future_synchronises") == {"value": 5000, "done": 1}


def test_pencils_in_place():
    assert run("pencils_in_place") == {"pencils": 1, "in_place": 1, "given_up": 1}


def test_colours_after_pencils():
    assert run("colours_after_pencils") == {"pencils": [1, 0], "same": 1}


def test_small_solves_take_their_share():
    assert run("small_solves_take_their_share") == {"solved": 2}


def test_blocking_wait():
    """A wait of some 90 ms takes less than half of its time from the core."""
    out = run("blocking_wait")
    print(out, flush=True)
    assert out["value"] == 5000
    assert out["wall_s"] > 0.02 and out["cpu_s"] < 0.5 * out["wall_s"]


def test_widths_in_one_launch():
    """Rows of up to 7 entries (6 and 7 of 6 to 9, each in one workgroup and in several)."""
    assert run("widths_in_one_launch") == {"taken": [1, 1, 1, 1, 0, 0, 0, 0]}


def test_without_memory():
    """Factorisation entry point, FP64 and FP32 pencils and their set-up, resident CG: each refused its workspace once."""
    assert run("without_memory") == {"refused": 5, "same": 1}
