"""The host-built work order of the triangular sweeps (sweep_plan.hpp) on the CPU, under the
address and undefined-behaviour sanitizers (sweep_plan_check.cpp)."""
import os
import subprocess

import pytest

HERE = os.path.dirname(os.path.abspath(__file__))
CSRC = os.path.join(HERE, "..", "voluma_amd", "csrc")


@pytest.fixture(scope="module")
def check(tmp_path_factory):
    exe = str(tmp_path_factory.mktemp("sweep_plan") / "check")
    subprocess.run(["g++", "-std=c++20", "-O1", "-g", "-fsanitize=address,undefined", "-fno-sanitize-recover=all",
                    "-I", CSRC, os.path.join(HERE, "sweep_plan_check.cpp"), "-o", exe], check=True)

    def run(*args):
        r = subprocess.run([exe, *map(str, args)], capture_output=True, text=True, timeout=300)
        assert r.returncode == 0, r.stdout + r.stderr
        words = r.stdout.split()
        return dict(zip(words[::2], map(int, words[1::2])))

    return run


@pytest.mark.parametrize("n", [8193, 200_000, 2_000_000])
def test_wait_limit_covers_every_step_in_turn(check, n):
    """A chain of cells has one row per level, and the last chunk waits for nearly all of
    them: the limit of a wait, at 0.3 µs a poll, is ten times what the steps take at the
    measured 0.4 µs."""
    got = check("limit", n)
    assert got["steps"] == n and got["chunks"] > 1
    assert got["polls"] * 0.3 >= 10 * 0.4 * n
