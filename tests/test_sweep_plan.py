"""The host-built work order of the triangular sweeps (sweep_plan.hpp) on the CPU, under the
address and undefined-behaviour sanitizers (sweep_plan_check.cpp)."""
import os
import subprocess

import numpy as np
import pytest

from helpers import sweep_graph

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


def _write(path, n, own, nei):
    l, u = np.minimum(own, nei), np.maximum(own, nei)
    with open(path, "wb") as f:
        f.write(b"".join(np.asarray(a, np.int32).tobytes() for a in ([n, l.size], l, u)))
    return path


SMALL = {"cell": (1, [], []), "apart": (3, [], []), "pair": (2, [0], [1]), "row": (100, range(99), range(1, 100))}


@pytest.mark.parametrize("name", list(SMALL) + ["chain", "one", "two", "wide", "far", "hub", "box", "scattered"])
@pytest.mark.parametrize("backward", [0, 1])
def test_plan_gives_the_sequential_loop(check, tmp_path, name, backward):
    """A plan worked through as the kernels do it (chunk by chunk, the steps of a level in
    either order, x copied as early or as late as it may be) reads only what is there by
    then and gives the sequential loop's bits: one sweep, several in one launch, and a
    substitution, in as many chunks as the rule makes and in others."""
    small = name in SMALL
    f = _write(tmp_path / "faces", *(SMALL[name] if small else sweep_graph(name)))
    for sweeps, old in ((1, 1), (2, 1), (1, 0)) if name == "scattered" else ((1, 1), (2, 1), (4, 1), (1, 0)):
        for chunks in (0, 1, 2, 7, 70) if small else (0,):
            got = check("sweep", f, backward, sweeps, chunks, old)
            if name in ("one", "two"):
                assert (got["chunks"] == 1) == (name == "one")
            if name in ("far", "scattered") and old:  # values past the halo
                assert (got["fromx"] > 10000) == (name == "scattered" or backward == 1)
