"""The balanced split's plan on the host: tests/cpp/test_runs.cpp, built once with g++."""
from __future__ import annotations

import functools
import subprocess
import tempfile
from pathlib import Path

ROOT = Path(__file__).resolve().parent.parent


@functools.lru_cache(maxsize=None)
def _exe() -> tuple[tempfile.TemporaryDirectory, str]:
    d = tempfile.TemporaryDirectory()
    exe = str(Path(d.name) / "test_runs")
    subprocess.run(["g++", "-O1", "-std=c++17", "-Wall", "-Wextra", "-Werror",
                    "-I", str(ROOT / "voltattn_amd" / "csrc"), str(ROOT / "tests" / "cpp" / "test_runs.cpp"),
                    "-o", exe], check=True)
    return d, exe


def run(*args):
    return subprocess.run([_exe()[1], *map(str, args)], capture_output=True, text=True, timeout=120)


def plan(lens, tile: int, groups: int, wgs: int) -> tuple[int, int, int]:
    """(runs, most pieces of a merge group, pieces of all cut merge groups) of a batch: `tile`
    positions per tile of the plan, `groups` merge groups per sequence, `wgs` work-groups."""
    r = run(256 // tile, wgs, groups, *(max(1, -(-L // tile)) for L in lens))
    assert r.returncode == 0, r.stderr
    return tuple(int(x) for x in r.stdout.split()[1::2])
