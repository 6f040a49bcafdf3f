"""CPU: the arithmetic of the balanced split (voltattn_amd/csrc/va_runs.hpp), which
tests/cpp/test_runs.cpp drives directly, the same code as the kernels': runs that differ
by at most a unit, every tile of every merge group in one item, its pieces in consecutive
runs and at most 64 of them, the plan around the lengths where the shortest run grows,
and no item past the last sequence when lengths change under a running kernel."""
from tests import runs_model


def test_runs():
    r = runs_model.run()
    assert r.returncode == 0, r.stderr
    assert "runs: ok" in r.stdout
