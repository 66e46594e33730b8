"""How many Krylov steps are enqueued for a given history of residuals: none in
vain where a solve ends in one step or converges at a steady or growing rate,
none ahead at all with the preconditioners whose step is long, and all but the
first and the last two where it converges slowly.  The rule is compiled here from the
header the solver uses; the loop is the solver's."""
import os
import subprocess

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
SRC = r"""
#include <cstdio>
#include <cstdlib>
#include "sg_ahead.hpp"
// argv: precond, target, then the residual after each step (the first is before)
int main(int argc, char** argv) {
  const int precond = atoi(argv[1]), n = argc - 4;
  const double target = atof(argv[2]);
  double res = atof(argv[3]), rate = 0.0;
  int queued = 0, ahead = 0, j = 0;
  for (; j < n; ++j) {
    if (queued == j) ++queued;
    if (sg::enqueue_ahead(precond, res, rate, target)) { ++queued; ++ahead; }
    const double before = res;
    res = atof(argv[4 + j]);
    rate = res / before;
    if (res <= target) { ++j; break; }
  }
  printf("%d %d %d\n", j, queued, ahead);
}
"""


@pytest.fixture(scope="module")
def steps(tmp_path_factory):
    d = tmp_path_factory.mktemp("ahead")
    (d / "ahead.cpp").write_text(SRC)
    exe = d / "ahead"
    subprocess.run(["g++", "-std=c++17", "-I" + os.path.join(ROOT, "structured_amd", "csrc"), str(d / "ahead.cpp"),
                    "-o", str(exe)], check=True)

    def run(precond, target, history):
        out = subprocess.run([str(exe), str(precond), repr(target)] + [repr(h) for h in history], check=True,
                             capture_output=True, text=True).stdout
        return tuple(map(int, out.split()))
    return run


HISTORIES = {
    "one step": [1.0, 1e-4],
    "two steps": [1.0, 0.05, 2e-4],
    "steady": [0.3 ** k for k in range(9)],
    "growing rate": [1.0, 0.5, 0.2, 0.06, 0.012, 1e-3, 5e-5],
    "slow": [0.9 ** k for k in range(70)],
}


@pytest.mark.parametrize("name", HISTORIES)
@pytest.mark.parametrize("precond", range(8))
def test_no_step_in_vain(steps, name, precond):
    needed, queued, ahead = steps(precond, 1e-3, HISTORIES[name])
    print(name, precond, needed, queued, ahead)
    assert queued == needed
    if precond in (3, 5):
        assert ahead == 0


def test_slow_convergence_runs_ahead(steps):
    needed, queued, ahead = steps(7, 1e-3, HISTORIES["slow"])
    assert needed == 66 and needed - ahead <= 4
