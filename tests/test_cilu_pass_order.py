"""The work-groups of a chunked-ILU pass finish with any number of them running
at a time: every column group appears once, and where an XCD runs its
work-groups in index order, one at a time or several, none waits for one that
cannot start.  The map from work-groups to column groups is compiled here from
the header the kernels use."""
import os
import subprocess

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
SRC = r"""
#include <cstdio>
#include <cstdlib>
#include "sg_pass_order.hpp"
int main(int argc, char** argv) {
  const int nchunk = atoi(argv[1]), ng = atoi(argv[2]), asc = atoi(argv[3]);
  for (int b = 0; b < sg::pass_blocks(nchunk, ng); ++b) {
    const sg::PassGroup p = sg::pass_group(b, ng, asc != 0);
    printf("%d %d %d\n", b, p.chunk, p.group);
  }
}
"""


@pytest.fixture(scope="module")
def order(tmp_path_factory):
    d = tmp_path_factory.mktemp("order")
    (d / "order.cpp").write_text(SRC)
    exe = d / "order"
    subprocess.run(["g++", "-std=c++17", "-I" + os.path.join(ROOT, "structured_amd", "csrc"), str(d / "order.cpp"),
                    "-o", str(exe)], check=True)

    def run(nchunk, ng, asc):
        out = subprocess.run([str(exe), str(nchunk), str(ng), str(int(asc))], check=True, capture_output=True, text=True)
        return [tuple(map(int, l.split())) for l in out.stdout.splitlines()]
    return run


@pytest.mark.parametrize("nchunk,ng", [(1, 1), (1, 6), (3, 6), (8, 4), (9, 3), (23, 6), (43, 3)])
@pytest.mark.parametrize("asc", [True, False])
@pytest.mark.parametrize("room", [1, 2, 5])
def test_every_group_runs(order, nchunk, ng, asc, room):
    blocks = order(nchunk, ng, asc)
    groups = [(c, g) for _, c, g in blocks if c < nchunk]
    assert sorted(groups) == [(c, g) for c in range(nchunk) for g in range(ng)]
    done = set()
    for xcd in range(8):
        queue = [(c, g) for b, c, g in blocks if b % 8 == xcd]
        running = []
        while queue or running:
            while queue and len(running) < room:
                running.append(queue.pop(0))
            ends = [(c, g) for c, g in running
                    if c >= nchunk or g == (0 if asc else ng - 1) or (c, g + (-1 if asc else 1)) in done]
            assert ends, "work-groups %s wait for one that is not started" % running
            done.update(ends)
            running = [r for r in running if r not in ends]
