"""The autotuner's search (csrc/tune_search.h) on made-up timings: it starts from
the choices in force, so it never ends slower than they are, skips what does not
fit and finds the optimum of a separable cost."""
import os
import subprocess

import pytest

SRC = r"""
#include <cstdio>
#include <cstdlib>
#include "tune_search.h"
using sf21::TuneChoice;
int main(int argc, char** argv) {
  const int n = atoi(argv[1]), nr = atoi(argv[2]), plane = atoi(argv[3]), mode = atoi(argv[4]);
  TuneChoice b{atoi(argv[5]), atoi(argv[6]), atoi(argv[7]), atoi(argv[8]), atoi(argv[9]), atoi(argv[10])};
  const TuneChoice s = b;
  double ms = -1;
  int calls = 0;
  auto timed = [&](const TuneChoice& t, double* out) {
    ++calls;
    const bool same = t.tile == s.tile && t.K == s.K && t.ct == s.ct && t.cw == s.cw && t.rw == s.rw && t.fp == s.fp;
    if (mode == 0) *out = same ? 1.0 : 2.0;                     // nothing beats the start
    else if (mode == 1)                                         // separable
      *out = 10 - (t.K == nr) - (t.tile == 8) - (t.fp == 1) - (t.ct == 32 && t.cw == 3) - (t.rw == 1);
    else if (mode == 2) { if (!same) return 1; *out = 5.0; }    // only the start fits
    else if (mode == 3) return 1;                               // nothing fits
    else if (mode == 4) { *out = 1.0; return calls == 4 ? -1 : 0; }
    return 0;
  };
  const int rc = sf21::tune_search(n, nr, plane != 0, timed, &b, &ms);
  printf("%d %d %d %d %d %d %d %g %d\n", rc, b.tile, b.K, b.ct, b.cw, b.rw, b.fp, ms, calls);
}
"""


@pytest.fixture(scope="module")
def search(tmp_path_factory):
    d = tmp_path_factory.mktemp("tune")
    (d / "main.cpp").write_text(SRC)
    inc = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "simfast21_amd", "csrc")
    subprocess.run(["g++", "-std=c++17", "-Wall", "-Werror", "-I", inc, str(d / "main.cpp"), "-o", str(d / "t")],
                   check=True)

    def run(*args):
        out = subprocess.run([str(d / "t"), *map(str, args)], check=True, capture_output=True, text=True)
        return [float(v) if "." in v else int(v) for v in out.stdout.split()]
    return run


@pytest.mark.parametrize("start", [(16, 47, 16, 1, 0, 1), (4, 20, 16, 0, 1, 0), (16, 5, 32, 3, 1, 1)])
@pytest.mark.parametrize("n,plane", [(256, 0), (192, 0), (128, 1)])
def test_never_slower_than_the_start(search, n, plane, start):
    assert search(n, 47, plane, 0, *start)[:8] == [0, *start, 1]
    assert search(n, 47, plane, 2, *start)[:8] == [0, *start, 5]


def test_finds_a_separable_optimum(search):
    for start in ((16, 20, 16, 1, 0, 0), (8, 47, 16, 0, 0, 1), (16, 16, 32, 3, 1, 1)):
        assert search(512, 47, 0, 1, *start)[:8] == [0, 8, 47, 32, 3, 1, 1, 5]
    # plane sides keep the choices of the passes they do not run
    assert search(128, 30, 1, 1, 16, 16, 16, 0, 0, 0)[:8] == [0, 8, 30, 16, 0, 0, 1, 7]


def test_nothing_fits_and_errors(search):
    assert search(256, 47, 0, 3, 16, 16, 16, 0, 0, 0)[0] == 1
    rc = search(256, 47, 0, 4, 16, 16, 16, 0, 0, 0)
    assert rc[0] == -1 and rc[-1] == 4
