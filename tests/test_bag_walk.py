"""The walk of a bag's rows (csrc/tbe_bag_walk.h), compiled for the host: every row once, in
order, in calls that stay inside the bag, up to bags of 2^31 - 1 rows, where a position
counter that runs past the bag overflows."""
import os
import subprocess

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))

SOURCE = r"""
#include <stdio.h>
#include <stdlib.h>
#include "tbe_bag_walk.h"
using namespace tbe;
static void check(bool ok, const char* what) { if (!ok) { printf("%s\n", what); exit(1); } }
int main(int argc, char** argv) {
  const int64_t start = atoll(argv[1]), L = atoll(argv[2]);
  const int step = atoi(argv[3]);
  // three stages over two register sets: what each holds, and what was consumed
  int64_t at[2] = {-1, -1}, rows[2] = {-1, -1}, next = start;
  int64_t steps = 0;
  if (L > 0) walk_steps(start, static_cast<int>(L), step,
    [&](auto s, int64_t p, int left) {
      check(p == start + L - left, "position and rows left disagree");
      at[s()] = p;
    },
    [&](auto s, int left) {
      check(at[s()] == start + L - left, "rows issued from another step's indices");
      rows[s()] = left < 0 ? 0 : left < step ? left : step;
    },
    [&](auto s, int left) {
      check(left > 0 && start + L - left == next, "rows consumed out of order");
      check(rows[s()] == (left < step ? left : step), "rows consumed of another step");
      next += rows[s()];
      check(++steps <= L / step + 1, "the walk does not end");
    });
  check(next == start + L, "rows left out");
  next = start;
  walk_chunks(start, static_cast<int>(L), step, [&](int64_t p, int n) {
    check(p == next && n > 0 && n <= step && next + n <= start + L, "chunk outside the bag");
    next += n;
  });
  check(next == start + L, "chunks left out");
  int64_t sum = 0;
  for (int w = 0; w < 4; ++w) {
    const BagShare s = bag_share(static_cast<int>(L), w, 4);
    check(s.first >= 0 && s.rows >= 0 && (s.rows == 0 || s.first == sum), "shares overlap");
    sum += s.rows;
  }
  check(sum == L, "shares left out");
  return 0;
}
"""


@pytest.fixture(scope="module")
def walk(tmp_path_factory):
    d = tmp_path_factory.mktemp("walk")
    (d / "walk.cpp").write_text(SOURCE)
    subprocess.run(["g++", "-std=c++17", "-O2", "-fsanitize=undefined", "-fno-sanitize-recover=all",
                    "-I" + os.path.join(ROOT, "fbgemm-ascend_amd", "csrc"), str(d / "walk.cpp"), "-o", str(d / "walk")],
                   check=True)
    return str(d / "walk")


SHORT = [0, 1, 7, 15, 16, 17, 63, 64, 65, 127, 128, 129, 192, 1000]
LONG = [2 ** 31 - 129, 2 ** 31 - 64, 2 ** 31 - 63, 2 ** 31 - 1]


@pytest.mark.parametrize("length,step", [(n, s) for n in SHORT for s in (8, 16, 64)] + [(n, 64) for n in LONG])
def test_every_row_once(walk, length, step):
    for start in (0, 5):
        r = subprocess.run([walk, str(start), str(length), str(step)], capture_output=True, text=True, timeout=120)
        assert r.returncode == 0, (r.stdout + r.stderr)[-500:]
