"""The support kernel's item lists, walked on the host.

A launch's jobs map every token of their window class exactly once, and a
class without tokens (a sliding window that has not opened yet in an early
block of a long prefix) has no items: an item of no tokens would still stream
its job's maps, and would look its row up one token before its range.
"""

from __future__ import annotations

import itertools
import shutil
import subprocess

import pytest

from .conftest import ROOT

PROGRAM = r"""
#include <cstdio>
#include <cstdlib>
#include "cb_items.h"
struct Args {
  int ncls, cls_unit_begin[4], cls_unit_end[4], cls_tok_first[4], cls_tok_count[4], cls_nchunks[4];
};
// argv: units and tokens of each class; prints class-order first token, then the items of every XCD.
int main(int argc, char** argv) {
  Args a{};
  a.ncls = (argc - 1) / 2;
  long unit = 0, token = 0;
  for (int c = 0; c < a.ncls; ++c) {
    const long n = std::atol(argv[1 + 2 * c]), t = std::atol(argv[2 + 2 * c]);
    a.cls_unit_begin[c] = unit;
    a.cls_unit_end[c] = unit += n;
    set_class_tokens(a, c, token, t, kSupTile);
    token += t;
  }
  for (int x = 0; x < 8; ++x) {
    SupItem it;
    for (long p = 0; support_list_item(a, x, p, [](int unit) { return unit; }, it); ++p)
      std::printf("%d %d %d %d\n", x, it.job, it.lo, it.hi);
  }
}
"""


@pytest.fixture(scope="module")
def walk(tmp_path_factory):
    compiler = shutil.which("g++")
    if not compiler:
        pytest.skip("g++ not available")
    work = tmp_path_factory.mktemp("items")
    (work / "walk.cpp").write_text(PROGRAM)
    subprocess.run([compiler, "-std=c++17", "-Wall", "-Werror", f"-I{ROOT / 'cachebridge_amd' / 'csrc'}",
                    str(work / "walk.cpp"), "-o", str(work / "walk")], check=True)

    def run(classes):
        out = subprocess.run([str(work / "walk"), *(str(v) for c in classes for v in c)], check=True,
                             capture_output=True, text=True).stdout
        return [tuple(map(int, line.split())) for line in out.splitlines()]

    return run


@pytest.mark.parametrize("units", [1, 7, 8, 40, 300])
@pytest.mark.parametrize("tokens", list(itertools.product([0, 1, 256, 700], repeat=3)))
def test_every_token_of_every_job_once_and_nothing_for_empty_classes(walk, units, tokens):
    classes = [(units, t) for t in tokens]
    seen = {}
    for xcd, unit, lo, hi in walk(classes):
        assert lo < hi <= lo + 256, (unit, lo, hi)
        assert (unit - unit // units * units) % 8 == xcd  # (its place in its class)
        seen.setdefault(unit, []).append((lo, hi))
    first = 0
    for c, (n, t) in enumerate(classes):
        for unit in range(c * n, (c + 1) * n):
            parts = sorted(seen.pop(unit, []))
            assert [p[0] for p in parts] == list(range(first, first + t, 256))
            assert not parts or parts[-1][1] == first + t
        first += t
    assert not seen
