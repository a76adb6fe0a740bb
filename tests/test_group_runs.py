"""How the sixteen-lane pooled kernel takes a lane group's bags (tbe_group_run.h), on the CPU: the kernel's walk over a
group's bags, written out with the header's rules, against one bag at a time.  Lengths that do not fit 32 bits, bounds
that fall and running sums that wrap neither lengthen a loop beyond the bags' own ids nor leave a bag without result."""
import os
import shutil
import subprocess

import pytest

CSRC = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "torchrec_amd", "csrc")

WALK = r"""
#include <cstdio>
#include <cstdlib>
#include <vector>
#include "tbe_group_run.h"
// stdin: for every group a count n, then n times (start, length as given).  Prints per group
// the rows walked, then for every bag its first position and its ids, in the order in which the kernel stores them.
int main() {
  int n;
  while (scanf("%d", &n) == 1) {
    std::vector<long long> start(n), given(n);
    std::vector<int> len(n);
    bool one_run = true;
    for (int i = 0; i < n; ++i) {
      if (scanf("%lld %lld", &start[i], &given[i]) != 2) return 1;
      len[i] = tra::bag_ids(given[i]);
    }
    for (int i = 0; i + 1 < n; ++i) one_run = one_run && tra::bags_join(start[i], len[i], start[i + 1]);
    long long rows = 0;
    std::vector<long long> out;
    for (int seg = 0; seg < (one_run ? 1 : n); ++seg) {
      const int last = one_run ? n - 1 : seg;
      const long long total = (long long)((unsigned long long)start[last] + len[last] - (unsigned long long)start[seg]);
      for (int b = seg; b <= last; ++b)
        if (len[b] == 0) out.insert(out.end(), {b, 0, 0});
      rows += total > 0 ? total : 0;
      long long end = 0;
      for (int b = seg; b <= last; ++b) {
        if (len[b] == 0) continue;
        if (end + len[b] > total) break;  // (the loop ends in front of the bag's end: never stored)
        out.insert(out.end(), {b, (long long)((unsigned long long)start[seg] + end), len[b]});
        end += len[b];
      }
    }
    printf("%lld", rows);
    for (long long x : out) printf(" %lld", x);
    printf("\n");
  }
  return 0;
}
"""


def _i32(x):
    return (x + 2**31) % 2**32 - 2**31


def _i64(x):
    return (x + 2**63) % 2**64 - 2**63


GROUPS = {
    "well formed": [3, 0, 7, 16, 1, 0, 0, 40],
    "one bag": [5],
    "negative": [3, -2, 7, -1, 4, 0],
    "cut to 3": [4, 2**32 + 3, 5, 6],
    "cut to nothing": [4, 2**40, 5, 6],
    "falls by 2^32 - 5": [4, 5 - 2**32, 5, 6],
    "beyond 31 bits": [1, 2**31 + 9, 2],
    "last bag cut": [1, 2, 2**33 + 1],
    "sum of 64 bits wraps": [2, 2**62, 2**62, 2**62, 7],
}


@pytest.mark.parametrize("wrap", [32, 64])
def test_group_walk(tmp_path, wrap):
    cxx = shutil.which("g++") or "/opt/rocm/bin/amdclang++"
    src, exe = tmp_path / "walk.cpp", tmp_path / "walk"
    src.write_text(WALK)
    subprocess.run([cxx, "-std=c++17", "-O1", "-I", CSRC, str(src), "-o", str(exe)], check=True)
    lines, wants = [], []
    for name, lengths in GROUPS.items():
        lengths = [_i32(x) for x in lengths] if wrap == 32 else list(lengths)
        if wrap == 32:
            lengths += [2**31 - 100, 50, 60, 8]  # (the running sum passes 2^31)
        at, bags = 1000, []
        for x in lengths:
            bags.append((at, x))
            at = _i32(at + x) if wrap == 32 else _i64(at + x)
        lines.append(" ".join([str(len(bags))] + [f"{s} {x}" for s, x in bags]))
        ids = [max(_i32(x), 0) for _, x in bags]
        wants.append((name, sum(ids), sorted((b, s if n else 0, n) for b, ((s, _), n) in enumerate(zip(bags, ids)))))
    got = subprocess.run([str(exe)], input="\n".join(lines) + "\n", capture_output=True, text=True, check=True).stdout
    for line, (name, rows, want) in zip(got.splitlines(), wants):
        v = [int(x) for x in line.split()]
        assert v[0] == rows, name
        assert sorted(zip(v[1::3], v[2::3], v[3::3])) == want, name
