"""How attention workgroups are dealt to the XCDs (xcd.hpp, plain C++ on the CPU): every (head, workgroup) once, no XCD with more than its
share, one head's workgroups together."""
from __future__ import annotations

import os
import subprocess

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))

CHECK = r"""
#include <stdio.h>
#include <vector>
#include "xcd.hpp"
int main() {
  for (int heads : {1, 2, 3, 4, 5, 6, 7, 8, 9, 10, 11, 12, 15, 16, 17, 24, 25, 40, 64})
    for (int n : {1, 2, 3, 5, 7, 8, 21, 25, 32, 63, 100, 257}) {
      const ti::XcdDeal d = ti::xcd_deal(heads, n);
      std::vector<int> seen(heads * n, 0);
      for (int x = 0; x < 8; ++x) {
        int first = heads, last = -1, work = 0;
        for (int i = 0; i < d.per + 9; ++i) {   // (a launch may hold more workgroups than the deal)
          const ti::XcdWork w = ti::xcd_work(d, x, i);
          if (w.head < 0) continue;
          if (w.head >= heads || w.j < 0 || w.j >= n) return printf("%d heads of %d: (%d, %d)\n", heads, n, w.head, w.j), 1;
          ++seen[w.head * n + w.j];
          first = w.head < first ? w.head : first;
          last = w.head > last ? w.head : last;
          ++work;
        }
        // an even share; heads that divide 8 deal theirs to 8 / heads XCDs
        const int even = 8 % heads ? (heads * n + 7) / 8 : (n + 8 / heads - 1) / (8 / heads);
        if (work > even) return printf("%d heads of %d: XCD %d has %d, even %d\n", heads, n, x, work, even), 1;
        if (work && last - first > (work - 1 + n - 1) / n) return printf("%d heads of %d: XCD %d holds heads %d .. %d\n", heads, n, x, first, last), 1;
      }
      for (int s : seen)
        if (s != 1) return printf("%d heads of %d: dealt %d times\n", heads, n, s), 1;
    }
  const ti::XcdDeal big = ti::xcd_deal(8, 262140);   // (1048560 rows of 16 query heads a kv-head)
  return big.per == 262140 ? 0 : 1;
}
"""


def test_every_workgroup_once_and_even_xcds(tmp_path):
    (tmp_path / "check.cpp").write_text(CHECK)
    exe = str(tmp_path / "check")
    subprocess.run(["g++", "-std=c++20", "-O1", "-I" + os.path.join(ROOT, "turboinfer_amd", "csrc", "kernels"), str(tmp_path / "check.cpp"), "-o", exe], check=True)
    r = subprocess.run([exe], capture_output=True, text=True)
    assert r.returncode == 0, r.stdout
