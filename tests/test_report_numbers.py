"""The numbers of the solves' reports (csrc/reports.h, plain C++): an iteration
takes its number from the box's owner before its launches, so that the solve
after one whose launch failed does not wait for a number already reported."""
import os
import shutil
import subprocess

import pytest

CSRC = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "nek5000_amd",
                    "csrc")

PROGRAM = r"""
#include <cstdio>
#include "reports.h"
using namespace nekamd;

// an iteration: its first launch reports, the second one may fail
static bool iteration(const Reports &reports, bool fails, BoxRef *asked) {
  *asked = reports.next();
  if (asked->b) asked->b->seq = asked->seq;
  return !fails;
}

int main() {
  HostBox box{};
  unsigned long long count = 0;
  BoxRef r;
  {  // a solve whose second iteration fails after its report
    const Reports reports{&box, &count};
    if (!iteration(reports, false, &r)) return 1;
    if (iteration(reports, true, &r)) return 2;
  }
  // the next solve's report has not been made yet
  const BoxRef next = Reports{&box, &count}.next();
  if (!(box.seq < next.seq)) return 3;
  // without a box there is no report, and no number is taken
  const unsigned long long before = count;
  if (Reports{nullptr, &count}.next().b != nullptr || count != before) return 4;
  return 0;
}
"""


def test_failed_launch_leaves_no_stale_report(tmp_path):
    cxx = shutil.which("g++") or shutil.which("c++")
    if cxx is None:
        pytest.skip("no C++ compiler")
    src, exe = tmp_path / "t.cpp", tmp_path / "t"
    src.write_text(PROGRAM)
    subprocess.run([cxx, "-std=c++17", "-Wall", "-Werror", "-I", CSRC, str(src), "-o", str(exe)],
                   check=True)
    assert subprocess.run([str(exe)]).returncode == 0
