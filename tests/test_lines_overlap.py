"""Whether two sets of lines share memory (ovx_overlap.hpp), compiled for the CPU
and compared with every pair of lines: equal and other strides, single lines,
lines between each other's, bases apart by less than a value."""
import os
import shutil
import subprocess

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))

SOURCE = """
#include "ovx_overlap.hpp"
#include <cstdlib>
int main()
{
  struct V { float x, y; };
  static char room[40000];
  long yes = 0;
  for (long t = 0; t < 1000000; ++t) {
    const long n = 1 + rand() % 9, la = 1 + rand() % 5, lb = 1 + rand() % 5;
    long lda = la > 1 ? n + rand() % 12 : (rand() % 3 ? n : 0), ldb = lb > 1 ? n + rand() % 12 : (rand() % 3 ? n : 0);
    if (rand() % 2 && la > 1 && lb > 1) lda = ldb = std::max(lda, ldb);
    const V *a = (const V *)(room + 16000 + 4 * (rand() % 240)), *b = (const V *)(room + 16000 + 4 * (rand() % 240));
    bool want = false;
    for (long i = 0; i < la; ++i)
      for (long j = 0; j < lb; ++j) want = want || (a + i * lda < b + j * ldb + n && b + j * ldb < a + i * lda + n);
    if (ovx::lines_meet(a, la, lda, b, lb, ldb, n) != want) return 1;
    yes += want;
  }
  return yes > 100000 && yes < 900000 ? 0 : 2;
}
"""


@pytest.mark.skipif(not shutil.which("g++"), reason="no g++")
def test_lines_meet_against_every_pair(tmp_path):
    src, exe = tmp_path / "meet.cpp", tmp_path / "meet"
    src.write_text(SOURCE)
    subprocess.run(["g++", "-O1", "-std=c++17", "-I" + os.path.join(ROOT, "openvsip_amd", "csrc"), str(src), "-o",
                    str(exe)], check=True)
    assert subprocess.run([str(exe)], timeout=60).returncode == 0
