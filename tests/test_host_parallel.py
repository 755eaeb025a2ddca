"""The host threads of the table build: every item once, and an exception of one item
reaches the caller (it used to end the process)."""
import os
import subprocess

CSRC = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "bigstickpublick_amd", "csrc")

PROGRAM = r"""
#include "bs_parallel.hpp"
#include <cstdio>
#include <new>
#include <string>
int main() {
  for (int n : {0, 1, 5, 1000}) {
    std::vector<std::atomic<int>> seen(n);
    for (auto& s : seen) s = 0;
    bs::parallel(n, [&](int i) { seen[i]++; });
    for (auto& s : seen) if (s != 1) return 1;
  }
  for (int bad : {0, 3, 999}) {
    try {
      bs::parallel(1000, [&](int i) { if (i == bad) throw std::bad_alloc(); });
      return 2;
    } catch (const std::bad_alloc&) {
    }
  }
  puts("ok");
}
"""


def test_parallel(tmp_path):
    src = tmp_path / "p.cpp"
    src.write_text(PROGRAM)
    exe = str(tmp_path / "p")
    subprocess.run(["g++", "-std=c++17", "-O1", "-pthread", "-I", CSRC, str(src), "-o", exe], check=True)
    r = subprocess.run([exe], capture_output=True, text=True, timeout=60)
    assert r.returncode == 0 and r.stdout == "ok\n", (r.returncode, r.stdout, r.stderr)
