"""The limit of a wait that depends on others' work (gsis_wait.h), compiled for
the host: it ends a stall, never a wait beside work that goes on."""
import subprocess

from helpers import PKG_DIR

CODE = """
#include <cstdio>
#include "gsis_wait.h"
int main() {
  const long long s = 100000000;  // ticks of a second
  {  // an hour beside gangs that end an iteration every 1.1 s
    gsis::StallLimit w(120 * s);
    long long over = 0;
    for (long long t = 0; t < 3600 * s; t += s / 100) over += w.over(t / (s + s / 10), 5 * s + t);
    std::printf("%lld\\n", over);
  }
  {  // a stall ends 120 s after the last change
    gsis::StallLimit w(120 * s);
    long long t = 0;
    while (!w.over(t < 500 * s ? t / s : 500, t)) t += s / 100;
    std::printf("%lld\\n", t / s);
  }
  gsis::StallLimit w(0);
  const bool a = w.over(7, 1000), b = w.over(7, 1001);
  std::printf("%d %d\\n", a, b);
}
"""


def test_a_wait_ends_by_a_stall_only(tmp_path):
    src, exe = tmp_path / "w.cpp", tmp_path / "w"
    src.write_text(CODE)
    subprocess.run(["g++", "-O1", "-std=c++17", f"-I{PKG_DIR / 'csrc'}", "-o", str(exe), str(src)], check=True)
    out = subprocess.run([str(exe)], capture_output=True, text=True, check=True, timeout=60).stdout.split()
    assert out == ["0", "620", "0", "1"]
