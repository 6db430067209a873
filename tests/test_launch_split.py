"""Host rules of how launches cut their work (csrc/launch_split.hpp), compiled and checked on the
CPU: a delivery's task count stays inside 32 bits whatever spikes, and rows are shared as before
where it does anyway."""
import os
import subprocess

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))

PROGRAM = r"""
#include "launch_split.hpp"
#include <cstdio>
int main() {
  for (int64_t units : {1ll, 63ll, 5000ll, 65536ll, 500000ll, 524288ll, 525000ll, 2000000ll, 16777216ll})
    for (int G : {1, 2, 15, 20, 32, 63, 64, 65, 200})
      for (int64_t row : {0ll, 1ll, 64ll, 65ll, 1000ll, 4033ll, 4096ll, 1000000ll})
        std::printf("%lld %d %lld %d\n", (long long)units, G, (long long)row, spk::deliver_row_waves(row, units, G));
}
"""


def test_delivery_tasks_fit_32_bits(tmp_path):
    src, exe = tmp_path / "t.cpp", tmp_path / "t"
    src.write_text(PROGRAM)
    subprocess.run(["g++", "-std=c++17", "-I", os.path.join(ROOT, "spike_amd", "csrc"), str(src), "-o", str(exe)],
                   check=True)
    limited = 0
    for line in subprocess.run([str(exe)], check=True, capture_output=True, text=True).stdout.splitlines():
        units, G, row, waves = map(int, line.split())
        want = min(64, max(1, -(-row // 64)))
        assert 1 <= waves <= want
        assert units * min(G, 64) * waves <= 2 ** 30
        if units * min(G, 64) * want <= 2 ** 30:
            assert waves == want
        else:
            limited += 1
    assert limited
