"""Every row or column group of every probe is some workgroup's work exactly once, whatever number of
groups a workgroup takes in turn (unit_map.h, compiled for the host)."""
import os
import subprocess

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))

PROGRAM = r"""
#include <cstdio>
#include <vector>
#include "unit_map.h"
template <int K> int check() {
  int bad = 0;
  for (int G : {8, 16, 24, 32, 40, 64, 80, 88, 96, 128, 256, 384, 512, 1024, 12, 20})
    for (int items : {1, 2, 3, 7, 26}) {
      if (G % K) continue;                                  // what the launches require
      std::vector<int> seen((size_t)items * G, 0);
      for (int bid = 0; bid < items * G / K; ++bid)
        for (int u = 0; u < K; ++u) {
          int item = -1, g = -1;
          totem::unit_map<K>(bid, u, G, item, g);
          if (item < 0 || item >= items || g < 0 || g >= G) { ++bad; continue; }
          ++seen[(size_t)item * G + g];
        }
      for (int n : seen) bad += n != 1;
    }
  return bad;
}
int main() {
  const int bad[] = {check<1>(), check<2>(), check<4>()};
  std::printf("%d %d %d\n", bad[0], bad[1], bad[2]);
}
"""


def test_every_group_once(tmp_path):
    src, exe = tmp_path / "map.cpp", tmp_path / "map"
    src.write_text(PROGRAM)
    subprocess.run(["g++", "-std=c++17", "-D__HIP_PLATFORM_AMD__", "-I/opt/rocm/include",
                    "-I" + os.path.join(ROOT, "totem_amd", "csrc"), str(src), "-o", str(exe)], check=True)
    assert subprocess.run([str(exe)], capture_output=True, text=True, check=True).stdout == "0 0 0\n"

