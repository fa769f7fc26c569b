"""The order in which an amax pass and the passes behind it take a tensor (csrc/kernels/read_twice.hpp), on the CPU: every vector and every piece
once, none past the end, the front last in the one and first in the others, the same 32 KiB on the same XCD."""
import os
import subprocess

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
SOURCE = r"""
#include <initializer_list>
#include <stdio.h>
#include <vector>
#include "read_twice.hpp"
using namespace mtrt_dev;
static long wrong = 0, checked = 0;
template <int LOADS>
void amax(int64_t nvec, int64_t grid, int64_t kept_vectors) {
  using Turns = AmaxTurns<LOADS>;
  const Turns t(nvec);
  std::vector<unsigned char> seen(nvec / Turns::kTurn + 1, 0);
  const int64_t kept = t.first_kept(kept_vectors);
  for (int64_t block = 0; block < grid; ++block)
    for (int64_t turn = block; turn < t.turns; turn += grid) {
      const int64_t first = t.first(turn), chunk = first / Turns::kTurn;
      ++checked;
      if (first < 0 || first >= nvec || first % Turns::kTurn || seen[chunk]++) { ++wrong; continue; }
      if (turn >= t.whole) continue;
      if (first + Turns::kTurn > nvec || chunk % 8 != turn % 8) ++wrong;
      if ((turn < kept) != (first >= kept_vectors / Turns::kGroup * Turns::kGroup)) ++wrong;
      if (turn >= 8 && t.first(turn - 8) != first + Turns::kGroup) ++wrong;
    }
  long taken = 0;
  for (unsigned char s : seen) taken += s;
  wrong += taken != (nvec + Turns::kTurn - 1) / Turns::kTurn;
}
template <uint32_t PER>
void pieces(uint32_t n, int64_t bytes, bool grouped) {
  std::vector<unsigned char> seen(n, 0);
  for (uint32_t id = 0; id < n; ++id) {
    const uint32_t p = piece_of<PER>(id, n, bytes);
    ++checked;
    if (p >= n || seen[p]++) { ++wrong; continue; }
    if (!grouped) wrong += p != id;
    else if (id < n / (8 * PER) * (8 * PER)) wrong += p / PER % 8 != id % 8 || p / (8 * PER) != id / (8 * PER);
  }
}
int main() {
  for (int64_t nvec : {0, 1, 255, 1023, 1024, 2047, 2049, 8191, 8192, 8193, 16383, 16384, 16385, 18433, 40000, 98304, 131071, 262145, 9000001})
    for (int64_t grid : {1, 7, 8, 9, 64, 512})
      for (int64_t kept : {0, 16384, 40000, 1 << 21}) {
        amax<4>(nvec, grid, kept);
        amax<8>(nvec, grid, kept);
      }
  for (uint32_t n = 1; n < 200; ++n)
    for (int64_t bytes : {int64_t(1), kReadTwiceBelow - 1, kReadTwiceBelow, int64_t(1) << 40}) {
      pieces<2>(n, bytes, bytes < kReadTwiceBelow);
      pieces<4>(n, bytes, bytes < kReadTwiceBelow);
    }
  printf("%ld %ld\n", checked, wrong);
}
"""


def test_every_vector_once_and_on_its_xcd(tmp_path):
    src, exe = tmp_path / "order.cpp", tmp_path / "order"
    src.write_text(SOURCE)
    subprocess.run(["g++", "-std=c++17", "-O2", "-I", os.path.join(ROOT, "tensorrt-incubator_amd", "csrc", "kernels"), "-o", str(exe), str(src)], check=True)
    checked, wrong = (int(v) for v in subprocess.run([str(exe)], check=True, stdout=subprocess.PIPE, text=True, timeout=100).stdout.split())
    assert checked > 100000 and wrong == 0
