"""NVFP4 along the second-to-last axis: where the dequantize pass looks for a vector's scales (csrc/kernels/nvfp4_index.hpp), on the CPU.
A tensor of 2^32 vectors is 64 GiB; below that the kernel divides in 32 bits."""
import os
import subprocess

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
SOURCE = r"""
#include <initializer_list>
#include <stdio.h>
#include "nvfp4_index.hpp"
using namespace nvfp4_cluster;
template <int G>
int64_t scale_of(int64_t v, int64_t nvec, int64_t d1) { return numbers_fit(nvec) ? scale_of_vector<true, G>(v, d1) : scale_of_vector<false, G>(v, d1); }
int main() {
  const int64_t big = int64_t(1) << 32;
  long checked = 0, wrong = 0;
  // rows of 1 ... 2^31 vectors, odd ones among them, in tensors on both sides of 2^32 vectors
  const int64_t groups[] = {1, 2, 3, 1000, 4099, 65536, (1 << 20) + 1, (1 << 27) + 5, (int64_t(1) << 31) - 1, int64_t(1) << 31};
  const int64_t totals[] = {1 << 12, big - 1, big, big + 1, 2 * big + 12345, 8 * big};
  for (int64_t g : groups)
    for (int64_t total : totals)
      for (int G : {4, 8}) {
        const int64_t d0 = (total / g + 15) / 16 * 16 + (total < g ? 16 : 0), nvec = d0 * g, d1 = g * G, scales = d0 / 16 * d1;
        int64_t near[] = {0, g, 16 * g, nvec / 2, big, 2 * big, nvec - 1};
        for (int64_t at : near)
          for (int64_t v = at - 2; v <= at + 2; ++v) {
            if (v < 0 || v >= nvec) continue;
            const int64_t row = v / g, column = v % g * G, want = row / 16 * d1 + column;
            const int64_t got = G == 4 ? scale_of<4>(v, nvec, d1) : scale_of<8>(v, nvec, d1);
            ++checked;
            if (got != want || got < 0 || got + G > scales) ++wrong;
          }
      }
  printf("%ld %ld\n", checked, wrong);
}
"""


def test_scales_of_vectors_on_both_sides_of_32_bits(tmp_path):
    src, exe = tmp_path / "index.cpp", tmp_path / "index"
    src.write_text(SOURCE)
    subprocess.run(["g++", "-std=c++17", "-O1", "-I", os.path.join(ROOT, "tensorrt-incubator_amd", "csrc", "kernels"), "-o", str(exe), str(src)], check=True)
    checked, wrong = (int(v) for v in subprocess.run([str(exe)], check=True, stdout=subprocess.PIPE, text=True, timeout=60).stdout.split())
    assert checked > 1000 and wrong == 0
