"""The quantize kernels form a quotient to a code as q0 = RN(x r), q = RN(q0 + RN(x - q0 s) r), r = RN(1/s)
(csrc/kernels/qdq.hip: quantize_fast1), which need not be the correctly rounded x / s.  This checks, on the CPU, that it lies on the same
side of every number where two codes can meet: those have at most 12 significant bits, and only an x / s beside the middle between such a
number and a neighbouring float could fall to the wrong side.  So for a scale s and each of the 2^11 numbers m of 12 bits: the three x
nearest to s m and to s times the middles below and above m, each by its quotient less than, equal to or greater than m, against the
IEEE quotient.  Powers of two in s and m change no rounding (the kernel divides outside of 2^-60 ... 2^60, test_gpu_quant_boundaries.py).

The normal run takes one in 64 of the 2^23 mantissas of s; MTRT_ALL_QUOTIENTS=1 takes all of them (1.5e11 quotients, 15 s on eight cores)."""
import os
import subprocess

import pytest

SOURCE = r"""
#include <math.h>
#include <stdint.h>
#include <stdio.h>
#include <stdlib.h>
#include <string.h>
static inline float from_bits(uint32_t u) { float f; memcpy(&f, &u, 4); return f; }
static inline uint32_t to_bits(float f) { uint32_t u; memcpy(&u, &f, 4); return u; }
static inline int side(float q, float m) { return (q > m) - (q < m); }
int main(int argc, char** argv) {
  const uint32_t step = (uint32_t)atoi(argv[1]);
  long long checked = 0, wrong = 0, single = 0;
  #pragma omp parallel for schedule(dynamic, 64) reduction(+ : checked, wrong, single)
  for (uint32_t i = 0; i < (1u << 23) / step; ++i) {
    const uint32_t mantissa = i * step + (i * 2654435761u >> 7) % step;      /* step 1: every one; else one of each step */
    const float s = from_bits(0x3F800000u | mantissa), r = 1.0f / s;
    int bad = 0, first = 0;
    for (int n = 2048; n < 4096; ++n) {
      const float m = (float)n;
      for (int d = -1; d <= 1; ++d) {
        const double target = 0.5 * ((double)m + (double)from_bits(to_bits(m) + (uint32_t)d));
        const uint32_t x0 = to_bits((float)((double)s * target));            /* 24 + 25 bits: the product is exact */
        for (int k = -1; k <= 1; ++k) {
          const float x = from_bits(x0 + (uint32_t)k);
          const float q0 = x * r, q = fmaf(fmaf(-q0, s, x), r, q0), ieee = x / s;
          bad += side(q, m) != side(ieee, m);
          first += side(q0, m) != side(ieee, m);
        }
      }
    }
    checked += 2048 * 9;
    wrong += bad;
    single += first;
  }
  printf("%lld %lld %lld\n", checked, wrong, single);
  return 0;
}
"""


def test_one_correction_leaves_every_code_as_it_is(tmp_path):
    src, exe = tmp_path / "quotient.c", tmp_path / "quotient"
    src.write_text(SOURCE)
    flags = ["-O3", "-ffp-contract=off", "-fno-trapping-math", "-fopenmp"]
    with open("/proc/cpuinfo") as f:
        info = f.read()
    fast = " fma " in info and " avx2 " in info
    subprocess.run(["gcc"] + flags + (["-mavx2", "-mfma"] if fast else []) + ["-o", str(exe), str(src), "-lm"], check=True)
    step = 1 if os.environ.get("MTRT_ALL_QUOTIENTS") == "1" else 64 if fast else 4096
    out = subprocess.run([str(exe), str(step)], check=True, stdout=subprocess.PIPE, text=True, timeout=110 if step > 1 else 3000).stdout.split()
    checked, wrong, uncorrected = (int(v) for v in out)
    assert checked == (1 << 23) // step * 2048 * 9
    assert wrong == 0
    assert uncorrected > 0                      # the correction is needed: without it some x fall to the wrong side
