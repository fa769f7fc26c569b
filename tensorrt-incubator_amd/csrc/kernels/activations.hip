// The activation side of a Linear, in one pass in front of its GEMM: rows of x [M, K] into rows of Kp elements, Kp = K rounded
// up to the GEMM's K slices, and, where the module quantizes its input, the codes (mtrt_act_codes_*) or the dequantized
// codes (mtrt_act_fake_*) instead of the values.  The padding is zero before it is quantized, so that a K that is no whole
// number of slices runs on the same kernels: its products are exact zeros, for the padded weights are zero and the padding
// is finite wherever x's own zeros are (with a scale of zero it has the largest code, as 0 / 0 is clamped to it, and that times
// the scale is zero again).  Same arithmetic, bit for bit, as mtrt_hip_quantize followed
// by mtrt_hip_dequantize with a per-tensor scale, in one launch that reads x once and writes the result once (as two they
// move 3 bytes per element more for 16-bit types; bf16 [999, 4096] to f8 and back 10.6 us as two launches).
//
// Bound by memory; a wave takes 128 groups of 16 bytes of one row, two per lane in flight, with 128-bit loads at element
// alignment (rows of x need not start on 16 bytes) and aligned stores.
#include "common.hpp"

namespace activations_cluster {

using namespace qdq_cluster;

constexpr int kActGroups = 2;                          // groups in flight per lane

// MODE: 0 values, 1 codes (one byte each), 2 dequantized codes
template <typename X, typename Q, int MODE, typename OUT>
__device__ __forceinline__ void act_rows(const typename X::storage* __restrict__ x, OUT* __restrict__ out, const float* __restrict__ scale,
                                         int64_t M, int64_t K, int64_t Kp) {
  using FG = FloatGroup<X>;
  constexpr int G = FG::G;
  const uint32_t groups = uint32_t(Kp / G);            // Kp is a whole number of groups
  const uint32_t chunks = (groups + kWave * kActGroups - 1) / (kWave * kActGroups);
  const int lane = threadIdx.x & (kWave - 1);
  const int64_t items = M * chunks, nwaves = waves_in_launch();
  const ExactDivisor dv(MODE == 0 ? 1.0f : scale[0]);
  for (int64_t item = wave_in_launch(); item < items; item += nwaves) {
    const int64_t row = item / chunks;
    const uint32_t g0 = uint32_t(item - row * chunks) * (kWave * kActGroups) + lane;
    u32x4 in[kActGroups];
#pragma unroll
    for (int u = 0; u < kActGroups; ++u) {
      const int64_t k = int64_t(g0 + u * kWave) * G;
      in[u] = (u32x4){0u, 0u, 0u, 0u};
      if (k + G <= K) {
        in[u] = *reinterpret_cast<const u32x4_unaligned*>(x + row * K + k);
      } else if (k < K) {                              // the group that holds the end of the row
#pragma unroll
        for (int e = 0; e < G; ++e) {
          if (k + e >= K) continue;
          const uint32_t bits = G == 4 ? f32_to_bits(Tile<X>::load1(x + row * K + k + e)) : uint32_t(*reinterpret_cast<const uint16_t*>(x + row * K + k + e));
          if (G == 4) in[u][e % 4] = bits;
          else in[u][(e >> 1) % 4] |= bits << (16 * (e & 1));
        }
      }
    }
#pragma unroll
    for (int u = 0; u < kActGroups; ++u) {
      const uint32_t g = g0 + u * kWave;
      if (g >= groups) continue;
      OUT* dst = out + row * Kp + int64_t(g) * G;
      if (MODE == 0) {
        *reinterpret_cast<u32x4*>(dst) = in[u];
      } else {
        float v[G];
        FG::unpack(in[u], v);
        quantize_group<Q>(dv, v, 0);
        uint32_t w[G / 4];
#pragma unroll
        for (int i = 0; i < G / 4; ++i) {
          w[i] = pack4<Q>(&v[4 * i], 0);
          if (MODE == 2) unpack4<Q>(w[i], &v[4 * i]);
        }
        if (MODE == 1) {
#pragma unroll
          for (int i = 0; i < G / 4; ++i) reinterpret_cast<uint32_t*>(dst)[i] = w[i];
        } else {
#pragma unroll
          for (int k = 0; k < G; ++k) v[k] = v[k] * dv.s;
          u32x4 t;
          if (G == 4) {
#pragma unroll
            for (int k = 0; k < 4; ++k) t[k] = f32_to_bits(v[k]);
          } else {
#pragma unroll
            for (int k = 0; k < 4; ++k) t[k] = narrow2<X>(v[(2 * k) % G], v[(2 * k + 1) % G]);
          }
          *reinterpret_cast<u32x4*>(dst) = t;
        }
      }
    }
  }
}

}  // namespace activations_cluster

// (x [M,K], out [M,Kp], scale: one f32, M, K, Kp) ; x aligned to its elements, out to 16 bytes, Kp % 16 == 0 and Kp >= K ;
// grid-stride over (row, chunk of 128 groups), block = 256.
#define MTRT_ACT_KERNEL(NAME, XT, QT, MODE, OUT)                                                                      \
  extern "C" __global__ void __launch_bounds__(256) NAME(const XT::storage* __restrict__ x, OUT* __restrict__ out,    \
                                                         const float* __restrict__ scale, int64_t M, int64_t K, int64_t Kp) { \
    activations_cluster::act_rows<XT, QT, MODE>(x, out, scale, M, K, Kp);                                             \
  }
MTRT_ACT_KERNEL(mtrt_act_pad_b16, F16, I8, 0, uint16_t)
MTRT_ACT_KERNEL(mtrt_act_codes_f16_i8, F16, I8, 1, int8_t)
#define MTRT_ACT_FOR_FLOAT(XN, XT)                                        \
  MTRT_ACT_KERNEL(mtrt_act_fake_##XN##_i8, XT, I8, 2, XT::storage)        \
  MTRT_ACT_KERNEL(mtrt_act_fake_##XN##_f8, XT, F8, 2, XT::storage)        \
  MTRT_ACT_KERNEL(mtrt_act_fake_##XN##_i4, XT, I4, 2, XT::storage)
MTRT_ACT_FOR_FLOAT(f32, F32)
MTRT_ACT_FOR_FLOAT(f16, F16)
MTRT_ACT_FOR_FLOAT(bf16, BF16)
