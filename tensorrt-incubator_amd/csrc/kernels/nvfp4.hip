// NVFP4 block quantize / dequantize for gfx950: the two-level scaling of tensorrt.dynamic_quantize
// (mlir-tensorrt/tensorrt/include/mlir-tensorrt-dialect/TensorRT/IR/TensorRTOps.td:3279-3358) in the
// program form of mlir-tensorrt/integrations/PJRT/test/JAX/test_q_dq_nvfp4.py:21-45, blocks of 16
// along the last axis (or, in the *_cols kernels at the end, the second-to-last), every op in f32 and in this order:
//     S_dec_x = max|x_block| / 6        S_enc = 2688 / tensor_amax
//     s8      = f8e4m3fn(S_dec_x * S_enc)                  (block scale, stored)
//     S_enc_x = S_enc / f32(s8)         q = f4e2m1fn(f16(x * S_enc_x))
//     y       = narrow(f32(q) * (f32(s8) * (tensor_amax / 2688)))
// Conversions to f4 go through f16, the only f4 truncation the reference defines (RNE, saturation
// to +-6, inf -> +-6, NaN -> 0: mlir-tensorrt/executor/lib/Passes/ExpandOps.cpp:471-694).  An all-zero
// block has s8 = 0, S_enc_x = inf and x * S_enc_x = NaN, which that conversion maps to code 0; the
// same chain is evaluated here, no block is special-cased.  Only the last step differs by value: the
// hardware conversion gives a NaN another code than the reference's table, so NaN products take the table.
//
// Data movement: as in the quantize/dequantize clusters a lane owns one 128-bit vector of the float
// operand per trip (4 f32 or 8 f16/bf16), so a block of 16 is held by 4 (or 2) neighbouring lanes
// and its amax is two (one) cross-lane exchanges; every lane of the block then evaluates the
// block's scalar chain itself.  A wave handles 2, 4 or 8 consecutive trips (2 to 8 KiB of the float operand);
// its codes (8 trips: 1 or 2 KiB) and block scales (128 or 256 B) are parked in the wave's own LDS region
// and written out as whole cache lines, 16 bytes per lane.
#include "common.hpp"
#include "nvfp4_index.hpp"
#include "read_twice.hpp"

namespace nvfp4_cluster {

using namespace mtrt_dev;
using qdq_cluster::FloatGroup;

typedef _Float16 h2 __attribute__((ext_vector_type(2)));
typedef float f2 __attribute__((ext_vector_type(2)));

constexpr int kThreads = 256;
// vectors per lane.  Codes and scales are a fifth of what a dequantize moves, so it needs little in flight: 2, 4 and 8 vectors take
// bf16 of 134 MB 25.0, 25.4 and 25.7 us, f32 of 268 MB 42.9, 43.8 and 46.6
constexpr int kDqTrips = 2;

// the reference's table on one f16 bit pattern (exact, slow): used for blocks that contain NaN
__device__ __forceinline__ uint32_t f16_bits_to_f4_exact(uint32_t h) {
  const uint32_t a = h & 0x7FFFu, sign = (h >> 12) & 8u;
  if (a > 0x7C00u) return 0;
  const uint32_t code = (a > 0x3400u) + (a >= 0x3A00u) + (a > 0x3D00u) + (a >= 0x3F00u) + (a > 0x4100u) + (a >= 0x4300u) +
                        (a > 0x4500u);
  return code | sign;
}
// G products -> G f16 values (RNE), two per word, product k in half k % 2 of word k / 2
template <int G>
__device__ __forceinline__ void products_to_f16(float (&w)[G], uint32_t (&h)[G / 2]) {
#pragma unroll
  for (int k = 0; k < G; k += 2) {
    // The empty asm keeps the products' own f32 rounding in front of the f16 rounding (see f32_to_f16_bits in
    // common.hpp: without it the multiply and the conversion merge into one instruction that rounds once).
    __asm__("" : "+v"(w[k]), "+v"(w[k + 1]));
    union { h2 v; uint32_t u; } c;
    c.v = (h2){(_Float16)w[k], (_Float16)w[k + 1]};
    h[k / 2] = c.u;
  }
}
// is any of the G values a NaN?  (one unordered compare per pair)
template <int G>
__device__ __forceinline__ bool any_nan(const float (&w)[G]) {
  bool r = false;
#pragma unroll
  for (int k = 0; k < G; k += 2) r = r || __builtin_isunordered(w[k], w[k + 1]);
  return r;
}
// G f16 values -> G f4E2M1FN codes, value k in nibble k: the hardware conversion writes one byte of its
// destination and keeps the others.  Right for ordinary values; NaN (code 0 by the reference's rule) is
// patched in by the caller per block.
template <int G>
__device__ __forceinline__ uint32_t f16_to_f4(const uint32_t (&h)[G / 2]) {
  union { uint32_t u; h2 v; } c;
  c.u = h[0];
  uint32_t codes = __builtin_amdgcn_cvt_scalef32_pk_fp4_f16(0u, c.v, 1.0f, 0);
  c.u = h[1];
  codes = __builtin_amdgcn_cvt_scalef32_pk_fp4_f16(codes, c.v, 1.0f, 1);
  if (G == 8) {
    c.u = h[2 % (G / 2)];
    codes = __builtin_amdgcn_cvt_scalef32_pk_fp4_f16(codes, c.v, 1.0f, 2);
    c.u = h[3 % (G / 2)];
    codes = __builtin_amdgcn_cvt_scalef32_pk_fp4_f16(codes, c.v, 1.0f, 3);
  }
  return codes;
}
// the reference's table on value k of the packed f16 words
template <int G>
__device__ __forceinline__ uint32_t f16_to_f4_exact(const uint32_t (&h)[G / 2], int k) {
  return f16_bits_to_f4_exact((h[k / 2] >> (16 * (k & 1))) & 0xFFFFu);
}
// x / 6 for x >= 0 (a block maximum), correctly rounded, in 5 instructions instead of the 11 of the IEEE divide
// expansion: q0 = RN(x r), q = RN(q0 + RN(x - 6 q0) r) with r = RN(1/6) (the remainder of a faithful quotient is
// exact in an FMA; Markstein's correction).  Compared with the IEEE quotient on EVERY non-negative f32 on the
// CPU: equal for +0 and for all of [2^-125, FLT_MAX]; below (the remainder is no longer exact) and for
// inf / NaN the lanes take the real divide, in a wave-uniform branch that ordinary data never enters.
__device__ __forceinline__ float divide_by_six(float x) {
  const float r = 1.0f / 6.0f;
  const float q0 = x * r;
  float q = __builtin_fmaf(__builtin_fmaf(-q0, 6.0f, x), r, q0);
  // x / 2 is exact, and a positive normal number or +0 exactly where the short form holds: any other class
  // (0x2BF = all ten classes but those two) takes the divide
  const bool other = __builtin_amdgcn_classf(x * 0.5f, 0x2BF);
  if (__builtin_amdgcn_ballot_w64(other) != 0) q = other ? x / 6.0f : q;
  return q;
}
// S_enc / f32(s8) for every scale byte, one IEEE divide per lane of the workgroup (256 lanes): a block's second
// divide becomes a look-up.  Every lane of the workgroup must get here (there is a barrier inside).
__device__ __forceinline__ void fill_inverse_scales(float* table, float s_enc) {
  for (uint32_t b = threadIdx.x; b < 256u; b += block_threads()) table[b] = s_enc / f8_to_f32<0>(b);
  __syncthreads();
}

// (x, q_packed, scales, tensor_amax, nvec) ; nvec 128-bit vectors of x, a multiple of the vectors per block.
// A wave's time is the trip to memory, the scale table and then its trips one after the other, so few trips keep small tensors short and
// many amortize the table (the rule and its figures: nvfp4_trips in clusters.cpp).  With few trips x is asked for before the table
// is filled; with eight other waves cover the wait.  A kernel for each number: the same bodies in one kernel took 0.3 to 0.9 us more (a launch
// fetches its instructions anew).
template <typename X, int TRIPS>
__device__ __forceinline__ void quantize_body(const typename X::storage* __restrict__ x, uint8_t* __restrict__ q,
                                              uint8_t* __restrict__ scales, const float* __restrict__ tensor_amax,
                                              int64_t nvec) {
  constexpr int G = FloatGroup<X>::G;                  // elements per vector: 4 or 8
  constexpr int LPB = 16 / G;                          // lanes per block: 4 or 2
  constexpr int kCodeBytes = G / 2;                    // code bytes per lane and trip
  constexpr int kSpanCodes = TRIPS * 64 * kCodeBytes;  // eight trips: 1 or 2 KiB per wave
  constexpr int kSpanScales = TRIPS * 64 / LPB;        // eight trips: 128 or 256 B per wave
  __shared__ __attribute__((aligned(16))) uint8_t lds[(kThreads / 64) * (kSpanCodes + kSpanScales)];
  __shared__ float inverse_scale[256];
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  uint8_t* my_codes = lds + wave * (kSpanCodes + kSpanScales);
  uint8_t* my_scales = my_codes + kSpanCodes;
  const uint32_t piece = TRIPS == 8 ? blockIdx.x : piece_of<8 / TRIPS>(blockIdx.x, gridDim.x, nvec * 16);   // behind an amax pass: see read_twice.hpp
  const int64_t span = (int64_t(piece) * (kThreads / 64) + wave) * (TRIPS * 64);        // first vector of this wave
  const float s_enc = 2688.0f / *tensor_amax;
  if (TRIPS == 8) fill_inverse_scales(inverse_scale, s_enc);
  if (TRIPS == 8 && span >= nvec) return;              // whole wave
  u32x4 t[TRIPS];
#pragma unroll
  for (int j = 0; j < TRIPS; ++j) {
    int64_t v = span + j * 64 + lane;
    v = v < nvec ? v : nvec - 1;                       // past the end: a valid vector, its results are not stored
    t[j] = __builtin_nontemporal_load(reinterpret_cast<const u32x4*>(x) + v);
  }
  if (TRIPS != 8) fill_inverse_scales(inverse_scale, s_enc);
  if (TRIPS != 8 && span >= nvec) return;
#pragma unroll
  for (int j = 0; j < TRIPS; ++j) {
    float v[G];
    FloatGroup<X>::unpack(t[j], v);
    float amax = 0.0f;
#pragma unroll
    for (int k = 0; k < G; ++k) amax = fmaxf(amax, fabsf(v[k]));
    amax = lanes_reduce<LPB>(amax, MaxF32());
    const float s_dec_x = divide_by_six(amax);
    uint32_t s8 = f32x2_to_f8_ieee(s_dec_x * s_enc, 0.0f) & 0xFFu;
    s8 = (s8 & 0x7Fu) == 0x7Fu ? 0x7Fu : s8;             // NaN (0 * inf when the tensor amax is 0): 0x7F whatever its sign, as the host class
    const float s_enc_x = inverse_scale[s8];             // = s_enc / f32(s8), the same IEEE quotient
    float w[G];
#pragma unroll
    for (int k = 0; k < G; ++k) w[k] = v[k] * s_enc_x;
    uint32_t h[G / 2];
    products_to_f16<G>(w, h);
    uint32_t codes = f16_to_f4<G>(h);
    // A NaN product (a NaN element; a zero times an infinite S_enc_x, which a scale byte of 0 or a tiny tensor
    // amax produce; anything times a NaN S_enc_x) has code 0 by the reference's rule, not the hardware's: lanes
    // that hold one convert again by the reference's table (a wave-uniform branch that is rarely taken)
    const bool special = any_nan<G>(w);
    if (__builtin_amdgcn_ballot_w64(special) != 0) {
      uint32_t exact = 0;
#pragma unroll
      for (int k = 0; k < G; ++k) exact |= f16_to_f4_exact<G>(h, k) << (4 * k);
      codes = special ? exact : codes;
    }
    if (G == 4) *reinterpret_cast<uint16_t*>(my_codes + (j * 64 + lane) * 2) = uint16_t(codes);
    else *reinterpret_cast<uint32_t*>(my_codes + (j * 64 + lane) * 4) = codes;
    if ((lane & (LPB - 1)) == 0) my_scales[(j * 64 + lane) / LPB] = uint8_t(s8);
  }
  // this wave's own LDS region only: program order suffices, no barrier
  const int64_t left = nvec - span;                    // vectors of this span that exist (>= 1)
  const int64_t code_bytes = (left < TRIPS * 64 ? left : TRIPS * 64) * kCodeBytes;
  const int64_t scale_bytes = (left < TRIPS * 64 ? left : TRIPS * 64) / LPB;
  uint8_t* qo = q + span * kCodeBytes;
  uint8_t* so = scales + span / LPB;
#pragma unroll
  for (int c = 0; c < (kSpanCodes + 1023) / 1024; ++c) {
    const int o = (c * 64 + lane) * 16;
    if (kSpanCodes % 1024 != 0 && o >= kSpanCodes) break;
    const u32x4 vv = *reinterpret_cast<const u32x4*>(my_codes + o);
    if (o + 16 <= code_bytes) {
      *reinterpret_cast<u32x4*>(qo + o) = vv;            // q is 16-byte aligned (checked by the host side)
    } else {
      for (int b = 0; b < 16; b += 2)                    // ragged end: code bytes come in pairs at least
        if (o + b < code_bytes) *reinterpret_cast<uint16_t*>(qo + o + b) = uint16_t(vv[b >> 2] >> (8 * (b & 3)));
    }
  }
  if (lane * 4 < kSpanScales) {
    const int o = lane * 4;
    const uint32_t vv = *reinterpret_cast<const uint32_t*>(my_scales + o);
    if (o + 4 <= scale_bytes && (reinterpret_cast<uintptr_t>(so) & 3) == 0) {
      *reinterpret_cast<uint32_t*>(so + o) = vv;
    } else {
      for (int b = 0; b < 4; ++b)
        if (o + b < scale_bytes) so[o + b] = uint8_t(vv >> (8 * b));
    }
  }
}

// (q_packed, scales, tensor_amax, y, nvec) ; nvec 128-bit vectors of y
template <typename Y>
__device__ __forceinline__ void dequantize_body(const uint8_t* __restrict__ q, const uint8_t* __restrict__ scales,
                                                const float* __restrict__ tensor_amax, typename Y::storage* __restrict__ y,
                                                int64_t nvec) {
  constexpr int G = FloatGroup<Y>::G;
  constexpr int LPB = 16 / G;
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  const int64_t span = (int64_t(blockIdx.x) * (kThreads / 64) + wave) * (kDqTrips * 64);
  if (span >= nvec) return;
  const float s_dec = *tensor_amax / 2688.0f;
  uint32_t codes[kDqTrips], s8[kDqTrips];
#pragma unroll
  for (int j = 0; j < kDqTrips; ++j) {
    int64_t v = span + j * 64 + lane;
    v = v < nvec ? v : nvec - 1;
    codes[j] = G == 4 ? uint32_t(*reinterpret_cast<const uint16_t*>(q + v * 2)) : *reinterpret_cast<const uint32_t*>(q + v * 4);
    s8[j] = scales[v / LPB];
  }
#pragma unroll
  for (int j = 0; j < kDqTrips; ++j) {
    const int64_t v = span + j * 64 + lane;
    const float u = f8_to_f32<0>(s8[j]) * s_dec;
    float out[G];
#pragma unroll
    for (int k = 0; k < G; k += 2) {
      f2 p;
      if (k == 0) p = __builtin_amdgcn_cvt_scalef32_pk_f32_fp4(codes[j], 1.0f, 0);
      else if (k == 2) p = __builtin_amdgcn_cvt_scalef32_pk_f32_fp4(codes[j], 1.0f, 1);
      else if (k == 4) p = __builtin_amdgcn_cvt_scalef32_pk_f32_fp4(codes[j], 1.0f, 2);
      else p = __builtin_amdgcn_cvt_scalef32_pk_f32_fp4(codes[j], 1.0f, 3);
      out[k] = p[0] * u;
      out[k + 1] = p[1] * u;
    }
    if (v < nvec) FloatGroup<Y>::store(y + v * G, out);
  }
}

// ---- blocks of 16 along the SECOND-TO-LAST axis ([d0, d1] view, d0 % 16 == 0) ----------------------
// A unit is G neighbouring columns of one block row.  The lanes l, l + 16, l + 32 and l + 48 of a wave share it, four of its
// sixteen rows each: the block amax is a maximum down the lane's own registers and two exchanges, and every lane computes the
// scales of a quarter of the columns.  Per row a wave reads 256 bytes and its workgroup 1 KiB of contiguous memory.
// Bound by memory where enough waves are in flight, by the length of a lane's work where few are.  With all sixteen rows in
// one lane (158 registers, three waves per SIMD), eight in each of two, and four in each of four (54 registers), us:
//   bf16 [4096, 8192] 29.8, 20.4, 16.5   [16384, 4096] 42.5, 32.4, 28.9   [7136, 528] 14.5, 8.4, 5.7   [16384, 64] 9.3, 5.8, 4.1
//   f32  [4096, 8192] 30.8, 26.9, 27.3   [16384, 4096] 55.0, 51.2, 52.3   [7136, 528] 9.6, 6.6, 5.4    [16384, 64] 6.5, 4.4, 3.4
// (x, q_packed, scales, tensor_amax, d0, d1) ; d1 % G == 0 ; four lanes per unit
template <typename X>
__device__ __forceinline__ void quantize_cols_body(const typename X::storage* __restrict__ x, uint8_t* __restrict__ q,
                                                   uint8_t* __restrict__ scales, const float* __restrict__ tensor_amax,
                                                   int64_t d0, int64_t d1) {
  constexpr int G = FloatGroup<X>::G;
  constexpr int R = 4;                                 // rows per lane
  __shared__ float inverse_scale[256];
  const uint32_t groups = uint32_t(d1 / G), units = uint32_t((d0 / 16) * groups);   // 2^32 units are a TiB of x: more than there is
  const uint32_t part = (threadIdx.x >> 4) & 3;
  uint32_t u = blockIdx.x * (kThreads / 4) + (threadIdx.x >> 6) * 16 + (threadIdx.x & 15);
  u = u < units ? u : units - 1;                       // past the end: the last unit once more, which stores the same bytes
  const uint32_t rb = u / groups;
  const int64_t c0 = int64_t(u - rb * groups) * G, row0 = int64_t(rb) * 16 + part * R;
  const typename X::storage* xp = x + row0 * d1 + c0;
  u32x4 t[R];
#pragma unroll
  for (int r = 0; r < R; ++r) t[r] = __builtin_nontemporal_load(reinterpret_cast<const u32x4*>(xp + r * d1));
  const float s_enc = 2688.0f / *tensor_amax;
  fill_inverse_scales(inverse_scale, s_enc);
  float amax[G];
#pragma unroll
  for (int k = 0; k < G; ++k) amax[k] = 0.0f;
#pragma unroll
  for (int r = 0; r < R; ++r) {
    float v[G];
    FloatGroup<X>::unpack(t[r], v);
#pragma unroll
    for (int k = 0; k < G; ++k) amax[k] = fmaxf(amax[k], fabsf(v[k]));
  }
  // Two swaps of lane groups leave each lane with the block maxima of a quarter of the columns (16-lane group j: columns
  // j G/4 ...); it computes their scales, and the same swaps hand those to all four lanes.
  uint32_t m[G / 2], s8[G / 4];
  float s_enc_x[G];
#pragma unroll
  for (int k = 0; k < G / 2; ++k) {
    const auto t2 = __builtin_amdgcn_permlane32_swap(f32_to_bits(amax[k]), f32_to_bits(amax[k + G / 2]), false, false);
    m[k] = f32_to_bits(fmaxf(bits_to_f32(t2[0]), bits_to_f32(t2[1])));
  }
#pragma unroll
  for (int k = 0; k < G / 4; ++k) {
    const auto t2 = __builtin_amdgcn_permlane16_swap(m[k], m[k + G / 4], false, false);
    const float s_dec_x = divide_by_six(fmaxf(bits_to_f32(t2[0]), bits_to_f32(t2[1])));
    uint32_t b = f32x2_to_f8_ieee(s_dec_x * s_enc, 0.0f) & 0xFFu;
    b = (b & 0x7Fu) == 0x7Fu ? 0x7Fu : b;
    s8[k] = b;
    const uint32_t inverse = f32_to_bits(inverse_scale[b]);   // = s_enc / f32(b), the same IEEE quotient
    const auto pair = __builtin_amdgcn_permlane16_swap(inverse, inverse, false, false);
#pragma unroll
    for (int p = 0; p < 2; ++p) {
      const auto halves = __builtin_amdgcn_permlane32_swap(pair[p], pair[p], false, false);
      s_enc_x[k + p * (G / 4)] = bits_to_f32(halves[0]);
      s_enc_x[k + p * (G / 4) + G / 2] = bits_to_f32(halves[1]);
    }
  }
  uint8_t* sp = scales + rb * d1 + c0 + part * (G / 4);
  if (G == 4) *sp = uint8_t(s8[0]);
  else *reinterpret_cast<uint16_t*>(sp) = uint16_t(s8[0] | (s8[1 % (G / 4)] << 8));
  uint8_t* qp = q + (row0 * d1 + c0) / 2;
#pragma unroll
  for (int r = 0; r < R; ++r) {
    float v[G], w[G];
    FloatGroup<X>::unpack(t[r], v);
#pragma unroll
    for (int k = 0; k < G; ++k) w[k] = v[k] * s_enc_x[k];
    uint32_t h[G / 2];
    products_to_f16<G>(w, h);
    uint32_t codes = f16_to_f4<G>(h);
    const bool special = any_nan<G>(w);                // a NaN product: the reference's table (see quantize_body)
    if (__builtin_amdgcn_ballot_w64(special) != 0) {
      uint32_t exact = 0;
#pragma unroll
      for (int k = 0; k < G; ++k) exact |= f16_to_f4_exact<G>(h, k) << (4 * k);
      codes = special ? exact : codes;
    }
    if (G == 4) *reinterpret_cast<uint16_t*>(qp + r * (d1 / 2)) = uint16_t(codes);
    else *reinterpret_cast<uint32_t*>(qp + r * (d1 / 2)) = codes;
  }
}

// (q_packed, scales, tensor_amax, y, d0, d1) ; one lane per output vector
template <typename Y, bool NARROW>
__device__ __forceinline__ void dequantize_cols_body(const uint8_t* __restrict__ q, const uint8_t* __restrict__ scales,
                                                     const float* __restrict__ tensor_amax,
                                                     typename Y::storage* __restrict__ y, int64_t d0, int64_t d1) {
  constexpr int G = FloatGroup<Y>::G;
  const int64_t nvec = d0 * (d1 / G);
  const float s_dec = *tensor_amax / 2688.0f;
  const int64_t stride = int64_t(gridDim.x) * kThreads;
  for (int64_t v = int64_t(blockIdx.x) * kThreads + threadIdx.x; v < nvec; v += stride) {
    const uint32_t codes = G == 4 ? uint32_t(*reinterpret_cast<const uint16_t*>(q + v * 2)) : *reinterpret_cast<const uint32_t*>(q + v * 4);
    const uint8_t* sp = scales + scale_of_vector<NARROW, G>(v, d1);
    uint32_t sw[2];
    sw[0] = *reinterpret_cast<const uint32_t*>(sp);
    sw[1] = G == 8 ? *reinterpret_cast<const uint32_t*>(sp + 4) : 0u;
    float out[G];
#pragma unroll
    for (int k = 0; k < G; k += 2) {
      f2 p;
      if (k == 0) p = __builtin_amdgcn_cvt_scalef32_pk_f32_fp4(codes, 1.0f, 0);
      else if (k == 2) p = __builtin_amdgcn_cvt_scalef32_pk_f32_fp4(codes, 1.0f, 1);
      else if (k == 4) p = __builtin_amdgcn_cvt_scalef32_pk_f32_fp4(codes, 1.0f, 2);
      else p = __builtin_amdgcn_cvt_scalef32_pk_f32_fp4(codes, 1.0f, 3);
      const uint32_t word = sw[k / 4];
      const float u0 = ((k & 3) == 0 ? f8_to_f32<0>(word) : f8_to_f32<2>(word)) * s_dec;
      const float u1 = ((k & 3) == 0 ? f8_to_f32<1>(word) : f8_to_f32<3>(word)) * s_dec;
      out[k] = p[0] * u0;
      out[k + 1] = p[1] * u1;
    }
    FloatGroup<Y>::store(y + v * G, out);
  }
}

}  // namespace nvfp4_cluster

// mtrt_nvfp4_q_<t>(x, q_packed, scales, tensor_amax, nvec), 8 trips, and with 2 and 4 mtrt_nvfp4_q2_<t>, mtrt_nvfp4_q4_<t> ;
// mtrt_nvfp4_dq_<t>(q_packed, scales, tensor_amax, y, nvec), 2 trips ; grid = ceil(nvec / (4 waves * 64 * trips)); block = 256; x / y and q_packed 16-byte aligned.
#define MTRT_NVFP4_QUANTIZE(NAME, XT, TRIPS)                                                                            \
  extern "C" __global__ void __launch_bounds__(nvfp4_cluster::kThreads) NAME(                                           \
      const XT::storage* x, uint8_t* q, uint8_t* scales, const float* tensor_amax, int64_t nvec) {                      \
    nvfp4_cluster::quantize_body<XT, TRIPS>(x, q, scales, tensor_amax, nvec);                                           \
  }
#define MTRT_NVFP4_KERNELS(XN, XT)                                                                                      \
  MTRT_NVFP4_QUANTIZE(mtrt_nvfp4_q2_##XN, XT, 2)                                                                        \
  MTRT_NVFP4_QUANTIZE(mtrt_nvfp4_q4_##XN, XT, 4)                                                                        \
  MTRT_NVFP4_QUANTIZE(mtrt_nvfp4_q_##XN, XT, 8)                                                                         \
  extern "C" __global__ void __launch_bounds__(nvfp4_cluster::kThreads) mtrt_nvfp4_dq_##XN(                              \
      const uint8_t* q, const uint8_t* scales, const float* tensor_amax, XT::storage* y, int64_t nvec) {                \
    nvfp4_cluster::dequantize_body<XT>(q, scales, tensor_amax, y, nvec);                                                \
  }
// Blocks along the second-to-last axis: mtrt_nvfp4_qc_<t>(x, q_packed, scales, tensor_amax, d0, d1) with
// grid = ceil((d0 / 16) * (d1 / G) / 64); mtrt_nvfp4_dqc_<t>(q_packed, scales, tensor_amax, y, d0, d1), below 2^32 vectors, and
// mtrt_nvfp4_dqc_far_<t>, any number of them: grid: any.  (Both divisions in one kernel, whichever way, cost every launch 0.25 us.)
// d1 % G == 0 (G = 4 for f32, 8 for f16 / bf16), x / y rows 16-byte aligned, scales 4- (G = 4) or 8-byte aligned.
#define MTRT_NVFP4_COL_KERNELS(XN, XT)                                                                                  \
  extern "C" __global__ void __launch_bounds__(nvfp4_cluster::kThreads) mtrt_nvfp4_qc_##XN(                              \
      const XT::storage* x, uint8_t* q, uint8_t* scales, const float* tensor_amax, int64_t d0, int64_t d1) {            \
    nvfp4_cluster::quantize_cols_body<XT>(x, q, scales, tensor_amax, d0, d1);                                           \
  }                                                                                                                     \
  extern "C" __global__ void __launch_bounds__(nvfp4_cluster::kThreads) mtrt_nvfp4_dqc_##XN(                             \
      const uint8_t* q, const uint8_t* scales, const float* tensor_amax, XT::storage* y, int64_t d0, int64_t d1) {      \
    nvfp4_cluster::dequantize_cols_body<XT, true>(q, scales, tensor_amax, y, d0, d1);                                   \
  }                                                                                                                     \
  extern "C" __global__ void __launch_bounds__(nvfp4_cluster::kThreads) mtrt_nvfp4_dqc_far_##XN(                         \
      const uint8_t* q, const uint8_t* scales, const float* tensor_amax, XT::storage* y, int64_t d0, int64_t d1) {      \
    nvfp4_cluster::dequantize_cols_body<XT, false>(q, scales, tensor_amax, y, d0, d1);                                  \
  }
MTRT_NVFP4_COL_KERNELS(f32, mtrt_dev::F32)
MTRT_NVFP4_COL_KERNELS(f16, mtrt_dev::F16)
MTRT_NVFP4_COL_KERNELS(bf16, mtrt_dev::BF16)
MTRT_NVFP4_KERNELS(f32, mtrt_dev::F32)
MTRT_NVFP4_KERNELS(f16, mtrt_dev::F16)
MTRT_NVFP4_KERNELS(bf16, mtrt_dev::BF16)
