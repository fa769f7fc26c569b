// W8A8 GEMM cluster for gfx950:
//     acc[m,n] = sum_k i32(a[m,k]) * i32(w[k,n])                 (exact int32)
//     y[m,n]   = f16((f32(acc[m,n]) * a_scale[m]) * w_scale[n])   (two f32 roundings, then f16)
// i.e. the dot_general + per-token / per-output-channel dequantize epilogue of a
// quantized Linear (tripy/nvtripy/frontend/module/linear.py:112-151), which the
// reference realises as a plain FMA loop nest without matrix cores
// (mlir-tensorrt/kernel/test/Kernel/TransformSchedules/fallback-schedule-matmul.mlir:24).
//
// Matrix cores want both operands contiguous along K per row/column.  Activations
// [M,K] already are.  Weights arrive as [K,N] (N contiguous); they are constants of
// the program, so they are re-laid once into [N,K] by mtrt_w8_prepack_kn_to_nk and
// the GEMM consumes that.  The main loop (tiling, pipeline, LDS layout, tile order,
// epilogue staging) is the shared one in gemm_core.hpp with v_mfma_i32_32x32x32_i8.
#include "gemm_frag.hpp"

namespace gemm_w8a8_cluster {

using namespace mtrt_dev;
using gemm_core::v4i;
typedef int v16i __attribute__((ext_vector_type(16)));

struct I8Traits {
  using Acc = v16i;
  using Scalar = int;
  static __device__ __forceinline__ Acc zero() {
    Acc z;
#pragma unroll
    for (int r = 0; r < 16; ++r) z[r] = 0;
    return z;
  }
  static __device__ __forceinline__ Acc mfma(v4i a, v4i b, Acc c) { return __builtin_amdgcn_mfma_i32_32x32x32_i8(a, b, c, 0, 0, 0); }
  // accumulators in ordinary vector registers (gemm_frag::run_wide)
  static __device__ __forceinline__ void mfma_vgpr(v4i a, v4i b, Acc& c) { __asm__ volatile("v_mfma_i32_32x32x32_i8 %0, %1, %2, %0" : "+v"(c) : "v"(a), "v"(b)); }
  static __device__ __forceinline__ void clear_vgpr(v4i a, v4i b, Acc& c) { __asm__ volatile("v_mfma_i32_32x32x32_i8 %0, %1, %2, 0" : "=v"(c) : "v"(a), "v"(b)); }
};

// The results of a quantized Linear: f16((f32(acc) * a_scale) * w_scale), then, with a bias, the f16 sum of that and it
// (two f16 roundings, as a separate addition gives).
__device__ __forceinline__ uint32_t add_bias2(uint32_t word, float b0, float b1) {
  return f32x2_to_f16x2_bits(f16_bits_to_f32(word & 0xFFFFu) + b0, f16_bits_to_f32(word >> 16) + b1);
}

// BN: columns of the workgroup's tile (the scratch holds 256 + 2 BN floats).  a_step: 1, or 0 for one scale for all rows.
// BIAS: whether there may be a bias (it is tested for null then).
template <int BN, bool BIAS = false>
struct ScaleEpilogueT {
  static constexpr int kScratch = 256 + (BIAS ? 2 : 1) * BN;
  const float* a_scale;
  const float* w_scale;
  uint32_t a_step;
  const uint16_t* bias;
  const float* sa;                                   // a_scale of this tile's 256 rows, in LDS
  const float* sw;                                   // w_scale of this tile's BN columns, in LDS; then the bias
  float as;
  __device__ __forceinline__ ScaleEpilogueT(const float* a, const float* w, uint32_t step = 1, const uint16_t* b = nullptr)
      : a_scale(a), w_scale(w), a_step(step), bias(b) {}
  __device__ __forceinline__ void setup(int8_t* scratch, int64_t m0, int64_t M, int64_t n0, int64_t N) {
    float* dst = reinterpret_cast<float*>(scratch);
    const int64_t row = m0 + threadIdx.x;              // the first 256 threads: 256 rows
    if (threadIdx.x < 256) dst[threadIdx.x] = row < M ? a_scale[row * a_step] : 0.0f;
    for (int c = threadIdx.x; c < BN; c += block_threads()) dst[256 + c] = n0 + c < N ? w_scale[n0 + c] : 0.0f;
    if (BIAS && bias)
      for (int c = threadIdx.x; c < BN; c += block_threads()) dst[256 + BN + c] = n0 + c < N ? f16_bits_to_f32(bias[n0 + c]) : 0.0f;
    sa = dst;
    sw = dst + 256;
  }
  __device__ __forceinline__ void row(int row_in_tile) { as = sa[row_in_tile]; }
  // the lane's column scales of one staging pass (HC column tiles of 32, four runs of four columns each), read from LDS
  // once and kept in registers for the pass's rows
  template <int HC>
  __device__ __forceinline__ void columns(int first_col_in_tile) {
#pragma unroll
    for (int jj = 0; jj < HC; ++jj)
#pragma unroll
      for (int q = 0; q < 4; ++q) {
        wsr[jj][q] = *reinterpret_cast<const f32x4*>(sw + first_col_in_tile + jj * 32 + q * 8);
        if (BIAS && bias) br[jj][q] = *reinterpret_cast<const f32x4*>(sw + BN + first_col_in_tile + jj * 32 + q * 8);
      }
  }
  __device__ __forceinline__ void convert4(const v16i& acc, int q, int jj, uint32_t (&words)[2]) const {
#pragma unroll
    for (int e = 0; e < 4; e += 2)
      words[e >> 1] = f32x2_to_f16x2_bits((float(acc[4 * q + e]) * as) * wsr[jj][q][e], (float(acc[4 * q + e + 1]) * as) * wsr[jj][q][e + 1]);
    if (BIAS && bias) {
#pragma unroll
      for (int e = 0; e < 4; e += 2) words[e >> 1] = add_bias2(words[e >> 1], br[jj][q][e], br[jj][q][e + 1]);
    }
  }
  f32x4 wsr[2][4], br[2][4];
};
using ScaleEpilogue = ScaleEpilogueT<256>;

// The entry points below have C linkage; they sit inside the namespace only so that
// its helper names do not meet those of the other clusters in the one-module build.

// (a [M,K] i8, w_nk [N,K] i8, a_scale [M] f32, w_scale [N] f32, y [M,N] f16, M, K, N, full_panels) ; K % 128 == 0,
// a and w_nk 16-byte aligned, both below 4 GiB.  The first full_panels * 256 columns are computed in
// 256 x 256 tiles, the rest in 256 x 128 tiles: with one workgroup per compute unit a launch runs in
// rounds, and a last round that would use few of the units is cut into twice as many tiles of half
// the length.  grid = even_blocks(full_panels * tiles_m) + even_blocks(half panels * tiles_m), block = 256 (each kind
// of tile dealt evenly to the XCDs, gemm_core::tile_of_even).
extern "C" __global__ void __launch_bounds__(gemm_core::THREADS, 1) mtrt_gemm_w8a8_nk(
    const int8_t* __restrict__ a, const int8_t* __restrict__ w, const float* __restrict__ a_scale,
    const float* __restrict__ w_scale, uint16_t* __restrict__ y, int64_t M, int64_t K, int64_t N, int64_t full_panels) {
  __shared__ __attribute__((aligned(16))) int8_t lds[gemm_core::LDS_BYTES];
  const int64_t tiles_m = (M + gemm_core::BM - 1) / gemm_core::BM;
  const int64_t full_blocks = gemm_core::even_blocks(full_panels * tiles_m);
  ScaleEpilogue epi{a_scale, w_scale};
  int64_t tile_m, panel;
  if (int64_t(blockIdx.x) < full_blocks) {
    if (!gemm_core::tile_of_even(blockIdx.x, uint32_t(full_blocks), tiles_m, full_panels, tiles_m, tile_m, panel)) return;
    gemm_core::run<I8Traits, 4>(a, w, K, epi, y, M, N, K / gemm_core::BKB, tile_m * 256, panel * 256, lds);
  } else {
    const int64_t n_full = full_panels * 256;
    if (!gemm_core::tile_of_even(blockIdx.x - uint32_t(full_blocks), gridDim.x - uint32_t(full_blocks), tiles_m, (N - n_full + 127) / 128,
                                 tiles_m, tile_m, panel))
      return;
    gemm_core::run<I8Traits, 2>(a, w, K, epi, y, M, N, K / gemm_core::BKB, tile_m * 256, n_full + panel * 128, lds);
  }
}

// ---- weights in fragment order (gemm_frag.hpp) ---------------------------------------------------------
// mtrt_gemm_w8a8_frag_t<rows>x<columns> (a [M,K] i8, w_frag, a_scale [M] f32, w_scale [N] f32, y [M,N] f16, M, K, N, Split,
// a_step, bias) ; K % 128 == 0, a and w_frag 16-byte aligned, a below 4 GiB; a_step 1, or 0 for a
// single a_scale; bias f16 [N] or null.
// grid = 8 * ceil(tiles * splits / 8), block = 256.  Tiles of 32 x 128, 64 x 128, 128 x 128 and 128 x 256 (two
// workgroups per compute unit), 128 x 384 and 256 x 256 (one; the last never split).  Which tile and how many splits: the host's
// estimate of the launch (frag_plan in clusters.cpp).  Measured, the one 256-row tile loop that these replaced -> now,
// us: (M, K, N) = (256, 4096, 4096) 21.8 -> 10.4, (398, 11520, 1856) 51.8 -> 19.3, (1024, 2048, 2048) 14.7 -> 8.8,
// (200, 12288, 512) 52.7 -> 10.6, (999, 4096, 11008) 46.5 -> 44.
// t128x256: 239 registers, so that one workgroup's first loads and its epilogue (6 us of a tile) lie under the other's loop, where a unit has more
// than one; a meeting fetches two 32 x 32 tiles of two parts at a time (gemm_frag::meet).  One and two to a unit, us: (3043, 768, 13632) 59.6, 42.2;
// (4011, 256, 12672) 46.5, 37.1; (2048, 4096, 11008) 91.1, 81.7; (999, 4096, 11008) 54.4, 48.3; where a unit has one tile (985, 1152, 4352) 12.0,
// 11.6; (1296, 4992, 4352) 32.9, 32.1; with K in two parts (2332, 10368, 1024) 38.4, 37.7.
#define MTRT_W8_FRAG_KERNEL(NAME, IT, JT, D, WG)                                                                          \
  extern "C" __global__ void __launch_bounds__(256, WG) NAME(                                                             \
      const int8_t* __restrict__ a, const int8_t* __restrict__ w_frag, const float* __restrict__ a_scale,                 \
      const float* __restrict__ w_scale, uint16_t* __restrict__ y, int64_t M, int64_t K, int64_t N,                       \
      gemm_frag::Split sp, uint32_t a_step, const uint16_t* __restrict__ bias) {                                          \
    using Epilogue = ScaleEpilogueT<128 * JT, true>;                                                                      \
    __shared__ __attribute__((aligned(16))) int8_t lds[gemm_frag::lds_bytes<IT, D>(Epilogue::kScratch)];                  \
    gemm_frag::Part part;                                                                                                 \
    if (!gemm_frag::part_of<32 * IT, 128 * JT>(blockIdx.x, gridDim.x, M, N, uint32_t(K) / 128, sp, part)) return; \
    Epilogue epi{a_scale, w_scale, a_step, bias};                                                                         \
    gemm_frag::run<I8Traits, IT, JT, D>(a, K, gemm_core::Values{w_frag}, epi, y, M, N, part, lds);                                           \
  }
MTRT_W8_FRAG_KERNEL(mtrt_gemm_w8a8_frag_t32x128, 1, 1, 4, 2)
MTRT_W8_FRAG_KERNEL(mtrt_gemm_w8a8_frag_t64x128, 2, 1, 4, 2)
MTRT_W8_FRAG_KERNEL(mtrt_gemm_w8a8_frag_t128x128, 4, 1, 2, 2)
MTRT_W8_FRAG_KERNEL(mtrt_gemm_w8a8_frag_t128x256, 4, 2, 2, 2)
MTRT_W8_FRAG_KERNEL(mtrt_gemm_w8a8_frag_t128x384, 4, 3, 2, 1)
MTRT_W8_FRAG_KERNEL(mtrt_gemm_w8a8_frag_t256x256, 8, 2, 2, 1)

// 256 x 384 tiles (gemm_frag::run_wide).  (a, w_frag, a_scale, w_scale, y, M, K, N [, a_step, bias]) as above.
// grid = 8 * ceil(ceil(M/256) * ceil(N/384) / 8), block = 256: the tiles dealt evenly to the XCDs, a panel's M tiles neighbours.
template <class Epilogue>
__device__ __forceinline__ void wide_kernel(const int8_t* __restrict__ a, const int8_t* __restrict__ w_frag, Epilogue& epi,
                                            uint16_t* __restrict__ y, int64_t M, int64_t K, int64_t N, int8_t* lds) {
  const int64_t tiles_m = (M + 255) / 256, panels = (N + gemm_frag::kWideBN - 1) / gemm_frag::kWideBN;
  int64_t tile_m, panel;
  if (!gemm_core::tile_of_even(blockIdx.x, gridDim.x, tiles_m, panels, tiles_m, tile_m, panel)) return;
  gemm_frag::run_wide<I8Traits>(a, K, gemm_core::Values{w_frag}, (N + 31) / 32, epi, y, M, N, K / 128, tile_m * 256, panel * gemm_frag::kWideBN, lds);
}
extern "C" __global__ void __launch_bounds__(256, 1) mtrt_gemm_w8a8_frag_t256x384(
    const int8_t* __restrict__ a, const int8_t* __restrict__ w_frag, const float* __restrict__ a_scale,
    const float* __restrict__ w_scale, uint16_t* __restrict__ y, int64_t M, int64_t K, int64_t N) {
  using Epilogue = ScaleEpilogueT<gemm_frag::kWideBN>;
  __shared__ __attribute__((aligned(16))) int8_t lds[gemm_frag::lds_bytes<8, 2>(Epilogue::kScratch)];
  Epilogue epi{a_scale, w_scale};
  wide_kernel(a, w_frag, epi, y, M, K, N, lds);
}
extern "C" __global__ void __launch_bounds__(256, 1) mtrt_gemm_w8a8_frag_t256x384_linear(
    const int8_t* __restrict__ a, const int8_t* __restrict__ w_frag, const float* __restrict__ a_scale,
    const float* __restrict__ w_scale, uint16_t* __restrict__ y, int64_t M, int64_t K, int64_t N, uint32_t a_step,
    const uint16_t* __restrict__ bias) {
  using Epilogue = ScaleEpilogueT<gemm_frag::kWideBN, true>;
  __shared__ __attribute__((aligned(16))) int8_t lds[gemm_frag::lds_bytes<8, 2>(Epilogue::kScratch)];
  Epilogue epi{a_scale, w_scale, a_step, bias};
  wide_kernel(a, w_frag, epi, y, M, K, N, lds);
}
// Weight re-layout into fragment order, from [K,N] (nk = 0) or [N,K] (nk = 1).  One 16-byte chunk per
// thread.  (w, w_frag, K, N, nk) ; w_frag holds 32 * ceil(N/32) * 128 * ceil(K/128) bytes, zeros where w has none.
extern "C" __global__ void __launch_bounds__(256) mtrt_w8_prepack_frag(const int8_t* __restrict__ w, v4i* __restrict__ w_frag,
                                                                     int64_t K, int64_t N, int32_t nk) {
  const int64_t slices = (K + 127) / 128, ntiles = (N + 31) / 32;
  const int64_t total = ntiles * slices * 256;
  for (int64_t id = int64_t(blockIdx.x) * block_threads() + threadIdx.x; id < total; id += int64_t(gridDim.x) * block_threads()) {
    const int lane = int(id & 63), p = int((id >> 6) & 3);
    const int64_t slice = (id >> 8) % slices, tile = (id >> 8) / slices;
    const int64_t n = tile * 32 + (lane & 31), k0 = slice * 128 + 32 * p + 16 * (lane >> 5);
    union { v4i v; int8_t b[16]; } c;
#pragma unroll
    for (int i = 0; i < 16; ++i) c.b[i] = n < N && k0 + i < K ? (nk ? w[n * K + k0 + i] : w[(k0 + i) * N + n]) : int8_t(0);
    w_frag[id] = c.v;
  }
}

// Epilogue of the kernels that finish one output at a time: as ScaleEpilogueT.
struct RowsScaleEpilogue {
  const float* a_scale;
  const float* w_scale;
  uint32_t a_step = 1;
  const uint16_t* bias = nullptr;
  __device__ __forceinline__ uint32_t finish(int sum, int64_t row, int64_t col) const {
    const uint32_t y = f32_to_f16_bits((float(sum) * a_scale[row * a_step]) * w_scale[col]);
    return bias ? f32_to_f16_bits(f16_bits_to_f32(y) + f16_bits_to_f32(bias[col])) : y;
  }
};

// ---- small M (<= 32): one workgroup per 32 columns, four waves split K -----------------------------------
// A launch of the tile kernel above lasts one tile's whole K loop however few rows it has (M = 16 at K = 4096,
// N = 11008: 21.7 us) although all it has to do is read the weights once (45 MB).  Here every workgroup owns one
// tile of 32 columns (or two, see `tiles` below) over all of K, its four waves a quarter of K each: a wave keeps
// a ring of four stages (8 * G rows x 128 k of activations each) of its own in LDS, filled by direct-to-LDS loads
// three slices ahead as whole 128-byte row segments (a fragment read straight from memory would touch 32 cache
// lines), and takes the weights from fragment order straight into registers: no barrier until the four partial
// sums (int32, exact in any order) meet in LDS.  G: groups of 8 activation rows per stage (M <= 8 * G); PAST: the weights
// pass the caches by.
namespace small_m {

template <int G, int WAVES, int JT, bool PAST>
__device__ __forceinline__ void run(const int8_t* __restrict__ a, const v4i* __restrict__ wfrag, const RowsScaleEpilogue& epi,
                                    uint16_t* __restrict__ y, int64_t M, int64_t K, int64_t N, int8_t* lds) {
  constexpr int kStages = 4, kStageBytes = 8 * G * 128;
  constexpr int kLoads = G + 4 * JT;                 // memory instructions per slice and wave
  const int lane = threadIdx.x & 63;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int frow = lane & 31, fhalf = lane >> 5;
  const int64_t slices = K / 128;
  const int64_t kb0 = slices * wave / WAVES, kb1 = slices * (wave + 1) / WAVES;
  int64_t tile[JT];
  const v4i* bp[JT];
#pragma unroll
  for (int j = 0; j < JT; ++j) {
    tile[j] = blockIdx.x + int64_t(j) * gridDim.x;
    bp[j] = wfrag + (tile[j] * slices) * 256 + lane;
  }
  int8_t* ring = lds + wave * (kStages * kStageBytes);

  // direct-to-LDS load g (of G) of a slice: rows 8g .. 8g+7, lane l <-> (row l >> 3, LDS chunk l & 7)
  uint32_t aoff[G];
#pragma unroll
  for (int g = 0; g < G; ++g) {
    const int lrow = g * 8 + (lane >> 3);
    const int64_t row = lrow < M ? lrow : M - 1;     // rows past M repeat the last row; never stored
    aoff[g] = uint32_t(row * K + (((lane & 7) ^ ((lrow >> 1) & 7)) << 4));
  }
  struct Slice {
    v4i w[JT][4];
  };
  // everything slice kb needs from memory: G + 4 JT loads, always, so that the waits can count
  auto fetch = [&](int64_t kb, int64_t clamp, Slice& dst) {
    kb = kb < clamp ? kb : clamp;
    int8_t* st = ring + int(kb & (kStages - 1)) * kStageBytes;
#pragma unroll
    for (int g = 0; g < G; ++g)
      __builtin_amdgcn_global_load_lds((gemm_core::global_void_t*)(a + kb * 128 + aoff[g]),
                                       (gemm_core::lds_void_t*)(st + g * 1024), 16, 0, 0);
    // register loads as opaque instructions, the waits placed by hand in `landed` (the compiler's own
    // bookkeeping drains every load carried around a loop before its first use)
#pragma unroll
    for (int j = 0; j < JT; ++j)
#pragma unroll
      for (int p = 0; p < 4; ++p) {
        const v4i* wsrc = bp[j] + kb * 256 + p * 64;
        if constexpr (PAST) __asm__ volatile("global_load_dwordx4 %0, %1, off nt" : "=v"(dst.w[j][p]) : "v"(wsrc) : "memory");
        else __asm__ volatile("global_load_dwordx4 %0, %1, off" : "=v"(dst.w[j][p]) : "v"(wsrc) : "memory");
      }
  };
  // all loads but those of `in_flight` younger slices have landed
  auto landed = [&](auto in_flight, Slice& sl) {
#pragma unroll
    for (int j = 0; j < JT; ++j)
#pragma unroll
      for (int p = 0; p < 4; ++p) __asm__ volatile("s_waitcnt vmcnt(%1)" : "+v"(sl.w[j][p]) : "n"(decltype(in_flight)::value * kLoads) : "memory");
  };

  v16i acc[JT];
#pragma unroll
  for (int j = 0; j < JT; ++j)
#pragma unroll
    for (int r = 0; r < 16; ++r) acc[j][r] = 0;
  auto multiply = [&](int64_t kb, const Slice& sl) {
    const int8_t* st = ring + int(kb & (kStages - 1)) * kStageBytes;
#pragma unroll
    for (int p = 0; p < 4; ++p) {
      const int arow = frow < 8 * G ? frow : 8 * G - 1;   // rows past the ring: any valid data, never stored
      const v4i fa = *reinterpret_cast<const v4i*>(st + gemm_core::lds_off(arow, 2 * p + fhalf));
#pragma unroll
      for (int j = 0; j < JT; ++j) acc[j] = __builtin_amdgcn_mfma_i32_32x32x32_i8(fa, sl.w[j][p], acc[j], 0, 0, 0);
    }
  };

  // Main part: groups of four slices with four register sets, so that nothing is copied (a copy would have
  // to wait for the load) and the loop has no branch; three slices stay in flight.  The last slices, at most three, are on
  // their way when it ends.
  if (kb0 < kb1) {
    using gemm_core::IntC;
    const int64_t kmain = kb0 + ((kb1 - kb0) & ~int64_t(3)), clamp = kb1 - 1;   // past the end: the last slice again, into the stage that holds it
    Slice s0, s1, s2, s3;
    fetch(kb0, clamp, s0);
    fetch(kb0 + 1, clamp, s1);
    fetch(kb0 + 2, clamp, s2);
    for (int64_t kb = kb0; kb < kmain; kb += 4) {
      fetch(kb + 3, clamp, s3);
      landed(IntC<3>{}, s0);
      multiply(kb, s0);
      fetch(kb + 4, clamp, s0);
      landed(IntC<3>{}, s1);
      multiply(kb + 1, s1);
      fetch(kb + 5, clamp, s1);
      landed(IntC<3>{}, s2);
      multiply(kb + 2, s2);
      fetch(kb + 6, clamp, s2);
      landed(IntC<3>{}, s3);
      multiply(kb + 3, s3);
    }
    // (surplus loads still target these registers: they stay allocated until those land)
    landed(IntC<2>{}, s0);
    if (kmain < kb1) multiply(kmain, s0);
    landed(IntC<1>{}, s1);
    if (kmain + 1 < kb1) multiply(kmain + 1, s1);
    landed(IntC<0>{}, s2);
    if (kmain + 2 < kb1) multiply(kmain + 2, s2);
  }
  __builtin_amdgcn_s_waitcnt(0x0070);                  // surplus loads have landed before the ring is reused
  int (*partial)[16][64] = reinterpret_cast<int (*)[16][64]>(lds);
#pragma unroll
  for (int j = 0; j < JT; ++j) {
    __syncthreads();
#pragma unroll
    for (int r = 0; r < 16; ++r) partial[wave][r][lane] = acc[j][r];
    __syncthreads();
    for (int e = threadIdx.x; e < 16 * 64; e += 64 * WAVES) {
      const int r = e >> 6, l = e & 63;
      int v = partial[0][r][l];
#pragma unroll
      for (int w = 1; w < WAVES; ++w) v = v + partial[w][r][l];
      const int64_t row = (r >> 2) * 8 + (l >> 5) * 4 + (r & 3);
      const int64_t c = tile[j] * 32 + (l & 31);
      if (row < M && c < N) y[row * N + c] = uint16_t(epi.finish(v, row, c));
    }
  }
}

// The grid is one workgroup per column tile, or, while that would leave some compute units with two workgroups
// and the rest with one (tiles between one and two times the compute units), one workgroup per compute unit:
// workgroup g then also takes tile g + gridDim.x if there is one, and reads the activations once for both.
template <int G, bool PAST>
__device__ __forceinline__ void tiles(const int8_t* __restrict__ a, const v4i* __restrict__ wfrag, const RowsScaleEpilogue& epi,
                                      uint16_t* __restrict__ y, int64_t M, int64_t K, int64_t N, int8_t* lds) {
  const int64_t ntiles = (N + 31) / 32;
  if (int64_t(blockIdx.x) + gridDim.x < ntiles)
    run<G, 4, 2, PAST>(a, wfrag, epi, y, M, K, N, lds);
  else
    run<G, 4, 1, PAST>(a, wfrag, epi, y, M, K, N, lds);
}

}  // namespace small_m

// (a [M,K] i8, w_frag (fragment order), a_scale [M] f32, w_scale [N] f32, y [M,N] f16, M, K, N, a_step, bias, past) ; K % 128 == 0, a
// and w_frag 16-byte aligned, M * K < 2^32; past: the weights are read past the caches (w8_few_rows_past in clusters.cpp); grid = ceil(N / 32) or
// the number of compute units (see small_m::tiles), block = 256.
// M <= 16:
extern "C" __global__ void __launch_bounds__(256) mtrt_gemm_w8a8_small16(
    const int8_t* __restrict__ a, const v4i* __restrict__ w_frag, const float* __restrict__ a_scale,
    const float* __restrict__ w_scale, uint16_t* __restrict__ y, int64_t M, int64_t K, int64_t N, uint32_t a_step,
    const uint16_t* __restrict__ bias, int32_t past) {
  __shared__ __attribute__((aligned(16))) int8_t lds[4 * 4 * 2 * 1024];
  const RowsScaleEpilogue epi{a_scale, w_scale, a_step, bias};
  if (past) small_m::tiles<2, true>(a, w_frag, epi, y, M, K, N, lds);
  else small_m::tiles<2, false>(a, w_frag, epi, y, M, K, N, lds);
}
// ... M <= 32, the same arguments; grid = ceil(N / 32) or the number of compute units: which one stands beside the launch.  Against eight waves to
// a tile that each bring their own rows, as in gemm_core::rows32 (there 64 rows still run so), us, (M, K, N), weights of three sets in turn: (32, 1152, 9216)
// 7.0, 5.5; (17, 2048, 11008) 9.3, 7.6; (32, 4096, 11008) 13.2, 11.4; (32, 8192, 11008) 24.7, 22.3; (17, 4096, 4096) 6.2, 5.9; from memory the third 17.0, 13.6;
// the other way up to six slices by no more tiles than units, (17, 384, 4096) 2.8, 3.0; (32, 640, 4096) 3.1, 3.5, from memory 3.8, 3.4; 4.2, 4.4.
extern "C" __global__ void __launch_bounds__(256) mtrt_gemm_w8a8_frag_rows32(
    const int8_t* __restrict__ a, const v4i* __restrict__ w_frag, const float* __restrict__ a_scale,
    const float* __restrict__ w_scale, uint16_t* __restrict__ y, int64_t M, int64_t K, int64_t N, uint32_t a_step,
    const uint16_t* __restrict__ bias, int32_t past) {
  __shared__ __attribute__((aligned(16))) int8_t lds[4 * 4 * 4 * 1024];
  const RowsScaleEpilogue epi{a_scale, w_scale, a_step, bias};
  if (past) small_m::tiles<4, true>(a, w_frag, epi, y, M, K, N, lds);
  else small_m::tiles<4, false>(a, w_frag, epi, y, M, K, N, lds);
}
// Any K (no alignment needs): one output element per lane, plain loops.  Only K = 0 is left to it (every
// other shape runs on the matrix cores).
extern "C" __global__ void __launch_bounds__(256) mtrt_gemm_w8a8_nk_any(
    const int8_t* __restrict__ a, const int8_t* __restrict__ w, const float* __restrict__ a_scale,
    const float* __restrict__ w_scale, uint16_t* __restrict__ y, int64_t M, int64_t K, int64_t N) {
  const int64_t total = M * N;
  for (int64_t e = int64_t(blockIdx.x) * block_threads() + threadIdx.x; e < total; e += int64_t(gridDim.x) * block_threads()) {
    const int64_t m = e / N, n = e - m * N;
    int acc = 0;
    for (int64_t k = 0; k < K; ++k) acc += int(a[m * K + k]) * int(w[n * K + k]);
    y[e] = uint16_t(f32_to_f16_bits((float(acc) * a_scale[m]) * w_scale[n]));
  }
}

// Up to 32 rows on [N,K] weights read as whole rows (gemm_core::rows32): (a [M,K] i8, w_nk [N,K] i8, a_scale, w_scale, y,
// M <= 32, K, N) ; K % 128 == 0, a and w_nk 16-byte aligned; grid: any, block = 512.
extern "C" __global__ void __launch_bounds__(512) mtrt_gemm_w8a8_nk_rows32(
    const int8_t* __restrict__ a, const int8_t* __restrict__ w_nk, const float* __restrict__ a_scale,
    const float* __restrict__ w_scale, uint16_t* __restrict__ y, int64_t M, int64_t K, int64_t N) {
  __shared__ __attribute__((aligned(16))) int8_t lds[gemm_core::rows32::lds_bytes<8>()];
  RowsScaleEpilogue epi{a_scale, w_scale};
  gemm_core::rows32::run<I8Traits, 8>(a, w_nk, K, epi, y, M, N, lds);
}
// ... and up to 64 rows: two activation row tiles against each weight fragment
extern "C" __global__ void __launch_bounds__(512) mtrt_gemm_w8a8_nk_rows64(
    const int8_t* __restrict__ a, const int8_t* __restrict__ w_nk, const float* __restrict__ a_scale,
    const float* __restrict__ w_scale, uint16_t* __restrict__ y, int64_t M, int64_t K, int64_t N) {
  __shared__ __attribute__((aligned(16))) int8_t lds[gemm_core::rows32::lds_bytes<8, 2>()];
  RowsScaleEpilogue epi{a_scale, w_scale};
  gemm_core::rows32::run<I8Traits, 8, 2>(a, w_nk, K, epi, y, M, N, lds);
}
// ... and up to 128 rows: four row tiles, four waves (block = 256)
extern "C" __global__ void __launch_bounds__(256) mtrt_gemm_w8a8_nk_rows128(
    const int8_t* __restrict__ a, const int8_t* __restrict__ w_nk, const float* __restrict__ a_scale,
    const float* __restrict__ w_scale, uint16_t* __restrict__ y, int64_t M, int64_t K, int64_t N) {
  __shared__ __attribute__((aligned(16))) int8_t lds[gemm_core::rows32::lds_bytes<4, 4>()];
  RowsScaleEpilogue epi{a_scale, w_scale};
  gemm_core::rows32::run<I8Traits, 4, 4>(a, w_nk, K, epi, y, M, N, lds);
}

// Up to 64 rows on fragment-order weights: the same kernel with the weight fragments straight from
// memory into registers.  (a [M,K] i8, w_frag, a_scale, w_scale, y, M, K, N, a_step, bias) ; K % 128 == 0, a and w_frag
// 16-byte aligned; a_step and bias as for the tiles; grid: any, block = 512.
#define MTRT_W8_FRAG_ROWS_KERNEL(NAME, MT)                                                                                \
  extern "C" __global__ void __launch_bounds__(512) NAME(                                                                 \
      const int8_t* __restrict__ a, const int8_t* __restrict__ w_frag, const float* __restrict__ a_scale,                 \
      const float* __restrict__ w_scale, uint16_t* __restrict__ y, int64_t M, int64_t K, int64_t N, uint32_t a_step,      \
      const uint16_t* __restrict__ bias) {                                                                                \
    __shared__ __attribute__((aligned(16))) int8_t lds[gemm_core::rows32::lds_bytes<8, MT, true>()];                      \
    RowsScaleEpilogue epi{a_scale, w_scale, a_step, bias};                                                                \
    gemm_core::rows32::run<I8Traits, 8, MT, true>(a, w_frag, K, epi, y, M, N, lds);                                       \
  }
MTRT_W8_FRAG_ROWS_KERNEL(mtrt_gemm_w8a8_frag_rows64, 2)

// ---- a decode step's Linear in ONE launch: f16 activations, quantized where they are used ------------------
// With one scale for all activations nothing has to be known before a row can be quantized, and at a decode step the pass
// in front of the GEMM is all launch: M = 1, K = N = 4096 was 2.9 us of quantization and 6.3 us of GEMM.  Here every
// workgroup quantizes the whole of x (at most 16 Ki elements, from L2) into LDS while its first weights are on their
// way.  It owns 16 columns, half a tile of the fragment order (v_mfma_i32_16x16x64_i8 takes a k-step pair's halves in four
// groups of lanes), so that 4096 columns fill the chip's 256 compute units; its 8 waves share K in slices of 128, four
// slices in flight each (8 KiB a wave).  The sums are exact integers: the result is that of the two launches, bit for bit.
// Bound by the weights' way from memory and, towards 16 Ki elements, by the quantization.  Kernel times in us against the
// two launches (whose gap comes on top), (M, K, N): (1, 4096, 4096) 4.9 against 2.9 + 6.6, (1, 14336, 4096) 12.5 against
// 3.7 + 12.0, (4, 4096, 4096) 5.9 against 3.4 + 6.6, (16, 1024, 16384) 10.8 against 3.9 + 8.9.  The LDS and the registers
// for x end it at 16 Ki elements, where it is still the shorter by a sixth and more.
namespace decode {

constexpr int kWaves = 8, kMaxRows = 16, kMaxElements = 16384, kAhead = 4;
constexpr int kXGroups = kMaxElements / 8 / (64 * kWaves);        // groups of 8 elements of x per lane at most
constexpr int kRowPad = 16;                                       // LDS bytes between the rows of codes: their banks differ

__device__ __forceinline__ void run(const uint16_t* __restrict__ x, const float* __restrict__ x_scale, const int8_t* __restrict__ w_frag,
                                    const RowsScaleEpilogue& epi, uint16_t* __restrict__ y, int M, int K, int Kp, int64_t N, int8_t* codes,
                                    int (*partial)[64][4]) {
  using qdq_cluster::ExactDivisor;
  using qdq_cluster::FloatGroup;
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  const int col = lane & 15, kgroup = lane >> 4;
  const int slices = Kp / 128, kb0 = slices * wave / kWaves, kb1 = slices * (wave + 1) / kWaves;
  const int64_t n0 = int64_t(blockIdx.x) * 16;

  // x first: what is asked for first arrives first
  const int row_groups = Kp / 8, groups = M * row_groups;
  u32x4 xin[kXGroups];
  int xrow[kXGroups], xk[kXGroups];
#pragma unroll
  for (int i = 0; i < kXGroups; ++i) {
    const int g = int(threadIdx.x) + i * 64 * kWaves;
    xrow[i] = g / row_groups;
    xk[i] = (g - xrow[i] * row_groups) * 8;
    xin[i] = (u32x4){0u, 0u, 0u, 0u};
    if (g < groups && xk[i] + 8 <= K) xin[i] = *reinterpret_cast<const qdq_cluster::u32x4_unaligned*>(x + int64_t(xrow[i]) * K + xk[i]);
  }
  const ExactDivisor dv(x_scale[0]);

  // lane (col, kgroup) of k-step pair p: bytes 64 p + 16 kgroup ... + 15 of its column
  const int8_t* wp = w_frag + (n0 / 32) * slices * 4096 + (kgroup >> 1) * 1024 + ((kgroup & 1) * 32 + int(n0 & 16) + col) * 16;
  const int last = kb1 > kb0 ? kb1 - 1 : 0;                        // a slice past the wave's last one is that one again
  v4i w[kAhead][2];
  const auto fetch = [&](int kb, v4i (&into)[2]) {
    const int8_t* from = wp + int64_t(kb < kb1 ? kb : last) * 4096;
#pragma unroll
    for (int p = 0; p < 2; ++p) into[p] = __builtin_nontemporal_load(reinterpret_cast<const v4i*>(from + p * 2048));
  };
#pragma unroll
  for (int s = 0; s < kAhead; ++s) fetch(kb0 + s, w[s]);

  const int pitch = Kp + kRowPad;
#pragma unroll
  for (int i = 0; i < kXGroups; ++i) {
    if (int(threadIdx.x) + i * 64 * kWaves >= groups) continue;
    const int left = K - xk[i];                                    // the group that holds a row's end, and the padding behind it
    if (left > 0 && left < 8) {
      for (int e = 0; e < left; ++e) {
        const uint32_t bits = uint32_t(x[int64_t(xrow[i]) * K + xk[i] + e]) << (16 * (e & 1));
#pragma unroll
        for (int k = 0; k < 4; ++k) xin[i][k] |= (e >> 1) == k ? bits : 0u;
      }
    }
    float v[8];
    FloatGroup<F16>::unpack(xin[i], v);
    qdq_cluster::quantize_group<I8>(dv, v, 0);
    const u32x2 c = {qdq_cluster::pack4<I8>(&v[0], 0), qdq_cluster::pack4<I8>(&v[4], 0)};
    *reinterpret_cast<u32x2*>(codes + xrow[i] * pitch + xk[i]) = c;
  }
  __syncthreads();

  v4i acc = {0, 0, 0, 0};
  const int8_t* arow = codes + (col < M ? col : M - 1) * pitch + kgroup * 16;   // as the first operand the lane's row; rows past M repeat the last
  for (int kb = kb0; kb < kb1; kb += kAhead) {
#pragma unroll
    for (int s = 0; s < kAhead; ++s) {
      v4i held[2] = {w[s][0], w[s][1]};
      if (kb + kAhead < kb1) fetch(kb + kAhead + s, w[s]);
      if (kb + s < kb1) {
#pragma unroll
        for (int p = 0; p < 2; ++p) {
          const v4i a = *reinterpret_cast<const v4i*>(arow + (kb + s) * 128 + p * 64);
          acc = __builtin_amdgcn_mfma_i32_16x16x64_i8(a, held[p], acc, 0, 0, 0);
        }
      }
    }
  }
  // lane (col, h = lane / 16) holds rows 4 h + r of its column in register r
#pragma unroll
  for (int r = 0; r < 4; ++r) partial[wave][lane][r] = acc[r];
  __syncthreads();
  if (threadIdx.x < 256) {
    const int l = threadIdx.x & 63, r = threadIdx.x >> 6;
    int v = partial[0][l][r];
#pragma unroll
    for (int k = 1; k < kWaves; ++k) v = v + partial[k][l][r];
    const int row = (l >> 4) * 4 + r;
    const int64_t c = n0 + (l & 15);
    if (row < M && c < N) y[int64_t(row) * N + c] = uint16_t(epi.finish(v, row, c));
  }
}

}  // namespace decode

// (x [M,K] f16, x_scale: one f32, w_frag (K padded to Kp), w_scale, y [M,N] f16, M <= 16, K, Kp, N, bias f16 or null) ;
// Kp = K rounded up to 128, M * Kp <= 16384, w_frag 16-byte aligned, x aligned to its elements; grid = ceil(N / 16), block = 512.
extern "C" __global__ void __launch_bounds__(512) mtrt_linear_w8a8_decode(
    const uint16_t* __restrict__ x, const float* __restrict__ x_scale, const int8_t* __restrict__ w_frag, const float* __restrict__ w_scale,
    uint16_t* __restrict__ y, int64_t M, int64_t K, int64_t Kp, int64_t N, const uint16_t* __restrict__ bias) {
  __shared__ __attribute__((aligned(16))) int8_t codes[decode::kMaxElements + decode::kMaxRows * decode::kRowPad];
  __shared__ __attribute__((aligned(16))) int partial[decode::kWaves][64][4];
  decode::run(x, x_scale, w_frag, RowsScaleEpilogue{x_scale, w_scale, 0, bias}, y, int(M), int(K), int(Kp), N, codes, partial);
}

// Any K and any operand alignment on the matrix cores, for the shapes the kernels above do not take (K not a
// multiple of 128, operands off 16-byte alignment, operands of 4 GiB and more): the 128 x 128 tile loop of
// gemm_core::edge.  (a [M,K] i8, w_nk [N,K] i8, a_scale [M] f32, w_scale [N] f32, y [M,N] f16, M, K, N, a_step, bias)
// grid: any (tiles are dealt round-robin), block = 256.
struct EdgeScaleEpilogue {
  const float* a_scale;
  const float* w_scale;
  uint32_t a_step;
  const uint16_t* bias;
  float as;
  __device__ __forceinline__ void row(int64_t row, bool valid) { as = valid ? a_scale[row * a_step] : 0.0f; }
  __device__ __forceinline__ uint32_t finish(int acc, int64_t col, bool valid) const {
    const uint32_t y = f32_to_f16_bits((float(acc) * as) * (valid ? w_scale[col] : 0.0f));
    return bias && valid ? f32_to_f16_bits(f16_bits_to_f32(y) + f16_bits_to_f32(bias[col])) : y;
  }
};

extern "C" __global__ void __launch_bounds__(256) mtrt_gemm_w8a8_nk_edge(
    const int8_t* __restrict__ a, const int8_t* __restrict__ w, const float* __restrict__ a_scale,
    const float* __restrict__ w_scale, uint16_t* __restrict__ y, int64_t M, int64_t K, int64_t N, uint32_t a_step,
    const uint16_t* __restrict__ bias) {
  __shared__ __attribute__((aligned(16))) int8_t lds[gemm_core::edge::kLdsBytes];
  EdgeScaleEpilogue epi{a_scale, w_scale, a_step, bias, 0.0f};
  gemm_core::edge::run<I8Traits>(a, w, K, epi, y, M, N, lds);
}

// Weight re-layout [K,N] -> [N,K], bytes.  64 x 64 tiles through LDS; both the global
// read and the global write are contiguous.  (w_kn, w_nk, K, N) grid = ceil(K/64)*ceil(N/64).
extern "C" __global__ void __launch_bounds__(256) mtrt_w8_prepack_kn_to_nk(const int8_t* __restrict__ w_kn,
                                                                         int8_t* __restrict__ w_nk, int64_t K, int64_t N) {
  __shared__ int8_t tile[64][65];
  const int64_t tiles_n = (N + 63) / 64;
  const int64_t k0 = int64_t(blockIdx.x / tiles_n) * 64, n0 = int64_t(blockIdx.x % tiles_n) * 64;
  const int tx = threadIdx.x & 63, ty = threadIdx.x >> 6;
#pragma unroll
  for (int i = 0; i < 16; ++i) {
    const int64_t k = k0 + ty + 4 * i, n = n0 + tx;
    if (k < K && n < N) tile[ty + 4 * i][tx] = w_kn[k * N + n];
  }
  __syncthreads();
#pragma unroll
  for (int i = 0; i < 16; ++i) {
    const int64_t n = n0 + ty + 4 * i, k = k0 + tx;
    if (k < K && n < N) w_nk[n * K + k] = tile[tx][ty + 4 * i];
  }
}

}  // namespace gemm_w8a8_cluster
