// Dense Linear: y[m,n] = narrow(sum_k f32(x[m,k]) * f32(w[n,k]) (+ f32(bias[n]))), f32 accumulation, all
// operands of one float type.  This is the float matmul of the quantized Linear in its fake-quant form
//   tripy/nvtripy/frontend/module/linear.py:112-151   (out = x' @ W'^T + b on the dequantized operands)
// for the parameter combinations the integer / int4 matrix-core clusters cannot express (f8 codes, scales
// along the input features, int4 blocks along the output features) and for the unquantized module.  The
// reference's own generator emits an FMA loop nest for such a matmul
// (mlir-tensorrt/kernel/test/Kernel/TransformSchedules/fallback-schedule-matmul.mlir:24); this is the same
// class of kernel, tiled through LDS: 64 x 64 outputs per workgroup, 4 x 4 per lane, K in slices of 16.
// w is [N,K] (K contiguous), the module's own weight layout; any M, N, K; no alignment needs.  It only serves
// K = 0 now: every other shape runs on the matrix cores (mtrt_gemm_dense_edge_* for rows that are not whole slices).
// 16-bit operands whose rows are whole 128-byte slices (K % 64 == 0, 16-byte aligned) go to the matrix cores
// instead (mtrt_gemm_dense_mfma_*): both operands are K-contiguous per row, which is the form the shared tile
// loop of gemm_core.hpp takes (both panels through LDS, 256 x 256 tiles, v_mfma_f32_32x32x16_{f16,bf16}; a
// product of two 16-bit floats is exact in f32), with the bias added to the f32 sum before the one narrowing.
#include "gemm_frag.hpp"

using namespace mtrt_dev;

namespace dense_cluster {

constexpr int kDenseTile = 64, kDenseK = 16;

template <typename X>
__device__ __forceinline__ void dense_body(const typename X::storage* __restrict__ x, const typename X::storage* __restrict__ w,
                                           const typename X::storage* __restrict__ bias, typename X::storage* __restrict__ y,
                                           int64_t M, int64_t K, int64_t N) {
  __shared__ float xs[kDenseK][kDenseTile + 1];
  __shared__ float ws[kDenseK][kDenseTile + 1];
  const int64_t tiles_n = (N + kDenseTile - 1) / kDenseTile;
  const int64_t m0 = int64_t(blockIdx.x / tiles_n) * kDenseTile, n0 = int64_t(blockIdx.x % tiles_n) * kDenseTile;
  const int tx = threadIdx.x & 15, ty = threadIdx.x >> 4;       // lane's 4 x 4 block: rows 4*ty.., columns 4*tx..
  const int lk = threadIdx.x & 15, lr = threadIdx.x >> 4;       // loader: k index, row index (+16 per step)
  float acc[4][4] = {};
  for (int64_t k0 = 0; k0 < K; k0 += kDenseK) {
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      const int r = lr + 16 * i;
      const int64_t k = k0 + lk;
      xs[lk][r] = (m0 + r < M && k < K) ? Tile<X>::load1(x + (m0 + r) * K + k) : 0.0f;
      ws[lk][r] = (n0 + r < N && k < K) ? Tile<X>::load1(w + (n0 + r) * K + k) : 0.0f;
    }
    __syncthreads();
#pragma unroll
    for (int kk = 0; kk < kDenseK; ++kk) {
      float a[4], b[4];
#pragma unroll
      for (int i = 0; i < 4; ++i) { a[i] = xs[kk][4 * ty + i]; b[i] = ws[kk][4 * tx + i]; }
#pragma unroll
      for (int i = 0; i < 4; ++i)
#pragma unroll
        for (int j = 0; j < 4; ++j) acc[i][j] = __builtin_fmaf(a[i], b[j], acc[i][j]);
    }
    __syncthreads();
  }
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    const int64_t m = m0 + 4 * ty + i;
    if (m >= M) continue;
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      const int64_t n = n0 + 4 * tx + j;
      if (n >= N) continue;
      float v = acc[i][j];
      if (bias) v = v + Tile<X>::load1(bias + n);
      Tile<X>::store1(y + m * N + n, v);
    }
  }
}

// ---- matrix-core form for f16 / bf16 --------------------------------------------------------------------
using gemm_core::v4i;
typedef float v16f __attribute__((ext_vector_type(16)));
typedef _Float16 v8h __attribute__((ext_vector_type(8)));
typedef __bf16 v8b __attribute__((ext_vector_type(8)));

template <typename X> struct HalfTraits;
template <> struct HalfTraits<F16> {
  using Acc = v16f;
  using Scalar = float;
  static __device__ __forceinline__ Acc zero() {
    Acc z;
#pragma unroll
    for (int r = 0; r < 16; ++r) z[r] = 0.0f;
    return z;
  }
  static __device__ __forceinline__ Acc mfma(v4i a, v4i b, Acc c) {
    union { v4i i; v8h h; } ua, ub;
    ua.i = a; ub.i = b;
    return __builtin_amdgcn_mfma_f32_32x32x16_f16(ua.h, ub.h, c, 0, 0, 0);
  }
  // accumulators in ordinary vector registers (gemm_frag::run_wide)
  static __device__ __forceinline__ void mfma_vgpr(v4i a, v4i b, Acc& c) { __asm__ volatile("v_mfma_f32_32x32x16_f16 %0, %1, %2, %0" : "+v"(c) : "v"(a), "v"(b)); }
  static __device__ __forceinline__ void clear_vgpr(v4i a, v4i b, Acc& c) { __asm__ volatile("v_mfma_f32_32x32x16_f16 %0, %1, %2, 0" : "=v"(c) : "v"(a), "v"(b)); }
};
template <> struct HalfTraits<BF16> {
  using Acc = v16f;
  using Scalar = float;
  static __device__ __forceinline__ Acc zero() { return HalfTraits<F16>::zero(); }
  static __device__ __forceinline__ Acc mfma(v4i a, v4i b, Acc c) {
    union { v4i i; v8b h; } ua, ub;
    ua.i = a; ub.i = b;
    return __builtin_amdgcn_mfma_f32_32x32x16_bf16(ua.h, ub.h, c, 0, 0, 0);
  }
  static __device__ __forceinline__ void mfma_vgpr(v4i a, v4i b, Acc& c) { __asm__ volatile("v_mfma_f32_32x32x16_bf16 %0, %1, %2, %0" : "+v"(c) : "v"(a), "v"(b)); }
  static __device__ __forceinline__ void clear_vgpr(v4i a, v4i b, Acc& c) { __asm__ volatile("v_mfma_f32_32x32x16_bf16 %0, %1, %2, 0" : "=v"(c) : "v"(a), "v"(b)); }
};

// f32 operands: a 16-byte fragment holds four k values per lane, and v_mfma_f32_32x32x2_f32 takes one per lane (the two
// halves of the wave supplying its two k values), so a fragment pair is four chained instructions; which k values
// meet in one instruction does not matter as long as both operands agree.
struct F32Traits {
  using Acc = v16f;
  using Scalar = float;
  static __device__ __forceinline__ Acc zero() { return HalfTraits<F16>::zero(); }
  static __device__ __forceinline__ Acc mfma(v4i a, v4i b, Acc c) {
#pragma unroll
    for (int e = 0; e < 4; ++e) c = __builtin_amdgcn_mfma_f32_32x32x2f32(bits_to_f32(uint32_t(a[e])), bits_to_f32(uint32_t(b[e])), c, 0, 0, 0);
    return c;
  }
};
struct BiasF32Epilogue {
  const float* bias;
  __device__ __forceinline__ void finish4(float (&v)[4], int64_t col, int64_t N) const {
    if (!bias) return;
#pragma unroll
    for (int e = 0; e < 4; ++e)
      if (col + e < N) v[e] = v[e] + bias[col + e];
  }
};

template <typename X> __device__ __forceinline__ uint32_t narrow16(float v);
template <> __device__ __forceinline__ uint32_t narrow16<F16>(float v) { return f32_to_f16_bits(v); }
template <> __device__ __forceinline__ uint32_t narrow16<BF16>(float v) { return f32_to_bf16_bits(v); }
template <typename X> __device__ __forceinline__ uint32_t narrow16x2(float lo, float hi);
template <> __device__ __forceinline__ uint32_t narrow16x2<F16>(float lo, float hi) { return f32x2_to_f16x2_bits(lo, hi); }
template <> __device__ __forceinline__ uint32_t narrow16x2<BF16>(float lo, float hi) { return f32x2_to_bf16x2_bits(lo, hi); }

// y = narrow(acc + f32(bias[n])); without a bias zeros are added, which changes no sum (an accumulator that starts at +0
// is never -0).  BN: columns of the tile (scratch floats)
template <typename X, int BN = 256>
struct BiasEpilogue {
  const typename X::storage* bias;
  const float* sb;                                   // bias of this tile's columns as f32, in LDS
  f32x4 br[2][4];
  __device__ __forceinline__ void setup(int8_t* scratch, int64_t, int64_t, int64_t n0, int64_t N) {
    float* dst = reinterpret_cast<float*>(scratch);
    for (int c = threadIdx.x; c < BN; c += block_threads()) dst[c] = (bias && n0 + c < N) ? Tile<X>::load1(bias + n0 + c) : 0.0f;
    sb = dst;
  }
  __device__ __forceinline__ void row(int) {}
  template <int HC>
  __device__ __forceinline__ void columns(int first_col_in_tile) {
#pragma unroll
    for (int jj = 0; jj < HC; ++jj)
#pragma unroll
      for (int q = 0; q < 4; ++q) br[jj][q] = *reinterpret_cast<const f32x4*>(sb + first_col_in_tile + jj * 32 + q * 8);
  }
  __device__ __forceinline__ void convert4(const v16f& acc, int q, int jj, uint32_t (&words)[2]) const {
#pragma unroll
    for (int e = 0; e < 4; e += 2) words[e >> 1] = narrow16x2<X>(acc[4 * q + e] + br[jj][q][e], acc[4 * q + e + 1] + br[jj][q][e + 1]);
  }
};

template <typename X>
__device__ __forceinline__ void dense_mfma_body(const typename X::storage* __restrict__ x, const typename X::storage* __restrict__ w,
                                                const typename X::storage* __restrict__ bias, uint16_t* __restrict__ y, int64_t M,
                                                int64_t K, int64_t N, int64_t full_panels, int8_t* lds) {
  const int64_t tiles_m = (M + gemm_core::BM - 1) / gemm_core::BM;
  const int64_t full_blocks = gemm_core::even_blocks(full_panels * tiles_m);
  BiasEpilogue<X> epi{bias, nullptr, {}};
  const int8_t* a8 = reinterpret_cast<const int8_t*>(x);
  const int8_t* w8 = reinterpret_cast<const int8_t*>(w);
  int64_t tile_m, panel;
  if (int64_t(blockIdx.x) < full_blocks) {
    if (!gemm_core::tile_of_even(blockIdx.x, uint32_t(full_blocks), tiles_m, full_panels, tiles_m, tile_m, panel)) return;
    gemm_core::run<HalfTraits<X>, 4>(a8, w8, K * 2, epi, y, M, N, K * 2 / gemm_core::BKB, tile_m * 256, panel * 256, lds);
  } else {
    const int64_t n_full = full_panels * 256;
    if (!gemm_core::tile_of_even(blockIdx.x - uint32_t(full_blocks), gridDim.x - uint32_t(full_blocks), tiles_m, (N - n_full + 127) / 128,
                                 tiles_m, tile_m, panel))
      return;
    gemm_core::run<HalfTraits<X>, 2>(a8, w8, K * 2, epi, y, M, N, K * 2 / gemm_core::BKB, tile_m * 256, n_full + panel * 128, lds);
  }
}

// Epilogues of the any-shape tile loop (gemm_core::edge): the same sum + bias, one narrowing.
template <typename X>
struct EdgeBiasEpilogue {
  const typename X::storage* bias;
  __device__ __forceinline__ void row(int64_t, bool) {}
  __device__ __forceinline__ uint32_t finish(float acc, int64_t col, bool valid) const {
    if (bias && valid) acc = acc + Tile<X>::load1(bias + col);
    return narrow16<X>(acc);
  }
};
struct EdgeBiasF32Epilogue {
  const float* bias;
  __device__ __forceinline__ void row(int64_t, bool) {}
  __device__ __forceinline__ float finish(float acc, int64_t col, bool valid) const { return bias && valid ? acc + bias[col] : acc; }
};

// Epilogues of the up-to-32-rows kernel (gemm_core::rows32)
template <typename X>
struct RowsBiasEpilogue {
  const typename X::storage* bias;
  __device__ __forceinline__ uint32_t finish(float sum, int64_t, int64_t col) const {
    if (bias) sum = sum + Tile<X>::load1(bias + col);
    return narrow16<X>(sum);
  }
};
struct RowsBiasF32Epilogue {
  const float* bias;
  __device__ __forceinline__ float finish(float sum, int64_t, int64_t col) const { return bias ? sum + bias[col] : sum; }
};

}  // namespace dense_cluster

// (x [M,K], w [N,K], bias [N] or null, y [M,N], M, K, N, full_panels) ; K % 64 == 0, x and w 16-byte aligned and below
// 4 GiB each; tiles and grid as mtrt_gemm_w8a8_nk (256 x 256 for the first full_panels * 256 columns, 256 x 128 after),
// block = 256.
#define MTRT_DENSE_MFMA_KERNEL(XN, XT)                                                                             \
  extern "C" __global__ void __launch_bounds__(gemm_core::THREADS, 1) mtrt_gemm_dense_mfma_##XN(                   \
      const XT::storage* __restrict__ x, const XT::storage* __restrict__ w, const XT::storage* __restrict__ bias,  \
      uint16_t* __restrict__ y, int64_t M, int64_t K, int64_t N, int64_t full_panels) {                            \
    __shared__ __attribute__((aligned(16))) int8_t lds[gemm_core::LDS_BYTES];                                      \
    dense_cluster::dense_mfma_body<XT>(x, w, bias, y, M, K, N, full_panels, lds);                                  \
  }
MTRT_DENSE_MFMA_KERNEL(f16, F16)
MTRT_DENSE_MFMA_KERNEL(bf16, BF16)

// ---- few rows of f32 -----------------------------------------------------------------------------------
// A wave takes COLS columns against ROWS rows, a lane four elements of K at a time, all in f32 (multiply-adds on the vector units);
// KW = 4: the four waves of a workgroup take the same columns and every fourth 256 elements of K.  More rows than ROWS are groups,
// on workgroups of one XCD that follow each other, so that its L2 has the weights from the first.  Bound by reading the weights up to
// four rows (M = 1, K = 4096, N = 11008: 26.7 us, 6.8 TB/s), with more by the rows' way through L1, which COLS columns share.  The
// matrix cores' f32 form works for 32 rows whatever M is and one workgroup walks 32 columns: us on 32 x 32 tiles, and here:
// (M, K, N) = (1, 4096, 11008) 52.5, 26.7; (1, 5449, 1344) 32.3, 6.8; (3, 2816, 4672) 19.0, 11.5; (8, 4096, 4096) 26.1, 15.8;
// (5, 12288, 256) 62, 9.8; (16, 1031, 260) 9.1, 4.3; (32, 4097, 4096), four groups, 38.7, 40.5.
// Any K of at least 4, any alignment of whole elements.
namespace dense_cluster {
namespace dot {
typedef float f32x4 __attribute__((ext_vector_type(4)));
typedef f32x4 f32x4_words __attribute__((aligned(4)));

// PAST: weights larger than the caches are read past them (M = 1, K = 4096, N = 11008: 28.9 -> 26.7 us; 29 MB in turns of six 6.8 -> 7.7)
template <bool PAST>
__device__ __forceinline__ f32x4 load(const f32x4_words* p) {
  return PAST ? __builtin_nontemporal_load(p) : *p;
}

template <int ROWS, int COLS, int KW, int UNROLL, bool PAST>
__device__ __forceinline__ void run(const float* __restrict__ x, const float* __restrict__ w, const float* __restrict__ bias,
                                    float* __restrict__ y, int64_t M, int64_t K, int64_t N, float* lds) {
  asm volatile("" : "+s"(K));   // what two forms of a kernel have in common is not computed, and held, for both
  const int lane = int(threadIdx.x & 63), wave = __builtin_amdgcn_readfirstlane(int(threadIdx.x >> 6));
  const uint32_t groups = (uint32_t(M) + ROWS - 1) / ROWS, turn = blockIdx.x >> 3;
  const int64_t row0 = turn % groups * ROWS, first = (int64_t(turn / groups * 8 + (blockIdx.x & 7)) * (4 / KW) + (KW == 1 ? wave : 0)) * COLS;
  if (first >= N) return;
  const float *xr[ROWS], *wr[COLS];
#pragma unroll
  for (int r = 0; r < ROWS; ++r) xr[r] = x + (row0 + r < M ? row0 + r : M - 1) * K;
#pragma unroll
  for (int c = 0; c < COLS; ++c) wr[c] = w + (first + c < N ? first + c : N - 1) * K;
  float acc[ROWS][COLS];
#pragma unroll
  for (int r = 0; r < ROWS; ++r)
#pragma unroll
    for (int c = 0; c < COLS; ++c) acc[r][c] = 0.0f;
  const int64_t whole = K / 256;
  const int slot = KW == 1 ? 0 : wave;
  int64_t b = slot;
#pragma unroll 1
  for (; b + (UNROLL - 1) * KW < whole; b += UNROLL * KW) {
    f32x4 wv[UNROLL][COLS];
#pragma unroll
    for (int u = 0; u < UNROLL; ++u)
#pragma unroll
      for (int c = 0; c < COLS; ++c) wv[u][c] = load<PAST>(reinterpret_cast<const f32x4_words*>(wr[c] + (b + u * KW) * 256 + lane * 4));
#pragma unroll
    for (int u = 0; u < UNROLL; ++u) {
      f32x4 xv[ROWS];
#pragma unroll
      for (int r = 0; r < ROWS; ++r) xv[r] = *reinterpret_cast<const f32x4_words*>(xr[r] + (b + u * KW) * 256 + lane * 4);
#pragma unroll
      for (int r = 0; r < ROWS; ++r)
#pragma unroll
        for (int c = 0; c < COLS; ++c)
#pragma unroll
          for (int e = 0; e < 4; ++e) acc[r][c] = __builtin_fmaf(xv[r][e], wv[u][c][e], acc[r][c]);
    }
  }
  // the rest in steps of 256: the last one ends at K, its lanes' vectors moved back to lie within the row, what they then hold twice zero
#pragma unroll 1
  for (; b * 256 < K; b += KW) {
    const int64_t k = b * 256 + lane * 4, at = k + 4 <= K ? k : K - 4;
    const int skip = int(k - at < 4 ? k - at : 4);
    f32x4 wv[COLS], xv[ROWS];
#pragma unroll
    for (int c = 0; c < COLS; ++c) wv[c] = load<PAST>(reinterpret_cast<const f32x4_words*>(wr[c] + at));
#pragma unroll
    for (int r = 0; r < ROWS; ++r) xv[r] = *reinterpret_cast<const f32x4_words*>(xr[r] + at);
#pragma unroll
    for (int e = 0; e < 4; ++e) {
#pragma unroll
      for (int c = 0; c < COLS; ++c) wv[c][e] = e < skip ? 0.0f : wv[c][e];
#pragma unroll
      for (int r = 0; r < ROWS; ++r) xv[r][e] = e < skip ? 0.0f : xv[r][e];
    }
#pragma unroll
    for (int r = 0; r < ROWS; ++r)
#pragma unroll
      for (int c = 0; c < COLS; ++c)
#pragma unroll
        for (int e = 0; e < 4; ++e) acc[r][c] = __builtin_fmaf(xv[r][e], wv[c][e], acc[r][c]);
  }
  // ROWS * COLS sums over the wave: each exchange halves the values a lane holds, then the rest of the lanes' bits are summed
  constexpr int V = ROWS * COLS;
  float v[V];
#pragma unroll
  for (int r = 0; r < ROWS; ++r)
#pragma unroll
    for (int c = 0; c < COLS; ++c) v[r * COLS + c] = acc[r][c];
  int id = 0;
#pragma unroll
  for (int h = V / 2, bit = 1; bit < 64; bit *= 2, h /= 2) {
    if (h >= 1) {
      const bool up = lane & bit;
      id = 2 * id + (up ? 1 : 0);
#pragma unroll
      for (int i = 0; i < h; ++i) {
        const float keep = up ? v[i + h] : v[i], give = up ? v[i] : v[i + h];
        v[i] = keep + __shfl_xor(give, bit, 64);
      }
    } else {
      v[0] = v[0] + __shfl_xor(v[0], bit, 64);
    }
  }
  // lane < V holds the sum of row id / COLS, column id % COLS
  if (KW > 1) {
    if (lane < V) lds[wave * V + lane] = v[0];
    __syncthreads();
    if (wave == 0 && lane < V) v[0] = (lds[lane] + lds[V + lane]) + (lds[2 * V + lane] + lds[3 * V + lane]);
  }
  const int64_t row = row0 + id / COLS, col = first + id % COLS;
  if ((KW == 1 || wave == 0) && lane < V && row < M && col < N) y[row * N + col] = bias ? v[0] + bias[col] : v[0];
}

template <int ROWS, int COLS, int KW, int UNROLL>
__device__ __forceinline__ void run_any(const float* x, const float* w, const float* bias, float* y, int64_t M, int64_t K, int64_t N, bool past, float* lds) {
  if (past)
    run<ROWS, COLS, KW, UNROLL, true>(x, w, bias, y, M, K, N, lds);
  else
    run<ROWS, COLS, KW, UNROLL, false>(x, w, bias, y, M, K, N, lds);
}
}  // namespace dot
}  // namespace dense_cluster

// Up to <rows> rows: (x [M,K], w [N,K], bias [N] or null, y [M,N], M, K, N, form) ; form bit 0: waves share K, bit 1: weights past the
// caches; grid = 8 * ceil(ceil(N / columns of a workgroup) / 8), block = 256.
#define MTRT_DENSE_DOT_KERNEL(NAME, ROWS, COLS, UNROLL)                                                            \
  extern "C" __global__ void __launch_bounds__(256) mtrt_gemm_dense_##NAME##_f32(                                  \
      const float* __restrict__ x, const float* __restrict__ w, const float* __restrict__ bias, float* __restrict__ y, int64_t M, \
      int64_t K, int64_t N, int32_t form) {                                                                        \
    __shared__ float lds[4 * ROWS * COLS];                                                                         \
    if (form & 1)                                                                                                  \
      dense_cluster::dot::run_any<ROWS, COLS, 4, UNROLL>(x, w, bias, y, M, K, N, form & 2, lds);                   \
    else                                                                                                           \
      dense_cluster::dot::run_any<ROWS, COLS, 1, UNROLL>(x, w, bias, y, M, K, N, form & 2, lds);                   \
  }
MTRT_DENSE_DOT_KERNEL(rows1, 1, 2, 4)
MTRT_DENSE_DOT_KERNEL(rows2, 2, 4, 4)
MTRT_DENSE_DOT_KERNEL(rows4, 4, 4, 4)
// ... any number in groups of eight: grid * ceil(M / 8); four columns to a wave, and eight (form bit 0 set)
MTRT_DENSE_DOT_KERNEL(rows8, 8, 4, 2)
extern "C" __global__ void __launch_bounds__(256) mtrt_gemm_dense_rows8_wide_f32(
    const float* __restrict__ x, const float* __restrict__ w, const float* __restrict__ bias, float* __restrict__ y, int64_t M,
    int64_t K, int64_t N, int32_t form) {
  __shared__ float lds[4 * 8 * 8];
  dense_cluster::dot::run_any<8, 8, 4, 1>(x, w, bias, y, M, K, N, form & 2, lds);
}

// Up to 32 rows, weights read once as whole rows (gemm_core::rows32): (x [M,K], w [N,K], bias or null, y, M <= 32, K, N) ;
// rows in whole 128-byte slices, x and w 16-byte aligned; grid: any, block = 512.
// f32: tiles != 0; or groups of eight rows on the vector units (dot::run, `form` as there), block = 256.
extern "C" __global__ void __launch_bounds__(512) mtrt_gemm_dense_rows32_f32(
    const float* __restrict__ x, const float* __restrict__ w, const float* __restrict__ bias, float* __restrict__ y, int64_t M,
    int64_t K, int64_t N, int32_t tiles, int32_t form) {
  __shared__ __attribute__((aligned(16))) int8_t lds[gemm_core::rows32::lds_bytes<8>()];
  if (tiles) {
    dense_cluster::RowsBiasF32Epilogue epi{bias};
    gemm_core::rows32::run<dense_cluster::F32Traits, 8>(reinterpret_cast<const int8_t*>(x), reinterpret_cast<const int8_t*>(w), K * 4, epi, y, M, N, lds);
  } else if (form & 1) {
    dense_cluster::dot::run<8, 4, 4, 2, false>(x, w, bias, y, M, K, N, reinterpret_cast<float*>(lds));
  } else {
    dense_cluster::dot::run<8, 4, 1, 2, false>(x, w, bias, y, M, K, N, reinterpret_cast<float*>(lds));
  }
}
#define MTRT_DENSE_ROWS32_KERNEL(XN, XT)                                                                           \
  extern "C" __global__ void __launch_bounds__(512) mtrt_gemm_dense_rows32_##XN(                                   \
      const XT::storage* __restrict__ x, const XT::storage* __restrict__ w, const XT::storage* __restrict__ bias,  \
      uint16_t* __restrict__ y, int64_t M, int64_t K, int64_t N) {                                                 \
    __shared__ __attribute__((aligned(16))) int8_t lds[gemm_core::rows32::lds_bytes<8>()];                         \
    dense_cluster::RowsBiasEpilogue<XT> epi{bias};                                                                 \
    gemm_core::rows32::run<dense_cluster::HalfTraits<XT>, 8>(reinterpret_cast<const int8_t*>(x), reinterpret_cast<const int8_t*>(w), K * 2, \
                                                             epi, y, M, N, lds);                                   \
  }
MTRT_DENSE_ROWS32_KERNEL(f16, F16)
MTRT_DENSE_ROWS32_KERNEL(bf16, BF16)
// f32, more rows (x, w, bias, y, M, K, N): 32 x 32 tiles, K shared by eight waves (any M; rows64 and rows128 differ in name only), or, _tall,
// the rows against each weight fragment at once; grid: any, block = 512 (rows128_tall: 256).  The matrix cores set the time of a tile
// column with all its rows (0.18 us to a 128-byte slice of K for every 32 rows, and 1 to 3 us to a round of tiles): it is level with the tiles at
// best, where the columns alone fill the chip once or twice and K is short: us, so and in tiles, (100, 512, 8192) 18.1 and 18.1, (40, 256, 16384)
// 12.7 and 13.0, (64, 512, 32768) 36.7 and 31.7, (64, 4096, 4096) 44.9 and 25.6, (109, 3072, 448) 62.7 and 19.2, (128, 4096, 1024) 82.7 and 23.8.
#define MTRT_DENSE_ROWS_F32_KERNEL(NAME, WAVES, MT, MANY)                                                          \
  extern "C" __global__ void __launch_bounds__(64 * WAVES) mtrt_gemm_dense_##NAME##_f32(                           \
      const float* __restrict__ x, const float* __restrict__ w, const float* __restrict__ bias, float* __restrict__ y, int64_t M, \
      int64_t K, int64_t N) {                                                                                      \
    __shared__ __attribute__((aligned(16))) int8_t lds[gemm_core::rows32::lds_bytes<WAVES, MT>()];                 \
    dense_cluster::RowsBiasF32Epilogue epi{bias};                                                                  \
    gemm_core::rows32::run<dense_cluster::F32Traits, WAVES, MT, false, MANY>(                                      \
        reinterpret_cast<const int8_t*>(x), reinterpret_cast<const int8_t*>(w), K * 4, epi, y, M, N, lds);         \
  }
// ... and up to 64 rows: two activation row tiles against each weight fragment
MTRT_DENSE_ROWS_F32_KERNEL(rows64, 8, 1, true)
MTRT_DENSE_ROWS_F32_KERNEL(rows64_tall, 8, 2, false)
#define MTRT_DENSE_ROWS64_KERNEL(XN, XT)                                                                           \
  extern "C" __global__ void __launch_bounds__(512) mtrt_gemm_dense_rows64_##XN(                                   \
      const XT::storage* __restrict__ x, const XT::storage* __restrict__ w, const XT::storage* __restrict__ bias,  \
      uint16_t* __restrict__ y, int64_t M, int64_t K, int64_t N) {                                                 \
    __shared__ __attribute__((aligned(16))) int8_t lds[gemm_core::rows32::lds_bytes<8, 2>()];                      \
    dense_cluster::RowsBiasEpilogue<XT> epi{bias};                                                                 \
    gemm_core::rows32::run<dense_cluster::HalfTraits<XT>, 8, 2>(reinterpret_cast<const int8_t*>(x), reinterpret_cast<const int8_t*>(w),     \
                                                                K * 2, epi, y, M, N, lds);                         \
  }
MTRT_DENSE_ROWS64_KERNEL(f16, F16)
MTRT_DENSE_ROWS64_KERNEL(bf16, BF16)
// ... and up to 128 rows: four row tiles, four waves (block = 256)
MTRT_DENSE_ROWS_F32_KERNEL(rows128, 8, 1, true)
MTRT_DENSE_ROWS_F32_KERNEL(rows128_tall, 4, 4, false)
#define MTRT_DENSE_ROWS128_KERNEL(XN, XT)                                                                          \
  extern "C" __global__ void __launch_bounds__(256) mtrt_gemm_dense_rows128_##XN(                                  \
      const XT::storage* __restrict__ x, const XT::storage* __restrict__ w, const XT::storage* __restrict__ bias,  \
      uint16_t* __restrict__ y, int64_t M, int64_t K, int64_t N) {                                                 \
    __shared__ __attribute__((aligned(16))) int8_t lds[gemm_core::rows32::lds_bytes<4, 4>()];                      \
    dense_cluster::RowsBiasEpilogue<XT> epi{bias};                                                                 \
    gemm_core::rows32::run<dense_cluster::HalfTraits<XT>, 4, 4>(reinterpret_cast<const int8_t*>(x), reinterpret_cast<const int8_t*>(w),     \
                                                                K * 2, epi, y, M, N, lds);                         \
  }
MTRT_DENSE_ROWS128_KERNEL(f16, F16)
MTRT_DENSE_ROWS128_KERNEL(bf16, BF16)

// ... and where the tiles are more than the compute units: four waves, four workgroups to a unit; grid: any, block = 256.  Bound by the
// matrix cores (a 32 x 32 x 2 instruction every 64 cycles: 157 TFLOP/s nominal) and, where the tiles fill the chip, by what they read through
// the L2s, 256 bytes of K for 32 x 32 outputs: no more than 108 TFLOP/s at any size.  Larger tiles read less and leave units idle
// where they are few.  us, 32 x 32, 128 x 128 and 256 x 128:
//   (200, 1024, 1024) 10.3, 84, 139      (300, 3072, 2048) 50, 236, 379       (512, 4096, 4096) 176, 311, 500      (768, 1024, 11008) 195, 229, 281
//   (2048, 512, 8192) 208, 163, 170      (4096, 64, 4096) 78.6, 46.2, 61.3    (120, 64, 65536) 42.4, 25.5, 55.5    (1024, 4096, 4096) 358, 319, 496
//   (2048, 4096, 4096) 672, 544, 502     (4096, 4096, 4096) 1303, 1075, 1007  (2048, 4096, 11008) 1689, 1614, 1504
// (256 x 256 tiles, tried before: 254 registers and all accumulators a lane, (2048, 512, 8192) 205, (4096, 4096, 4096) 1001, (2048, 4096, 11008) 1508.)
// All of them sum K in four parts or more, then the parts: the error against 64 bits is half of one chain's (K = 4096: 4.5e-7 and 9.0e-7 of the result).
MTRT_DENSE_ROWS_F32_KERNEL(mfma, 4, 1, true)

// ... 32 x 32 tiles, K shared by eight waves of up to eight workgroups (gemm_core::rows32::SplitK): (x, w, bias, y, M, K, N, SplitK), grid: any, block = 512;
// _ragged: rows of at least 16 bytes that are no whole slices, any alignment.  Bound by the matrix cores of the units that have a workgroup, and where K is
// short by 3 us of meeting.  us, whole and in 2, 3, 4, 6 and 8 parts (the units hold 256): (66, 11072, 576), 54 tiles, 60.0; 34.6, 26.8, 22.6, 30.5, 26.9; (96,
// 12288, 300), 30 tiles, 64.9; 37.5, 27.6, 23.1, 19.0, 17.9; (109, 3072, 448), 56 tiles, 20.7; 15.1, 12.7, 12.1, 16.1, 15.9; (257, 12288, 512), 144, 69.3; 71.6,
// 52.5, 60.0; (231, 10496, 1318), 336, 108; 89, 81, 89; (200, 2048, 1024), 224, 16.3; 20.6; (70, 608, 942), 90, 7.7; 8.4.  (128 registers instead of 137, so
// that a unit has two workgroups: 36 bytes of scratch, 2 % slower where it has one and 3 % faster where two.)  The error against 64 bits is 0.3 to 0.7 of the
// whole walk's.
#define MTRT_DENSE_SPLIT_F32_KERNEL(NAME, RAGGED)                                                                  \
  extern "C" __global__ void __launch_bounds__(512) mtrt_gemm_dense_##NAME##_f32(                                  \
      const float* __restrict__ x, const float* __restrict__ w, const float* __restrict__ bias, float* __restrict__ y, int64_t M, \
      int64_t K, int64_t N, gemm_core::rows32::SplitK split) {                                                     \
    __shared__ __attribute__((aligned(16))) int8_t lds[gemm_core::rows32::lds_bytes<8>()];                         \
    dense_cluster::RowsBiasF32Epilogue epi{bias};                                                                  \
    gemm_core::rows32::run<dense_cluster::F32Traits, 8, 1, false, true, RAGGED, gemm_core::Values, true>(          \
        reinterpret_cast<const int8_t*>(x), reinterpret_cast<const int8_t*>(w), K * 4, epi, y, M, N, lds, nullptr, &split); \
  }
MTRT_DENSE_SPLIT_F32_KERNEL(split, false)
MTRT_DENSE_SPLIT_F32_KERNEL(split_ragged, true)

// ... 128 x 128 tiles: (x, w, bias, y, M, K, N) ; grid: any, block = 256.
extern "C" __global__ void __launch_bounds__(256, 2) mtrt_gemm_dense_t128x128_f32(
    const float* __restrict__ x, const float* __restrict__ w, const float* __restrict__ bias, float* __restrict__ y, int64_t M,
    int64_t K, int64_t N) {
  __shared__ __attribute__((aligned(16))) int8_t lds[gemm_core::edge::kLdsBytes];
  dense_cluster::EdgeBiasF32Epilogue epi{bias};
  gemm_core::edge::run<dense_cluster::F32Traits, 4>(reinterpret_cast<const int8_t*>(x), reinterpret_cast<const int8_t*>(w), K * 4, epi, y, M, N, lds);
}
// ... 256 x 128 tiles: (x, w, bias, y, M, K, N) ; x and w below 4 GiB each; grid = 8 * ceil(ceil(M/256) * ceil(N/128) / 8), block = 256.
extern "C" __global__ void __launch_bounds__(gemm_core::THREADS, 1) mtrt_gemm_dense_t256x128_f32(
    const float* __restrict__ x, const float* __restrict__ w, const float* __restrict__ bias, float* __restrict__ y, int64_t M,
    int64_t K, int64_t N) {
  __shared__ __attribute__((aligned(16))) int8_t lds[gemm_core::LDS_BYTES];
  const int64_t tiles_m = (M + 255) / 256;
  int64_t tile_m, panel;
  if (!gemm_core::tile_of_even(blockIdx.x, gridDim.x, tiles_m, (N + 127) / 128, tiles_m, tile_m, panel)) return;
  dense_cluster::BiasF32Epilogue epi{bias};
  gemm_core::run<dense_cluster::F32Traits, 2, 4>(reinterpret_cast<const int8_t*>(x), reinterpret_cast<const int8_t*>(w), K * 4, epi, y, M, N,
                                                 K * 4 / gemm_core::BKB, tile_m * 256, panel * 128, lds);
}

// ---- weights in fragment order (gemm_frag.hpp) ---------------------------------------------------------
// What a module's Linear runs on: its weights are re-laid once per parameter set.  Against the loops above, which bring both
// operands through LDS in 256-row tiles (f16, us): (M, K, N) = (999, 4096, 11008) 113 -> 83, (2048, 4096, 11008) 197 -> 147,
// (256, 4096, 4096) 58 -> 16, (398, 11520, 1856) 165 -> 30, (1024, 2048, 2048) 32 -> 12.5, (200, 12288, 512) 164 -> 12.7.
// mtrt_gemm_dense_frag_<type>_t<rows>x<columns> (x [M,K], w_frag, bias [N] or null, y [M,N], M, K, N, Split) ;
// K % 64 == 0, x and w_frag 16-byte aligned, x below 4 GiB; the rest as mtrt_gemm_w8a8_frag_t<rows>x<columns>.
// mtrt_gemm_dense_frag_<type>_f8_...: float8 codes in their place (mtrt_wf8_prepack_frag), their scales w_scale (f32 [N]) the last argument.  Half the bytes on the way to a
// unit (a slice of a 128 x 384 tile: 40 instead of 64 KiB) and from memory, for 16 (bf16) or 8 (f16) vector instructions to a fragment of eight
// weights, which a wave issues beside the IT MFMAs that use it: what bounds it is the weights' way, in tiles of few rows those instructions.  Time of the
// kernel with codes over that with values, bf16, weights from memory: (24, 4096, 11008) 0.76, (128, ..) 0.81, (512, ..) 0.87, (1024, ..) 0.96, (2048, ..) 1.04;
// f16 0.74, 0.75, 0.81, 0.94, 1.01; from the Infinity Cache (K, N) = (4096, 4096) bf16 1.05, 1.21, 1.31, 1.14, 1.12, and f16 0.95, 1.05, 1.04, 1.04,
// 1.03.  Whole calls, us, values and codes, twelve modules in turn, which come from memory either way, bf16 (24, 4096, 11008) 23.9, 19.3; (256, ..) 44.6, 40.6; (1024, ..) 88.9, 90.6;
// (2048, ..) 152.7, 156.1; f16 24.0, 18.9; 44.6, 39.7; 90.7, 92.4; 163.8, 163.2; of three modules in turn, whose codes the Infinity Cache holds and whose values it does not, bf16 (1024, ..) 91.5,
// 89.4; (2048, ..) 156.8, 153.0; (4096, ..) 313, 308; f16 93.0, 89.6; 166, 157; 332, 318.  (By sets of four waves that share K, as W4A16's 32- and 64-row tiles are: no faster, the wave's own instructions are the limit.)
#define MTRT_DENSE_FRAG_KERNEL(XN, XT, WT, WPARAM, WARGS, IT, JT, D, WG, TILE)                                            \
  extern "C" __global__ void __launch_bounds__(256, WG) mtrt_gemm_dense_frag_##XN##_##TILE(                               \
      const int8_t* __restrict__ x, const int8_t* __restrict__ w_frag, const XT::storage* __restrict__ bias,              \
      uint16_t* __restrict__ y, int64_t M, int64_t K, int64_t N, gemm_frag::Split sp MTRT_UNWRAP WPARAM) {    \
    __shared__ __attribute__((aligned(16))) int8_t lds[gemm_frag::lds_bytes<IT, D>(128 * JT)];                            \
    gemm_frag::Part part;                                                                                                 \
    if (!gemm_frag::part_of<32 * IT, 128 * JT>(blockIdx.x, gridDim.x, M, N, uint32_t(K) / 64, sp, part)) return; \
    dense_cluster::BiasEpilogue<XT, 128 * JT> epi{bias, nullptr, {}};                                                     \
    gemm_frag::run<dense_cluster::HalfTraits<XT>, IT, JT, D>(x, 2 * K, WT{MTRT_UNWRAP WARGS}, epi, y, M, N, part, lds);               \
  }
// ... 256 x 384 tiles: (x, w_frag, bias, y, M, K, N) ; grid = 8 * ceil(ceil(M/256) * ceil(N/384) / 8), block = 256.
// ... up to 32 and 64 rows, a wave for itself (gemm_core::rows32): the same arguments; grid: any, block = 512.
#define MTRT_DENSE_FRAG_KERNELS(XN, XT, WT, WPARAM, WARGS, WSCALE)                                                       \
  MTRT_DENSE_FRAG_KERNEL(XN, XT, WT, WPARAM, WARGS, 1, 1, 4, 2, t32x128)                         \
  MTRT_DENSE_FRAG_KERNEL(XN, XT, WT, WPARAM, WARGS, 2, 1, 4, 2, t64x128)                         \
  MTRT_DENSE_FRAG_KERNEL(XN, XT, WT, WPARAM, WARGS, 4, 1, 2, 2, t128x128)                        \
  MTRT_DENSE_FRAG_KERNEL(XN, XT, WT, WPARAM, WARGS, 4, 2, 2, 2, t128x256)                        \
  MTRT_DENSE_FRAG_KERNEL(XN, XT, WT, WPARAM, WARGS, 4, 3, 2, 1, t128x384)                        \
  MTRT_DENSE_FRAG_KERNEL(XN, XT, WT, WPARAM, WARGS, 8, 2, 2, 1, t256x256)                        \
  extern "C" __global__ void __launch_bounds__(256, 1) mtrt_gemm_dense_frag_##XN##_t256x384(                              \
      const int8_t* __restrict__ x, const int8_t* __restrict__ w_frag, const XT::storage* __restrict__ bias,              \
      uint16_t* __restrict__ y, int64_t M, int64_t K, int64_t N MTRT_UNWRAP WPARAM) {                                     \
    __shared__ __attribute__((aligned(16))) int8_t lds[gemm_frag::lds_bytes<8, 2>(gemm_frag::kWideBN)];                   \
    const int64_t tiles_m = (M + 255) / 256, panels = (N + gemm_frag::kWideBN - 1) / gemm_frag::kWideBN;                  \
    int64_t tile_m, panel;                                                                                                \
    if (!gemm_core::tile_of_even(blockIdx.x, gridDim.x, tiles_m, panels, tiles_m, tile_m, panel)) return;                 \
    dense_cluster::BiasEpilogue<XT, gemm_frag::kWideBN> epi{bias, nullptr, {}};                                           \
    gemm_frag::run_wide<dense_cluster::HalfTraits<XT>>(x, 2 * K, WT{MTRT_UNWRAP WARGS}, (N + 31) / 32, epi, y, M, N, K / 64, tile_m * 256, \
                                                       panel * gemm_frag::kWideBN, lds);                                  \
  }                                                                                                                       \
  extern "C" __global__ void __launch_bounds__(512) mtrt_gemm_dense_frag_##XN##_rows32(                                   \
      const int8_t* __restrict__ x, const int8_t* __restrict__ w_frag, const XT::storage* __restrict__ bias,              \
      uint16_t* __restrict__ y, int64_t M, int64_t K, int64_t N MTRT_UNWRAP WPARAM) {                                     \
    __shared__ __attribute__((aligned(16))) int8_t lds[gemm_core::rows32::lds_bytes<8, 1, true>()];                       \
    dense_cluster::RowsBiasEpilogue<XT> epi{bias};                                                                        \
    gemm_core::rows32::run<dense_cluster::HalfTraits<XT>, 8, 1, true, false, false, WT>(x, w_frag, 2 * K, epi, y, M, N, lds, WSCALE); \
  }                                                                                                                       \
  extern "C" __global__ void __launch_bounds__(512) mtrt_gemm_dense_frag_##XN##_rows64(                                   \
      const int8_t* __restrict__ x, const int8_t* __restrict__ w_frag, const XT::storage* __restrict__ bias,              \
      uint16_t* __restrict__ y, int64_t M, int64_t K, int64_t N MTRT_UNWRAP WPARAM) {                                     \
    __shared__ __attribute__((aligned(16))) int8_t lds[gemm_core::rows32::lds_bytes<8, 2, true>()];                       \
    dense_cluster::RowsBiasEpilogue<XT> epi{bias};                                                                        \
    gemm_core::rows32::run<dense_cluster::HalfTraits<XT>, 8, 2, true, false, false, WT>(x, w_frag, 2 * K, epi, y, M, N, lds, WSCALE); \
  }
#define MTRT_UNWRAP(...) __VA_ARGS__
MTRT_DENSE_FRAG_KERNELS(f16, F16, gemm_core::Values, (), (w_frag), nullptr)
MTRT_DENSE_FRAG_KERNELS(bf16, BF16, gemm_core::Values, (), (w_frag), nullptr)
MTRT_DENSE_FRAG_KERNELS(f16_f8, F16, gemm_core::F8Codes<F16>, (, const float* __restrict__ w_scale), (w_frag, w_scale), w_scale)
MTRT_DENSE_FRAG_KERNELS(bf16_f8, BF16, gemm_core::F8Codes<BF16>, (, const float* __restrict__ w_scale), (w_frag, w_scale), w_scale)

// ---- up to 16 rows on fragment-order weights in ONE launch -----------------------------------------------
// x goes into LDS whole, quantized and dequantized on its way where the module quantizes its input (the arithmetic of mtrt_act_fake_*,
// bit for bit), while the first weights are on theirs: at a decode step the pass in front of the GEMM is all launch, and the
// eight waves of gemm_core::rows32 each read all rows of their slices again, through the L1 that the weights come by.  A workgroup owns
// 16 columns, half a tile of the fragment order (v_mfma_f32_16x16x32 takes a k-step pair's halves in four groups of lanes); its
// eight waves share K in slices of 128 bytes, four slices in flight each.  Bound by the weights' way from memory and, with several
// thousand elements, by their quantization in every workgroup.  bf16, us, rows32 and here (M, K, N): (1, 4096, 4096) 8.1, 7.0; (1, 4096, 11008)
// 21.7, 16.2; (2, 14336, 512) 15.4, 10.2; (8, 2048, 16384) 15.8, 12.4; (16, 1024, 16384) 9.8, 8.4; (16, 512, 512) 3.5, 3.5; with float8
// inputs, two launches and here: (1, 3968, 896) 9.3, 4.7; (1, 4096, 4096) 11.1, 7.0; (1, 4096, 11008) 25.0, 16.3; (8, 2048, 16384) 19.0, 14.5.
// Weights above 48 MB are read past the caches ((1, 4096, 11008) 17.0 -> 16.2; 33 MB in turns of six 8.4 -> 9.8).
namespace dense_cluster {
namespace rows16 {
typedef float v4f __attribute__((ext_vector_type(4)));
constexpr int kWaves = 8, kMaxRows = 16;
constexpr int kRowPad = 16;                                        // LDS bytes between the rows: their banks differ

template <typename X> __device__ __forceinline__ v4f mfma(v4i a, v4i b, v4f c);
template <> __device__ __forceinline__ v4f mfma<F16>(v4i a, v4i b, v4f c) {
  union { v4i i; v8h h; } ua, ub;
  ua.i = a; ub.i = b;
  return __builtin_amdgcn_mfma_f32_16x16x32_f16(ua.h, ub.h, c, 0, 0, 0);
}
template <> __device__ __forceinline__ v4f mfma<BF16>(v4i a, v4i b, v4f c) {
  union { v4i i; v8b h; } ua, ub;
  ua.i = a; ub.i = b;
  return __builtin_amdgcn_mfma_f32_16x16x32_bf16(ua.h, ub.h, c, 0, 0, 0);
}

struct Plain {};

template <typename X, typename Q, class W, int kXGroups, bool PAST>
__device__ __forceinline__ void run(const uint16_t* __restrict__ x, const float* __restrict__ x_scale, const W& weights,
                                    const RowsBiasEpilogue<X>& epi, uint16_t* __restrict__ y, int M, int K, int Kp, int64_t N, int8_t* rows,
                                    float (*partial)[64][4]) {
  using qdq_cluster::ExactDivisor;
  using qdq_cluster::FloatGroup;
  using Raw = typename W::Raw;
  constexpr bool kQuantized = !std::is_same<Q, Plain>::value;
  constexpr int kAhead = W::kCodes ? 8 : 4;                        // slices: the same bytes on their way
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  const int col = lane & 15, kgroup = lane >> 4;
  const int slices = Kp / 64, kb0 = slices * wave / kWaves, kb1 = slices * (wave + 1) / kWaves;
  const int64_t n0 = int64_t(blockIdx.x) * 16;

  // x first: what is asked for first arrives first
  const int row_groups = Kp / 8, groups = M * row_groups, pitch = 2 * Kp + kRowPad;
  u32x4 xin[kXGroups];
#pragma unroll
  for (int i = 0; i < kXGroups; ++i) {
    const int g = int(threadIdx.x) + i * 64 * kWaves, row = g / row_groups, k = (g - row * row_groups) * 8;
    xin[i] = (u32x4){0u, 0u, 0u, 0u};
    if (g < groups && k + 8 <= K) xin[i] = *reinterpret_cast<const qdq_cluster::u32x4_unaligned*>(x + int64_t(row) * K + k);
  }
  const float scale = kQuantized ? x_scale[0] : 1.0f;

  // lane (col, kgroup) of k-step pair p: bytes 64 p + 16 kgroup ... + 15 of its column's slice (codes: half as many)
  const int8_t* wp = weights.frag + (n0 / 32) * slices * (4 * W::kStepBytes) + (kgroup >> 1) * W::kStepBytes + ((kgroup & 1) * 32 + int(n0 & 16) + col) * int(sizeof(Raw));
  typename W::Scale w_scale{};
  if constexpr (W::kCodes) w_scale = W::scale_of(weights.scale, n0 + col, N);
  const int last = kb1 > kb0 ? kb1 - 1 : 0;                        // a slice past the wave's last one is that one again
  Raw w[kAhead][2];
  const auto fetch = [&](int kb, Raw (&into)[2]) {
    const int8_t* from = wp + int64_t(kb < kb1 ? kb : last) * (4 * W::kStepBytes);
#pragma unroll
    for (int p = 0; p < 2; ++p) {
      const Raw* at = reinterpret_cast<const Raw*>(from + p * (2 * W::kStepBytes));
      into[p] = PAST ? __builtin_nontemporal_load(at) : *at;
    }
  };
#pragma unroll
  for (int s = 0; s < kAhead; ++s) fetch(kb0 + s, w[s]);

  const ExactDivisor dv(scale);
#pragma unroll
  for (int i = 0; i < kXGroups; ++i) {
    const int g = int(threadIdx.x) + i * 64 * kWaves, row = g / row_groups, xk = (g - row * row_groups) * 8;
    if (g >= groups) continue;
    const int left = K - xk;                                     // the group that holds a row's end, and the padding behind it
    if (left > 0 && left < 8) {
      for (int e = 0; e < left; ++e) {
        const uint32_t bits = uint32_t(x[int64_t(row) * K + xk + e]) << (16 * (e & 1));
#pragma unroll
        for (int k = 0; k < 4; ++k) xin[i][k] |= (e >> 1) == k ? bits : 0u;
      }
    }
    u32x4 t = xin[i];
    if constexpr (kQuantized) {
      float v[8];
      FloatGroup<X>::unpack(xin[i], v);
      qdq_cluster::quantize_group<Q>(dv, v, 0);
#pragma unroll
      for (int h = 0; h < 2; ++h) qdq_cluster::unpack4<Q>(qdq_cluster::pack4<Q>(&v[4 * h], 0), &v[4 * h]);
#pragma unroll
      for (int k = 0; k < 8; ++k) v[k] = v[k] * scale;
#pragma unroll
      for (int k = 0; k < 4; ++k) t[k] = qdq_cluster::narrow2<X>(v[2 * k], v[2 * k + 1]);
    }
    *reinterpret_cast<u32x4*>(rows + row * pitch + 2 * xk) = t;
  }
  __syncthreads();

  v4f acc = {0.0f, 0.0f, 0.0f, 0.0f};
  const int8_t* arow = rows + (col < M ? col : M - 1) * pitch + kgroup * 16;   // as the first operand the lane's row; rows past M repeat the last
  for (int kb = kb0; kb < kb1; kb += kAhead) {
#pragma unroll
    for (int s = 0; s < kAhead; ++s) {
      v4i held[2];
#pragma unroll
      for (int p = 0; p < 2; ++p) {
        if constexpr (W::kCodes) {
          W::dequantize(uint32_t(w[s][p][0]), w_scale, 0, held[p]);
          W::dequantize(uint32_t(w[s][p][1]), w_scale, 1, held[p]);
        } else {
          held[p] = w[s][p];
        }
      }
      if (kb + kAhead < kb1) fetch(kb + kAhead + s, w[s]);
      if (kb + s < kb1) {
#pragma unroll
        for (int p = 0; p < 2; ++p) {
          const v4i a = *reinterpret_cast<const v4i*>(arow + (kb + s) * 128 + p * 64);
          acc = mfma<X>(a, held[p], acc);
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
    float v = partial[0][l][r];
#pragma unroll
    for (int k = 1; k < kWaves; ++k) v = v + partial[k][l][r];
    const int row = (l >> 4) * 4 + r;
    const int64_t c = n0 + (l & 15);
    if (row < M && c < N) y[int64_t(row) * N + c] = uint16_t(epi.finish(v, row, c));
  }
}

template <typename X, typename Q, int kXGroups, class W>
__device__ __forceinline__ void run_any(const uint16_t* x, const float* x_scale, const W& weights, const uint16_t* bias, uint16_t* y, int64_t M, int64_t K,
                                        int64_t Kp, int64_t N, bool past, int8_t* rows, float (*partial)[64][4]) {
  const RowsBiasEpilogue<X> epi{bias};
  if (past)
    run<X, Q, W, kXGroups, true>(x, x_scale, weights, epi, y, int(M), int(K), int(Kp), N, rows, partial);
  else
    run<X, Q, W, kXGroups, false>(x, x_scale, weights, epi, y, int(M), int(K), int(Kp), N, rows, partial);
}
}  // namespace rows16
}  // namespace dense_cluster

// (x [M,K], x_scale: one f32 (null without codes), w_frag (K padded to Kp), bias [N] or null, y [M,N], M <= 16, K, Kp, N, past) ; Kp = K rounded
// up to 64, M * Kp <= 16384 (32768 for _long: twice the registers and LDS for x, one workgroup to a compute unit), w_frag 16-byte
// aligned, x aligned to its elements; past: weights read past the caches; grid = ceil(N / 16), block = 512.
// Of x that is not quantized or goes through float8 codes (a module of float8 weights), one more argument: w_scale, f32 [N] where w_frag holds float8
// codes, else null.  Half the bytes: bf16, us, values and codes, (1, 4096, 4096) 7.2, 5.9; (1, 4096, 11008) 16.4, 11.0; (8, 2048, 16384) in f16 17.5, 13.4.
#define MTRT_DENSE_ROWS16_BODY(GROUPS)                                                                                    \
  using namespace dense_cluster::rows16;                                                                                  \
  __shared__ __attribute__((aligned(16))) int8_t rows[GROUPS * 64 * kWaves * 16 + kMaxRows * kRowPad];                    \
  __shared__ __attribute__((aligned(16))) float partial[kWaves][64][4];
#define MTRT_DENSE_ROWS16_KERNEL(NAME, XT, QT, GROUPS)                                                                    \
  extern "C" __global__ void __launch_bounds__(512) mtrt_gemm_dense_frag_##NAME(                                          \
      const uint16_t* __restrict__ x, const float* __restrict__ x_scale, const int8_t* __restrict__ w_frag, const uint16_t* __restrict__ bias, \
      uint16_t* __restrict__ y, int64_t M, int64_t K, int64_t Kp, int64_t N, int32_t past) {                              \
    MTRT_DENSE_ROWS16_BODY(GROUPS)                                                                                        \
    run_any<XT, QT, GROUPS>(x, x_scale, gemm_core::Values{w_frag}, bias, y, M, K, Kp, N, past, rows, partial);            \
  }
#define MTRT_DENSE_ROWS16_CODES_KERNEL(NAME, XT, QT, GROUPS)                                                              \
  extern "C" __global__ void __launch_bounds__(512) mtrt_gemm_dense_frag_##NAME(                                          \
      const uint16_t* __restrict__ x, const float* __restrict__ x_scale, const int8_t* __restrict__ w_frag, const uint16_t* __restrict__ bias, \
      uint16_t* __restrict__ y, int64_t M, int64_t K, int64_t Kp, int64_t N, int32_t past, const float* __restrict__ w_scale) { \
    MTRT_DENSE_ROWS16_BODY(GROUPS)                                                                                        \
    if (w_scale)                                                                                                          \
      run_any<XT, QT, GROUPS>(x, x_scale, gemm_core::F8Codes<XT>{w_frag, w_scale}, bias, y, M, K, Kp, N, past, rows, partial); \
    else                                                                                                                  \
      run_any<XT, QT, GROUPS>(x, x_scale, gemm_core::Values{w_frag}, bias, y, M, K, Kp, N, past, rows, partial);          \
  }
#define MTRT_DENSE_ROWS16_KERNELS(XN, XT)                               \
  MTRT_DENSE_ROWS16_CODES_KERNEL(XN##_rows16, XT, Plain, 4)             \
  MTRT_DENSE_ROWS16_KERNEL(XN##_rows16_i8, XT, I8, 4)                   \
  MTRT_DENSE_ROWS16_CODES_KERNEL(XN##_rows16_f8, XT, F8, 4)             \
  MTRT_DENSE_ROWS16_KERNEL(XN##_rows16_i4, XT, I4, 4)                   \
  MTRT_DENSE_ROWS16_CODES_KERNEL(XN##_rows16_long, XT, Plain, 8)        \
  MTRT_DENSE_ROWS16_KERNEL(XN##_rows16_long_i8, XT, I8, 8)              \
  MTRT_DENSE_ROWS16_CODES_KERNEL(XN##_rows16_long_f8, XT, F8, 8)        \
  MTRT_DENSE_ROWS16_KERNEL(XN##_rows16_long_i4, XT, I4, 8)
MTRT_DENSE_ROWS16_KERNELS(f16, F16)
MTRT_DENSE_ROWS16_KERNELS(bf16, BF16)

// Re-layout of float8 codes [N,K] into the fragment order of 16-bit products, the eight codes of a lane and k-step per thread: (w, w_frag,
// K, N) ; w_frag holds 32 * ceil(N/32) * 64 * ceil(K/64) bytes, zeros where w has no element.
extern "C" __global__ void __launch_bounds__(256) mtrt_wf8_prepack_frag(const uint8_t* __restrict__ w, u32x2* __restrict__ w_frag,
                                                                      int64_t K, int64_t N) {
  const int64_t slices = (K + 63) / 64, ntiles = (N + 31) / 32;
  const int64_t total = ntiles * slices * 256;
  for (int64_t id = int64_t(blockIdx.x) * block_threads() + threadIdx.x; id < total; id += int64_t(gridDim.x) * block_threads()) {
    const int lane = int(id & 63), p = int((id >> 6) & 3);
    const int64_t slice = (id >> 8) % slices, tile = (id >> 8) / slices;
    const int64_t n = tile * 32 + (lane & 31), k0 = slice * 64 + 16 * p + 8 * (lane >> 5);
    u32x2 v = {0u, 0u};
#pragma unroll
    for (int e = 0; e < 8; ++e)
      if (n < N && k0 + e < K) v[e >> 2] |= uint32_t(w[n * K + k0 + e]) << (8 * (e & 3));
    w_frag[id] = v;
  }
}

// Re-layout of 16-bit weights [N,K] into fragment order, one 16-byte chunk per thread: (w, w_frag, K, N) ; w_frag holds
// 32 * ceil(N/32) * 128 * ceil(K/64) bytes, zeros where w has no element.
extern "C" __global__ void __launch_bounds__(256) mtrt_w16_prepack_frag(const uint16_t* __restrict__ w, u32x4* __restrict__ w_frag,
                                                                      int64_t K, int64_t N) {
  const int64_t slices = (K + 63) / 64, ntiles = (N + 31) / 32;
  const int64_t total = ntiles * slices * 256;
  for (int64_t id = int64_t(blockIdx.x) * block_threads() + threadIdx.x; id < total; id += int64_t(gridDim.x) * block_threads()) {
    const int lane = int(id & 63), p = int((id >> 6) & 3);
    const int64_t slice = (id >> 8) % slices, tile = (id >> 8) / slices;
    const int64_t n = tile * 32 + (lane & 31), k0 = slice * 64 + 16 * p + 8 * (lane >> 5);
    u32x4 v = {0u, 0u, 0u, 0u};
    if (n < N) {
      if (k0 + 8 <= K) {
        v = *reinterpret_cast<const gemm_core::u32x4_halves*>(w + n * K + k0);
      } else {
#pragma unroll
        for (int e = 0; e < 8; ++e)
          if (k0 + e < K) v[e >> 1] |= uint32_t(w[n * K + k0 + e]) << (16 * (e & 1));
      }
    }
    w_frag[id] = v;
  }
}

// Any K and any alignment on the matrix cores: (x [M,K], w [N,K], bias [N] or null, y [M,N], M, K, N, waves) ; grid: any.
// waves = 0, block = 256: 128 x 128 tiles dealt round-robin, each walked down all of K.  waves = 4 or 8, block = 64 waves, rows of at
// least 16 bytes: 32 x 32 tiles whose K the waves share (gemm_core::rows32).  The large tile is bound by the one workgroup's walk
// where there are fewer tiles than compute units, whatever the rows: us, large and small, f32 (1, 5449, 1344) 404 and 33,
// (9, 1192, 3456) 92 and 11, (300, 2049, 1000) 163 and 31, (900, 1023, 1030) 95 and 37, (2000, 901, 2000) 86 and 118; f16 (1, 5449, 1344)
// 87 and 15, (64, 2050, 2048) 38 and 9.7, (512, 2049, 2048) 45 and 31, (700, 1023, 8200) 49 and 92.
#define MTRT_DENSE_EDGE_KERNEL(XN, XT, YT, TRAITS, EDGE, ROWS)                                                     \
  extern "C" __global__ void __launch_bounds__(512) mtrt_gemm_dense_edge_##XN(                                     \
      const XT::storage* __restrict__ x, const XT::storage* __restrict__ w, const XT::storage* __restrict__ bias,  \
      YT* __restrict__ y, int64_t M, int64_t K, int64_t N, int32_t waves) {                                        \
    constexpr int kSmall = gemm_core::rows32::lds_bytes<8>(), kLarge = gemm_core::edge::kLdsBytes;                 \
    __shared__ __attribute__((aligned(16))) int8_t lds[kSmall > kLarge ? kSmall : kLarge];                         \
    const int8_t *x8 = reinterpret_cast<const int8_t*>(x), *w8 = reinterpret_cast<const int8_t*>(w);               \
    const int64_t row_bytes = K * int64_t(sizeof(XT::storage));                                                    \
    dense_cluster::ROWS rows_epi{bias};                                                                            \
    if (waves == 8) {                                                                                              \
      gemm_core::rows32::run<dense_cluster::TRAITS, 8, 1, false, true, true>(x8, w8, row_bytes, rows_epi, y, M, N, lds); \
    } else if (waves == 4) {                                                                                       \
      gemm_core::rows32::run<dense_cluster::TRAITS, 4, 1, false, true, true>(x8, w8, row_bytes, rows_epi, y, M, N, lds); \
    } else {                                                                                                       \
      dense_cluster::EDGE epi{bias};                                                                               \
      gemm_core::edge::run<dense_cluster::TRAITS>(x8, w8, row_bytes, epi, y, M, N, lds);                           \
    }                                                                                                              \
  }
MTRT_DENSE_EDGE_KERNEL(f32, F32, float, F32Traits, EdgeBiasF32Epilogue, RowsBiasF32Epilogue)
MTRT_DENSE_EDGE_KERNEL(f16, F16, uint16_t, HalfTraits<F16>, EdgeBiasEpilogue<F16>, RowsBiasEpilogue<F16>)
MTRT_DENSE_EDGE_KERNEL(bf16, BF16, uint16_t, HalfTraits<BF16>, EdgeBiasEpilogue<BF16>, RowsBiasEpilogue<BF16>)

// (x [M,K], w [N,K], bias [N] or null, y [M,N], M, K, N) ; grid = ceil(M/64) * ceil(N/64), block = 256
#define MTRT_DENSE_KERNEL(XN, XT)                                                                                  \
  extern "C" __global__ void __launch_bounds__(256) mtrt_gemm_dense_##XN(                                          \
      const XT::storage* x, const XT::storage* w, const XT::storage* bias, XT::storage* y, int64_t M, int64_t K,   \
      int64_t N) { dense_cluster::dense_body<XT>(x, w, bias, y, M, K, N); }
MTRT_DENSE_KERNEL(f32, F32)
MTRT_DENSE_KERNEL(f16, F16)
MTRT_DENSE_KERNEL(bf16, BF16)
