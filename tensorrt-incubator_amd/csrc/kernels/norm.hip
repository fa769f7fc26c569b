// Fused elementwise+reduce clusters over the last dimension: LayerNorm and softmax.
//
// LayerNorm (the decomposition the reference recognises,
//   mlir-tensorrt/tensorrt/lib/TensorRT/Transforms/RaiseNormalizations.pdll:277-308;
//   user API tripy/nvtripy/frontend/module/layernorm.py:30-70):
//     xf = f32(x); mu = sum(xf)/D; d = xf - mu; var = sum(d*d)/D;
//     y = narrow(((d * (1/sqrt(var + eps))) * f32(gamma)) + f32(beta))
// softmax (mlir-tensorrt/compiler/lib/Dialect/StablehloExt/Utils/StablehloMatchers.cpp:311-335;
//   tripy/nvtripy/frontend/ops/softmax.py:30-82):
//     xf = f32(x); m = max(xf); e = exp(xf - m); s = sum(e); y = narrow(e / s)   [computed as e * (1/s)]
//
// The reference's code generator emits at least three (LayerNorm) or four (softmax)
// kernels for these, each re-reading the tensor, with one thread walking a whole
// row (mlir-tensorrt/kernel/lib/Utils/TilingUtils.cpp:669-677).  Here each row is
// read from HBM exactly once: ONE WAVE OWNS ONE ROW, the row lives in that wave's
// registers (NV 128-bit vectors per lane, lane l holding vectors l, l+64, ...: every
// load instruction of the wave covers 1 KiB of contiguous HBM), and both row
// reductions are cross-lane exchanges with no LDS and no barrier.  Longer rows (up to
// 1024 * 16 vectors) are owned by a workgroup in the same way ("_g" kernels); rows that
// fit neither scheme (D not a multiple of the vector width, or longer still) use the
// workgroup-per-row "_any" kernels, which re-read the row from cache.
//
// All arithmetic is f32 with the operation order above; reductions are trees
// rather than the host's left-to-right sums, which the float tolerance covers.
#include "common.hpp"

using namespace mtrt_dev;

namespace norm_cluster {

constexpr int kNormThreads = 256;
constexpr int kRowsPerBlock = kNormThreads / kWave;

template <typename X> struct Vec;     // one 128-bit vector <-> floats
template <> struct Vec<F32> {
  static constexpr int kElems = 4;
  static constexpr uint32_t kMinusInf = 0xFF800000u;   // in every element of a word
  static __device__ __forceinline__ void unpack(u32x4 t, float* v) {
#pragma unroll
    for (int j = 0; j < 4; ++j) v[j] = bits_to_f32(t[j]);
  }
  static __device__ __forceinline__ u32x4 pack(const float* v) {
    u32x4 t;
#pragma unroll
    for (int j = 0; j < 4; ++j) t[j] = f32_to_bits(v[j]);
    return t;
  }
};
template <> struct Vec<BF16> {
  static constexpr int kElems = 8;
  static constexpr uint32_t kMinusInf = 0xFF80FF80u;
  static __device__ __forceinline__ void unpack(u32x4 t, float* v) {
#pragma unroll
    for (int j = 0; j < 4; ++j) { v[2 * j] = bits_to_f32(t[j] << 16); v[2 * j + 1] = bits_to_f32(t[j] & 0xFFFF0000u); }
  }
  static __device__ __forceinline__ u32x4 pack(const float* v) {
    u32x4 t;
#pragma unroll
    for (int j = 0; j < 4; ++j) t[j] = f32x2_to_bf16x2_bits(v[2 * j], v[2 * j + 1]);
    return t;
  }
};
template <> struct Vec<F16> {
  static constexpr int kElems = 8;
  static constexpr uint32_t kMinusInf = 0xFC00FC00u;
  static __device__ __forceinline__ void unpack(u32x4 t, float* v) {
#pragma unroll
    for (int j = 0; j < 4; ++j) { v[2 * j] = f16_bits_to_f32(t[j] & 0xFFFFu); v[2 * j + 1] = f16_bits_to_f32(t[j] >> 16); }
  }
  static __device__ __forceinline__ u32x4 pack(const float* v) {
    u32x4 t;
#pragma unroll
    for (int j = 0; j < 4; ++j) t[j] = f32x2_to_f16x2_bits(v[2 * j], v[2 * j + 1]);
    return t;
  }
};

// Where a softmax row that starts off a cache line is cut: an access of the wave covers whole lines but at the row's two ends.  `head` elements in
// front of the first 16-byte boundary move one per lane, with those behind the last whole vector; `shift` is that vector's place in its
// line, and so the number of lanes that the first access leaves out (as far as a row that fills its lanes allows).
// What bounds these rows is memory: an access that starts inside a line leaves a part of it to the next one, which is fetched and written as a part.
// us, vectors from the row's first element on, on 16-byte boundaries, and on lines, f16 [48000, 1500] 51.9, 51.4, 48.5; [8000, 9001] 58.7, 52.3, 49.5; bf16
// [1084, 43165] 54.4, 46.9, 44.7; whole vectors, f16 [24000, 3000] 49.9, 48.7.  (Staged through LDS, four rows' whole
// range at once, 48.3 for the first, but 52.9 with 1503 elements and 66 with 4500; LayerNorm bf16 [1500, 9011] 16.0 -> 14.0, but [700, 10243] 8.7 -> 9.4: behind
// a head its parameters' vectors lie off their boundaries.)
// A head puts the row's elements into other lanes, so its sum is taken in 64 bits: what the order of the terms changes there is about a 2^-28th of the f32
// result's last place, so that equal rows at different places in a line differ only where that much decides a rounding.  (48.5 -> 49.3 and 44.7 -> 47.0 for the first and the third; the longer part is the exchange.)
// A shift alone is undone by one exchange of the lanes' sums: the same bits.
// It costs more than it saves, and is taken all the same so that a row's bits do not follow the size of its tensor, in 16-bit rows of a wave that are read
// through the caches, where the line that two rows share is fetched once anyhow (us, uncut and cut, f16 [5998, 5001] 20.9, 22.2; [2999, 5001] 11.7, 12.2; bf16 [5997, 2501]
// 10.8, 11.1; f16 [19960, 1503] 19.4, 19.8; of a workgroup [1499, 20001] 22.3, 20.8), and in small tensors of four vectors a lane ([2661, 1503] 5.23, 5.34; [5322, 1503] 8.3, 7.3).
struct RowCut { int head, shift; };
template <bool CUT> struct RowSum { using type = float; using op = SumF32; };
template <> struct RowSum<true> { using type = double; using op = SumF64; };
// Of the places that a lane's vectors j = 0, 1, ... have, whether one is the row's, and the nearest that is: only the first can lie in front of a row that is CUT.
template <bool CUT> __device__ __forceinline__ bool within(int j, int place, int shift, int end) { return place < end && (!CUT || j > 0 || place >= shift); }
template <bool CUT> __device__ __forceinline__ int held(int j, int place, int shift, int end) { return !CUT || j > 0 ? min(place, end - 1) : max(shift, min(place, end - 1)); }
template <typename X, int VECTORS>
__device__ __forceinline__ RowCut cut_row(const typename X::storage* xr, const typename X::storage* yr, int64_t d) {
  const uint32_t at = uint32_t(reinterpret_cast<uintptr_t>(xr)), to = uint32_t(reinterpret_cast<uintptr_t>(yr));
  const bool both = ((at ^ to) & 15u) == 0;            // (else no cut puts both on boundaries)
  const int head = both ? int((0u - at) & 15u) / int(sizeof(typename X::storage)) : 0;
  return {head, both ? min(int((at + 15u) / 16u) & 7, VECTORS - (int(d) - head) / Vec<X>::kElems) : 0};
}

// Load the wave's row into registers: NV vectors per lane, those in places [shift, end) the row's (see RowCut).  Every lane always loads (the
// other places re-read the row's first or last vector and are replaced by `fill` afterwards), so the
// loads are issued back to back with no branches between them; with FULL (the row fills all
// 64 * NV vectors) the replacement disappears as well.
template <typename X, int NV, bool FULL, bool PAST, bool CUT>
__device__ __forceinline__ void load_row(const u32x4* __restrict__ row, int shift, int end, int lane, float fill,
                                         float (&v)[NV * Vec<X>::kElems]) {
  constexpr int E = Vec<X>::kElems;
  u32x4 t[NV];
#pragma unroll
  for (int j = 0; j < NV; ++j) {
    const int idx = lane + kWave * j;
    const u32x4* p = row + (FULL ? idx : held<CUT>(j, idx, shift, end));
    t[j] = PAST ? __builtin_nontemporal_load(p) : *p;
  }
#pragma unroll
  for (int j = 0; j < NV; ++j) {
    Vec<X>::unpack(t[j], &v[j * E]);
    if (!FULL) {
      const bool live = within<CUT>(j, lane + kWave * j, shift, end);
#pragma unroll
      for (int k = 0; k < E; ++k) v[j * E + k] = live ? v[j * E + k] : fill;
    }
  }
}

// LayerNorm reads past the caches always, softmax but in the kernels whose names end in t (softmax_reads_past in clusters.cpp).  (LayerNorm, us, past and
// through, three tensors in turn; each from memory; with a launch that makes x in front and one that reads y behind, all three: f32 [256, 4096] 4.8, 4.8; 5.8, 6.2;
// 11.9, 12.0; [512, 4096] 5.2, 5.2; 6.1, 6.5; 16.7, 17.5; bf16 [512, 4096] 4.4, 4.4; 5.0, 5.4; 11.7, 11.9; [1024, 4096] 4.5, 4.6; 5.6, 6.0; 15.0, 15.4; f16
// [2796, 1500] 5.7, 5.5; 6.5, 6.5; 21.3, 21.7; bf16 [250, 14165] 6.6, 6.4; 7.2, 7.5; 16.3, 16.6.)
// What is written goes past the caches whatever its size.  (Left to them, a large result is shorter by what the launches behind it then write back:
// alone softmax bf16 of 134 MB 44.1 -> 46.8 us where each result has memory of its own, 44.3 -> 46.7 from memory, with a copy of 268 MB behind each 133.2 ->
// 135.7, between the launches that make x and take y 128.7 -> 127.6; LayerNorm bf16 [8178, 4096] 22.6 -> 21.4, 23.0 -> 22.3, 113.6 -> 116.8, 62.0 -> 60.6; of 101 MB
// 37.0 -> 39.0, 37.6 -> 39.3, 128.0 -> 132.1, 95.3 -> 96.4.)

// Hides a vector's provenance from the optimiser (no instruction is emitted).
__device__ __forceinline__ void opaque(u32x4& t) { __asm__ volatile("" : "+v"(t)); }

// A row's reduction over its wave.  The exchanges of the vector unit shorten a wave's chain, which is what few rows wait for and most
// forms gain from; where the waves of aligned short rows fill the chip, LDS takes instructions off the vector unit.  us, LDS and vector unit:
// LayerNorm f16 [8, 4096] 4.3, 3.9, f32 [22, 1984] 3.9, 3.5, f32 [77101, 204] 26.3, 24.9; softmax f32 [179, 1405] 3.5, 3.1, bf16 [76538, 411] 27.8,
// 25.8; the other way LayerNorm bf16 [20000, 1024] 15.8, 16.2, [26061, 512] 11.6, 11.9, softmax bf16 [5120, 1024] 5.1, 5.7, f32 [2560, 816] 4.5, 5.1.
// Whole f32 rows of 2048 take 5.0 us where [1280, 2048] lies in the caches from the call before, and 4.7 by LDS; with every call's tensors new it is
// 5.8 and 5.9, [300, 2048] 3.5 and 3.7, so they stay on the vector unit.
template <bool LDS, typename Op>
__device__ __forceinline__ float row_reduce(float v, Op op) { return LDS ? wave_reduce_lds(v, op) : wave_reduce(v, op); }

// The row stays in registers in its STORAGE form (NV 128-bit vectors per lane) and is widened
// again in each of the three passes: for 16-bit types that halves the live registers compared
// with keeping f32 values (a widening is one shift or mask per element), and the higher
// occupancy it buys is worth more to this memory-bound kernel than the extra VALU work.
// RESIDENT: the form held to 64 registers.  In f32 the exchanges need one more, which lay in private memory: by LDS there (us, f32 [5500,
// 2048] 17.3, 16.5; [7000, 2048] 21.1, 20.3; [7000, 1100] 13.8, 13.1; [8192, 2048] 24.0, 23.5).
template <typename X, int NV, bool FULL, bool RESIDENT>
__device__ __forceinline__ void layernorm_row(const typename X::storage* __restrict__ x,
                                              const typename X::storage* __restrict__ gamma,
                                              const typename X::storage* __restrict__ beta,
                                              typename X::storage* __restrict__ y, int64_t row, int64_t d, float eps) {
  constexpr int E = Vec<X>::kElems;
  const int lane = threadIdx.x & (kWave - 1);
  const int nvec = int(d / E);
  const u32x4* xr = reinterpret_cast<const u32x4*>(x + row * d);
  u32x4 t[NV];
#pragma unroll
  for (int j = 0; j < NV; ++j) {
    const int idx = lane + kWave * j;
    t[j] = __builtin_nontemporal_load(xr + (FULL ? idx : min(idx, nvec - 1)));
  }

  constexpr bool kLds = NV == 2 || NV == 4 || (NV == 1 && E == 8) || (RESIDENT && E == 4);
  const float fd = float(d);
  float sum = 0.0f;
#pragma unroll
  for (int j = 0; j < NV; ++j) {
    const bool live = FULL || lane + kWave * j < nvec;
    float v[E];
    Vec<X>::unpack(t[j], v);
#pragma unroll
    for (int k = 0; k < E; ++k) sum = sum + (live ? v[k] : 0.0f);
  }
  const float mu = row_reduce<kLds>(sum, SumF32()) / fd;
  float sq = 0.0f;
#pragma unroll
  for (int j = 0; j < NV; ++j) {
    const bool live = FULL || lane + kWave * j < nvec;
    float v[E];
    opaque(t[j]);                                    // widen again instead of keeping pass 1's values live
    Vec<X>::unpack(t[j], v);
#pragma unroll
    for (int k = 0; k < E; ++k) {
      const float dv = v[k] - mu;
      sq = sq + (live ? dv * dv : 0.0f);
    }
  }
  const float var = row_reduce<kLds>(sq, SumF32()) / fd;
  const float rstd = 1.0f / sqrtf(var + eps);

  const u32x4* gv = reinterpret_cast<const u32x4*>(gamma);
  const u32x4* bv = reinterpret_cast<const u32x4*>(beta);
  u32x4* yr = reinterpret_cast<u32x4*>(y + row * d);
#pragma unroll
  for (int j = 0; j < NV; ++j) {
    const int idx = lane + kWave * j;
    const int idc = FULL ? idx : min(idx, nvec - 1);
    float v[E], g[E], b[E], o[E];
    opaque(t[j]);
    Vec<X>::unpack(t[j], v);
    Vec<X>::unpack(gv[idc], g);
    Vec<X>::unpack(bv[idc], b);
#pragma unroll
    for (int k = 0; k < E; ++k) o[k] = (((v[k] - mu) * rstd) * g[k]) + b[k];
    if (FULL || idx < nvec) __builtin_nontemporal_store(Vec<X>::pack(o), yr + idx);
  }
}

template <typename X, int NV, bool RESIDENT = false>
__device__ __forceinline__ void layernorm_rows(const typename X::storage* __restrict__ x,
                                               const typename X::storage* __restrict__ gamma,
                                               const typename X::storage* __restrict__ beta,
                                               typename X::storage* __restrict__ y, int64_t rows, int64_t d, float eps) {
  // the wave index as a scalar: the row pointers are then wave-uniform and the accesses need one lane offset, not an address pair each
  const int64_t row = int64_t(blockIdx.x) * kRowsPerBlock + __builtin_amdgcn_readfirstlane(int(threadIdx.x / kWave));
  if (row >= rows) return;                           // whole wave leaves together
  if (d == int64_t(Vec<X>::kElems) * kWave * NV)
    layernorm_row<X, NV, true, RESIDENT>(x, gamma, beta, y, row, d, eps);
  else
    layernorm_row<X, NV, false, RESIDENT>(x, gamma, beta, y, row, d, eps);
}

template <typename X, int NV, bool FULL, bool PAST, bool CUT>
__device__ __forceinline__ void softmax_row(const typename X::storage* __restrict__ x, typename X::storage* __restrict__ y,
                                            int64_t row, int64_t d) {
  constexpr int E = Vec<X>::kElems;
  const int lane = threadIdx.x & (kWave - 1);
  const int nvec = int(d / E);
  const u32x4* xr = reinterpret_cast<const u32x4*>(x + row * d);
  const int shift = !CUT ? 0 : cut_row<X, kWave * NV>(x + row * d, y + row * d, d).shift, end = nvec + shift;
  float v[NV * E];
  load_row<X, NV, FULL, PAST, CUT>(xr - shift, shift, end, lane, -INFINITY, v);

  constexpr bool kLds = NV == 2 || NV == 4;
  float mx = -INFINITY;
#pragma unroll
  for (int i = 0; i < NV * E; ++i) mx = fmaxf(mx, v[i]);
  mx = row_reduce<kLds>(mx, MaxF32());
  float s = 0.0f;
#pragma unroll
  for (int i = 0; i < NV * E; ++i) {
    v[i] = __expf(v[i] - mx);                        // exp(-inf) = 0 for the fill lanes
    s = s + v[i];
  }
  if (CUT) s = __shfl(s, (lane + shift) & (kWave - 1));   // each lane's sum to the lane that has it where the row starts on a line
  s = row_reduce<kLds>(s, SumF32());
  // e / s as e * (1/s): one correctly rounded reciprocal per row instead of a divide per element; at most one
  // f32 ulp from the quotient.  Together with the hardware exponential (2^(d * log2 e), a few f32 ulps off for
  // |d| ~ 10) that is far below what the order of the row sum already changes: with an exponential good to one
  // ulp and a remainder-corrected quotient the share of f16 outputs that differ from the host's by one ulp
  // stayed at 0.05 % (4096 x 4096, sigma 2) and the launch took 1 us longer, so the short forms are kept.
  const float inv = 1.0f / s;
  u32x4* yr = reinterpret_cast<u32x4*>(y + row * d) - shift;
#pragma unroll
  for (int j = 0; j < NV; ++j) {
    const int idx = lane + kWave * j;
    float o[E];
#pragma unroll
    for (int k = 0; k < E; ++k) o[k] = v[j * E + k] * inv;
    if (FULL || within<CUT>(j, idx, shift, end)) __builtin_nontemporal_store(Vec<X>::pack(o), yr + idx);
  }
}

template <typename X, int NV, bool PAST, bool CUT>
__device__ __forceinline__ void softmax_rows(const typename X::storage* __restrict__ x, typename X::storage* __restrict__ y,
                                             int64_t rows, int64_t d) {
  // the wave index as a scalar: the row pointers are then wave-uniform and the accesses need one lane offset, not an address pair each
  const int64_t row = int64_t(blockIdx.x) * kRowsPerBlock + __builtin_amdgcn_readfirstlane(int(threadIdx.x / kWave));
  if (row >= rows) return;
  if (PAST && d == int64_t(Vec<X>::kElems) * kWave * NV)   // (whole cache lines)
    softmax_row<X, NV, true, true, false>(x, y, row, d);
  else
    softmax_row<X, NV, false, PAST, CUT>(x, y, row, d);
}

// ---- rows longer than one wave's registers, and rows of any length or alignment: a GROUP of lanes owns one row ----
// THREADS lanes hold the row, NV vectors each (lane l the vectors l, l + THREADS, ...), in storage form; the row
// reductions are a cross-lane exchange per wave and, when the group is a whole workgroup (256 or 1024 lanes), a
// meeting of the waves' values in LDS.  The row is still read from HBM exactly once.  Workgroup-sized groups
// cover 64 * 16 < D / E <= 1024 * 16 vectors (hidden sizes above 8192, vocabulary-sized softmax rows).
// RAGGED: D need not be a multiple of the vector width E and nothing need be 16-byte aligned: the D / E whole
// vectors of a row are moved by 128-bit accesses at element alignment (the hardware splits those that straddle
// a line), the D % E elements behind them one each by the group's first lanes.  With THREADS = 64 that is the
// one-wave-per-row scheme for rows such as 197, 1500 or 50257 elements.
template <bool RAGGED> struct RowVector { typedef u32x4 type; };
template <> struct RowVector<true> { typedef u32x4 type __attribute__((aligned(2))); };

template <int THREADS, typename T, typename Op>
__device__ __forceinline__ T group_reduce(T v, Op op, void* shared) {
  T* lds = static_cast<T*>(shared);
  if constexpr (THREADS < kWave) return lanes_reduce<THREADS>(v, op);   // several rows per wave: exchanges stay inside the row's lanes
  v = wave_reduce(v, op);
  if (THREADS == kWave) return v;
  __syncthreads();                                   // lds may still be read from the previous reduction
  if ((threadIdx.x & (kWave - 1)) == 0) lds[threadIdx.x / kWave] = v;
  __syncthreads();
  T r = lds[0];
#pragma unroll
  for (int w = 1; w < THREADS / kWave; ++w) r = op(r, lds[w]);
  return r;                                          // the same value, combined in the same order, in every lane
}

// Whether vector j of any lane of this wave lies in the row (the same for the whole wave): what lies past it for all is not asked for, nor
// worked on.  A row takes the kernel with the next power of two of vectors, so that may be near half of them.  ALL: every vector is worked on;
// which is the faster one stands beside row_form in clusters.cpp.  (Without either and the fill below, f32 softmax rows of 16388 to
// 32768 elements off whole vectors took twice the vectors too, for want of registers: [2000, 25001] 102 us, [800, 18001] 41.5.)
template <int THREADS, bool ALL>
__device__ __forceinline__ bool wave_has(int j, int nvec) {
  return ALL || (THREADS > kWave ? __builtin_amdgcn_readfirstlane(int(threadIdx.x & ~63u)) : 0) + THREADS * j < nvec;
}

template <typename X, int NV, int THREADS, bool FULL, bool ALL, bool RAGGED>
__device__ __forceinline__ void layernorm_group_row(const typename X::storage* __restrict__ x,
                                                    const typename X::storage* __restrict__ gamma,
                                                    const typename X::storage* __restrict__ beta,
                                                    typename X::storage* __restrict__ y, int64_t row, int64_t d, float eps,
                                                    double* lds) {
  constexpr int E = Vec<X>::kElems;
  using V = typename RowVector<RAGGED>::type;
  const int lane = int(threadIdx.x) & (THREADS - 1);
  const int nvec = int(d / E), tail = RAGGED ? int(d - int64_t(nvec) * E) : 0;
  const V* xr = reinterpret_cast<const V*>(x + row * d);
  const bool extra = RAGGED && lane < tail;          // this lane also owns element nvec * E + lane
  const int ec = nvec * E + lane;
  // Asked for with the vectors, by every lane: in a branch, or behind them, it is a second trip to memory (us, behind and with them, f16 [24000, 1501] 30.7, 30.3; [64,
  // 3001] 5.04, 4.92; bf16 [3000, 1001] 4.94, 4.85; f32 [300, 9001] 7.37, 7.21; [24000, 1501] 57.6, 57.9).
  typename X::storage xb = 0;
  if constexpr (RAGGED) xb = (x + row * d)[min(ec, int(d) - 1)];
  u32x4 t[NV];
#pragma unroll
  for (int j = 0; j < NV; ++j) {
    if (!wave_has<THREADS, ALL>(j, nvec)) break;
    const int idx = lane + THREADS * j;
    if (RAGGED && ALL && nvec == 0) t[j] = (u32x4){0u, 0u, 0u, 0u};   // a row shorter than one vector: only the scalar elements below
    else t[j] = __builtin_nontemporal_load(xr + (FULL ? idx : min(idx, nvec - 1)));
  }
  const float xe = extra ? Tile<X>::load1(&xb) : 0.0f;
  const float fd = float(d);
  float sum = xe;
#pragma unroll
  for (int j = 0; j < NV; ++j) {
    if (!wave_has<THREADS, ALL>(j, nvec)) break;
    const bool live = FULL || lane + THREADS * j < nvec;
    float v[E];
    Vec<X>::unpack(t[j], v);
#pragma unroll
    for (int k = 0; k < E; ++k) sum = sum + (live ? v[k] : 0.0f);
  }
  const float mu = group_reduce<THREADS>(sum, SumF32(), lds) / fd;
  float sq = extra ? (xe - mu) * (xe - mu) : 0.0f;
#pragma unroll
  for (int j = 0; j < NV; ++j) {
    if (!wave_has<THREADS, ALL>(j, nvec)) break;
    const bool live = FULL || lane + THREADS * j < nvec;
    float v[E];
    opaque(t[j]);                                    // widen again instead of keeping pass 1's values live
    Vec<X>::unpack(t[j], v);
#pragma unroll
    for (int k = 0; k < E; ++k) {
      const float dv = v[k] - mu;
      sq = sq + (live ? dv * dv : 0.0f);
    }
  }
  const float var = group_reduce<THREADS>(sq, SumF32(), lds) / fd;
  const float rstd = 1.0f / sqrtf(var + eps);
  const V* gv = reinterpret_cast<const V*>(gamma);
  const V* bv = reinterpret_cast<const V*>(beta);
  V* yr = reinterpret_cast<V*>(y + row * d);
#pragma unroll
  for (int j = 0; j < NV; ++j) {
    if (!wave_has<THREADS, ALL>(j, nvec)) break;
    const int idx = lane + THREADS * j;
    const int idc = FULL ? idx : min(idx, nvec - 1);
    if (RAGGED && ALL && nvec == 0) continue;          // no whole vector: nothing to read or store here
    float v[E], g[E], b[E], o[E];
    opaque(t[j]);
    Vec<X>::unpack(t[j], v);
    Vec<X>::unpack(gv[idc], g);
    Vec<X>::unpack(bv[idc], b);
#pragma unroll
    for (int k = 0; k < E; ++k) o[k] = (((v[k] - mu) * rstd) * g[k]) + b[k];
    if (FULL || idx < nvec) __builtin_nontemporal_store(Vec<X>::pack(o), yr + idx);
  }
  if (extra)
    Tile<X>::store1(y + row * d + ec, (((xe - mu) * rstd) * Tile<X>::load1(gamma + ec)) + Tile<X>::load1(beta + ec));
}

// The group's row: a workgroup-sized group takes row blockIdx.x, wave-sized groups the rows 4 * blockIdx.x + wave,
// groups of 8, 16 or 32 lanes (short rows, several to a wave) the rows (256 / THREADS) * blockIdx.x + group.
template <int THREADS>
__device__ __forceinline__ int64_t group_row() {
  if (THREADS == kWave)
    return int64_t(blockIdx.x) * kRowsPerBlock + __builtin_amdgcn_readfirstlane(int(threadIdx.x / kWave));
  if (THREADS < kWave)
    return int64_t(blockIdx.x) * (kNormThreads / THREADS) + int(threadIdx.x) / THREADS;
  return blockIdx.x;
}

template <typename X, int NV, int THREADS, bool RAGGED, bool ENDS>
__device__ __forceinline__ void layernorm_group(const typename X::storage* __restrict__ x,
                                                const typename X::storage* __restrict__ gamma,
                                                const typename X::storage* __restrict__ beta,
                                                typename X::storage* __restrict__ y, int64_t rows, int64_t d, float eps) {
  __shared__ double lds[THREADS >= kWave ? THREADS / kWave : 1];
  const int64_t row = group_row<THREADS>();
  if (row >= rows) return;                           // groups of a wave or less only (no barrier follows there); grid = rows otherwise
  if (!RAGGED && (!ENDS || THREADS == 1024 || NV == 8) && d == int64_t(Vec<X>::kElems) * THREADS * NV)
    layernorm_group_row<X, NV, THREADS, true, true, false>(x, gamma, beta, y, row, d, eps, lds);
  else
    layernorm_group_row<X, NV, THREADS, false, !ENDS, RAGGED>(x, gamma, beta, y, row, d, eps, lds);
}

// KEEP: the exponentials stay in registers (f32) between the sum and the output pass; without it they are
// computed again from the stored row (the 1024-lane form has 128 registers per lane, not enough for both where a lane holds
// more than 64 elements).
template <typename X, int NV, int THREADS, bool FULL, bool ALL, bool KEEP, bool RAGGED, bool PAST>
__device__ __forceinline__ void softmax_group_row(const typename X::storage* __restrict__ x, typename X::storage* __restrict__ y,
                                                  int64_t row, int64_t d, double* lds) {
  constexpr int E = Vec<X>::kElems;
  using V = typename RowVector<RAGGED>::type;
  const int lane = int(threadIdx.x) & (THREADS - 1);
  // Fewer vectors, or 32-bit elements of which a line has half as many: what the 64-bit sums cost is more (uncut and cut, bf16 [96000, 750] 51.3, 54.6; f32
  // [20, 20001] 4.5, 5.1; [20, 50001] 8.1, 8.7; [3000, 1001] 4.8, 5.0, for [24000, 1501] 51.4, 48.6; [500, 50001] 43.9, 40.3).
  constexpr bool kCut = RAGGED && THREADS >= kWave && NV > 2 && sizeof(typename X::storage) == 2;
  using Sum = typename RowSum<kCut>::type;
  using Add = typename RowSum<kCut>::op;
  RowCut cut = {0, 0};
  if constexpr (kCut) cut = cut_row<X, THREADS * NV>(x + row * d, y + row * d, d);
  // Uncut rows' vectors are counted from the 64-bit length: of a 32-bit quotient the compiler works each vector's place against the row's end out again in every
  // pass, where it otherwise keeps the lanes' masks in scalar registers (us, 32 bits and 64, f32 [300, 9001] 6.8, 5.9; [300, 5001] 4.9, 4.6; [300, 60001] 35.5, 33.2;
  // f16 [300, 18000] 8.05, 7.77).
  const int nvec = kCut ? (int(d) - cut.head) / E : int(d / E), tail = RAGGED ? int(d) - nvec * E : 0, end = nvec + cut.shift;
  const V* xr = reinterpret_cast<const V*>(x + row * d + cut.head) - cut.shift;
  const bool extra = RAGGED && lane < tail;          // this lane also owns an element outside the vectors
  const int ec = (lane < cut.head ? 0 : nvec * E) + lane;
  // Asked for with the vectors, by every lane, as in LayerNorm (us, behind and with them, f32 [124584, 301] 51.9, 50.5; [24983, 1501] 51.5, 50.9; [600, 25001] 22.1, 21.1; f16
  // [79893, 751] 42.6, 41.7; bf16 [149625, 401] 46.6, 45.5; f16 [79207, 101] 8.8, 8.4; slower f32 [399, 25001] 15.0, 15.4; [300, 5001] 4.53, 4.57).
  typename X::storage xb = 0;
  if constexpr (RAGGED) xb = (x + row * d)[min(ec, int(d) - 1)];
  u32x4 t[NV];
#pragma unroll
  for (int j = 0; j < NV; ++j) {
    if (!wave_has<THREADS, ALL>(j, end)) break;
    const int idx = lane + THREADS * j;
    if (!RAGGED || !ALL || nvec > 0)                  // (a row shorter than one vector: only the scalar elements below)
      t[j] = PAST ? __builtin_nontemporal_load(xr + (FULL ? idx : held<kCut>(j, idx, cut.shift, end))) : xr[FULL ? idx : held<kCut>(j, idx, cut.shift, end)];
  }
  // What lies past the row becomes -infinity where it is loaded: it changes no maximum and its exponential is zero, and the passes
  // below need not tell it from the row (us, f16 [1084, 50000] 61.2 -> 53.0, f32 [2000, 25001] 102 -> 97, bf16 [200, 8191] 7.5 -> 7.1; [48000, 1500] as before).
  if (!FULL) {
#pragma unroll
    for (int j = 0; j < NV; ++j) {
      if (!wave_has<THREADS, ALL>(j, end)) break;
      const bool live = within<kCut>(j, lane + THREADS * j, cut.shift, end);
#pragma unroll
      for (int k = 0; k < 4; ++k) t[j][k] = live ? t[j][k] : Vec<X>::kMinusInf;
    }
  }
  const float xe = extra ? Tile<X>::load1(&xb) : -INFINITY;
  float mx = xe;
#pragma unroll
  for (int j = 0; j < NV; ++j) {
    if (!wave_has<THREADS, ALL>(j, end)) break;
    float v[E];
    Vec<X>::unpack(t[j], v);
#pragma unroll
    for (int k = 0; k < E; ++k) mx = fmaxf(mx, v[k]);
  }
  mx = group_reduce<THREADS>(mx, MaxF32(), lds);
  float e[KEEP ? NV * E : 1];
  const float ee = extra ? __expf(xe - mx) : 0.0f;
  constexpr int kSums = kCut ? 4 : 1;                  // (a chain of 64-bit additions is long)
  Sum s[kSums] = {};
  s[0] = ee;
#pragma unroll
  for (int j = 0; j < NV; ++j) {
    if (!wave_has<THREADS, ALL>(j, end)) break;
    float v[E];
    opaque(t[j]);
    Vec<X>::unpack(t[j], v);
#pragma unroll
    for (int k = 0; k < E; ++k) {
      const float ev = __expf(v[k] - mx);
      if (KEEP) e[j * E + k] = ev;
      s[k % kSums] = s[k % kSums] + ev;
    }
  }
  if (kCut) s[0] = (s[0] + s[kSums / 2]) + (s[kSums / 4] + s[kSums - 1]);
  const float inv = 1.0f / float(group_reduce<THREADS>(s[0], Add(), lds));                         // e * (1/s), as in softmax_row
  V* yr = reinterpret_cast<V*>(y + row * d + cut.head) - cut.shift;
#pragma unroll
  for (int j = 0; j < NV; ++j) {
    if (!wave_has<THREADS, ALL>(j, end)) break;
    const int idx = lane + THREADS * j;
    float o[E];
    if (KEEP) {
#pragma unroll
      for (int k = 0; k < E; ++k) o[k] = e[j * E + k] * inv;
    } else {
      float v[E];
      opaque(t[j]);
      Vec<X>::unpack(t[j], v);
#pragma unroll
      for (int k = 0; k < E; ++k) o[k] = __expf(v[k] - mx) * inv;
    }
    if (FULL || within<kCut>(j, idx, cut.shift, end)) __builtin_nontemporal_store(Vec<X>::pack(o), yr + idx);
  }
  if (extra) Tile<X>::store1(y + row * d + ec, ee * inv);
}

template <typename X, int NV, int THREADS, bool RAGGED, bool ENDS, bool PAST>
__device__ __forceinline__ void softmax_group(const typename X::storage* __restrict__ x, typename X::storage* __restrict__ y,
                                              int64_t rows, int64_t d) {
  __shared__ double lds[THREADS >= kWave ? THREADS / kWave : 1];
  constexpr bool kKeep = THREADS <= 256 || NV * Vec<X>::kElems <= 64;
  const int64_t row = group_row<THREADS>();
  if (row >= rows) return;                           // groups of a wave or less only (no barrier follows there); grid = rows otherwise
  if (PAST && !RAGGED && !(ENDS && THREADS < 1024) && d == int64_t(Vec<X>::kElems) * THREADS * NV)   // (whole cache lines)
    softmax_group_row<X, NV, THREADS, true, true, kKeep, false, true>(x, y, row, d, lds);
  else
    softmax_group_row<X, NV, THREADS, false, !ENDS, kKeep, RAGGED, PAST>(x, y, row, d, lds);
}

// ---- any D, any alignment: one workgroup per row, row re-read from cache -------------
template <typename Op>
__device__ __forceinline__ float block_reduce(float v, Op op, float* lds) {
  v = wave_reduce(v, op);
  const int wave = threadIdx.x / kWave;
  __syncthreads();                                   // lds may still be read from the previous round
  if ((threadIdx.x & (kWave - 1)) == 0) lds[wave] = v;
  __syncthreads();
  float r = lds[0];
#pragma unroll
  for (int w = 1; w < kNormThreads / kWave; ++w) r = op(r, lds[w]);
  return r;
}

// Rows of any length and alignment: whole vectors by 128-bit accesses at element alignment, the d % E elements behind
// them one per lane; the row is read three times (the second and third time from cache).
template <typename X>
__device__ __forceinline__ void layernorm_any(const typename X::storage* __restrict__ x,
                                              const typename X::storage* __restrict__ gamma,
                                              const typename X::storage* __restrict__ beta,
                                              typename X::storage* __restrict__ y, int64_t rows, int64_t d, float eps) {
  constexpr int E = Vec<X>::kElems;
  using V = typename RowVector<true>::type;
  __shared__ float lds[kNormThreads / kWave];
  const int64_t nvec = d / E, tail0 = nvec * E;
  const V* gv = reinterpret_cast<const V*>(gamma);
  const V* bv = reinterpret_cast<const V*>(beta);
  for (int64_t row = blockIdx.x; row < rows; row += gridDim.x) {
    const typename X::storage* xr = x + row * d;
    const V* xv = reinterpret_cast<const V*>(xr);
    float sum = 0.0f;
    for (int64_t v = threadIdx.x; v < nvec; v += kNormThreads) {
      float f[E];
      Vec<X>::unpack(xv[v], f);
#pragma unroll
      for (int k = 0; k < E; ++k) sum = sum + f[k];
    }
    for (int64_t c = tail0 + threadIdx.x; c < d; c += kNormThreads) sum = sum + Tile<X>::load1(xr + c);
    const float mu = block_reduce(sum, SumF32(), lds) / float(d);
    float sq = 0.0f;
    for (int64_t v = threadIdx.x; v < nvec; v += kNormThreads) {
      float f[E];
      Vec<X>::unpack(xv[v], f);
#pragma unroll
      for (int k = 0; k < E; ++k) { const float dv = f[k] - mu; sq = sq + dv * dv; }
    }
    for (int64_t c = tail0 + threadIdx.x; c < d; c += kNormThreads) { const float dv = Tile<X>::load1(xr + c) - mu; sq = sq + dv * dv; }
    const float var = block_reduce(sq, SumF32(), lds) / float(d);
    const float rstd = 1.0f / sqrtf(var + eps);
    V* yv = reinterpret_cast<V*>(y + row * d);
    for (int64_t v = threadIdx.x; v < nvec; v += kNormThreads) {
      float f[E], g[E], b[E], o[E];
      Vec<X>::unpack(xv[v], f);
      Vec<X>::unpack(gv[v], g);
      Vec<X>::unpack(bv[v], b);
#pragma unroll
      for (int k = 0; k < E; ++k) o[k] = (((f[k] - mu) * rstd) * g[k]) + b[k];
      yv[v] = Vec<X>::pack(o);
    }
    for (int64_t c = tail0 + threadIdx.x; c < d; c += kNormThreads) {
      const float dv = Tile<X>::load1(xr + c) - mu;
      Tile<X>::store1(y + row * d + c, ((dv * rstd) * Tile<X>::load1(gamma + c)) + Tile<X>::load1(beta + c));
    }
  }
}

template <typename X>
__device__ __forceinline__ void softmax_any(const typename X::storage* __restrict__ x, typename X::storage* __restrict__ y,
                                            int64_t rows, int64_t d) {
  constexpr int E = Vec<X>::kElems;
  using V = typename RowVector<true>::type;
  __shared__ float lds[kNormThreads / kWave];
  const int64_t nvec = d / E, tail0 = nvec * E;
  for (int64_t row = blockIdx.x; row < rows; row += gridDim.x) {
    const typename X::storage* xr = x + row * d;
    const V* xv = reinterpret_cast<const V*>(xr);
    float mx = -INFINITY;
    for (int64_t v = threadIdx.x; v < nvec; v += kNormThreads) {
      float f[E];
      Vec<X>::unpack(xv[v], f);
#pragma unroll
      for (int k = 0; k < E; ++k) mx = fmaxf(mx, f[k]);
    }
    for (int64_t c = tail0 + threadIdx.x; c < d; c += kNormThreads) mx = fmaxf(mx, Tile<X>::load1(xr + c));
    mx = block_reduce(mx, MaxF32(), lds);
    float s = 0.0f;
    for (int64_t v = threadIdx.x; v < nvec; v += kNormThreads) {
      float f[E];
      Vec<X>::unpack(xv[v], f);
#pragma unroll
      for (int k = 0; k < E; ++k) s = s + __expf(f[k] - mx);
    }
    for (int64_t c = tail0 + threadIdx.x; c < d; c += kNormThreads) s = s + __expf(Tile<X>::load1(xr + c) - mx);
    s = block_reduce(s, SumF32(), lds);
    const float inv = 1.0f / s;
    V* yv = reinterpret_cast<V*>(y + row * d);
    for (int64_t v = threadIdx.x; v < nvec; v += kNormThreads) {
      float f[E], o[E];
      Vec<X>::unpack(xv[v], f);
#pragma unroll
      for (int k = 0; k < E; ++k) o[k] = __expf(f[k] - mx) * inv;
      yv[v] = Vec<X>::pack(o);
    }
    for (int64_t c = tail0 + threadIdx.x; c < d; c += kNormThreads)
      Tile<X>::store1(y + row * d + c, __expf(Tile<X>::load1(xr + c) - mx) * inv);
  }
}

}  // namespace norm_cluster
using namespace norm_cluster;

// _v8r: the eight-vector LayerNorm held to 64 registers, eight waves per SIMD.  It is the slower kernel per
// row (the affine parameters are fetched one vector at a time), but when the whole tensor then fits on the
// chip at once while the default kernel (five waves per SIMD) would need a second, partly filled round, the
// launch is one read phase followed by one write phase and ends sooner (bf16 [8192, 4096]: 26.6 -> 24.3 us;
// [4096, 4096] 11.3 -> 12.7 us and [16384, 4096] 47.4 -> 50.4 us, hence only inside that window).
// Entry points.  mtrt_layernorm_<t>_v<NV>(x, gamma, beta, y, rows, d, eps)
//                mtrt_softmax_<t>_v<NV>(x, y, rows, d)         NV = vectors per lane
// Softmax kernels, here and below, with a t at the end: rows read through the caches, which don't fill all vectors; with a c: rows that are cut, past the caches (those
// through them are, too).  A body of its own for either kind: both in one kernel are as slow for small tensors as the cut alone, whose code a launch has to fetch.
#define MTRT_LN_OCCUPANCY_1
#define MTRT_LN_OCCUPANCY_2
#define MTRT_LN_OCCUPANCY_4
#define MTRT_LN_OCCUPANCY_8 __attribute__((amdgpu_waves_per_eu(5, 5)))
#define MTRT_LN_OCCUPANCY_16
#define MTRT_NORM_KERNELS(XN, XT, NV)                                                                         \
  extern "C" __global__ void __launch_bounds__(kNormThreads) MTRT_LN_OCCUPANCY_##NV mtrt_layernorm_##XN##_v##NV(                      \
      const XT::storage* x, const XT::storage* gamma, const XT::storage* beta, XT::storage* y, int64_t rows,  \
      int64_t d, float eps) { layernorm_rows<XT, NV>(x, gamma, beta, y, rows, d, eps); }                      \
  extern "C" __global__ void __launch_bounds__(kNormThreads) mtrt_softmax_##XN##_v##NV(                        \
      const XT::storage* x, XT::storage* y, int64_t rows, int64_t d) { softmax_rows<XT, NV, true, false>(x, y, rows, d); }  \
  extern "C" __global__ void __launch_bounds__(kNormThreads) mtrt_softmax_##XN##_v##NV##t(                     \
      const XT::storage* x, XT::storage* y, int64_t rows, int64_t d) { softmax_rows<XT, NV, false, true>(x, y, rows, d); }  \
  extern "C" __global__ void __launch_bounds__(kNormThreads) mtrt_softmax_##XN##_v##NV##c(                     \
      const XT::storage* x, XT::storage* y, int64_t rows, int64_t d) { softmax_rows<XT, NV, true, true>(x, y, rows, d); }

#define MTRT_NORM_FOR_TYPE(XN, XT)                                                                            \
  MTRT_NORM_KERNELS(XN, XT, 1) MTRT_NORM_KERNELS(XN, XT, 2) MTRT_NORM_KERNELS(XN, XT, 4)                       \
  MTRT_NORM_KERNELS(XN, XT, 8) MTRT_NORM_KERNELS(XN, XT, 16)                                                   \
  extern "C" __global__ void __launch_bounds__(kNormThreads) __attribute__((amdgpu_waves_per_eu(8, 8)))        \
  mtrt_layernorm_##XN##_v8r(const XT::storage* x, const XT::storage* gamma, const XT::storage* beta,           \
                            XT::storage* y, int64_t rows, int64_t d, float eps) {                              \
    layernorm_rows<XT, 8, true>(x, gamma, beta, y, rows, d, eps);                                              \
  }                                                                                                            \
  extern "C" __global__ void __launch_bounds__(kNormThreads) mtrt_layernorm_##XN##_any(                        \
      const XT::storage* x, const XT::storage* gamma, const XT::storage* beta, XT::storage* y, int64_t rows,  \
      int64_t d, float eps) { layernorm_any<XT>(x, gamma, beta, y, rows, d, eps); }                           \
  extern "C" __global__ void __launch_bounds__(kNormThreads) mtrt_softmax_##XN##_any(                          \
      const XT::storage* x, XT::storage* y, int64_t rows, int64_t d) { softmax_any<XT>(x, y, rows, d); }

// One workgroup per row: mtrt_layernorm_<t>_g<THREADS>v<NV>(x, gamma, beta, y, rows, d, eps), mtrt_softmax_<t>_g<THREADS>v<NV>(x, y, rows, d)
//   grid = rows, block = THREADS; d % E == 0, d / E <= THREADS * NV, operands 16-byte aligned.
// Ragged rows: mtrt_{layernorm,softmax}_<t>_u<THREADS>v<NV>, same arguments; any d >= 1 with d / E <= THREADS * NV,
//   operands aligned to their element; THREADS <= 64 (NV = 1 below 64): grid = ceil(rows / (256 / THREADS)), block = 256;
//   else grid = rows, block = THREADS.
#define MTRT_LAYERNORM_GROUP_KERNEL(XN, XT, NV, THREADS, TAG, RAGGED, BLOCK, ENDS, END)                        \
  extern "C" __global__ void __launch_bounds__(BLOCK) mtrt_layernorm_##XN##_##TAG##THREADS##v##NV##END(        \
      const XT::storage* x, const XT::storage* gamma, const XT::storage* beta, XT::storage* y, int64_t rows,  \
      int64_t d, float eps) { layernorm_group<XT, NV, THREADS, RAGGED, ENDS>(x, gamma, beta, y, rows, d, eps); }
#define MTRT_SOFTMAX_GROUP_KERNEL(XN, XT, NV, THREADS, TAG, RAGGED, BLOCK, ENDS, END)                          \
  extern "C" __global__ void __launch_bounds__(BLOCK) mtrt_softmax_##XN##_##TAG##THREADS##v##NV##END(          \
      const XT::storage* x, XT::storage* y, int64_t rows, int64_t d) { softmax_group<XT, NV, THREADS, RAGGED, ENDS, true>(x, y, rows, d); }   \
  extern "C" __global__ void __launch_bounds__(BLOCK) mtrt_softmax_##XN##_##TAG##THREADS##v##NV##END##t(       \
      const XT::storage* x, XT::storage* y, int64_t rows, int64_t d) { softmax_group<XT, NV, THREADS, RAGGED, ENDS, false>(x, y, rows, d); }
// (f32 LayerNorm at element alignment: nearly full rows, [2000, 15001], 49.4 us with every vector worked on and 51.1 without)
#define MTRT_NORM_GROUP_KERNELS(XN, XT, NV, THREADS, TAG, RAGGED, BLOCK)                                       \
  MTRT_LAYERNORM_GROUP_KERNEL(XN, XT, NV, THREADS, TAG, RAGGED, BLOCK, (THREADS == 1024 && !(RAGGED && Vec<XT>::kElems == 4)), )               \
  MTRT_SOFTMAX_GROUP_KERNEL(XN, XT, NV, THREADS, TAG, RAGGED, BLOCK, (THREADS == 1024), )
#define MTRT_NORM_GROUPS_FOR_TYPE(XN, XT)                                                                      \
  MTRT_NORM_GROUP_KERNELS(XN, XT, 8, 256, g, false, 256) MTRT_NORM_GROUP_KERNELS(XN, XT, 16, 256, g, false, 256)      \
  MTRT_NORM_GROUP_KERNELS(XN, XT, 8, 1024, g, false, 1024) MTRT_NORM_GROUP_KERNELS(XN, XT, 16, 1024, g, false, 1024)  \
  MTRT_NORM_GROUP_KERNELS(XN, XT, 1, 8, u, true, 256) MTRT_NORM_GROUP_KERNELS(XN, XT, 1, 16, u, true, 256)            \
  MTRT_NORM_GROUP_KERNELS(XN, XT, 1, 32, u, true, 256)                                                                \
  MTRT_NORM_GROUP_KERNELS(XN, XT, 1, 64, u, true, 256) MTRT_NORM_GROUP_KERNELS(XN, XT, 2, 64, u, true, 256)           \
  MTRT_NORM_GROUP_KERNELS(XN, XT, 4, 64, u, true, 256) MTRT_NORM_GROUP_KERNELS(XN, XT, 16, 64, u, true, 256)          \
  MTRT_NORM_GROUP_KERNELS(XN, XT, 16, 256, u, true, 256) MTRT_NORM_GROUP_KERNELS(XN, XT, 16, 1024, u, true, 1024)     \
  MTRT_SOFTMAX_GROUP_KERNEL(XN, XT, 8, 64, u, true, 256, false, ) MTRT_SOFTMAX_GROUP_KERNEL(XN, XT, 8, 256, u, true, 256, false, )  \
  MTRT_SOFTMAX_GROUP_KERNEL(XN, XT, 8, 1024, u, true, 1024, true, )
// (f32 LayerNorm takes the 16-vector forms there: unaligned_nv in clusters.cpp)
#define MTRT_NORM_GROUPS_OF_8_RAGGED_16_BIT(XN, XT)                                                            \
  MTRT_LAYERNORM_GROUP_KERNEL(XN, XT, 8, 64, u, true, 256, false, ) MTRT_LAYERNORM_GROUP_KERNEL(XN, XT, 8, 256, u, true, 256, false, )  \
  MTRT_LAYERNORM_GROUP_KERNEL(XN, XT, 8, 1024, u, true, 1024, true, )

MTRT_NORM_FOR_TYPE(f32, F32)
MTRT_NORM_FOR_TYPE(f16, F16)
MTRT_NORM_FOR_TYPE(bf16, BF16)
MTRT_NORM_GROUPS_FOR_TYPE(f32, F32)
MTRT_NORM_GROUPS_FOR_TYPE(f16, F16)
MTRT_NORM_GROUPS_FOR_TYPE(bf16, BF16)
MTRT_NORM_GROUPS_OF_8_RAGGED_16_BIT(f16, F16)
MTRT_NORM_GROUPS_OF_8_RAGGED_16_BIT(bf16, BF16)

// Both forms of a kernel where either is the faster one for some rows (row_form in clusters.cpp).  The names above are those that work on every
// vector, with 1024 lanes those that stop at the row's end; here the other ones: `e`, stop at the row's end (rows that do not fill
// all vectors, or without a body of its own for those that do), and `a`, every vector.
#define MTRT_NORM_OTHER_FORMS_16_BIT(XN, XT)                                                                   \
  MTRT_LAYERNORM_GROUP_KERNEL(XN, XT, 8, 256, g, false, 256, true, e) MTRT_LAYERNORM_GROUP_KERNEL(XN, XT, 16, 256, g, false, 256, true, e)  \
  MTRT_LAYERNORM_GROUP_KERNEL(XN, XT, 4, 64, u, true, 256, true, e) MTRT_LAYERNORM_GROUP_KERNEL(XN, XT, 8, 64, u, true, 256, true, e)       \
  MTRT_LAYERNORM_GROUP_KERNEL(XN, XT, 16, 64, u, true, 256, true, e)                                                                        \
  MTRT_LAYERNORM_GROUP_KERNEL(XN, XT, 8, 256, u, true, 256, true, e) MTRT_LAYERNORM_GROUP_KERNEL(XN, XT, 16, 256, u, true, 256, true, e)    \
  MTRT_SOFTMAX_GROUP_KERNEL(XN, XT, 8, 256, g, false, 256, true, e) MTRT_SOFTMAX_GROUP_KERNEL(XN, XT, 16, 256, g, false, 256, true, e)      \
  MTRT_SOFTMAX_GROUP_KERNEL(XN, XT, 8, 256, u, true, 256, true, e) MTRT_SOFTMAX_GROUP_KERNEL(XN, XT, 16, 256, u, true, 256, true, e)
#define MTRT_NORM_OTHER_FORMS(XN, XT)                                                                          \
  MTRT_LAYERNORM_GROUP_KERNEL(XN, XT, 8, 1024, g, false, 1024, false, a)                                       \
  MTRT_SOFTMAX_GROUP_KERNEL(XN, XT, 8, 1024, g, false, 1024, false, a) MTRT_SOFTMAX_GROUP_KERNEL(XN, XT, 16, 1024, g, false, 1024, false, a)
MTRT_LAYERNORM_GROUP_KERNEL(f16, F16, 16, 1024, g, false, 1024, false, a)
MTRT_LAYERNORM_GROUP_KERNEL(bf16, BF16, 16, 1024, g, false, 1024, false, a)
MTRT_NORM_OTHER_FORMS_16_BIT(f16, F16)
MTRT_NORM_OTHER_FORMS_16_BIT(bf16, BF16)
MTRT_NORM_OTHER_FORMS(f32, F32)
MTRT_NORM_OTHER_FORMS(f16, F16)
MTRT_NORM_OTHER_FORMS(bf16, BF16)
MTRT_LAYERNORM_GROUP_KERNEL(f32, F32, 8, 256, g, false, 256, true, e)
MTRT_SOFTMAX_GROUP_KERNEL(f32, F32, 8, 1024, u, true, 1024, false, a)
MTRT_SOFTMAX_GROUP_KERNEL(f32, F32, 16, 1024, u, true, 1024, false, a)

// Softmax of 16-bit rows of 32769 to 65536 elements where there are more rows than compute units: the exponentials are computed again in the output pass
// instead of kept, 62 or 64 registers instead of 84 to 103, so that a unit has two rows and one's arithmetic lies under the other's way to memory; the same bits.
// What bounds it: memory and the vector units, each idle for a part of a row.  `r`: to the row's end, `ra`: every vector.  us, kept and computed
// again, bf16 [1084, 43165] 46.8, 41.1; [2000, 34000] 60.4, 52.2; [512, 50000] 24.4, 21.1; [300, 40000] 15.9, 14.6; rows past 0.8 of the vectors [1084, 64000] 59.1,
// 57.5, every vector 54.1; [300, 64000] 22.2, 21.7, 19.0; up to a row to a unit [230, 40000] 9.6, 10.2; [230, 64000] 14.0, 15.4, 14.5.
#define MTRT_SOFTMAX_TWO_ROWS_KERNEL(XN, XT, TAG, RAGGED, ALL, NAME, PAST)                                     \
  extern "C" __global__ void __launch_bounds__(1024) __attribute__((amdgpu_waves_per_eu(8, 8))) mtrt_softmax_##XN##_##TAG##1024v8##NAME(  \
      const XT::storage* x, XT::storage* y, int64_t rows, int64_t d) {                                         \
    __shared__ double lds[16];                                                                                 \
    const int64_t row = blockIdx.x;                                                                            \
    if (row < rows) softmax_group_row<XT, 8, 1024, false, ALL, false, RAGGED, PAST>(x, y, row, d, lds);        \
  }
#define MTRT_SOFTMAX_TWO_ROWS_KERNELS(XN, XT)                                                                  \
  MTRT_SOFTMAX_TWO_ROWS_KERNEL(XN, XT, g, false, false, r, true) MTRT_SOFTMAX_TWO_ROWS_KERNEL(XN, XT, g, false, false, rt, false)  \
  MTRT_SOFTMAX_TWO_ROWS_KERNEL(XN, XT, g, false, true, ra, true) MTRT_SOFTMAX_TWO_ROWS_KERNEL(XN, XT, g, false, true, rat, false)  \
  MTRT_SOFTMAX_TWO_ROWS_KERNEL(XN, XT, u, true, false, r, true) MTRT_SOFTMAX_TWO_ROWS_KERNEL(XN, XT, u, true, false, rt, false)
MTRT_SOFTMAX_TWO_ROWS_KERNELS(f16, F16)
MTRT_SOFTMAX_TWO_ROWS_KERNELS(bf16, BF16)
