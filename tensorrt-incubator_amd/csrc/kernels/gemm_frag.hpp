// The tile loop of the GEMMs whose weights are held in fragment order (int8, f16, bf16): weights from memory straight
// into registers, activations through a ring of LDS stages, any tile of IT x 32 rows by 4 JT x 32 columns, K cut over
// several workgroups where a launch would otherwise leave compute units idle.
//
// Fragment order (mtrt_w8_prepack_frag, mtrt_w16_prepack_frag): for each tile of 32 columns and each slice of 128 bytes
// of K four 1 KiB blocks, one per k-step p; in a block lane l = 32 h + (n % 32) owns the 16 bytes 128 slice + 32 p + 16 h
// .. + 15 of column n: the B operand of the 32 x 32 matrix instruction of that k-step, whatever the type (16 int8 or
// 8 sixteen-bit values), and every load of a wave reads 1 KiB of contiguous memory.  Float8 codes of 16-bit products (mtrt_wf8_prepack_frag,
// gemm_core::F8Codes) lie the same way in half the bytes, eight codes to a lane and k-step.
//
// Why one loop for many tiles.  A 256-row tile gives the fewest bytes per MFMA, but a launch lasts one tile's whole K
// loop: with M in the hundreds, or a short N, such tiles occupied 10 to 60 of the 256 compute units (M = 398, K = 11520,
// N = 1856 int8: 30 half tiles, 75 us for 17 G operations).  Smaller tiles and, when even those are too few, several
// workgroups per tile that share its K range put the whole chip on the problem; what a compute unit's L1 takes in (24 to
// 34 bytes per clock) then sets the time, so the tile is the largest one that fills the chip.
//
// Structure (one workgroup of four waves per compute unit, one wave per SIMD, 1 x 4 waves):
//   * every wave owns all IT * 32 rows of its JT * 32 columns, so a weight fragment is loaded by one wave only;
//   * the weights of D slices (4 D k-steps) sit in a register ring: those of a k-step are asked for again as soon as it is
//     over; the activations of D slices ahead are under way into LDS (direct-to-LDS loads, XOR-swizzled 128-byte rows,
//     a power of two of at least D + 2 stages);
//   * activation fragments are read AN ahead of their use as one stream of opaque instructions;
//   * memory instructions are issued in a fixed order and waited for by count (see Order); surplus loads past the end of
//     K fetch one fixed line.
// K split: workgroups (tile, 0 .. S - 1) run slices [S_i, S_i+1) each.  All of them write their partial tile to the
// workspace with write-through stores and take a ticket; the last one adds the partial tiles in split order (the same
// bits whoever is last) and runs the epilogue.  Nobody waits.  The ticket word is returned to zero.
#pragma once
#include "gemm_core.hpp"

namespace gemm_frag {

using namespace gemm_core;

template <int I, int N, class F>
__device__ __forceinline__ void static_for(F&& f) {
  if constexpr (I < N) {
    f(IntC<I>{});
    static_for<I + 1, N>(f);
  }
}

// 16 bytes (of codes: 8) per lane of k-step T of a weight slice: scalar base, 32-bit lane offset, the k-step as the instruction's offset
template <int T>
__device__ __forceinline__ void load_w(v2i& dst, uint32_t lane_off, const int8_t* base) {
  __asm__ volatile("global_load_dwordx2 %0, %1, %2 offset:%3" : "=v"(dst) : "v"(lane_off), "s"(base), "n"(T * 512) : "memory");
}
template <int T>
__device__ __forceinline__ void load_w(v4i& dst, uint32_t lane_off, const int8_t* base) {
  __asm__ volatile("global_load_dwordx4 %0, %1, %2 offset:%3" : "=v"(dst) : "v"(lane_off), "s"(base), "n"(T * 1024) : "memory");
}

// The memory instructions of a wave, in issue order: per k-step first its direct-to-LDS loads, then JT weight loads.
// In k-step T of slice s: the activations of slice s + D, the weights of the k-step 4 D - 1 further on.  Codes are dequantized during the k-step
// before the one that uses them, so their registers are free, and wanted again, a k-step earlier: 4 D further on, and the counts are the same.
template <int IT, int JT, int D>
struct Order {
  static constexpr int kLoads = IT;                    // direct-to-LDS loads per wave and slice (32 IT rows, 4 waves, 8 rows each)
  static constexpr int kRing = 4 * D;                  // k-steps of weights in registers
  static constexpr int dma(int t) { return IT >= 4 ? IT / 4 : (t < IT ? 1 : 0); }
  static constexpr int first(int t) { return IT >= 4 ? t * (IT / 4) : t; }       // first load of k-step t
  static constexpr int last_step() { return IT >= 4 ? 3 : IT - 1; }              // k-step of a slice's last direct-to-LDS load
  // issued after the weights of a k-step and before that k-step begins (at k-step T): kRing - 2 whole k-steps
  static constexpr int weights_in_flight(int t) {
    int n = 0;
    for (int i = 1; i <= kRing - 2; ++i) n += JT + dma(((t - i) % 4 + 4) % 4);
    return n;
  }
  // issued after the last load of slice s + 1's activations and before k-step `at` of slice s
  static constexpr int activations_in_flight(int at) {
    int n = JT + (3 - last_step()) * JT + (D - 2) * (kLoads + 4 * JT);
    for (int t = 0; t < at; ++t) n += dma(t) + JT;
    return n;
  }
  // ... of slice 0, at the end of the prologue
  // (no weights go with the first loads of all: a slice whose only load comes in k-step 0 has JT fewer behind it)
  static constexpr int activations_in_flight_at_start() {
    return (last_step() == 0 ? 0 : JT) + (3 - last_step()) * JT + (D - 1) * (kLoads + 4 * JT);
  }
  // codes: those of the first k-step, issued with the first loads of all, at the end of the prologue
  static constexpr int first_codes_in_flight() {
    int n = 0;
    for (int i = 1; i < 4 * D; ++i) n += JT + dma(i % 4);
    return n;
  }
};

template <int IT, int D>
constexpr int stages() { return D + 2 <= 4 ? 4 : 8; }
// LDS of a workgroup: the ring of activation stages, afterwards the staging of the outputs (at most 128 rows per wave at
// a time) and `scratch_floats` of the epilogue
template <int IT, int D>
constexpr int lds_bytes(int scratch_floats) {
  const int ring = stages<IT, D>() * IT * 32 * 128, out = 4 * 32 * (IT < 4 ? IT : 4) * kOutRow + 4 * scratch_floats;
  return ring > out ? ring : out;
}

// One workgroup's part of the problem.
struct Part {
  int64_t m0, n0;                                      // first row and column of the tile
  uint32_t slice0, nslices;                            // K range in slices of 128 bytes
  uint32_t splits, split;                              // workgroups on this tile, and which one this is
  uint32_t* ticket;                                    // splits > 1: zero, returned to zero
  f32x4* partial;                                      // splits > 1: this tile's partial tiles, split after split
};

__device__ __forceinline__ void store_through(f32x4* p, f32x4 v) {
  __asm__ volatile("global_store_dwordx4 %0, %1, off sc1" ::"v"(p), "v"(v) : "memory");
}

// device-coherent: this workgroup's L2 may hold old values of the line
template <int Q>
__device__ __forceinline__ void load_through(f32x4& dst, const f32x4* src) {
  __asm__ volatile("global_load_dwordx4 %0, %1, off offset:%2 sc1" : "=v"(dst) : "v"(src), "n"(Q * 1024) : "memory");
}

// Adds up the partial tiles of a split tile; true for the workgroup that is to run the epilogue.  Four waves hold the tile;
// further waves of the workgroup (active = false) only take part in the barriers.  SUMS: tiles times parts that a trip to memory brings (what the
// registers beside the accumulators hold), two parts of as many tiles as that is rather than four of half as many: parts past the last are fetched
// all the same, and most splits are into two or three.  us, four parts and two at a time, W4A16 (136, 4224, 3904) 15.2, 14.7; (282, 3840, 2880) 15.2, 14.7;
// (106, 10496, 6784) 25.7, 25.2; f16 (1493, 8448, 1152) 36.1, 35.4; more parts the same.
template <class Scalar, int SUMS, int IT, int JT, class Acc>
__device__ __forceinline__ bool meet(Acc (&acc)[IT][JT], const Part& part, int8_t* lds, int wave, bool active = true) {
  constexpr int kTiles = IT * JT, kPer = 4 * kTiles;   // 32 x 32 tiles of the wave; 16-byte pieces per lane
  const int lane = threadIdx.x & 63;
  f32x4* mine = part.partial + (uint64_t(part.split) * 4 + wave) * (kPer * 64) + lane;
  if (active) {
#pragma unroll
    for (int i = 0; i < IT; ++i)
#pragma unroll
      for (int j = 0; j < JT; ++j)
#pragma unroll
        for (int q = 0; q < 4; ++q) {
          f32x4 v;
#pragma unroll
          for (int e = 0; e < 4; ++e) v[e] = __builtin_bit_cast(float, Scalar(acc[i][j][4 * q + e]));
          store_through(mine + ((i * JT + j) * 4 + q) * 64, v);
        }
  }
  __asm__ volatile("s_waitcnt vmcnt(0)" ::: "memory");  // written through: visible to the whole device
  __syncthreads();
  uint32_t* seen = reinterpret_cast<uint32_t*>(lds);
  if (threadIdx.x == 0) *seen = __hip_atomic_fetch_add(part.ticket, 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
  __syncthreads();
  if (*seen != part.splits - 1) return false;
  if (threadIdx.x == 0) __hip_atomic_store(part.ticket, 0u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
  if (!active) return true;
  // a round trip to memory for each group of G tiles, KB splits at a time
  constexpr int KB = SUMS / 2 <= kTiles ? 2 : 4, G = SUMS / KB;
  static_assert(kTiles % G == 0, "whole groups of tiles");
  const f32x4* all = part.partial + uint64_t(wave) * (kPer * 64) + lane;
#pragma unroll
  for (int g = 0; g < kTiles; g += G) {
    for (uint32_t k0 = 0; k0 < part.splits; k0 += KB) {
      f32x4 v[G][KB][4];
#pragma unroll
      for (int u = 0; u < G; ++u)
#pragma unroll
        for (int k = 0; k < KB; ++k) {
          const uint32_t from = k0 + k < part.splits ? k0 + k : part.splits - 1;
          const f32x4* src = all + uint64_t(from) * (4 * kPer * 64) + (g + u) * 4 * 64;
          load_through<0>(v[u][k][0], src);
          load_through<1>(v[u][k][1], src);
          load_through<2>(v[u][k][2], src);
          load_through<3>(v[u][k][3], src);
        }
#pragma unroll
      for (int u = 0; u < G; ++u)
#pragma unroll
        for (int k = 0; k < KB; ++k)
#pragma unroll
          for (int q = 0; q < 4; ++q) __asm__ volatile("s_waitcnt vmcnt(0)" : "+v"(v[u][k][q])::"memory");
#pragma unroll
      for (int u = 0; u < G; ++u) {
        Acc& sum = acc[(g + u) / JT][(g + u) % JT];
#pragma unroll
        for (int k = 0; k < KB; ++k) {
          if (k0 + k >= part.splits) break;            // (uniform)
          const bool start = k0 + k == 0;
#pragma unroll
          for (int r = 0; r < 16; ++r) {
            const float word = v[u][k][r >> 2][r & 3];
            const Scalar x = __builtin_bit_cast(Scalar, word);
            sum[r] = start ? x : sum[r] + x;
          }
        }
      }
    }
  }
  return true;
}

// Traits: Acc (sixteen accumulators), zero(), mfma(weight fragment, activation fragment, acc).  W: gemm_core::Values, or codes, whose fragments are
// dequantized a k-step ahead, spread over the MFMAs of the k-step before.
template <class Traits, int IT, int JT, int D, class W, class Epilogue, typename Y>
__device__ __forceinline__ void run(const int8_t* __restrict__ a, int64_t row_bytes, const W& weights, Epilogue& epi,
                                    Y* __restrict__ y, int64_t M, int64_t N, const Part& part, int8_t* lds) {
  using Acc = typename Traits::Acc;
  using O = Order<IT, JT, D>;
  constexpr int R = O::kRing, NS = stages<IT, D>(), AN = 4, kStageBytes = IT * 32 * 128;
  constexpr int TB = (4 * IT - AN) / IT;               // the first k-step that reads a fragment of the next slice
  static_assert(D % 2 == 0 && O::weights_in_flight(3) < 64 && O::activations_in_flight(TB) < 64 && O::activations_in_flight_at_start() < 64, "wait counter range");
  int thread = threadIdx.x;
  if constexpr (W::kCodes) __asm__ volatile("" : "+v"(thread));   // (the lane is not held through the loop for the epilogue: 256 x 256 tiles have no register left)
  const int lane = thread & 63;
  const int slot = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int frow = lane & 31, fhalf = lane >> 5;
  const int64_t total_slices = row_bytes / 128, ntiles = (N + 31) / 32;
  // (scalars: what a load adds to its base must sit in scalar registers)
  const uint32_t nslices = __builtin_amdgcn_readfirstlane(part.nslices), slice0 = __builtin_amdgcn_readfirstlane(part.slice0);

  Acc acc[IT][JT];
  DmaLoaderT<IT> al;
  al.init(a + uint64_t(slice0) * 128, M, row_bytes, part.m0);
  v4i fa[2][AN];
  typename W::Raw wr[R][JT];
  v4i fb[2][JT];                                       // codes: the fragments of this k-step and the next
  typename W::Scale ws[JT];
  const int8_t* wsrc[JT];                              // the first slice of each column tile (uniform)
  const uint32_t wlane = uint32_t(lane) * uint32_t(sizeof(typename W::Raw));
  constexpr int kSliceBytes = 4 * W::kStepBytes;
#pragma unroll
  for (int j = 0; j < JT; ++j) {
    int64_t tile = int64_t(__builtin_amdgcn_readfirstlane(uint32_t(part.n0 / 32))) + slot * JT + j;
    tile = tile < ntiles ? tile : ntiles - 1;          // tiles past N: some valid data, never stored
    wsrc[j] = weights.frag + (tile * total_slices + slice0) * kSliceBytes;
    if constexpr (W::kCodes) ws[j] = W::scale_of(weights.scale, part.n0 + (slot * JT + j) * 32 + frow, N);
  }
  // all ones for a slice of this part, zero past its end: such a load reads one fixed line of the first slice
  auto keep = [&](uint32_t slice) { return uint32_t(int32_t(slice - nslices) >> 31); };
  const uint32_t lds_base = uint32_t(uintptr_t((lds_void_t*)lds));
  uint32_t a_lane[4];
#pragma unroll
  for (int p = 0; p < 4; ++p) a_lane[p] = lds_base + uint32_t(lds_off(frow, 2 * p + fhalf));
  auto read_a = [&](v4i& dst, uint32_t addr, auto tile) {
    constexpr int I = decltype(tile)::value;
    __asm__ volatile("ds_read_b128 %0, %1 offset:%2" : "=v"(dst) : "v"(addr), "n"(I * 4096) : "memory");
  };
  auto stage_off = [&](uint32_t slice) { return (slice & uint32_t(NS - 1)) * uint32_t(kStageBytes); };

  // the loads of k-step T of slice `s` (position U in the unrolled loop, or the prologue's virtual slices): activations of
  // slice s + D into its stage, weights of k-step 4 (s + D) + T - 1
  auto issue_dma = [&](auto step, uint32_t slice) {
    constexpr int T = decltype(step)::value;
    if constexpr (O::dma(T) > 0) {
      const uint32_t k = keep(slice);
      const int8_t* src = al.base + uint64_t(slice & k) * 128;
      int8_t* st = lds + stage_off(slice);
#pragma unroll
      for (int g = 0; g < O::dma(T); ++g) {
        uint32_t off = al.off[O::first(T) + g] & k;
        __asm__ volatile("" : "+v"(off));
        __builtin_amdgcn_global_load_lds((global_void_t*)(src + off), (lds_void_t*)(st + (al.wave_u * IT + O::first(T) + g) * 1024), 16, 0, 0);
      }
    }
  };
  // (slot of the register ring, k-step inside its slice, slice): column tile j
  auto issue_w = [&](auto slot_c, auto step, uint32_t slice, int j) {
    const uint32_t k = keep(slice);
    load_w<decltype(step)::value>(wr[decltype(slot_c)::value][j], wlane & k, wsrc[j] + uint64_t(__builtin_amdgcn_readfirstlane(slice & k)) * kSliceBytes);
  };

  static_for<0, 4 * D>([&](auto v) {                   // the D slices in front of the first, as the loop would have issued them
    constexpr int V = decltype(v)::value, SD = V / 4, T = V % 4;
    issue_dma(IntC<T>{}, SD);
    if constexpr (W::kCodes) {
#pragma unroll
      for (int j = 0; j < JT; ++j) issue_w(IntC<V>{}, IntC<T>{}, SD, j);
    } else if constexpr (V > 0) {
#pragma unroll
      for (int j = 0; j < JT; ++j) issue_w(IntC<(V - 1) % R>{}, IntC<(V - 1) % 4>{}, (V - 1) / 4, j);
    }
  });
  __builtin_amdgcn_sched_barrier(0);
  {                                                    // accumulators cleared by the matrix cores under those loads
    v4i none = {0, 0, 0, 0};
#pragma unroll
    for (int i = 0; i < IT; ++i)
#pragma unroll
      for (int j = 0; j < JT; ++j) {
        __asm__ volatile("" : "+v"(none));
        acc[i][j] = Traits::mfma(none, none, Traits::zero());
      }
    __builtin_amdgcn_sched_barrier(0);
  }
  __asm__ volatile("s_waitcnt vmcnt(%0)" ::"n"(O::activations_in_flight_at_start()) : "memory");
  __asm__ volatile("s_barrier" ::: "memory");
  static_for<0, AN>([&](auto n) {                      // fragments 0 .. AN - 1 of the stream
    constexpr int X = decltype(n)::value;
    read_a(fa[0][X], a_lane[X / IT] + stage_off(0), IntC<X % IT>{});
  });
  auto dequantize = [&](auto slot_c, int j, int half, v4i& fragment) { W::dequantize(uint32_t(wr[decltype(slot_c)::value][j][half]), ws[j], half, fragment); };
  if constexpr (W::kCodes) {
#pragma unroll
    for (int j = 0; j < JT; ++j) {
      __asm__ volatile("s_waitcnt vmcnt(%1)" : "+v"(wr[0][j]) : "n"(O::first_codes_in_flight()) : "memory");
      dequantize(IntC<0>{}, j, 0, fb[0][j]);
      dequantize(IntC<0>{}, j, 1, fb[0][j]);
    }
    __builtin_amdgcn_sched_barrier(0);
  }

  // k-step T of the slice at position U of the unrolled loop (slice s)
  auto kstep = [&](auto pos, auto step, uint32_t s) {
    constexpr int U = decltype(pos)::value, T = decltype(step)::value, Q = U * 4 + T, SLOT = Q % R;
    constexpr int WANTED = W::kCodes ? (Q + 1) % R : SLOT;   // codes: the next k-step's, dequantized under this one's MFMAs
    if constexpr (T == TB) {
      // the activations of slice s + 1 have landed for every wave; the stage filled next is not one that is being read
      __asm__ volatile("s_waitcnt vmcnt(%0)" ::"n"(O::activations_in_flight(TB)) : "memory");
      __asm__ volatile("s_barrier" ::: "memory");
    }
#pragma unroll
    for (int j = 0; j < JT; ++j) __asm__ volatile("s_waitcnt vmcnt(%1)" : "+v"(wr[WANTED][j]) : "n"(O::weights_in_flight(T)) : "memory");
    const uint32_t here = stage_off(s), next = stage_off(s + 1);
    static_for<0, IT>([&](auto cc) {
      constexpr int c = decltype(cc)::value, X = Q * IT + c, SET = (X / AN) % 2, AI = X % AN;
      constexpr int X2 = T * IT + c + AN, T2 = X2 / IT;  // the fragment read now, AN further on in the stream
      __asm__ volatile("s_waitcnt lgkmcnt(%1)" : "+v"(fa[SET][AI]) : "n"(AN - 1) : "memory");
#pragma unroll
      for (int j = 0; j < JT; ++j) {
        if constexpr (W::kCodes) acc[c][j] = Traits::mfma(fb[Q % 2][j], fa[SET][AI], acc[c][j]);
        else acc[c][j] = Traits::mfma(wr[SLOT][j], fa[SET][AI], acc[c][j]);
      }
      read_a(fa[1 - SET][AI], a_lane[T2 % 4] + (T2 >= 4 ? next : here), IntC<X2 % IT>{});
      if constexpr (c == 0) issue_dma(step, s + D);
      // the registers of the k-step before this one (codes: of this one), for their next use
#pragma unroll
      for (int j = 0; j < JT; ++j)
        if ((1 + j < IT ? 1 + j : IT - 1) == c) {
          if constexpr (W::kCodes) issue_w(IntC<SLOT>{}, step, s + D, j);
          else issue_w(IntC<(Q + R - 1) % R>{}, IntC<(T + 3) % 4>{}, T == 0 ? s + D - 1 : s + D, j);
        }
      if constexpr (W::kCodes) {
#pragma unroll
        for (int u = 0; u < 2 * JT; ++u)
          if ((u * IT) / (2 * JT) == c) dequantize(IntC<WANTED>{}, u >> 1, u & 1, fb[1 - Q % 2][u >> 1]);
      }
      __builtin_amdgcn_sched_barrier(0);
    });
  };
  uint32_t s = 0;
  for (; s + D - 1 < nslices; s += D)
    static_for<0, 4 * D>([&](auto q) { kstep(IntC<decltype(q)::value / 4>{}, IntC<decltype(q)::value % 4>{}, s + decltype(q)::value / 4); });
  static_for<0, D - 1>([&](auto p) {
    constexpr int P = decltype(p)::value;
    if (s + P < nslices) static_for<0, 4>([&](auto t) { kstep(p, t, s + P); });
  });
  __builtin_amdgcn_s_waitcnt(0x0070);                  // the surplus loads and fragment reads have landed: their
#pragma unroll                                         // registers stay allocated up to here
  for (int i = 0; i < AN; ++i) __asm__ volatile("s_waitcnt lgkmcnt(0)" ::"v"(fa[0][i]), "v"(fa[1][i]) : "memory");
#pragma unroll
  for (int q = 0; q < R; ++q)
#pragma unroll
    for (int j = 0; j < JT; ++j) __asm__ volatile("s_waitcnt vmcnt(0)" ::"v"(wr[q][j]) : "memory");
  __syncthreads();
  // (a tile whose accumulators fill half of the register file is never split: the partial sums would not fit beside them)
  if constexpr (IT * JT < 16) {
    if (part.splits > 1 && !meet<typename Traits::Scalar, (IT * JT < 2 || IT * JT >= 8 ? 4 : 8)>(acc, part, lds, slot)) return;
  }
  write_tile<JT, 4, 4>(acc, epi, y, M, N, part.m0, part.n0, lds, slot, true);
}

// ---- 256 x 384 tiles: four waves of 256 x 96 -------------------------------------------------------------
// The widest tile the register file holds: 384 accumulator registers per lane.  Every wave owns all 256 rows of 96
// columns, so each weight fragment is loaded by ONE wave (the 2 x 2 waves above load each twice) and a workgroup
// moves 80 KiB per slice for 384 MFMAs where the 256 x 256 tile moves 96 KiB for 256: on zero operands the loop runs at
// 95 % of its MFMA time.  What it takes:
//   * With one wave per SIMD the compiler gives the matrix instructions accumulation registers only, 256 per lane.
//     The third column tile's accumulators therefore live in ordinary vector registers, through MFMAs written as
//     instructions (the compiler does not see inside: s_nops in front of the epilogue let the matrix cores finish).
//   * That leaves about 120 vector registers for everything else.  Activation fragments are read HALF a k-step
//     ahead (two sets of four: chunks 0..3 of a k-step read its row tiles 4..7, chunks 4..7 row tiles 0..3 of the
//     next k-step); the weights of a k-step (3 x 16 bytes per lane) sit in a ring of four k-steps and are asked for
//     again as soon as the k-step is over, three k-steps before their next use.
//   * Memory instructions are issued in a fixed order per k-step (chunk 0: activations, chunks 1..3: weights,
//     chunk 4: activations) and waited for by count: when a k-step starts, eleven have been issued since its weights
//     were asked for; the activations of slice s+1 were asked for during slice s-1 and have landed by the same count
//     in front of k-step 3, where the workgroup meets.
// int8 at M = 2048, K = 4096, N = 11008 (232 tiles, one round) 77.5 us; 128 x 384 tiles there take 80.5, 256 x 256 ones 89.6.
constexpr int kWideBN = 384, kStageBytes = 256 * 128;  // columns; one slice of the activation panel

template <class Traits, class W, class Epilogue>
__device__ __forceinline__ void run_wide(const int8_t* __restrict__ a, int64_t a_row_bytes, const W& weights,
                                         int64_t ntiles, Epilogue& epi, uint16_t* __restrict__ y, int64_t M, int64_t N,
                                         int64_t slices, int64_t m0, int64_t n0, int8_t* lds) {
  constexpr int IT = 8, JT = 3, AN = 4, kG = 8;
  constexpr int JA = 2;                                // column tiles whose accumulators the compiler places
  constexpr int kFly = 11;                             // memory instructions issued since a k-step's weights were asked for
  const int lane = threadIdx.x & 63;
  const int slot = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);   // = the wave's column: 1 x 4 waves
  const int frow = lane & 31, fhalf = lane >> 5;

  typename Traits::Acc acc[IT][JT];
  const uint32_t nslices = uint32_t(slices), last = nslices - 1;
  DmaLoaderT<kG> al;
  al.init(a, M, a_row_bytes, m0);
  v4i fa[2][AN];
  typename W::Raw wr[4][JT];
  v4i fb[2][JT];                                       // codes: the fragments of this k-step and the next
  typename W::Scale ws[JT];
  const int8_t* wsrc[JT];                              // slice 0 of each column tile (uniform)
  uint32_t wlane = uint32_t(lane) * uint32_t(sizeof(typename W::Raw));
#pragma unroll
  for (int j = 0; j < JT; ++j) {
    int64_t tile = n0 / 32 + slot * JT + j;
    tile = tile < ntiles ? tile : ntiles - 1;          // tiles past N: some valid data, never stored
    wsrc[j] = weights.frag + tile * slices * (4 * W::kStepBytes);
    if constexpr (W::kCodes) ws[j] = W::scale_of(weights.scale, n0 + (slot * JT + j) * 32 + frow, N);
  }
  auto fetch_w = [&](auto tt, typename W::Raw& dst, int j, uint32_t slice) {
    load_w<decltype(tt)::value>(dst, wlane, wsrc[j] + uint64_t(slice) * (4 * W::kStepBytes));
  };
  const uint32_t lds_base = uint32_t(uintptr_t((lds_void_t*)lds));
  uint32_t a_lane[4];
#pragma unroll
  for (int p = 0; p < 4; ++p) a_lane[p] = lds_base + uint32_t(lds_off(frow, 2 * p + fhalf));
  auto read_a = [&](v4i& dst, uint32_t addr, auto tile) {
    constexpr int I = decltype(tile)::value;
    __asm__ volatile("ds_read_b128 %0, %1 offset:%2" : "=v"(dst) : "v"(addr), "n"(I * 4096) : "memory");
  };
  // the reads form one stream, four chunks ahead of their use: three younger ones may be outstanding
  auto landed_a = [&](v4i& frag) { __asm__ volatile("s_waitcnt lgkmcnt(3)" : "+v"(frag)::"memory"); };
  auto stage_off = [&](uint32_t slice) { return uint32_t(slice & 3) * uint32_t(kStageBytes); };
  auto stage = [&](uint32_t slice) { return lds + stage_off(slice); };
  auto at_most_last = [&](uint32_t slice) { return slice - ((uint32_t(last - slice) >> 31) * (slice - last)); };  // scalar min

  // slice 0 and its weights for k-steps 0..2 (k-step 3's are asked for in k-step 0, like every slice's; codes: all four), then slice 1
  const uint32_t one = at_most_last(1);
#pragma unroll
  for (int g = 0; g < kG; ++g) al.dma_at(al.slice_base(0), stage(0), g);
  static_for<0, W::kCodes ? 4 : 3>([&](auto t) {
    constexpr int T = decltype(t)::value;
#pragma unroll
    for (int j = 0; j < JT; ++j) fetch_w(t, wr[T][j], j, 0);
  });
#pragma unroll
  for (int g = 0; g < kG; ++g) al.dma_at(al.slice_base(one), stage(1), g);
  __builtin_amdgcn_sched_barrier(0);
  {                                                    // accumulators cleared by the matrix cores under those loads
    v4i none = {0, 0, 0, 0};
#pragma unroll
    for (int i = 0; i < IT; ++i)
#pragma unroll
      for (int j = 0; j < JT; ++j) {
        __asm__ volatile("" : "+v"(none));
        if (j < JA) acc[i][j] = Traits::mfma(none, none, Traits::zero());
        else Traits::clear_vgpr(none, none, acc[i][j]);
      }
    __builtin_amdgcn_sched_barrier(0);
  }
#pragma unroll
  for (int t = 0; t < (W::kCodes ? 4 : 3); ++t) __asm__ volatile("s_waitcnt vmcnt(0)" : "+v"(wr[t][0]), "+v"(wr[t][1]), "+v"(wr[t][2])::"memory");
  drain_and_barrier();
  static_for<0, AN>([&](auto i) { read_a(fa[0][decltype(i)::value], a_lane[0] + stage_off(0), i); });
  auto dequantize = [&](int t, int j, int half) { W::dequantize(uint32_t(wr[t][j][half]), ws[j], half, fb[t & 1][j]); };
  if constexpr (W::kCodes) {
#pragma unroll
    for (int u = 0; u < 2 * JT; ++u) dequantize(0, u >> 1, u & 1);
    __builtin_amdgcn_sched_barrier(0);
  }

  // k-step T of slice s0 (the next slice: s1): eight fenced chunks; chunk c multiplies row tile c by the three weight
  // fragments of the k-step.  ca: LDS offset of the stage this k-step reads, ra: of the stage the next k-step reads.
  auto kstep = [&](auto step, uint32_t ca, uint32_t ra, uint32_t s0, uint32_t s1, const int8_t* src, int8_t* nd) {
    constexpr int T = decltype(step)::value;
    const uint32_t raddr = a_lane[(T + 1) & 3] + ra, caddr = a_lane[T] + ca;
    constexpr int WANTED = W::kCodes ? (T + 1) & 3 : T;  // codes: the next k-step's, dequantized under this one's MFMAs
    __asm__ volatile("s_waitcnt vmcnt(%3)" : "+v"(wr[WANTED][0]), "+v"(wr[WANTED][1]), "+v"(wr[WANTED][2]) : "n"(kFly) : "memory");
    static_for<0, IT>([&](auto cc) {
      constexpr int c = decltype(cc)::value;
      constexpr int ASET = c / AN, AI = c % AN;
      landed_a(fa[ASET][AI]);
#pragma unroll
      for (int j = 0; j < JT; ++j) {
        v4i w;
        if constexpr (W::kCodes) w = fb[T & 1][j];
        else w = wr[T][j];
        if (j < JA) acc[c][j] = Traits::mfma(w, fa[ASET][AI], acc[c][j]);
        else Traits::mfma_vgpr(w, fa[ASET][AI], acc[c][j]);
      }
      if constexpr (c < AN) read_a(fa[1][c], caddr, IntC<c + AN>{});           // row tile c + 4 of this k-step
      else read_a(fa[0][c - AN], raddr, IntC<c - AN>{});                       // row tile c - 4 of the next
      if constexpr (c == 0) al.dma_at(src, nd, 2 * T);
      if constexpr (c == 4) al.dma_at(src, nd, 2 * T + 1);
      if constexpr (c >= 1 && c <= 3) {                // the registers of the k-step before this one (codes: of this one), for their next use
        if constexpr (W::kCodes) fetch_w(step, wr[T][c - 1], c - 1, s1);
        else if constexpr (T == 0) fetch_w(IntC<3>{}, wr[3][c - 1], c - 1, s0);
        else fetch_w(IntC<T - 1>{}, wr[T - 1][c - 1], c - 1, s1);
      }
      if constexpr (W::kCodes && c < 2 * JT) dequantize(WANTED, c >> 1, c & 1);
      __builtin_amdgcn_sched_barrier(0);
    });
  };
  for (uint32_t s = 0; s < nslices; ++s) {
    const uint32_t pa = stage_off(s);
    const uint32_t s1 = at_most_last(s + 1), s2 = at_most_last(s + 2);
    const int8_t* src = al.slice_base(s2);             // the slice fetched during this one (past the end: the last again,
    int8_t* nd = stage(s + 2);                         //  into a stage nobody reads)
    kstep(IntC<0>{}, pa, pa, s, s1, src, nd);
    kstep(IntC<1>{}, pa, pa, s, s1, src, nd);
    kstep(IntC<2>{}, pa, pa, s, s1, src, nd);
    // the activations of slice s+1 have landed (fifteen memory instructions were issued since the last of them); the
    // fragment reads in flight belong to stages that are not written before the next barrier but one
    __asm__ volatile("s_waitcnt vmcnt(%0)" ::"n"(kFly) : "memory");
    __asm__ volatile("s_barrier" ::: "memory");
    kstep(IntC<3>{}, pa, stage_off(s + 1), s, s1, src, nd);
  }
  __builtin_amdgcn_s_waitcnt(0x0070);                  // the surplus loads and fragment reads have landed: their
#pragma unroll                                         // registers stay allocated up to here
  for (int i = 0; i < AN; ++i) __asm__ volatile("s_waitcnt lgkmcnt(0)" ::"v"(fa[0][i]), "v"(fa[1][i]) : "memory");
#pragma unroll
  for (int t = 0; t < 4; ++t) __asm__ volatile("s_waitcnt vmcnt(0)" ::"v"(wr[t][0]), "v"(wr[t][1]), "v"(wr[t][2]) : "memory");
  __asm__ volatile("s_nop 15\n\ts_nop 15" ::: "memory");   // the matrix cores are done with the accumulators in vector registers

  write_tile<JT, 4, 4>(acc, epi, y, M, N, m0, n0, lds, slot, true);
}


// The K split of a launch, by value among the kernel's arguments (clusters.cpp: FragSplit).
struct Split {
  uint32_t splits, per;                                // parts, and slices in each but the last, which has the rest (at least one)
  f32x4* partial;                                      // splits > 1: BM * BN / 4 pieces per part, the parts of a tile together
  uint32_t* tickets;                                   // splits > 1: a zeroed word per tile
};

// Which part of the problem workgroup `id` of `nblocks` takes: (split, tile) items dealt evenly to the eight XCDs in
// split-major order, so that an XCD works on as few K ranges as possible (with eight splits on one: every operand byte is
// then fetched into one L2 only).  group: row tiles that keep a panel together (tile_at).
// (M, N and K are below 2^31: 32 bits throughout.  This code is in front of the launch's first load; with 64-bit divisions
// it was half a microsecond.)
template <int BM, int BN>
__device__ __forceinline__ bool part_of(uint32_t id, uint32_t nblocks, int64_t M, int64_t N, uint32_t slices, const Split& sp, Part& part,
                                        uint32_t group = ~0u) {
  const uint32_t tiles_m = (uint32_t(M) + (BM - 1)) / BM, panels = (uint32_t(N) + (BN - 1)) / BN, tiles = tiles_m * panels;
  uint32_t t = (id & 7) * (nblocks >> 3) + (id >> 3);
  if (t >= tiles * sp.splits) return false;
  part.slice0 = 0;
  part.nslices = slices;
  part.splits = sp.splits;
  part.split = 0;
  if (sp.splits > 1) {
    part.split = t / tiles;
    t -= part.split * tiles;
    part.slice0 = part.split * sp.per;
    part.nslices = part.split + 1 < sp.splits ? sp.per : slices - part.slice0;
    part.ticket = sp.tickets + t;
    part.partial = sp.partial + uint64_t(t) * sp.splits * (BM * BN / 4);
  }
  int64_t tile_m, panel;
  tile_at(t, tiles_m, panels, group, tile_m, panel);
  part.m0 = tile_m * BM;
  part.n0 = panel * BN;
  return true;
}

}  // namespace gemm_frag
