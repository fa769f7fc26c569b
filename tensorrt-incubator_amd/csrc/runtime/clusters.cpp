// Part 2 of the C ABI: one entry point per kernel cluster.  Each validates its
// operands on the host (so that no launch can address memory outside them), picks
// the kernel variant and launch shape for gfx950, builds the argument array in the
// reference's kernelParams convention and launches from the built-in module.
// This is the hand-written counterpart of the get-function + launch pairs the
// reference compiler emits for its generated kernels
// (mlir-tensorrt/compiler/lib/Passes/1_Core/KernelToCUDA/KernelToCUDA.cpp:151-186;
//  mlir-tensorrt/compiler/lib/Passes/2_Host/HostToExecutor/CUDAToExecutor/CUDAToExecutor.cpp:355-413).
#include "runtime_internal.hpp"
#include "../kernels/nvfp4_index.hpp"
#include "../kernels/read_twice.hpp"

#include <algorithm>
#include <atomic>
#include <cstdlib>

using namespace mtrt_rt;

namespace {

constexpr int kTile = 16;           // elements per lane per trip in qdq.hip
constexpr uint32_t kBlock = 256;
constexpr uint32_t kMaxGrid = 1u << 20;
// A launch has fewer than 2^32 work items.  kLoopGrid: most workgroups (of up to 512 lanes) of kernels that loop over their tiles.
constexpr int64_t kLoopGrid = int64_t(1) << 22;
constexpr bool launchable(int64_t grid, int64_t block) { return grid * block < (int64_t(1) << 32); }
// The one-wave-per-row kernels (layernorm / softmax `_v*`) map rows to waves from the workgroup index and do
// not loop, so their grid must cover every row: ceil(rows / 4) workgroups, which blocks_for() caps at
// kMaxGrid.  Tensors with more rows take the `_any` kernels, which loop over rows.
constexpr int64_t kMaxRowsPerWaveKernels = int64_t(kMaxGrid) * (kBlock / 64);

// ---- launch-time estimates behind the GEMM dispatch ------------------------------------------------------------
// Every choice between two GEMM kernels compares two estimates of the launch time in microseconds.  All constants
// live here, each with the measurement that set it (one MI355X, 256 compute units, times from HIP events over
// rotating operands; `rounds` = ceil(tiles / compute units), `row bytes` = K * element size).  They are fits to a
// few points, good to about 10 %: near a crossover either kernel is within that of the other, so a box whose power
// state moves the times by a few per cent picks differently without losing more than that.
namespace tuning {
// Tile loop against [N,K] operands (both panels through LDS), per round of 256 x 256 tiles: a fixed part plus the
// K loop.  int8: M = 16, K = 4096, N = 11008 32.7 us; M = 1, K = N = 4096 27.6 us; M = 32, K = N = 8192 57.1 us
// (8 + 0.006 * 4096 = 32.6, 8 + 0.006 * 8192 = 57.2).
constexpr double kTileFixedUs = 8.0, kTileUsPerRowByte = 0.006;
// Wave-private kernels that read the weights once (gemm_core::rows32), up to 64 rows: a fixed part plus the weight
// bytes at the rate the kernel streams them.  [N,K] int8 weights 3.4 TB/s (M = 16, K = 4096, N = 11008 13.0 us;
// M = 32, K = N = 8192 18.2 us); f16 / bf16 / f32 [N,K] weights 4.0 TB/s (dense f16 M = 16, K = 4096, N = 11008 23.4 us).
constexpr double kRowsFixedUs = 3.0, kRowsBytesPerUs = 3.4e6, kRowsWideBytesPerUs = 4.0e6;
// The same kernels with four row tiles (65 to 128 rows): one workgroup per compute unit at a time, so rounds of 32-column
// tiles, each the length of its K loop: 3.7 ns per row byte (int8 M = 128, K = N = 4096 18.4 us, K = N = 8192 30.7 us).
constexpr double kRows128FixedUs = 3.0, kRows128UsPerRowByte = 0.0037;
// Float products of few rows read weights above these bytes past the caches (us, past and through, f32: M = 1, 180 MB 26.7, 28.9; M = 3, 53 MB
// 11.5, 12.0; M = 1, 29 MB 7.7, 6.8; bf16: 90 MB 16.2, 17.0; 67 MB 12.4, 13.4; 33 MB 9.8, 8.4).
constexpr int64_t kWeightsPastBytes = int64_t(48) << 20;
// int8 and int4 weights of few rows are read past the caches: a decode step comes back to a layer's weights when all other layers' have been through, so
// that they lie in memory, and from there they take longer through the caches.  (us, past and through, weights of three sets in turn, which the Infinity
// Cache holds, and from memory: W4A16 (1, 4096, 11008) 6.8, 7.4; 7.7, 7.8; (8, 4096, 4096) 3.9, 3.9; 4.8, 5.0; (16, 4096, 11008) 8.6, 8.2; 9.1, 9.3; (32, 8192, 8192)
// 13.5, 11.5; 13.9, 14.5; W8A8 (1, 4096, 8192) 7.4, 7.5; 7.9, 8.7; (16, 4096, 6144) 6.9, 6.5; 7.5, 7.8; (16, 4096, 11008) 11.8, 10.4; 12.6, 12.8.)
// But for W8A8, from kThroughFromFewTiles or kThroughFrom to kThroughUpTo, where a workgroup's own rate is the bound, which from the Infinity Cache is 57 to 67
// GB/s past the caches and 100 through them: with at most half a tile of 32 columns to a unit, and with 17 to 32 rows, which come in beside the weights.  Past the
// caches these take longer there than eight waves to a tile did, through them they do in neither place.  The eight waves, past and through: (16, 8192, 2048) 7.7,
// 8.7, 6.8; 10.9, 9.7, 9.9; (8, 11008, 4096) 9.8, 11.6, 9.1; 14.2, 12.0, 12.6; (16, 14336, 4096) 12.2, 16.2, 11.6; 18.4, 16.7, 17.3; (4, 2688, 4096) 4.7, 4.2, 3.9; 6.3,
// 5.1, 5.3; (24, 4096, 2048) 5.6, 6.7, 5.4; 8.1, 7.2, 7.3; (32, 14336, 1024) 12.2, 15.9, 11.8; 19.4, 18.7, 18.8; (32, 6144, 9216) 16.0, 17.1, 13.8; 21.9, 17.9, 17.8; (32,
// 8192, 8192) 14.1, 15.6, 14.3; 17.5, 16.3, 17.4.  Smaller (8, 14336, 512) 9.1, 7.2, 7.2; 14.3, 12.4, 12.8; (32, 1152, 9216) 6.7, 5.4, 4.7; 9.0, 6.5, 6.7; larger (32, 12288, 8192)
// 21.9, 20.5, 21.3; 22.8, 21.2, 21.9.
constexpr int64_t kThroughFromFewTiles = int64_t(8) << 20, kThroughFrom = int64_t(16) << 20, kThroughUpTo = int64_t(64) << 20;
// f32 products of few rows on the vector units: K from which four waves share it; the fewest weights (below, the tiles take 3 to 4 us
// too); what several groups of rows read through the L2s.
constexpr int64_t kDotOwnColumnsBelow = 1536, kDotMinWeights = 16384;
constexpr double kDotGroupBytesPerUs = 7.5e6;
// Any-K kernel: rounds of 128 x 128 tiles, each a walk down K in steps of 128 bytes a row, against 32 x 32 tiles, two workgroups of four
// waves to a compute unit (f32, up to one workgroup a unit: eight waves).  Fitted to 34 products, M 1 ... 2000, K 6 ... 12287, N 7 ... 11000,
// f32 and f16; the faster form is taken in each of them.
constexpr double kEdgeFixedUs = 4.0, kEdgeF32StepUs = 2.45, kEdge16StepUs = 1.2;
// f32 products of whole slices, us to a slice of 128 bytes of K.  By rounds of 32-column tiles with all rows (up to 32, 64 and 128 of them): fitted to 27
// products, M 16 ... 128, K 256 ... 12288, N 256 ... 16384, of up to two rounds (what a round costs beside its slices is left out).
constexpr double kF32FixedUs = 3.0, kF32Rows32StepUs = 0.18, kF32Rows64StepUs = 0.36, kF32Rows128StepUs = 0.68, kF32RowsRounds = 2;
// By 32 x 32 tiles: one or none to a compute unit, and every two to a unit; by 128 x 128 tiles, the rest up to one to a unit and every two to a unit;
// by rounds of 256 x 128 tiles.  Fitted to 57 products, M 33 ... 65536, K 32 ... 11008, N 96 ... 65536; the form with the least estimate is the
// fastest in each, or within 2 percent of it.
constexpr double kF32FewTilesStepUs = 0.2, kF32TilesUs = 1.8, kF32TilesStepUs = 0.32;
// ... K split over workgroups: fixed and meeting, then by rounds of one workgroup to a unit (measured beside the kernels)
constexpr double kF32SplitUs = 4.0, kF32SplitRoundUs = 3.0, kF32SplitStepUs = 0.18, kF32SplitPromise = 0.95;
constexpr double kF32T128OneUs = 10.0, kF32T128OneStepUs = 2.36, kF32T128TwoUs = 14.0, kF32T128TwoStepUs = 4.12;
constexpr double kF32T256RoundUs = 30.0, kF32T256StepUs = 3.68;
constexpr double kEdgeSmallFixedUs = 3.0, kEdgeSmallFewStepUs = 0.2, kEdgeSmallStepUs = 0.5;
// W4A16 tile choice: a full round of 256 x 256 tiles takes 3.25 times a full round of 128 x 128 tiles (for four times
// the work), and a last round filled to a fraction f of the units takes 0.56 + 0.44 f^2 of a full one (fewer units
// share the power budget).  Fitted over M = 48 ... 4096 at (K, N) = (4096, 4096), (4096, 11008), (11008, 4096),
// (8192, 8192), (5120, 13824), (4096, 14336), (8192, 28672), (4096, 2048), 16 to 256 tiles in the last round; where
// the rule changed the choice: K = N = 4096, M = 2048 83.6 -> 77.1 us; N = 11008, M = 1536 193.2 -> 175.0 us.
constexpr double kW4BigRoundPerSmallRound = 3.25, kW4PartialRoundBase = 0.56, kW4PartialRoundSlope = 0.44;
// ... and a round of 256 x 384 tiles takes 1.5 x 0.95 of a round of 256 x 256 tiles (K = 4096, N = 11008, the benchmark's
// data, old and new in one process: M = 4096, 3 rounds against 2, 298.4 -> 286.8 us; M = 8192 600 -> 571; M = 2048, two
// rounds against one, 181 -> 145).
constexpr double kW4WideRoundPerBigRound = 1.5 * 0.95;
// ... and a round of 128 x 256 tiles 1.9 rounds of 128 x 128 tiles.
constexpr double kW4Mid256RoundPerSmallRound = 1.9;
// W4A16 tiles in time: n = tiles * splits workgroups of s = slices / splits slices of 64 k each, in L = ceil(n / units)
// rounds the last of which is filled to f:
//   fixed + (e + c s) (L - 1 + p + (1 - p) f^2) + (splits > 1 ? meet + meet_each * splits : 0)   us
// (a launch that leaves units idle is shorter, more so for the large tiles: the clock is power's).  Fitted to 17000
// launches of 621 log-uniform shapes, M 33 ... 4096, K 256 ... 14336, N 64 ... 16384, 1 to 12 splits.
// That is a full chip's law.  However few tiles there are, one of them takes least + least_slice * s, which a launch of few
// large tiles runs into (fitted to the launches of at most half as many unsplit tiles as units of 380 shapes of the same range).
// With it, M, K, N, us: (92, 640, 6336) t128x128 7.2, t32x128 5.2; (805, 1536, 768) 11.3, 8.4; (91, 1152, 8896) 9.4, 7.1; (748, 64, 127) 5.5, 3.3; (304, 704,
// 238) 8.1, 5.6; of 575 products of K up to 512, or 1024 by at most 256 columns, none slower and the geometric mean 0.73 of what it is without.
// t64x128's row was fitted to a kernel that is no more.  On 2779 launches of the present one its estimates are 1.3 % long on average and 9 % off
// (r.m.s.); a row fitted to those is 7 % off, and the choice with it 1.8 % longer than the fastest one, with this one 1.6 % (985 products of 33 to 4096
// rows, those 575 among them; 1.32 times as long at worst, (695, 128, 2098) 6.1 and 4.6).
struct W4Tile {
  const char *suffix;                                  // of the kernel's name
  int rows, columns, threads;
  bool splits;                                         // whether its K may be split
  double fixed, e, c, p, meet, meet_each, least, least_slice;
};
constexpr W4Tile kW4Tiles[] = {
    {"t32x128", 32, 128, 256, true, 2.64, 0.89, 0.197, 1.0, 1.59, 0.334, 0.0, 0.0},
    {"t64x128", 64, 128, 512, true, 0.99, 3.35, 0.252, 0.83, 2.59, 0.46, 0.0, 0.0},
    {"t64x256", 64, 256, 256, true, 0.0, 4.38, 0.497, 0.79, 4.02, 0.645, 3.39, 0.422},
    {"t128x128", 128, 128, 512, true, 0.0, 5.76, 0.523, 0.474, 3.54, 0.725, 4.3, 0.282},
    {"t128x256", 128, 256, 256, true, 0.0, 5.98, 1.046, 0.467, 5.8, 1.19, 4.16, 0.55},
    {"t256x256", 256, 256, 256, false, 0.0, 7.3, 1.589, 0.615, 0.0, 0.0, 5.99, 1.0},
    {"t256x384", 256, 384, 256, false, 0.0, 8.46, 2.637, 0.525, 0.0, 0.0, 7.59, 1.415},
};
// 32-row tiles by two and four sets of four waves (run_sets in gemm_w4a16.hip) take shorter slices and a later start: from 17 slices to a
// workgroup, and four sets from 24 where each workgroup has a compute unit.  us, one, two and four sets, by slices, unsplit: up to 8 two sets take
// 1.16 times as long as one, 13 to 16 as long, 21 to 28 0.955, 41 to 80 0.884 (and four 0.81), more 0.853 (0.72).  Fitted like the tiles above to
// 555 launches of 300 shapes, M 33 ... 2048; a form takes over the tile's own plan, and another tile's where it promises a tenth: over those
// shapes 2.6 % less time on average, (75, 7680, 10368) 36.9 -> 26.4, (147, 6016, 5888) 28.0 -> 21.3, (62, 3072, 8640) 14.5 -> 11.6.
constexpr W4Tile kW4Sets[] = {
    {"t32x128x2", 32, 128, 512, true, 4.175, 0.137, 0.207, 0.593, 1.573, 0.371, 3.056, 0.183},
    {"t32x128x4", 32, 128, 1024, true, 0.306, 5.059, 0.178, 0.775, 1.789, 0.370, 4.241, 0.139},
};
constexpr int64_t kW4TwoSetsFrom = 17, kW4FourSetsFrom = 24, kW4FourSetsSameSplitFrom = 32;
constexpr double kW4SetsPromise = 0.9;
// The tile by rounds (above) is the better founded choice where the estimates are close: another tile or a split has to
// promise a tenth (over those 380 shapes none is slower so than without the bound; with no such promise the worst is 1.15 times as long).
constexpr double kW4Promise = 0.9;
// Tiles on fragment-order weights (gemm_frag.hpp).  A launch of `tiles * splits` workgroups, L = ceil of that over the
// compute units, each running s = slices / splits slices of 128 bytes of K, is estimated as
//   max(first + first_slice * s, L * (next + next_slice * s)) + (splits > 1 ? meet + meet_each * splits : 0)   us.
// Fitted to 8500 launches (int8 and f16, 220 log-uniform shapes each: M 17 ... 4096, K 256 ... 14336, N 64 ... 16384, every
// tile, 1 to 8 splits); the tile and split the estimate takes are within 1.1 % of the fastest ones in the geometric mean
// and within 22 % at worst.  int8 and the 16-bit types move the same bytes per slice and share the constants.
struct FragTile {
  const char *suffix;                                  // of the kernel's name
  int rows, columns;
  bool splits;                                         // whether its K may be split
  double first, first_slice, next, next_slice, meet, meet_each;
};
constexpr FragTile kFragTiles[] = {
    {"t32x128", 32, 128, true, 3.16, 0.144, 1.86, 0.206, 1.65, 0.456},
    {"t64x128", 64, 128, true, 3.99, 0.128, 2.82, 0.243, 2.48, 0.70},
    {"t128x128", 128, 128, true, 4.54, 0.20, 3.61, 0.359, 3.8, 1.03},
    {"t128x256", 128, 256, true, 6.9, 0.127, 6.13, 0.51, 5.14, 1.55},
    {"t128x384", 128, 384, true, 2.82, 0.78, 8.22, 0.724, 6.9, 2.2},
    {"t256x256", 256, 256, false, 11.0, 0.25, 8.63, 0.912, 0.0, 0.0},
    {"t256x384", 256, 384, false, 12.3, 0.764, 9.99, 1.346, 0.0, 0.0},
};
// Two 128 x 256 tiles share a unit: L > 1 of them, each with all of K, take `first` + L * (each + slice * s) us.  Fitted to 70 products of 200 to
// 4096 rows beside the others' estimates: (3043, 768, 13632) 49.3 -> 42.2, (2006, 896, 14784) 38.3 -> 32.2.  So from one slice on: over 330 products
// of one to eight slices the choice is 2.2 % longer than the fastest one, 3.7 % with the pairs from five slices on only; where that
// changes it, int8 (940, 512, 12416) 14.7 -> 11.3, f16 (3715, 128, 8839) 32.3 -> 25.2; worst (1399, 256, 12352) 15.1 -> 16.2.
constexpr double kFragPairsUs = 1.24, kFragPairsEachUs = 2.68, kFragPairsSliceUs = 0.515;
// The wave-private kernels up to 32 and 64 rows on the same weights (gemm_core::rows32): L = ceil of their 32-column tiles
// over the compute units; int8 M = 16, K = N = 4096 5.7 us, (32, 3968, 11328) 13.2; M = 64, K = N = 4096 8.5, (54, 12032, 8682) 32.6.
constexpr double kFragRows32Us = 2.0, kFragRows32TileUs = 1.2, kFragRows32SliceUs = 0.08, kFragRows32LaterSliceUs = 0.13;
constexpr double kFragRows64Us = 1.6, kFragRows64TileUs = 1.9, kFragRows64SliceUs = 0.165;
} // namespace tuning

// gemm_frag::Split, the kernels' argument of this layout.
struct FragSplit {
  uint32_t splits = 1, per = 0;
  void *partial = nullptr;
  uint32_t *tickets = nullptr;
};
// `splits` parts of equal length; fewer where the last ones would have nothing left.
FragSplit split_of(int64_t slices, int splits) {
  const int64_t per = (slices + splits - 1) / splits;
  return {uint32_t((slices + per - 1) / per), uint32_t(per), nullptr, nullptr};
}

// A plan follows from the extents alone and costs 0.4 us; a call asks for it two or three times (its workspace, then the launch), so
// each thread keeps the last one of each kind.
template <class Plan>
class LastPlan {
public:
  template <class Make>
  const Plan &of(int64_t M, int64_t N, int64_t K, int64_t units, bool may_split, Make &&make) {
    const int64_t asked[] = {M, N, K, units, may_split};
    if (!std::equal(asked, asked + 5, key)) {
      plan = make();
      std::copy(asked, asked + 5, key);
    }
    return plan;
  }

private:
  int64_t key[5] = {-1, -1, -1, -1, -1};               // (extents are not negative)
  Plan plan;
};

// The tile and the K split of a GEMM on fragment-order weights (see tuning::kFragTiles).
struct FragPlan {
  const tuning::FragTile *tile = nullptr;
  int64_t tiles = 0;
  FragSplit split;
  double us = 0.0;
  uint32_t grid() const { return uint32_t(8 * ((tiles * int64_t(split.splits) + 7) / 8)); }
  int64_t workspace() const { return split.splits > 1 ? tiles * int64_t(split.splits) * tile->rows * tile->columns * 4 : 0; }
};
FragPlan make_frag_plan(int64_t M, int64_t N, int64_t slices, int64_t units, bool may_split) {
  static constexpr int kSplits[] = {1, 2, 3, 4, 6, 8};
  FragPlan best;
  for (const tuning::FragTile &t : tuning::kFragTiles) {
    const int64_t tiles = ((M + t.rows - 1) / t.rows) * ((N + t.columns - 1) / t.columns);
    if (tiles > int64_t(kMaxGrid) * 1024 - 8)
      continue;
    for (int splits : kSplits) {
      // a part of at least two slices, a ticket for every split tile, and no more workgroups than two rounds hold
      if (splits > 1 && (!may_split || !t.splits || slices < 2 * splits || tiles > int64_t(kTickets) || tiles * splits > 2 * units))
        break;
      const FragSplit split = split_of(slices, splits);
      const double s = double(split.per), rounds = double((tiles * int64_t(split.splits) + units - 1) / units);
      const bool pairs = splits == 1 && t.rows == 128 && t.columns == 256 && rounds > 1.0;
      const double full = pairs ? tuning::kFragPairsUs + rounds * (tuning::kFragPairsEachUs + tuning::kFragPairsSliceUs * s)
                                : rounds * (t.next + t.next_slice * s);
      const double us = std::max(t.first + t.first_slice * s, full) +
                        (split.splits > 1 ? t.meet + t.meet_each * split.splits : 0.0);
      if (!best.tile || us < best.us)
        best = {&t, tiles, split, us};
    }
  }
  return best;
}
FragPlan frag_plan(int64_t M, int64_t N, int64_t slices, int64_t units, bool may_split) {
  static thread_local LastPlan<FragPlan> last;
  return last.of(M, N, slices, units, may_split, [&] { return make_frag_plan(M, N, slices, units, may_split); });
}
double frag_rows_us(int64_t M, int64_t N, int64_t slices, int64_t units) {
  using namespace tuning;
  const double rounds = double(((N + 31) / 32 + units - 1) / units), s = double(slices);
  if (M <= 32)
    return kFragRows32Us + rounds * (kFragRows32TileUs + s * (rounds > 1.0 ? kFragRows32LaterSliceUs : kFragRows32SliceUs));
  return kFragRows64Us + rounds * (kFragRows64TileUs + s * kFragRows64SliceUs);
}


// Tile and K split of a W4A16 launch of more than 32 rows.
struct W4Plan {
  const tuning::W4Tile *tile = nullptr;
  int64_t tiles = 0;
  FragSplit split;
  double us = 0.0;
  bool narrow = false;                                 // 128 x 64 tiles: matrices of at most 64 columns, where 128 x 128 would run
  uint32_t grid() const { return uint32_t(8 * ((tiles * int64_t(split.splits) + 7) / 8)); }
  int64_t workspace() const { return split.splits > 1 ? tiles * int64_t(split.splits) * tile->rows * tile->columns * 4 : 0; }
};
W4Plan make_w4_plan(int64_t M, int64_t K, int64_t N, int64_t units, bool may_split) {
  using namespace tuning;
  static constexpr int kSplits[] = {1, 2, 3, 4, 6, 8};
  const int64_t slices = K / 64;
  auto tiles_of = [&](const W4Tile &t) { return ((M + t.rows - 1) / t.rows) * ((N + t.columns - 1) / t.columns); };
  auto plan_of = [&](const W4Tile &t, int splits) {
    W4Plan p;
    p.tile = &t;
    p.tiles = tiles_of(t);
    p.split = split_of(slices, splits);
    const int64_t n = p.tiles * p.split.splits, full = (n - 1) / units;
    const double s = double(p.split.per), f = double(n - full * units) / double(units);
    p.us = std::max(t.fixed + (t.e + t.c * s) * (double(full) + t.p + (1.0 - t.p) * f * f), t.least + t.least_slice * s) +
           (p.split.splits > 1 ? t.meet + t.meet_each * p.split.splits : 0.0);
    return p;
  };
  auto fits = [](int64_t tiles) { return tiles <= int64_t(kMaxGrid) * 1024 - 8; };
  // 128- and 256-row tiles by rounds
  auto rounds = [units](int64_t tiles) {
    const double f = double(tiles % units) / double(units);
    return double(tiles / units) + (tiles % units ? kW4PartialRoundBase + kW4PartialRoundSlope * f * f : 0.0);
  };
  const W4Tile &t128 = kW4Tiles[3], &t256w = kW4Tiles[4], &big = kW4Tiles[5], &wide = kW4Tiles[6];
  const double cost128 = rounds(tiles_of(t128)), cost256w = N > 64 ? kW4Mid256RoundPerSmallRound * rounds(tiles_of(t256w)) : cost128;
  const double cost_big = kW4BigRoundPerSmallRound * rounds(tiles_of(big));
  const double cost_wide = kW4BigRoundPerSmallRound * kW4WideRoundPerBigRound * rounds(tiles_of(wide));
  const double smaller = std::min(cost128, cost256w);
  const W4Tile *by_rounds = cost_wide < cost_big && cost_wide < smaller ? &wide : cost_big < smaller ? &big : cost256w < cost128 ? &t256w : &t128;
  if (!fits(tiles_of(*by_rounds)))
    by_rounds = &wide;
  W4Plan best;
  if (M > 64 && fits(tiles_of(*by_rounds))) {
    best = plan_of(*by_rounds, 1);
    best.narrow = by_rounds == &t128 && N <= 64;
    best.us *= kW4Promise;
  }
  for (const W4Tile &t : kW4Tiles) {
    if (!fits(tiles_of(t)))
      continue;
    for (int splits : kSplits) {
      // as for frag_plan: a part of at least two slices, a ticket for every split tile, at most two rounds of workgroups
      if (splits > 1 && (!may_split || !t.splits || slices < 2 * splits || tiles_of(t) > int64_t(kTickets) || tiles_of(t) * splits > 2 * units))
        break;
      const W4Plan p = plan_of(t, splits);
      if (!best.tile || p.us < best.us)
        best = p;
    }
  }
  const W4Tile &one = kW4Tiles[0], &two = kW4Sets[0], &four = kW4Sets[1];
  if (!best.tile || !fits(tiles_of(one)))
    return best;
  W4Plan sets;
  for (const W4Tile *t : {&two, &four}) {
    for (int splits : kSplits) {
      if (splits > 1 && (!may_split || slices < 2 * splits || tiles_of(*t) > int64_t(kTickets) || tiles_of(*t) * splits > 2 * units))
        break;
      const W4Plan p = plan_of(*t, splits);
      if (t == &two ? p.split.per < kW4TwoSetsFrom : p.split.per < kW4FourSetsFrom || p.tiles * p.split.splits > units)
        continue;
      if (!sets.tile || p.us < sets.us)
        sets = p;
    }
  }
  if (sets.tile && sets.us < kW4SetsPromise * best.us)
    return sets;
  if (best.tile == &one && best.split.per >= kW4TwoSetsFrom)
    best.tile = best.split.per >= kW4FourSetsSameSplitFrom && best.tiles * best.split.splits <= units ? &four : &two;
  return best;
}
W4Plan w4_plan(int64_t M, int64_t K, int64_t N, int64_t units, bool may_split) {
  static thread_local LastPlan<W4Plan> last;
  return last.of(M, N, K, units, may_split, [&] { return make_w4_plan(M, K, N, units, may_split); });
}

const char *float_name(int32_t dt) {
  switch (dt) {
  case MTRT_F32: return "f32";
  case MTRT_F16: return "f16";
  case MTRT_BF16: return "bf16";
  }
  return nullptr;
}
const char *code_name(int32_t dt) {
  switch (dt) {
  case MTRT_I8: return "i8";
  case MTRT_F8E4M3FN: return "f8";
  case MTRT_I4: return "i4";
  case MTRT_I4_PACKED: return "i4p";
  case MTRT_F4_PACKED: return "f4p";
  }
  return nullptr;
}
int float_bytes(int32_t dt) { return dt == MTRT_F32 ? 4 : 2; }

bool aligned(const void *p, uintptr_t a) { return (reinterpret_cast<uintptr_t>(p) & (a - 1)) == 0; }

// Element count of a [d0, d1] operand without signed overflow: false when the product does not fit in 63 bits.
bool element_count(int64_t d0, int64_t d1, int64_t *n) { return !__builtin_mul_overflow(d0, d1, n); }
// Matrix extents of the GEMM entry points: below 2^31 each, so that every product of two of them (and twice that)
// fits in 63 bits.
constexpr int64_t kMaxMatrixExtent = (int64_t(1) << 31) - 1;

// 256 x 256 tiles, one workgroup to a compute unit at a time; a last round that would fill at most half of the units (or a launch that
// does) has its panels cut into 256 x 128 halves.  Each kind is dealt evenly to the XCDs.
struct Panels {
  int64_t full, full_tiles, half_tiles, grid;
};
Panels panels_of(int64_t M, int64_t N, int64_t units) {
  const int64_t panels = (N + 255) / 256, tiles_m = (M + 255) / 256, tiles = panels * tiles_m, rest = tiles % units;
  Panels p;
  p.full = tiles * 2 <= units ? 0 : rest > 0 && rest * 2 <= units ? panels - (rest + tiles_m - 1) / tiles_m : panels;
  p.full_tiles = p.full * tiles_m;
  p.half_tiles = std::max<int64_t>(0, (N - p.full * 256 + 127) / 128) * tiles_m;   // (full panels may reach past N)
  p.grid = 8 * ((p.full_tiles + 7) / 8) + 8 * ((p.half_tiles + 7) / 8);
  return p;
}

uint32_t blocks_for(int64_t units, uint32_t per_block) {
  const int64_t b = (units + per_block - 1) / per_block;
  return uint32_t(std::max<int64_t>(1, std::min<int64_t>(b, kMaxGrid)));
}

// The memory of a split launch: the caller's workspace and a ticket per tile.  False where either is missing: the caller then
// takes the plan without a split.
template <class Plan>
bool bind_split(DeviceState *st, hipStream_t stream, Plan &plan, void *workspace, int64_t workspace_bytes) {
  if (!plan.tile || plan.split.splits <= 1)
    return true;
  if (!workspace || !aligned(workspace, 16) || workspace_bytes < plan.workspace())
    return false;
  plan.split.partial = workspace;
  plan.split.tickets = split_tickets(st, stream, uint32_t(plan.tiles));
  return plan.split.tickets != nullptr;
}

constexpr int32_t kCodesPast = 1 << 8;  // kFlagCodesPast of the kernels (common.hpp)

// Quantize and dequantize in one pass, one scale: the kernel with the wave's number in a scalar register, for tensors of more than four
// workgroups to a unit (three, to float8) and up to 9 Mi elements.  us, the number per lane and scalar: bf16 -> i8 of 4, 4.02, 5, 6, 8, 12
// and 32 Mi 5.2, 5.3; 6.25, 5.5; 7.0, 6.2; 7.6, 7.2; 9.5, 9.3; 12.6, 13.4; 27.6, 29.7; bf16 -> f8 of 3, 3.02, 4, 5 and 8 Mi 4.6, 4.8; 5.4, 4.8;
// 6.1, 5.4; 7.5, 6.5; 9.6, 9.4; f32 -> i8 of 4, 4.02, 5, 8, 20 and 48 Mi 7.4, 7.6; 8.95, 7.95; 9.95, 9.0; 15.2, 14.4; 32.9, 33.9; 69.7, 72.2;
// behind an amax the two are level.  f32 -> f8 loses (8 Mi 14.8, 15.9).
bool fused_scalar(int32_t x_dtype, int32_t q_dtype, int64_t n) {
  const bool codes = q_dtype == MTRT_I8 || q_dtype == MTRT_I4 || (q_dtype == MTRT_F8E4M3FN && x_dtype != MTRT_F32);
  return codes && n > (int64_t(q_dtype == MTRT_F8E4M3FN ? 3 : 4) << 20) && n < (int64_t(9) << 20);
}

// Column scales: four rows of a scale block to a wave instead of eight, for blocks that have no more and tensors of which eight rows would give
// a compute unit less than six waves.  By the waves that eight rows make, us, four and eight rows: quantize bf16 -> i4, 80 waves 2.9, 3.7;
// 528 3.7, 4.0; 1024 4.0, 4.2; 1504 5.0, 5.2; 2048 6.2, 5.95; 2519 5.7, 5.4; 4096 11.1, 10.4; 11264 25.1, 25.1; in blocks of four rows, 4096 6.8, 7.9; of
// one, 32768 23.8, 32.2; f32 -> i8, 2048 4.55, 4.5; 3008 6.0, 5.8; 22016 38.5, 37.3.  To quantize and dequantize in one pass, bf16 -> i4, 1504 6.6, 7.3;
// 2048 9.3, 8.5.  A dequantize by itself takes four as well at any size (384 2.8, 3.2; 2048 4.2, 4.5; 11264 22.5, 22.6), but behind a quantize it
// finds the codes in its XCD's L2 only where both take the same rows (four behind eight: bf16 [768, 9152] to i4 and back 12.8, and 10.9).
bool few_column_rows(int64_t nb, int64_t waves, int64_t units) { return nb <= 4 || waves <= 6 * units; }

// mode: 0 quantize, 1 dequantize, 2 fused.  codes_past: nobody is known to read the codes next (see CodeGroup in qdq.hip)
int32_t qdq_dispatch(int mode, hipStream_t stream, const void *x, int32_t x_dtype, void *q,
                     int32_t q_dtype, void *y, const float *scale, int32_t kind, int64_t d0,
                     int64_t d1, int64_t nb, int32_t flags, bool codes_past = false) {
  clear_error();
  const char *xn = float_name(x_dtype);
  const char *qn = code_name(q_dtype);
  if (!xn)
    return set_error(MTRT_INVALID_ARGUMENT, "float operand dtype %d is not one of f32/f16/bf16", x_dtype);
  if (!qn)
    return set_error(MTRT_INVALID_ARGUMENT, "quantized dtype %d is not one of i8/f8E4M3FN/i4/i4-packed", q_dtype);
  if (d0 < 0 || d1 < 0)
    return set_error(MTRT_INVALID_ARGUMENT, "negative extent [%lld, %lld]", (long long)d0, (long long)d1);
  if (kind < MTRT_SCALE_UNIFORM || kind > MTRT_SCALE_COL)
    return set_error(MTRT_INVALID_ARGUMENT, "unknown scale kind %d", kind);
  if (kind != MTRT_SCALE_UNIFORM && nb <= 0)
    return set_error(MTRT_INVALID_ARGUMENT, "scale kind %d needs a positive scale count / block size, got %lld",
                     kind, (long long)nb);
  if (kind == MTRT_SCALE_COL && d0 % nb != 0)
    return set_error(MTRT_INVALID_ARGUMENT, "block size %lld does not divide the blocked extent %lld",
                     (long long)nb, (long long)d0);
  if (flags & ~(MTRT_Q_ROUND_TO_INT | MTRT_F8_REFHOST | MTRT_F8_VIA_F16))
    return set_error(MTRT_INVALID_ARGUMENT, "unknown flag bits 0x%x", flags);
  if ((flags & MTRT_F8_REFHOST) && (flags & MTRT_F8_VIA_F16))
    return set_error(MTRT_INVALID_ARGUMENT, "MTRT_F8_REFHOST and MTRT_F8_VIA_F16 name two different conversions; pass one");
  int64_t n;
  if (!element_count(d0, d1, &n) || n >= (int64_t(1) << 35))
    return set_error(MTRT_INVALID_ARGUMENT, "[%lld, %lld] elements exceed the supported 2^35", (long long)d0, (long long)d1);
  if (n == 0)
    return MTRT_OK;
  if (!scale || !q || (mode != 1 && !x) || (mode != 0 && !y))
    return set_error(MTRT_INVALID_ARGUMENT, "null operand");
  if (!aligned(mode == 1 ? y : x, float_bytes(x_dtype)) || (mode == 2 && !aligned(y, float_bytes(x_dtype))))
    return set_error(MTRT_INVALID_ARGUMENT, "float operand is not aligned to its element size");
  if (d1 == 0)
    return MTRT_OK;
  if (kind == MTRT_SCALE_UNIFORM)
    nb = 1;

  DeviceState *st = device_state();
  if (!st)
    return MTRT_RUNTIME_ERROR;

  // The group kernels move one 128-bit vector of the float operand (G elements)
  // per lane per instruction: they need that operand 128-bit aligned, the codes
  // aligned to the G codes a lane moves at once, and - whenever the scale changes
  // along or across rows - rows that are whole groups.
  const int group = x_dtype == MTRT_F32 ? 4 : 8;
  const bool nibbles = q_dtype == MTRT_I4_PACKED || q_dtype == MTRT_F4_PACKED;
  const uintptr_t q_align = nibbles ? group / 2 : group;
  bool tiles = aligned(q, q_align) && (mode == 1 || aligned(x, 16)) && (mode == 0 || aligned(y, 16));
  // The row- and column-scaled group kernels keep group, row and scale-block indices in 32 bits; a tensor
  // beyond that (64 GiB of f32 and more) takes the element-wise kernel, which indexes in 64 bits throughout.
  if (kind != MTRT_SCALE_UNIFORM)
    tiles = tiles && (d1 % group == 0) && n / group < (int64_t(1) << 32) && nb < (int64_t(1) << 32);
  if (kind == MTRT_SCALE_COL)
    tiles = tiles && aligned(scale, 16);

  // Row or column scales on rows that are not whole groups, or on operands not aligned for group accesses: a wave
  // per 64 groups of one row with accesses at element alignment (codes one per byte only: a packed byte can
  // straddle rows).  Everything else that is not `tiles`: one element per lane.
  // A per-tensor scale on unaligned operands is the row kind on one row of n elements.
  const bool ragged = !tiles && !nibbles;
  if (ragged && kind == MTRT_SCALE_UNIFORM) {
    kind = MTRT_SCALE_ROW;
    d0 = 1;
    d1 = n;
  }
  static const char *kModeName[] = {"q", "dq", "qdq"};
  static const char *kKindName[] = {"uniform", "row", "col"};
  static const char *kRaggedName[] = {"", "rowu", "colu"};
  const bool strips = tiles && kind == MTRT_SCALE_COL;
  const int64_t row_strips = (d1 / group + 63) / 64;    // of 64 groups
  const bool few_rows = strips && few_column_rows(nb, d0 / nb * ((nb + 7) / 8) * row_strips, num_compute_units(st));
  KernelName name("mtrt_");
  name + kModeName[mode] + "_" + (tiles ? kKindName[kind] : (ragged ? kRaggedName[kind] : "any")) + "_" + xn + "_" + qn + (strips && !few_rows ? "r8" : "");

  if (mode == 2 && tiles && kind == MTRT_SCALE_UNIFORM && fused_scalar(x_dtype, q_dtype, n))
    name + "s";

  int64_t n_arg = n, d1_arg = d1, nb_arg = nb;
  int32_t kind_arg = kind, flags_arg = flags | (codes_past ? kCodesPast : 0);
  const void *x_arg = x;
  void *q_arg = q, *y_arg = y;
  const float *s_arg = scale;
  void *args[11];
  int na = 0;
  if (mode != 1) args[na++] = &x_arg;
  args[na++] = &q_arg;
  if (mode != 0) args[na++] = &y_arg;
  args[na++] = &s_arg;
  args[na++] = &n_arg;
  args[na++] = &d1_arg;
  args[na++] = &nb_arg;
  if (ragged) {                                        // row pitches of the float operand(s) and of the codes: contiguous here
    args[na++] = &d1_arg;
    args[na++] = &d1_arg;
  }
  if (!tiles && !ragged) args[na++] = &kind_arg;
  if (mode != 1) args[na++] = &flags_arg;

  if (strips) {
    // one wave per (scale block, chunk of its rows, strip of 64 groups of columns): see qdq_col_strips
    const int64_t rows = few_rows ? 4 : 8, items = d0 / nb * ((nb + rows - 1) / rows) * row_strips;
    return launch(st, name, blocks_for(items, kBlock / 64), kBlock, stream, args);
  }
  if (ragged) {
    const int64_t chunks = std::max<int64_t>(1, (d1 / group + 63) / 64);
    return launch(st, name, blocks_for(d0 * chunks, kBlock / 64), kBlock, stream, args);
  }
  const int64_t units = tiles ? (n + kTile - 1) / kTile : (nibbles ? (n + 1) / 2 : n);
  return launch(st, name, blocks_for(units, kBlock), kBlock, stream, args);
}

int32_t pick_nv(int64_t nvec_per_row) {
  for (int nv : {1, 2, 4, 8, 16})
    if (nvec_per_row <= int64_t(64) * nv)
      return nv;
  return 0;
}

// The element-aligned (`_u`) LayerNorm kernels on f32 rows with eight vectors per lane come out of the compiler with 230 registers per
// lane (one wave per SIMD: f32 [4096, 8190] took 114 us against softmax's 45).  Their 16-vector forms take under 130, so those rows use
// them (a lane past the end of the row holds nothing).
int unaligned_nv(int32_t dtype, int nv, bool layernorm) { return dtype == MTRT_F32 && nv == 8 && layernorm ? 16 : nv; }

// Rows too long for one wave: a workgroup of 256 or 1024 lanes with 8 or 16 vectors per lane owns the row.
// Returns false when the row is longer than 1024 * 16 vectors.
bool pick_group(int64_t nvec_per_row, int *threads, int *nv) {
  for (int t : {256, 1024})
    for (int v : {8, 16})
      if (nvec_per_row <= int64_t(t) * v) {
        *threads = t;
        *nv = v;
        return true;
      }
  return false;
}

// Two forms of a kernel (norm.hip): one works on every vector, the other stops at a row's end, which asks for less and needs fewer registers, but
// takes its vectors one after the other.  That one is the faster up to a share of the vectors that a row fills, which depends on the
// rows to a compute unit: few have nothing to hide the way to memory behind; `window` is where they fit on the chip at once in
// this form and not in the other.  Lines from 3050 shapes (5 to 6000 rows and 100 MB, shares 0.53 to 1, f32 and bf16), each where the forms
// are level; us, every vector and to the row's end:
//   LayerNorm bf16 [1500, 9011] 18.7, 14.7; [4000, 10243] 46.9, 40.8; [3633, 13760] 38.7, 42.8; [500, 27523] 14.7, 15.5; [1500, 31128] 37.8, 44.2;
//   [500, 47184] 24.3, 17.6; [1500, 36043] 78.5, 56.7; f32 [500, 4504] 5.6, 5.9; [1500, 5120] 13.0, 10.5; [1000, 27524] 48.9, 49.4
//   from 7 rows to a unit at element alignment [1800, 23595] 48.9, 45.8; [4000, 26179] 104.7, 103.1; [2800, 28179] 79.7, 81.6
//   softmax bf16 [1500, 10240] 13.7, 9.8; [768, 11792] 7.6, 8.1; [4000, 13763] 48.5, 45.9; [2000, 27520] 39.3, 41.7; [1000, 40963] 51.2, 43.0; f32 [2000,
//   18023] 63.6, 52.4
// Kernels that are not listed have one form; fewer than 8 rows, a few us whichever it is, take the one without a letter.
struct RowForm {
  bool layernorm, wide, ragged;                        // wide: f32
  int lanes, nv;
  double lo, hi;                                       // the window, rows to a compute unit
  double few, window, many;                            // largest share to stop at the row's end: up to lo, up to hi, beyond
  double whole = 0;                                    // whole rows too (its body for those has fewer registers): from here on
  double upto = 1e30;                                  // the entry holds up to here; the kernel's next one beyond
};
constexpr RowForm kRowForms[] = {
    {true, false, false, 256, 8, 5, 8, 0, 0.75, 0, 5},
    {true, false, false, 256, 16, 3, 5, 0, 1, 0.63},
    {true, false, false, 1024, 8, 0, 0, 0, 0, 0.95},
    {true, false, false, 1024, 16, 0, 0, 0, 0, 0.92},
    {true, false, true, 64, 4, 0, 0, 0, 0, 0.77},
    {true, false, true, 64, 8, 0, 0, 0, 0, 0.85},
    {true, false, true, 64, 16, 0, 0, 0, 0, 0.75},
    {true, false, true, 256, 8, 2.5, 2.5, 0.72, 0, 0.9},
    {true, false, true, 256, 16, 2.5, 4, 0.66, 0.95, 0.66, 0, 7},
    {true, false, true, 256, 16, 0, 0, 0, 0, 0.82},
    {true, true, false, 256, 8, 4, 4, 0, 0, 0.96},
    {true, true, false, 1024, 8, 0, 0, 0, 0, 0.7},
    {false, false, false, 256, 8, 3.5, 6, 0, 0.96, 0},
    {false, false, false, 256, 16, 2, 4, 0, 0.85, 0},
    {false, false, false, 1024, 8, 0, 0, 0, 0, 0.85},
    {false, false, false, 1024, 16, 0, 0, 0, 0, 0.9},
    {false, false, true, 256, 8, 2.5, 4, 0.66, 1, 0.85},
    {false, false, true, 256, 16, 1.1, 4, 0.66, 1, 0.85},
    {false, true, false, 1024, 8, 1, 1, 0.7, 0, 0.95},
    {false, true, false, 1024, 16, 0, 0, 0, 0, 0.75},
    {false, true, true, 1024, 8, 1, 1, 0.8, 0, 1},
    {false, true, true, 1024, 16, 0, 0, 0, 0, 0.8},
};
const char *row_form(bool layernorm, int32_t dtype, bool ragged, int lanes, int nv, int64_t rows, int64_t nvec_per_row, int64_t units) {
  const double to_a_unit = double(rows) / double(units), share = double(nvec_per_row) / double(lanes * nv);
  for (const RowForm &r : kRowForms)
    if (rows >= 8 && r.layernorm == layernorm && r.wide == (dtype == MTRT_F32) && r.ragged == ragged && r.lanes == lanes && r.nv == nv && to_a_unit <= r.upto) {
      const bool ends = share <= (to_a_unit <= r.lo ? r.few : to_a_unit <= r.hi ? r.window : r.many) || (share == 1 && r.whole > 0 && to_a_unit > r.whole);
      return lanes == 1024 ? (ends ? "" : "a") : (ends ? "e" : "");
    }
  return "";
}

// ... and the softmax kernels of two rows to a unit, where there are rows for them (norm.hip has the figures).
const char *softmax_form(int32_t dtype, bool ragged, int lanes, int nv, int64_t rows, int64_t nvec_per_row, int64_t units) {
  if (dtype != MTRT_F32 && lanes == 1024 && nv == 8 && rows > units)
    return !ragged && 10 * nvec_per_row > 8 * int64_t(lanes * nv) ? "ra" : "r";
  return row_form(false, dtype, ragged, lanes, nv, rows, nvec_per_row, units);
}

// Softmax rows that are no whole cache lines, of 20 to 80 MiB together, are read through the caches: the line that two rows share is fetched once, and what an
// earlier launch has left in the Infinity Cache comes from there.  Whole lines gain from the second alone, and a launch that has just made x, or memory, is the
// more common place for it to come from.  us, past and through, (rows, columns): three tensors in turn; each from memory; with a launch that makes x in front and
// one that reads y behind, all three.  No whole lines: f16 (17476, 1500) 19.8, 17.2; 20.7, 20.8; 64.2, 62.2; (8735, 3001) 21.3, 17.8; 22.3, 22.4; 64.7, 61.8; bf16
// (4368, 9001) 32.9, 26.3; 33.6, 34.1; 88.5, 84.4; f32 (12750, 1028) 19.5, 16.6; 20.3, 20.0; 58.1, 56.7; half lines (6553, 2000) 18.9, 16.4; 19.8, 20.3; 56.5, 57.0.
// Whole lines: f16 (25600, 1024) 17.7, 16.1; 18.7, 19.5; 54.7, 56.8; (4096, 4096) 11.4, 10.8; 12.8, 13.4; 37.1, 39.3; f32 (12800, 1024) 18.0, 16.5; 19.1, 19.7;
// 53.6, 56.7; (3268, 6016) 26.7, 23.4; 27.7, 28.8; 79.2, 80.6.  Smaller tensors of either kind: f16 (2097, 1500) 4.6, 4.4; 5.2, 5.3; 18.6, 18.9; f32 (698, 4501) 5.2,
// 5.6; 5.8, 6.3; 18.7, 19.0; larger ones: f16 (38447, 1500) 41.2, 41.0; 42.1, 42.0; f32 (6406, 4501) 40.5, 41.0; 41.5, 42.1.
bool softmax_reads_past(int64_t rows, int64_t row_bytes) {
  return row_bytes % 128 == 0 || rows * row_bytes <= int64_t(20) << 20 || rows * row_bytes > int64_t(80) << 20;
}

// Softmax rows of whole vectors that start off a cache line are cut there (norm.hip) in tensors of 14 MiB and more.  us, uncut and cut, f16 [2000, 3000] 5.48, 5.59; bf16
// [200, 5000] 4.26, 4.39; [600, 5000] 5.11, 5.18; f32 [3000, 1000] 4.82, 4.88; from 20 MB f16 [3333, 3000] 8.5, 8.2; bf16 [2000, 5000] 7.9, 7.6; f32 [24000, 1500] 48.7,
// 47.4.  Whole lines have nothing to cut, and pay for it the same (f16 [3000, 1984] 4.68, 4.81).
bool softmax_cuts(const void *x, int64_t rows, int64_t row_bytes) {
  return (row_bytes % 128 != 0 || !aligned(x, 128)) && rows * row_bytes >= int64_t(14) << 20;
}

} // namespace

extern "C" {

int32_t mtrt_hip_amax(mtrt_stream_t stream, const void *x, int32_t dtype, int64_t n, float qmax,
                      float *amax_out, float *scale_out) {
  clear_error();
  const char *xn = float_name(dtype);
  if (!xn)
    return set_error(MTRT_INVALID_ARGUMENT, "amax input dtype %d is not one of f32/f16/bf16", dtype);
  if (n < 0)
    return set_error(MTRT_INVALID_ARGUMENT, "negative element count %lld", (long long)n);
  if (n > 0 && !x)
    return set_error(MTRT_INVALID_ARGUMENT, "null input");
  if (!aligned(x, float_bytes(dtype)))
    return set_error(MTRT_INVALID_ARGUMENT, "input is not aligned to its element size");
  DeviceState *st = device_state();
  if (!st)
    return MTRT_RUNTIME_ERROR;
  uint32_t *slot = reduction_slot(st, as_hip(stream));
  if (!slot)
    return MTRT_RUNTIME_ERROR;
  // Two workgroups per CU (8 waves), each lane keeping eight 128-bit loads in flight; fewer when the tensor is small.
  // Measured on bf16 [16384, 8192] with four loads a lane: 1 / 2 / 3 / 4 / 8 / 16 workgroups per CU take 51.3 / 40.7 / 41.8 /
  // 41.9 / 45.7 / 48.2 us (fewer arrivals at the reduction tree).
  const int per_vec = dtype == MTRT_F32 ? 4 : 8;
  const int64_t nvec = n / per_vec;
  const uint32_t grid = uint32_t(std::max<int64_t>(
      1, std::min<int64_t>((nvec + int64_t(kBlock) * 8 - 1) / (int64_t(kBlock) * 8), int64_t(num_compute_units(st)) * 2)));
  const void *x_arg = x;
  int64_t n_arg = n;
  float qmax_arg = qmax;
  void *args[] = {&x_arg, &n_arg, &qmax_arg, &amax_out, &scale_out, &slot};
  return launch(st, KernelName("mtrt_amax_") + xn, grid, kBlock, as_hip(stream), args);
}

int32_t mtrt_hip_amax_scales(mtrt_stream_t stream, const void *x, int32_t dtype, int32_t scale_kind, int64_t d0, int64_t d1,
                             int64_t nb, float qmax, float *amax_out, float *scale_out) {
  clear_error();
  const char *xn = float_name(dtype);
  if (!xn)
    return set_error(MTRT_INVALID_ARGUMENT, "amax input dtype %d is not one of f32/f16/bf16", dtype);
  if (d0 < 0 || d1 < 0)
    return set_error(MTRT_INVALID_ARGUMENT, "negative extent [%lld, %lld]", (long long)d0, (long long)d1);
  if (scale_kind < MTRT_SCALE_UNIFORM || scale_kind > MTRT_SCALE_COL)
    return set_error(MTRT_INVALID_ARGUMENT, "unknown scale kind %d", scale_kind);
  int64_t n;
  if (!element_count(d0, d1, &n))
    return set_error(MTRT_INVALID_ARGUMENT, "[%lld, %lld] elements do not fit a 64-bit count", (long long)d0, (long long)d1);
  if (scale_kind == MTRT_SCALE_UNIFORM)
    return mtrt_hip_amax(stream, x, dtype, n, qmax, amax_out, scale_out);
  if (nb <= 0)
    return set_error(MTRT_INVALID_ARGUMENT, "scale kind %d needs a positive scale count / block size, got %lld", scale_kind,
                     (long long)nb);
  if (scale_kind == MTRT_SCALE_ROW && nb > d0 && d0 > 0)
    return set_error(MTRT_INVALID_ARGUMENT, "%lld scales for %lld rows", (long long)nb, (long long)d0);
  if (scale_kind == MTRT_SCALE_COL && d0 % nb != 0)
    return set_error(MTRT_INVALID_ARGUMENT, "block size %lld does not divide the blocked extent %lld", (long long)nb,
                     (long long)d0);
  if (d0 == 0 || d1 == 0)
    return MTRT_OK;                                    // no scale element has an input
  if (!x || (!amax_out && !scale_out))
    return set_error(MTRT_INVALID_ARGUMENT, "null operand");
  if (!aligned(x, float_bytes(dtype)))
    return set_error(MTRT_INVALID_ARGUMENT, "input is not aligned to its element size");
  DeviceState *st = device_state();
  if (!st)
    return MTRT_RUNTIME_ERROR;
  const int group = dtype == MTRT_F32 ? 4 : 8;
  const bool vec = d1 % group == 0 && aligned(x, 16);
  void *args[] = {&x, &d0, &d1, &nb, &qmax, &amax_out, &scale_out};
  if (scale_kind == MTRT_SCALE_ROW && vec && nb < 4 * int64_t(num_compute_units(st)) && nb <= d0) {
    // Few scales (one wave each would leave most of the chip idle): the tiles of a scale's rows (1024 vectors each)
    // are shared by several workgroups that meet in the output word by atomic max, about two workgroups per compute
    // unit in all; then the finishing launch.  Measured on f16 [65536, 1024]: nb = 64 945.6 us, nb = 8 7684 us as one
    // wave per scale; [8, 8M] with nb = 8 2387 us.
    const int64_t units = num_compute_units(st), nvec = d1 / group;
    const int64_t tiles = ((d0 + nb - 1) / nb) * ((nvec + 1023) / 1024);     // of the scale with the most rows
    const int64_t parts = std::max<int64_t>(1, std::min<int64_t>((2 * units + nb - 1) / nb, (tiles + 3) / 4));
    if (parts > 1) {
      int64_t count = nb;
      uint32_t *stage = reinterpret_cast<uint32_t *>(amax_out ? amax_out : scale_out);
      uint8_t *stage_bytes = reinterpret_cast<uint8_t *>(stage);
      uint32_t zero = 0;
      int32_t width = 4;
      void *fill_args[] = {&stage_bytes, &count, &zero, &width};
      int32_t rc = launch(st, KernelName("mtrt_fill"), blocks_for(count, kBlock), kBlock, as_hip(stream), fill_args);
      if (rc != MTRT_OK)
        return rc;
      int64_t parts_arg = parts;
      void *split_args[] = {&x, &d0, &d1, &nb, &parts_arg, &stage};
      rc = launch(st, KernelName("mtrt_amax_rows_split_") + xn, uint32_t(nb * parts), kBlock, as_hip(stream), split_args);
      if (rc != MTRT_OK)
        return rc;
      void *finish_args[] = {&stage, &count, &qmax, &amax_out, &scale_out};
      return launch(st, KernelName("mtrt_amax_finish_") + xn, blocks_for(count, kBlock), kBlock, as_hip(stream), finish_args);
    }
  }
  if (scale_kind == MTRT_SCALE_ROW) {
    const int64_t blocks = (nb + 3) / 4;
    if (blocks > int64_t(kMaxGrid) * 1024)
      return set_error(MTRT_INVALID_ARGUMENT, "%lld scales are too many for one launch", (long long)nb);
    return launch(st, KernelName(vec ? "mtrt_amax_rows_" : "mtrt_amax_rows_any_") + xn, uint32_t(blocks), kBlock,
                  as_hip(stream), args);
  }
  // A row length that is not whole vectors, or an unaligned operand: one lane per (block, column) while that gives
  // every compute unit a thousand lanes (f16 [8192, 8190], blocks of 128 rows: 44.7 us against 51.1 us for the
  // vector form at element alignment); with fewer, longer blocks the `_u` kernels, which move whole vectors at
  // element alignment, count a last partial vector and can share a block's rows (one block of 8192 rows: 2085 us
  // as one lane per column, 112.6 us shared).
  if (vec || (d0 / nb) * d1 < int64_t(num_compute_units(st)) * 1024) {
    const char *u = vec ? "" : "u_";
    const int64_t blocks = (d0 / nb) * (((d1 + group - 1) / group + 63) / 64), units = num_compute_units(st);
    if (blocks < 2 * units && nb >= 128 && (d0 / nb) * d1 < (int64_t(1) << 31)) {
      // Few, long blocks (one per-channel scale per column of a [K, N] weight): too few workgroups to pull the
      // tensor through.  Each block's rows are dealt to several workgroups (at least 32 rows each, about two
      // workgroups per compute unit in all, at most 16 per block: the atomics on one line are served one after
      // the other) that meet in the output itself, zeroed first, by atomic max on bit patterns; a last small
      // launch turns the patterns into amax and scale.  Measured on [4096, 11008], nb = 4096: f16 157.6 us as 22
      // workgroups, 24.3 / 26.3 / 32.3 / 40.8 us with 12 / 24 / 47 / 70 parts; f32 148.7 us, 37.5 / 36.8 / 36.3 us
      // with 6 / 12 / 24 parts.
      const int64_t want = std::min<int64_t>({(2 * units + blocks - 1) / blocks, nb / 32, int64_t(16)});
      const int64_t rows_per_part = (((nb + want - 1) / want) + 3) / 4 * 4, parts = (nb + rows_per_part - 1) / rows_per_part;
      int64_t count = (d0 / nb) * d1;
      uint32_t *stage = reinterpret_cast<uint32_t *>(amax_out ? amax_out : scale_out);
      uint8_t *stage_bytes = reinterpret_cast<uint8_t *>(stage);
      uint32_t zero = 0;
      int32_t width = 4;
      void *fill_args[] = {&stage_bytes, &count, &zero, &width};
      int32_t rc = launch(st, KernelName("mtrt_fill"), blocks_for(count, kBlock), kBlock, as_hip(stream), fill_args);
      if (rc != MTRT_OK)
        return rc;
      int64_t rpp = rows_per_part;
      void *split_args[] = {&x, &d0, &d1, &nb, &rpp, &stage};
      rc = launch(st, KernelName("mtrt_amax_cols_split_") + u + xn, uint32_t(blocks * parts), kBlock, as_hip(stream), split_args);
      if (rc != MTRT_OK)
        return rc;
      void *finish_args[] = {&stage, &count, &qmax, &amax_out, &scale_out};
      return launch(st, KernelName("mtrt_amax_finish_") + xn, blocks_for(count, kBlock), kBlock, as_hip(stream), finish_args);
    }
    if (blocks <= int64_t(kMaxGrid) * 1024)
      return launch(st, KernelName("mtrt_amax_cols_") + u + xn, uint32_t(blocks), kBlock, as_hip(stream), args);
  }
  return launch(st, KernelName("mtrt_amax_cols_any_") + xn, blocks_for((d0 / nb) * d1, kBlock), kBlock, as_hip(stream), args);
}

int32_t mtrt_hip_quantize(mtrt_stream_t stream, const void *x, int32_t x_dtype, void *q, int32_t q_dtype,
                          const float *scale, int32_t scale_kind, int64_t d0, int64_t d1, int64_t nb,
                          int32_t flags) {
  return qdq_dispatch(0, as_hip(stream), x, x_dtype, q, q_dtype, nullptr, scale, scale_kind, d0, d1, nb, flags);
}

int32_t mtrt_hip_dequantize(mtrt_stream_t stream, const void *q, int32_t q_dtype, void *y, int32_t y_dtype,
                            const float *scale, int32_t scale_kind, int64_t d0, int64_t d1, int64_t nb) {
  return qdq_dispatch(1, as_hip(stream), nullptr, y_dtype, const_cast<void *>(q), q_dtype, y, scale, scale_kind,
                      d0, d1, nb, 0);
}

int32_t mtrt_hip_quantize_dequantize(mtrt_stream_t stream, const void *x, int32_t x_dtype, void *q,
                                     int32_t q_dtype, void *y, const float *scale, int32_t scale_kind,
                                     int64_t d0, int64_t d1, int64_t nb, int32_t flags) {
  return qdq_dispatch(2, as_hip(stream), x, x_dtype, q, q_dtype, y, scale, scale_kind, d0, d1, nb, flags);
}

namespace {
std::atomic<int32_t> g_wait_limit{1 << 16};

// Highest and lowest element offset a [d0, d1] view with these strides touches, relative to its base.
bool view_extent(int64_t offset, int64_t d0, int64_t d1, int64_t s0, int64_t s1, int64_t *lo, int64_t *hi) {
  const __int128 a = __int128(d0 - 1) * s0, b = __int128(d1 - 1) * s1;
  const __int128 l = offset + (a < 0 ? a : 0) + (b < 0 ? b : 0), h = offset + (a > 0 ? a : 0) + (b > 0 ? b : 0);
  if (l < -(__int128(1) << 62) || h > (__int128(1) << 62))
    return false;
  *lo = int64_t(l);
  *hi = int64_t(h);
  return true;
}

int32_t view_dispatch(bool quantize, hipStream_t stream, const void *f, int32_t f_dtype, const mtrt_hip_view2d *fv, const void *q,
                      int32_t q_dtype, const mtrt_hip_view2d *qv, const float *scale, int32_t kind, int64_t d0, int64_t d1,
                      int64_t nb, int32_t flags) {
  clear_error();
  const char *xn = float_name(f_dtype);
  if (!xn)
    return set_error(MTRT_INVALID_ARGUMENT, "float operand dtype %d is not one of f32/f16/bf16", f_dtype);
  if (q_dtype != MTRT_I8 && q_dtype != MTRT_F8E4M3FN && q_dtype != MTRT_I4)
    return set_error(MTRT_INVALID_ARGUMENT, "views carry one code per byte (i8, f8E4M3FN, i4); dtype %d is packed or unknown", q_dtype);
  if (!fv || !qv)
    return set_error(MTRT_INVALID_ARGUMENT, "null view descriptor");
  if (d0 < 0 || d1 < 0)
    return set_error(MTRT_INVALID_ARGUMENT, "negative extent [%lld, %lld]", (long long)d0, (long long)d1);
  if (kind < MTRT_SCALE_UNIFORM || kind > MTRT_SCALE_COL)
    return set_error(MTRT_INVALID_ARGUMENT, "unknown scale kind %d", kind);
  if (kind != MTRT_SCALE_UNIFORM && nb <= 0)
    return set_error(MTRT_INVALID_ARGUMENT, "scale kind %d needs a positive scale count / block size, got %lld", kind, (long long)nb);
  if (kind == MTRT_SCALE_COL && d0 % nb != 0)
    return set_error(MTRT_INVALID_ARGUMENT, "block size %lld does not divide the blocked extent %lld", (long long)nb, (long long)d0);
  if (flags & ~(MTRT_Q_ROUND_TO_INT | MTRT_F8_REFHOST | MTRT_F8_VIA_F16) || ((flags & MTRT_F8_REFHOST) && (flags & MTRT_F8_VIA_F16)))
    return set_error(MTRT_INVALID_ARGUMENT, "bad flag bits 0x%x", flags);
  if (d0 == 0 || d1 == 0)
    return MTRT_OK;
  int64_t n;
  if (!element_count(d0, d1, &n) || n >= (int64_t(1) << 40))
    return set_error(MTRT_INVALID_ARGUMENT, "view of [%lld, %lld] elements is too large", (long long)d0, (long long)d1);
  if (!f || !q || !scale)
    return set_error(MTRT_INVALID_ARGUMENT, "null operand");
  if (!aligned(f, float_bytes(f_dtype)))
    return set_error(MTRT_INVALID_ARGUMENT, "float operand is not aligned to its element size");
  // a view must stay at or above its base pointer (the allocation starts there); its upper end is the caller's word
  int64_t lo, hi;
  if (!view_extent(fv->offset, d0, d1, fv->stride0, fv->stride1, &lo, &hi) || lo < 0 ||
      !view_extent(qv->offset, d0, d1, qv->stride0, qv->stride1, &lo, &hi) || lo < 0)
    return set_error(MTRT_INVALID_ARGUMENT, "view reaches below its base pointer or overflows 62-bit offsets");
  DeviceState *st = device_state();
  if (!st)
    return MTRT_RUNTIME_ERROR;
  if (kind == MTRT_SCALE_UNIFORM)
    nb = 1;
  int64_t fo = fv->offset, fs0 = fv->stride0, fs1 = fv->stride1, qo = qv->offset, qs0 = qv->stride0, qs1 = qv->stride1;
  if (fs1 == 1 && qs1 == 1 && (d0 == 1 || (fs0 == d1 && qs0 == d1))) {
    // Dense in both operands (what a launch with whole row-major tensors passes): the contiguous entry points' own
    // dispatch on the offset pointers, tile kernels when aligned (f16 [8192, 8192] to i8: 56 us row by row, 41 us so).
    void *fp = const_cast<char *>(static_cast<const char *>(f)) + fo * float_bytes(f_dtype);
    void *qp = const_cast<char *>(static_cast<const char *>(q)) + qo;
    if (quantize)
      return qdq_dispatch(0, stream, fp, f_dtype, qp, q_dtype, nullptr, scale, kind, d0, d1, nb, flags);
    return qdq_dispatch(1, stream, nullptr, f_dtype, qp, q_dtype, fp, scale, kind, d0, d1, nb, flags);
  }
  if (fs1 == 1 && qs1 == 1) {
    // Rows that are contiguous in both operands (row and column slices of row-major tensors, offset sub-tensors): the
    // row-walking kernels of the contiguous entry points, with the views' row strides as pitches (f16 [8192, 8192]
    // column slice: 1.3 TB/s one element per lane).  A per-tensor scale is the row kind with one scale.
    const int group = f_dtype == MTRT_F32 ? 4 : 8;
    const int32_t rkind = kind == MTRT_SCALE_COL ? MTRT_SCALE_COL : MTRT_SCALE_ROW;
    const void *fp = static_cast<const char *>(f) + fo * float_bytes(f_dtype);
    const void *qp = static_cast<const char *>(q) + qo;
    KernelName rname(quantize ? "mtrt_q_" : "mtrt_dq_");
    rname + (rkind == MTRT_SCALE_COL ? "colu_" : "rowu_") + xn + "_" + code_name(q_dtype);
    const int64_t chunks = std::max<int64_t>(1, (d1 / group + 63) / 64);
    const uint32_t rgrid = blocks_for(d0 * chunks, kBlock / 64);
    if (quantize) {
      void *rargs[] = {&fp, &qp, &scale, &n, &d1, &nb, &fs0, &qs0, &flags};
      return launch(st, rname, rgrid, kBlock, stream, rargs);
    }
    void *rargs[] = {&qp, &fp, &scale, &n, &d1, &nb, &fs0, &qs0};
    return launch(st, rname, rgrid, kBlock, stream, rargs);
  }
  // An operand that runs fastest along its first dimension (a transpose): 64 x 64 tiles through LDS, each side walked
  // along its own grain.  Otherwise one element per lane.
  auto magnitude = [](int64_t v) { return v < 0 ? -v : v; };
  const bool tiled = magnitude(fs0) < magnitude(fs1) || magnitude(qs0) < magnitude(qs1);
  KernelName name(quantize ? (tiled ? "mtrt_q_viewt_" : "mtrt_q_view_") : (tiled ? "mtrt_dq_viewt_" : "mtrt_dq_view_"));
  name + xn + "_" + code_name(q_dtype);
  const uint32_t grid = tiled ? uint32_t(std::min<int64_t>(((d0 + 63) / 64) * ((d1 + 63) / 64), int64_t(kMaxGrid) * 1024))
                              : blocks_for(n, kBlock);
  if (quantize) {
    void *args[] = {&f, &fo, &d0, &d1, &fs0, &fs1, &q, &qo, &d0, &d1, &qs0, &qs1, &scale, &nb, &kind, &flags};
    return launch(st, name, grid, kBlock, stream, args);
  }
  void *args[] = {&q, &qo, &d0, &d1, &qs0, &qs1, &f, &fo, &d0, &d1, &fs0, &fs1, &scale, &nb, &kind};
  return launch(st, name, grid, kBlock, stream, args);
}
} // namespace

int32_t mtrt_hip_quantize_view(mtrt_stream_t stream, const void *x, int32_t x_dtype, const mtrt_hip_view2d *x_view, void *q,
                               int32_t q_dtype, const mtrt_hip_view2d *q_view, const float *scale, int32_t scale_kind,
                               int64_t d0, int64_t d1, int64_t nb, int32_t flags) {
  return view_dispatch(true, as_hip(stream), x, x_dtype, x_view, q, q_dtype, q_view, scale, scale_kind, d0, d1, nb, flags);
}

int32_t mtrt_hip_dequantize_view(mtrt_stream_t stream, const void *q, int32_t q_dtype, const mtrt_hip_view2d *q_view, void *y,
                                 int32_t y_dtype, const mtrt_hip_view2d *y_view, const float *scale, int32_t scale_kind,
                                 int64_t d0, int64_t d1, int64_t nb) {
  return view_dispatch(false, as_hip(stream), y, y_dtype, y_view, q, q_dtype, q_view, scale, scale_kind, d0, d1, nb, 0);
}

static bool apart(const void *a, int64_t a_bytes, const void *b, int64_t b_bytes) {
  const uint64_t p = reinterpret_cast<uint64_t>(a), r = reinterpret_cast<uint64_t>(b);
  return p + uint64_t(a_bytes) <= r || r + uint64_t(b_bytes) <= p;
}

int32_t mtrt_hip_set_wait_limit(int32_t polls) {
  return g_wait_limit.exchange(polls < 0 ? 0 : polls);
}

int32_t mtrt_hip_dynamic_quantize_dequantize(mtrt_stream_t stream, const void *x, int32_t x_dtype, void *q, int32_t q_dtype,
                                             void *y, int64_t n, float qmax, float *amax_out, float *scale_out,
                                             int32_t flags) {
  clear_error();
  const char *xn = float_name(x_dtype);
  if (!xn)
    return set_error(MTRT_INVALID_ARGUMENT, "float operand dtype %d is not one of f32/f16/bf16", x_dtype);
  if (q_dtype != MTRT_I8 && q_dtype != MTRT_F8E4M3FN)
    return set_error(MTRT_INVALID_ARGUMENT, "dynamic per-tensor quantization targets i8 or f8E4M3FN, got dtype %d", q_dtype);
  if (n < 0)
    return set_error(MTRT_INVALID_ARGUMENT, "negative element count %lld", (long long)n);
  if (n > 0 && (!x || !q))
    return set_error(MTRT_INVALID_ARGUMENT, "null operand");
  if (!scale_out)
    return set_error(MTRT_INVALID_ARGUMENT, "scale_out must point at device memory for one f32 (the quantize step reads the scale there)");
  if (flags & ~(MTRT_Q_ROUND_TO_INT | MTRT_F8_REFHOST | MTRT_F8_VIA_F16))
    return set_error(MTRT_INVALID_ARGUMENT, "unknown flag bits 0x%x", flags);
  DeviceState *st = device_state();
  if (!st)
    return MTRT_RUNTIME_ERROR;
  const int group = x_dtype == MTRT_F32 ? 4 : 8;
  // one workgroup per compute unit at most, and one slot of the exchange per workgroup (256 of them)
  const int64_t nvec = n / group, units = std::min(num_compute_units(st), 256);
  // (The 16-vector form of the 16-bit -> f8 pairs does not fit the 128 registers a lane of a 1024-lane workgroup has
  // and would keep some of the row in scratch memory; a kernel that needs more than a little scratch pays some 10 us
  // per launch for its allocation, more than the second launch costs, so those pairs stop at 4 vectors per lane.)
  const int max_nv = group == 8 && q_dtype == MTRT_F8E4M3FN ? 4 : 16;
  const bool one_launch = n > 0 && n % group == 0 && aligned(x, 16) && aligned(q, group) && (!y || aligned(y, 16)) &&
                          nvec <= units * 1024 * max_nv && !((flags & MTRT_F8_REFHOST) && (flags & MTRT_F8_VIA_F16));
  if (one_launch) {
    uint32_t *slot = reduction_slot(st, as_hip(stream));
    if (!slot)
      return MTRT_RUNTIME_ERROR;
    // Vectors a lane: as few as leave the exchange a number of workgroups that starts without delay, half to three quarters of the units;
    // beyond four, as few as hold the tensor.  us, f32 -> i8 (bf16 -> f8), 1, 2, 3 and 4 vectors: 0.5 MB 4.8, 5.1, 5.2, 5.5 (4.8, 5.3, 6.1,
    // 7.1); 1 MB 5.3, 5.8, 6.4, 6.7 (5.7, 6.4, 7.1, 8.3); 2 MB 6.9, 6.8, 7.2, 7.7 (6.4, 7.0, 7.9, 9.1); 4 MB 9.2, 8.2, 8.2, 8.4 (8.8, 8.2, 8.8,
    // 9.6); 8 MB -, 10.1, 9.8, 9.7 (-, 10.3, 10.2, 10.7); f32 -> i8 of 20, 32 and 48 MB, 5, 8 and 12 vectors against 16: 13.9, 18.4; 18.4, 21.9;
    // 25.2, 26.7 (bf16 -> i8 15.3, 22.4; 20.8, 24.1; 28.4, 30.3).
    const int64_t per = units * 1024;
    int32_t nv = nvec <= per / 2 ? 1 : nvec <= per * 3 / 2 ? 2 : nvec <= per * 9 / 4 ? 3 : nvec <= per * 4 ? 4 : int32_t((nvec + per - 1) / per);
    const uint32_t grid = uint32_t((nvec + int64_t(1024) * nv - 1) / (int64_t(1024) * nv));
    // The smallest tensors' workgroups read all of x instead of waiting for each other, unless results lie over it: us, with the exchange and
    // so, f32 64 KiB 3.6, 3.2; 128 KiB 4.1, 3.7; 256 KiB 4.2, 4.8; 16 bits, twice the instructions a vector, 64 KiB 3.9, 3.7; 128 KiB 4.3, 4.4.
    const int64_t bytes = n * float_bytes(x_dtype);
    const bool alone = nvec <= (group == 4 ? 8192 : 4096) && apart(x, bytes, q, n) && (!y || apart(x, bytes, y, bytes));
    int32_t limit = alone ? -1 : g_wait_limit.load();
    void *args[] = {&x, &q, &y, &n, &qmax, &amax_out, &scale_out, &slot, &flags, &limit, &nv};
    return launch(st, KernelName("mtrt_dynqdq_") + xn + "_" + code_name(q_dtype) + "_v" + (nv <= 4 ? 4 : 16), grid, 1024,
                  as_hip(stream), args);
  }
  // Does not fit in the registers of one grid (or is not vector-aligned): the reduction, then the element-wise pass.
  const int32_t st1 = mtrt_hip_amax(stream, x, x_dtype, n, qmax, amax_out, scale_out);
  if (st1 != MTRT_OK)
    return st1;
  if (y)
    return qdq_dispatch(2, as_hip(stream), x, x_dtype, q, q_dtype, y, scale_out, MTRT_SCALE_UNIFORM, 1, n, 1, flags);
  return qdq_dispatch(0, as_hip(stream), x, x_dtype, q, q_dtype, nullptr, scale_out, MTRT_SCALE_UNIFORM, 1, n, 1, flags, true);
}

int32_t mtrt_hip_dynamic_quantize_rows(mtrt_stream_t stream, const void *x, int32_t x_dtype, void *q, int32_t q_dtype,
                                       int64_t rows, int64_t d, float qmax, float *amax_out, float *scale_out,
                                       int32_t flags) {
  clear_error();
  const char *xn = float_name(x_dtype);
  if (!xn)
    return set_error(MTRT_INVALID_ARGUMENT, "float operand dtype %d is not one of f32/f16/bf16", x_dtype);
  if (q_dtype != MTRT_I8 && q_dtype != MTRT_F8E4M3FN)
    return set_error(MTRT_INVALID_ARGUMENT, "dynamic per-row quantization targets i8 or f8E4M3FN, got dtype %d", q_dtype);
  if (rows < 0 || d < 0)
    return set_error(MTRT_INVALID_ARGUMENT, "negative extent [%lld, %lld]", (long long)rows, (long long)d);
  int64_t n;
  if (!element_count(rows, d, &n) || n >= (int64_t(1) << 35))
    return set_error(MTRT_INVALID_ARGUMENT, "[%lld, %lld] elements exceed the supported 2^35", (long long)rows, (long long)d);
  if (flags & ~(MTRT_Q_ROUND_TO_INT | MTRT_F8_REFHOST | MTRT_F8_VIA_F16))
    return set_error(MTRT_INVALID_ARGUMENT, "unknown flag bits 0x%x", flags);
  if ((flags & MTRT_F8_REFHOST) && (flags & MTRT_F8_VIA_F16))
    return set_error(MTRT_INVALID_ARGUMENT, "MTRT_F8_REFHOST and MTRT_F8_VIA_F16 name two different conversions; pass one");
  if (n == 0)
    return MTRT_OK;                                    // no row has an element: nothing is written
  if (!x || !q)
    return set_error(MTRT_INVALID_ARGUMENT, "null operand");
  if (!scale_out)
    return set_error(MTRT_INVALID_ARGUMENT, "scale_out must point at device memory for one f32 per row");
  if (!aligned(x, float_bytes(x_dtype)))
    return set_error(MTRT_INVALID_ARGUMENT, "float operand is not aligned to its element size");
  DeviceState *st = device_state();
  if (!st)
    return MTRT_RUNTIME_ERROR;
  // One launch while a row fits in the registers of a wave (up to 64 x 16 vectors) or of a workgroup's four waves
  // (up to 256 x 16 vectors): the row is read once.  Other rows (not whole vectors, operands off alignment, longer)
  // run as the two launches whose results this call is defined by.
  const int group = x_dtype == MTRT_F32 ? 4 : 8;
  const int64_t nvec = d / group;
  // A wave holds up to 8 vectors per lane, a workgroup's lanes up to 16; the 16-bit -> f8 pairs stop at 8 (their
  // 16-vector form would spill to scratch memory, whose allocation costs a launch some 10 us).
  const int max_group_nv = group == 8 && q_dtype == MTRT_F8E4M3FN ? 8 : 16;
  if (d % group == 0 && aligned(x, 16) && aligned(q, group) && nvec <= 256 * max_group_nv) {
    // A wave per row while that fills the chip (at least four waves per SIMD); with fewer rows the four waves of a
    // workgroup share each row, which puts four times the waves on the same loads (f16 [2048, 4096] 8.5 -> 7.5 us,
    // [4096, 4096] 12.7 -> 11.8 us; [8192, 4096] 22.7 against 23.4 us the other way).  Rows shorter than one vector
    // per lane of a workgroup stay with the wave form.
    const bool few_rows = rows <= int64_t(16) * num_compute_units(st) && nvec >= 256;
    const bool per_wave = nvec <= 64 * 8 && !few_rows;
    const int64_t lanes = per_wave ? 64 : 256;
    int nv = 1;
    while (lanes * nv < nvec)
      nv *= 2;
    const int64_t grid = per_wave ? (rows + 3) / 4 : rows;
    if (grid <= int64_t(kMaxGrid)) {
      void *args[] = {&x, &q, &rows, &d, &qmax, &amax_out, &scale_out, &flags};
      return launch(st, KernelName("mtrt_dynq_rows_") + xn + "_" + code_name(q_dtype) + (per_wave ? "_v" : "_g4v") + nv,
                    uint32_t(grid), kBlock, as_hip(stream), args);
    }
  }
  const int32_t st1 = mtrt_hip_amax_scales(stream, x, x_dtype, MTRT_SCALE_ROW, rows, d, rows, qmax, amax_out, scale_out);
  if (st1 != MTRT_OK)
    return st1;
  return qdq_dispatch(0, as_hip(stream), x, x_dtype, q, q_dtype, nullptr, scale_out, MTRT_SCALE_ROW, rows, d, rows, flags);
}

namespace {
// Vectors that a lane quantizes.  Few where the tensor gives each compute unit little, so that no wave works through a long chain of its own; 8
// where the launch is long; 2 again where the Infinity Cache keeps nothing of what the amax pass has read.  amax, quantize and dequantize
// in a row with 2, 4 and 8, us, bf16 (f32): 1 MiB 8.5, 8.8, 9.6 (8.3, 8.6, 9.2); 4 MiB 9.8, 10.1, 10.9 (9.6, 9.9, 10.5); 8 MiB 11.6, 11.8, 12.3
// (11.0, 11.1, 11.7); 16 MiB 14.9, 14.8, 15.3 (14.1, 13.9, 14.5); 32 MiB 23.3, 22.6, 22.8 (20.9, 20.2, 20.4); 48 MiB 32.1, 31.4, 31.1 (28.8, 27.7,
// 27.5); 128 MiB 72.4, 71.1, 71.4 (67.2, 67.1, 66.8); 192 MiB 108.5, 107.7, 109.1 (100.1, 101.2, 102.9); 256 MiB 142.4, 141.8, 143.9 (130.6, 133.0, 135.4).
int64_t nvfp4_trips(int64_t nvec, int64_t units) {
  const int64_t per = units * kBlock;
  if (nvec <= 8 * per || (nvec * 16 >= mtrt_dev::kReadTwiceBelow && nvec <= int64_t(1) << 32))   // (a launch has less than 2^32 work items)
    return 2;
  return nvec <= 32 * per ? 4 : 8;
}

int32_t nvfp4_dispatch(bool quantize, hipStream_t stream, const void *xy, int32_t dtype, const void *q, const void *scales,
                       const float *tensor_amax, int64_t d0, int64_t d1, int32_t block_axis) {
  clear_error();
  const char *xn = float_name(dtype);
  if (!xn)
    return set_error(MTRT_INVALID_ARGUMENT, "float operand dtype %d is not one of f32/f16/bf16", dtype);
  if (d0 < 0 || d1 < 0)
    return set_error(MTRT_INVALID_ARGUMENT, "negative extent [%lld, %lld]", (long long)d0, (long long)d1);
  if (block_axis != 0 && block_axis != 1)
    return set_error(MTRT_INVALID_ARGUMENT, "invalid axis! Axis can be either last (1) or second last (0) dimension of the [d0, d1] view, got %d",
                     block_axis);
  int64_t n;
  if (!element_count(d0, d1, &n) || n >= (int64_t(1) << 40))
    return set_error(MTRT_INVALID_ARGUMENT, "tensor of [%lld, %lld] elements is too large", (long long)d0, (long long)d1);
  const int64_t blocked = block_axis ? d1 : d0;
  if (blocked % 16 != 0)
    return set_error(MTRT_INVALID_ARGUMENT, "shape(input)[axis] must be divisible by 16, got %lld", (long long)blocked);
  if (d0 == 0 || d1 == 0)
    return MTRT_OK;
  if (!xy || !q || !scales || !tensor_amax)
    return set_error(MTRT_INVALID_ARGUMENT, "null operand");
  if (!aligned(xy, 16) || !aligned(q, 16) || !aligned(tensor_amax, 4) || !aligned(scales, 8))
    return set_error(MTRT_INVALID_ARGUMENT, "the float operand and the codes must be 16-byte aligned, the scales 8-byte aligned");
  DeviceState *st = device_state();
  if (!st)
    return MTRT_RUNTIME_ERROR;
  const int group = dtype == MTRT_F32 ? 4 : 8;
  if (block_axis == 0) {
    if (d1 % group != 0)
      return set_error(MTRT_INVALID_ARGUMENT, "blocks along the second-to-last axis need the last extent %% %d == 0, got %lld",
                       group, (long long)d1);
    const int64_t units = quantize ? 4 * (d0 / 16) * (d1 / group) : d0 * (d1 / group);   // lanes
    if ((units + kBlock - 1) / kBlock > int64_t(kMaxGrid) * 1024)
      return set_error(MTRT_INVALID_ARGUMENT, "tensor of %lld elements is too large", (long long)n);
    if (quantize) {
      void *args[] = {&xy, &q, &scales, &tensor_amax, &d0, &d1};
      return launch(st, KernelName("mtrt_nvfp4_qc_") + xn, uint32_t((units + kBlock - 1) / kBlock), kBlock, stream, args);
    }
    void *args[] = {&q, &scales, &tensor_amax, &xy, &d0, &d1};
    const int64_t blocks = std::min<int64_t>((units + kBlock - 1) / kBlock, int64_t(num_compute_units(st)) * 64);
    return launch(st, KernelName(nvfp4_cluster::numbers_fit(units) ? "mtrt_nvfp4_dqc_" : "mtrt_nvfp4_dqc_far_") + xn, uint32_t(blocks), kBlock, stream, args);
  }
  int64_t nvec = n / group;
  const int64_t trips = quantize ? nvfp4_trips(nvec, num_compute_units(st)) : 2;   // (kDqTrips)
  const int64_t per_block = kBlock * trips;
  const int64_t blocks = (nvec + per_block - 1) / per_block;
  if (blocks > int64_t(kMaxGrid) * 1024)
    return set_error(MTRT_INVALID_ARGUMENT, "tensor of %lld elements is too large", (long long)n);
  if (quantize) {
    void *args[] = {&xy, &q, &scales, &tensor_amax, &nvec};
    return launch(st, KernelName(trips == 2 ? "mtrt_nvfp4_q2_" : trips == 4 ? "mtrt_nvfp4_q4_" : "mtrt_nvfp4_q_") + xn, uint32_t(blocks), kBlock, stream, args);
  }
  // as many launches as it takes: each of whole workgroups, and a workgroup's vectors are whole blocks of 16
  const int64_t most = ((int64_t(1) << 32) / kBlock - 1) * per_block;
  for (int64_t at = 0; at < nvec; at += most) {
    int64_t some = std::min(most, nvec - at);
    const void *q_at = static_cast<const char *>(q) + at * group / 2, *s_at = static_cast<const char *>(scales) + at * group / 16,
               *y_at = static_cast<const char *>(xy) + at * 16;
    void *args[] = {&q_at, &s_at, &tensor_amax, &y_at, &some};
    const int32_t status = launch(st, KernelName("mtrt_nvfp4_dq_") + xn, uint32_t((some + per_block - 1) / per_block), kBlock, stream, args);
    if (status != MTRT_OK)
      return status;
  }
  return MTRT_OK;
}
} // namespace

int32_t mtrt_hip_nvfp4_quantize(mtrt_stream_t stream, const void *x, int32_t x_dtype, void *q_packed, void *scales,
                                const float *tensor_amax, int64_t d0, int64_t d1, int32_t block_axis) {
  return nvfp4_dispatch(true, as_hip(stream), x, x_dtype, q_packed, scales, tensor_amax, d0, d1, block_axis);
}

int32_t mtrt_hip_nvfp4_dequantize(mtrt_stream_t stream, const void *q_packed, const void *scales,
                                  const float *tensor_amax, void *y, int32_t y_dtype, int64_t d0, int64_t d1,
                                  int32_t block_axis) {
  return nvfp4_dispatch(false, as_hip(stream), y, y_dtype, q_packed, scales, tensor_amax, d0, d1, block_axis);
}

int32_t mtrt_hip_layernorm(mtrt_stream_t stream, const void *x, const void *gamma, const void *beta, void *y,
                           int32_t dtype, int64_t rows, int64_t d, float eps) {
  clear_error();
  const char *xn = float_name(dtype);
  if (!xn)
    return set_error(MTRT_INVALID_ARGUMENT, "layernorm dtype %d is not one of f32/f16/bf16", dtype);
  if (rows < 0 || d < 0)
    return set_error(MTRT_INVALID_ARGUMENT, "negative extent [%lld, %lld]", (long long)rows, (long long)d);
  int64_t n;
  if (!element_count(rows, d, &n) || n >= (int64_t(1) << 40))
    return set_error(MTRT_INVALID_ARGUMENT, "[%lld, %lld] elements exceed the supported 2^40", (long long)rows, (long long)d);
  if (rows == 0 || d == 0)
    return MTRT_OK;
  if (!x || !gamma || !beta || !y)
    return set_error(MTRT_INVALID_ARGUMENT, "null operand");
  const int eb = float_bytes(dtype);
  if (!aligned(x, eb) || !aligned(y, eb) || !aligned(gamma, eb) || !aligned(beta, eb))
    return set_error(MTRT_INVALID_ARGUMENT, "operand is not aligned to its element size");
  DeviceState *st = device_state();
  if (!st)
    return MTRT_RUNTIME_ERROR;
  const int per_vec = 16 / eb;
  const bool vec_ok = d % per_vec == 0 && aligned(x, 16) && aligned(y, 16) && aligned(gamma, 16) && aligned(beta, 16);
  const int nv = vec_ok ? pick_nv(d / per_vec) : 0;
  int64_t rows_arg = rows, d_arg = d;
  float eps_arg = eps;
  void *args[] = {&x, &gamma, &beta, &y, &rows_arg, &d_arg, &eps_arg};
  // Rows of at most 32 vectors: 8, 16 or 32 lanes per row, several rows to a wave (whatever the alignment).
  if (d / per_vec <= 32 && rows <= kMaxRowsPerWaveKernels) {
    const int lanes = d / per_vec <= 8 ? 8 : (d / per_vec <= 16 ? 16 : 32);
    return launch(st, KernelName("mtrt_layernorm_") + xn + "_u" + lanes + "v1", blocks_for(rows, kBlock / lanes), kBlock, as_hip(stream), args);
  }
  if (nv && rows <= kMaxRowsPerWaveKernels) {
    // One wave per row.  The eight-vector kernel runs five waves per SIMD; when that leaves a second, partly
    // filled round and eight waves per SIMD would hold every row at once, its 64-register form is faster.
    const int64_t simds = int64_t(num_compute_units(st)) * 4;
    const bool resident = nv == 8 && rows > 5 * simds && rows <= 8 * simds;
    return launch(st, KernelName("mtrt_layernorm_") + xn + "_v" + nv + (resident ? "r" : ""),
                  blocks_for(rows, kBlock / 64), kBlock, as_hip(stream), args);
  }
  int threads, gnv;
  if (vec_ok && !nv && rows <= int64_t(kMaxGrid) * 1024 && pick_group(d / per_vec, &threads, &gnv))
    return launch(st, KernelName("mtrt_layernorm_") + xn + "_g" + threads + "v" + gnv + row_form(true, dtype, false, threads, gnv, rows, d / per_vec, num_compute_units(st)), uint32_t(rows), uint32_t(threads),
                  as_hip(stream), args);
  // Row lengths that are not whole vectors, or operands that are not 16-byte aligned: the same two schemes with
  // 128-bit accesses at element alignment and the last d % per_vec elements of a row moved one by one.
  if (!vec_ok && d >= per_vec) {
    int rnv = pick_nv(d / per_vec);
    if (rnv && rows <= kMaxRowsPerWaveKernels) {
      rnv = unaligned_nv(dtype, rnv, true);
      return launch(st, KernelName("mtrt_layernorm_") + xn + "_u64v" + rnv + row_form(true, dtype, true, 64, rnv, rows, d / per_vec, num_compute_units(st)), blocks_for(rows, kBlock / 64), kBlock, as_hip(stream), args);
    }
    if (!rnv && rows <= int64_t(kMaxGrid) * 1024 && pick_group(d / per_vec, &threads, &gnv)) {
      gnv = unaligned_nv(dtype, gnv, true);
      return launch(st, KernelName("mtrt_layernorm_") + xn + "_u" + threads + "v" + gnv + row_form(true, dtype, true, threads, gnv, rows, d / per_vec, num_compute_units(st)), uint32_t(rows), uint32_t(threads),
                    as_hip(stream), args);
    }
  }
  return launch(st, KernelName("mtrt_layernorm_") + xn + "_any",
                uint32_t(std::min<int64_t>(rows, int64_t(num_compute_units(st)) * 8)), kBlock, as_hip(stream), args);
}

int32_t mtrt_hip_softmax(mtrt_stream_t stream, const void *x, void *y, int32_t dtype, int64_t rows, int64_t d) {
  clear_error();
  const char *xn = float_name(dtype);
  if (!xn)
    return set_error(MTRT_INVALID_ARGUMENT, "softmax dtype %d is not one of f32/f16/bf16", dtype);
  if (rows < 0 || d < 0)
    return set_error(MTRT_INVALID_ARGUMENT, "negative extent [%lld, %lld]", (long long)rows, (long long)d);
  int64_t n;
  if (!element_count(rows, d, &n) || n >= (int64_t(1) << 40))
    return set_error(MTRT_INVALID_ARGUMENT, "[%lld, %lld] elements exceed the supported 2^40", (long long)rows, (long long)d);
  if (rows == 0 || d == 0)
    return MTRT_OK;
  if (!x || !y)
    return set_error(MTRT_INVALID_ARGUMENT, "null operand");
  const int eb = float_bytes(dtype);
  if (!aligned(x, eb) || !aligned(y, eb))
    return set_error(MTRT_INVALID_ARGUMENT, "operand is not aligned to its element size");
  DeviceState *st = device_state();
  if (!st)
    return MTRT_RUNTIME_ERROR;
  const int per_vec = 16 / eb;
  const bool vec_ok = d % per_vec == 0 && aligned(x, 16) && aligned(y, 16);
  const int nv = vec_ok ? pick_nv(d / per_vec) : 0;
  int64_t rows_arg = rows, d_arg = d;
  void *args[] = {&x, &y, &rows_arg, &d_arg};
  const char *through = softmax_reads_past(rows, d * eb) ? "" : "t";
  // Rows of at most 32 vectors: 8, 16 or 32 lanes per row, several rows to a wave (whatever the alignment).
  if (d / per_vec <= 32 && rows <= kMaxRowsPerWaveKernels) {
    const int lanes = d / per_vec <= 8 ? 8 : (d / per_vec <= 16 ? 16 : 32);
    return launch(st, KernelName("mtrt_softmax_") + xn + "_u" + lanes + "v1" + through, blocks_for(rows, kBlock / lanes), kBlock, as_hip(stream), args);
  }
  if (nv && rows <= kMaxRowsPerWaveKernels)
    return launch(st, KernelName("mtrt_softmax_") + xn + "_v" + nv + (!*through && softmax_cuts(x, rows, d * eb) ? "c" : through),
                  blocks_for(rows, kBlock / 64), kBlock, as_hip(stream), args);
  int threads, gnv;
  if (vec_ok && !nv && rows <= int64_t(kMaxGrid) * 1024 && pick_group(d / per_vec, &threads, &gnv))
    return launch(st, KernelName("mtrt_softmax_") + xn + "_g" + threads + "v" + gnv + softmax_form(dtype, false, threads, gnv, rows, d / per_vec, num_compute_units(st)) + through, uint32_t(rows), uint32_t(threads),
                  as_hip(stream), args);
  // Row lengths that are not whole vectors, or operands that are not 16-byte aligned: the same two schemes with
  // 128-bit accesses at element alignment and the last d % per_vec elements of a row moved one by one.
  if (!vec_ok && d >= per_vec) {
    int rnv = pick_nv(d / per_vec);
    if (rnv && rows <= kMaxRowsPerWaveKernels) {
      rnv = unaligned_nv(dtype, rnv, false);
      return launch(st, KernelName("mtrt_softmax_") + xn + "_u64v" + rnv + through, blocks_for(rows, kBlock / 64), kBlock, as_hip(stream), args);
    }
    if (!rnv && rows <= int64_t(kMaxGrid) * 1024 && pick_group(d / per_vec, &threads, &gnv)) {
      gnv = unaligned_nv(dtype, gnv, false);
      return launch(st, KernelName("mtrt_softmax_") + xn + "_u" + threads + "v" + gnv + softmax_form(dtype, true, threads, gnv, rows, d / per_vec, num_compute_units(st)) + through, uint32_t(rows), uint32_t(threads),
                    as_hip(stream), args);
    }
  }
  return launch(st, KernelName("mtrt_softmax_") + xn + "_any",
                uint32_t(std::min<int64_t>(rows, int64_t(num_compute_units(st)) * 8)), kBlock, as_hip(stream), args);
}

int32_t mtrt_hip_gemm_w8a8_prepack(mtrt_stream_t stream, const void *w_kn, void *w_nk, int64_t K, int64_t N) {
  clear_error();
  if (K < 0 || N < 0 || K > kMaxMatrixExtent || N > kMaxMatrixExtent)
    return set_error(MTRT_INVALID_ARGUMENT, "extents [%lld, %lld] are negative or beyond 2^31 - 1", (long long)K, (long long)N);
  if (K == 0 || N == 0)
    return MTRT_OK;
  if (!w_kn || !w_nk)
    return set_error(MTRT_INVALID_ARGUMENT, "null operand");
  DeviceState *st = device_state();
  if (!st)
    return MTRT_RUNTIME_ERROR;
  const int64_t tiles = ((K + 63) / 64) * ((N + 63) / 64);
  if (tiles > int64_t(kMaxGrid) * 1024)
    return set_error(MTRT_INVALID_ARGUMENT, "weight matrix [%lld, %lld] is too large", (long long)K, (long long)N);
  void *args[] = {&w_kn, &w_nk, &K, &N};
  return launch(st, KernelName("mtrt_w8_prepack_kn_to_nk"), uint32_t(tiles), kBlock, as_hip(stream), args);
}

int32_t mtrt_hip_gemm_w8a8(mtrt_stream_t stream, const void *a, const void *w_nk, const float *a_scale,
                           const float *w_scale, void *y, int64_t M, int64_t K, int64_t N) {
  clear_error();
  if (M < 0 || K < 0 || N < 0)
    return set_error(MTRT_INVALID_ARGUMENT, "negative extent M=%lld K=%lld N=%lld", (long long)M, (long long)K,
                     (long long)N);
  if (M > kMaxMatrixExtent || K > kMaxMatrixExtent || N > kMaxMatrixExtent)
    return set_error(MTRT_INVALID_ARGUMENT, "matrix extents are limited to 2^31 - 1, got M=%lld K=%lld N=%lld", (long long)M,
                     (long long)K, (long long)N);
  if (M == 0 || N == 0)
    return MTRT_OK;
  if (!a_scale || !w_scale || !y || (K > 0 && (!a || !w_nk)))
    return set_error(MTRT_INVALID_ARGUMENT, "null operand");
  if (!aligned(y, 2))
    return set_error(MTRT_INVALID_ARGUMENT, "output is not aligned to its element size");
  DeviceState *st = device_state();
  if (!st)
    return MTRT_RUNTIME_ERROR;
  void *args[] = {&a, &w_nk, &a_scale, &w_scale, &y, &M, &K, &N};
  // The matrix-core kernel moves 128-byte K slices with 16-byte accesses.
  if (K > 0 && K % 128 == 0 && aligned(a, 16) && aligned(w_nk, 16) && M * K < (int64_t(1) << 32) &&
      N * K < (int64_t(1) << 32)) {
    // Up to 32 rows are bound by reading the weights once: one workgroup per 32 weight rows, its eight waves splitting K
    // and reading whole rows (3.4 TB/s of weights; the fragment-order entry point reaches 4).  A tile launch lasts
    // one 256-row tile's whole K loop per round whatever M is (about 8 us + 6 ns per k: M = 16, K = 4096, N = 11008
    // 32.7 us against 13.4; M = 32, K = N = 8192 57.1 against 18.6; M = 1, K = N = 4096 27.6 against 11.2), so it
    // only wins on very large weights.  33 to 64 rows take the form with two activation row tiles per weight fragment.
    const double tile_rounds = double(((N + 255) / 256 + num_compute_units(st) - 1) / num_compute_units(st));
    const double small_us = tuning::kRowsFixedUs + double(N) * double(K) / tuning::kRowsBytesPerUs;
    const double tile_us = (tuning::kTileFixedUs + tuning::kTileUsPerRowByte * double(K)) * tile_rounds;
    // 65 to 128 rows: four row tiles per weight fragment, one workgroup of four waves per compute unit at a time, so
    // the launch runs in rounds of about 3.7 ns per k (M = 128, K = N = 4096: 33 -> 18.4 us; K = N = 8192: 57 -> 30.7;
    // N = 11008 needs two rounds and equals the tile launch)
    const int64_t tiles32 = (N + 31) / 32;
    const double mid_us = tuning::kRows128FixedUs + tuning::kRows128UsPerRowByte * double(K) *
                                                        double((tiles32 + num_compute_units(st) - 1) / num_compute_units(st));
    if (M <= 64 ? small_us < tile_us : M <= 128 && mid_us < tile_us) {
      return launch(st, KernelName(M <= 32 ? "mtrt_gemm_w8a8_nk_rows32" : M <= 64 ? "mtrt_gemm_w8a8_nk_rows64" : "mtrt_gemm_w8a8_nk_rows128"),
                    uint32_t(std::min<int64_t>(tiles32, kLoopGrid)), M <= 64 ? 512 : 256, as_hip(stream), args);
    }
    Panels panels = panels_of(M, N, num_compute_units(st));
    if (panels.grid <= int64_t(kMaxGrid) * 1024) {
      void *fast_args[] = {&a, &w_nk, &a_scale, &w_scale, &y, &M, &K, &N, &panels.full};
      return launch(st, KernelName("mtrt_gemm_w8a8_nk"), uint32_t(panels.grid), kBlock, as_hip(stream), fast_args);
    }
  }
  if (K > 0) {
    // Any other K or alignment still goes to the matrix cores: 128 x 128 tiles with byte-aligned loads and a
    // zero-padded last k-step (M=4096 K=4100 N=11008: 1.2 s on the one-element-per-lane kernel below).
    const int64_t tiles = ((M + 127) / 128) * ((N + 127) / 128);
    uint32_t a_step = 1;
    const void *bias = nullptr;
    void *edge_args[] = {&a, &w_nk, &a_scale, &w_scale, &y, &M, &K, &N, &a_step, &bias};
    return launch(st, KernelName("mtrt_gemm_w8a8_nk_edge"), uint32_t(std::min<int64_t>(tiles, int64_t(kMaxGrid) * 1024)), kBlock,
                  as_hip(stream), edge_args);
  }
  return launch(st, KernelName("mtrt_gemm_w8a8_nk_any"), blocks_for(M * N, kBlock), kBlock, as_hip(stream), args);
}

int64_t mtrt_hip_gemm_w8a8_fragments_bytes(int64_t K, int64_t N) {
  if (K <= 0 || N <= 0 || K % 128 != 0 || K > kMaxMatrixExtent || N > kMaxMatrixExtent)
    return 0;
  return ((N + 31) / 32) * 32 * K;
}

int32_t mtrt_hip_gemm_w8a8_prepack_fragments(mtrt_stream_t stream, const void *w, int32_t w_is_nk, void *w_frag,
                                             int64_t K, int64_t N) {
  clear_error();
  if (K <= 0 || N <= 0 || K % 128 != 0 || K > kMaxMatrixExtent || N > kMaxMatrixExtent)
    return set_error(MTRT_INVALID_ARGUMENT, "fragment order needs positive extents below 2^31 and K %% 128 == 0, got K=%lld N=%lld",
                     (long long)K, (long long)N);
  if (!w || !w_frag)
    return set_error(MTRT_INVALID_ARGUMENT, "null operand");
  if (!aligned(w_frag, 16))
    return set_error(MTRT_INVALID_ARGUMENT, "fragment buffer must be 16-byte aligned");
  DeviceState *st = device_state();
  if (!st)
    return MTRT_RUNTIME_ERROR;
  const int64_t chunks = mtrt_hip_gemm_w8a8_fragments_bytes(K, N) / 16;
  void *args[] = {&w, &w_frag, &K, &N, &w_is_nk};
  return launch(st, KernelName("mtrt_w8_prepack_frag"), blocks_for(chunks, kBlock), kBlock, as_hip(stream), args);
}

namespace {
// Which kernel a W8A8 call on fragment-order weights takes.  Up to 32 rows: the four-wave kernels that read the weights once, with LDS for 16 or
// for 32 rows.
// 33 to 64 rows: the wave-private kernel or a tile, by estimate.  Above: the tile and K split frag_plan estimates fastest.
struct W8Plan {
  enum { kRows, kTile } kind;
  FragPlan tile;
};
W8Plan w8_plan(int64_t M, int64_t K, int64_t N, int64_t units, bool may_split) {
  if (M <= 32)
    return {W8Plan::kRows, {}};
  const FragPlan tile = frag_plan(M, N, K / 128, units, may_split);
  if (M <= 64 && frag_rows_us(M, N, K / 128, units) < tile.us)
    return {W8Plan::kRows, {}};
  return {W8Plan::kTile, tile};
}

// Whether the weights of up to 32 rows are read past the caches.
bool w8_few_rows_past(int64_t M, int64_t K, int64_t N, int64_t units) {
  const bool few_tiles = 2 * ((N + 31) / 32) <= units;
  return (M <= 16 && !few_tiles) || K * N < (few_tiles ? tuning::kThroughFromFewTiles : tuning::kThroughFrom) || K * N > tuning::kThroughUpTo;
}

// a_step: 1 for a scale per row, 0 for one scale; bias: f16 [N] or null; workspace: for K-split tiles, may be null.
int32_t w8a8_fragments(hipStream_t stream, const void *a, const void *w_frag, const float *a_scale, uint32_t a_step, const float *w_scale,
                       const void *bias, void *y, int64_t M, int64_t K, int64_t N, void *workspace, int64_t workspace_bytes) {
  if (M < 0 || K <= 0 || N < 0 || K % 128 != 0)
    return set_error(MTRT_INVALID_ARGUMENT, "fragment-order GEMM needs K %% 128 == 0 and non-negative extents, got M=%lld K=%lld N=%lld",
                     (long long)M, (long long)K, (long long)N);
  if (M > kMaxMatrixExtent || K > kMaxMatrixExtent || N > kMaxMatrixExtent)
    return set_error(MTRT_INVALID_ARGUMENT, "matrix extents are limited to 2^31 - 1, got M=%lld K=%lld N=%lld", (long long)M,
                     (long long)K, (long long)N);
  if (M == 0 || N == 0)
    return MTRT_OK;
  if (!a || !w_frag || !a_scale || !w_scale || !y)
    return set_error(MTRT_INVALID_ARGUMENT, "null operand");
  if (!aligned(y, 2) || !aligned(a, 16) || !aligned(w_frag, 16) || !aligned(bias, 2))
    return set_error(MTRT_INVALID_ARGUMENT, "a and w_frag must be 16-byte aligned, y and bias 2-byte aligned");
  if (M * K >= (int64_t(1) << 32))
    return set_error(MTRT_INVALID_ARGUMENT, "activations of %lld bytes exceed the kernel's 32-bit offsets", (long long)(M * K));
  DeviceState *st = device_state();
  if (!st)
    return MTRT_RUNTIME_ERROR;
  const int64_t units = num_compute_units(st), tiles32 = (N + 31) / 32;
  W8Plan plan = w8_plan(M, K, N, units, true);
  if (plan.kind == W8Plan::kTile && !bind_split(st, stream, plan.tile, workspace, workspace_bytes))
    plan = w8_plan(M, K, N, units, false);
  if (M <= 32 && tiles32 < (int64_t(1) << 24)) {
    // One workgroup per 32-column tile, its four waves splitting K; between one and two tiles per compute unit one workgroup per unit
    // instead, the first ones taking a second tile and the rows once for both: from 9 rows on (as for the int4 weights), and with more than 16
    // rows where K is long for the tiles that are left over (us, a workgroup to a tile and to a unit: 32 rows, K = 1152 and 288 tiles 4.8, 5.5; 2048 and 288
    // 8.0, 8.0, from memory 9.8, 9.1; 2048 and 344 8.1, 8.5; 4096 and 288 11.2, 10.6; 4096 and 444 12.5, 13.0; 6144 and 444 19.3, 18.2; 8192
    // and 512 30.7, 30.4).
    const bool over = tiles32 > units && tiles32 <= 2 * units;
    const bool pairs = over && (M > 16 ? K >= 2048 && (tiles32 - units) * 8192 <= K * units : M > 8);
    const uint32_t grid = uint32_t(pairs ? units : tiles32);
    int32_t past = w8_few_rows_past(M, K, N, units);
    void *args[] = {&a, &w_frag, &a_scale, &w_scale, &y, &M, &K, &N, &a_step, &bias, &past};
    return launch(st, KernelName(M <= 16 ? "mtrt_gemm_w8a8_small16" : "mtrt_gemm_w8a8_frag_rows32"), grid, kBlock, stream, args);
  }
  if (plan.kind == W8Plan::kRows) {
    void *args[] = {&a, &w_frag, &a_scale, &w_scale, &y, &M, &K, &N, &a_step, &bias};
    return launch(st, KernelName("mtrt_gemm_w8a8_frag_rows64"), uint32_t(std::min<int64_t>(tiles32, kLoopGrid)), 512, stream, args);
  }
  FragPlan &p = plan.tile;
  if (!p.tile)
    return set_error(MTRT_INVALID_ARGUMENT, "problem [%lld, %lld] needs too many tiles", (long long)M, (long long)N);
  if (p.tile->rows == 256 && p.tile->columns == 384) {
    void *args[] = {&a, &w_frag, &a_scale, &w_scale, &y, &M, &K, &N, &a_step, &bias};
    const bool plain = a_step == 1 && !bias;
    return launch(st, KernelName(plain ? "mtrt_gemm_w8a8_frag_t256x384" : "mtrt_gemm_w8a8_frag_t256x384_linear"), p.grid(), 256, stream, args);
  }
  void *args[] = {&a, &w_frag, &a_scale, &w_scale, &y, &M, &K, &N, &p.split, &a_step, &bias};
  return launch(st, KernelName("mtrt_gemm_w8a8_frag_") + p.tile->suffix, p.grid(), 256, stream, args);
}
} // namespace

int32_t mtrt_hip_gemm_w8a8_fragments(mtrt_stream_t stream, const void *a, const void *w_frag, const float *a_scale,
                                     const float *w_scale, void *y, int64_t M, int64_t K, int64_t N) {
  clear_error();
  return w8a8_fragments(as_hip(stream), a, w_frag, a_scale, 1, w_scale, nullptr, y, M, K, N, nullptr, 0);
}

int64_t mtrt_hip_gemm_w8a8_fragments_workspace(int64_t M, int64_t K, int64_t N) {
  if (M <= 32 || K <= 0 || N <= 0 || M > kMaxMatrixExtent || K > kMaxMatrixExtent || N > kMaxMatrixExtent)
    return 0;
  DeviceState *st = device_state();
  if (!st)
    return 0;
  const W8Plan plan = w8_plan(M, K, N, num_compute_units(st), true);
  return plan.kind == W8Plan::kTile && plan.tile.tile ? plan.tile.workspace() : 0;
}

int32_t mtrt_hip_gemm_w8a8_fragments_ws(mtrt_stream_t stream, const void *a, const void *w_frag, const float *a_scale,
                                        const float *w_scale, void *y, int64_t M, int64_t K, int64_t N, void *workspace,
                                        int64_t workspace_bytes) {
  clear_error();
  return w8a8_fragments(as_hip(stream), a, w_frag, a_scale, 1, w_scale, nullptr, y, M, K, N, workspace, workspace_bytes);
}

namespace {
// f32 products of few rows on the vector units (against the matrix cores' tiles: beside the kernels).  K below 1536 leaves four waves
// that share it unequal parts, so each takes columns of its own where that still gives every compute unit a workgroup (us, shared and
// own: (4, 448, 7680) 5.9, 4.8; (9, 1192, 3456) 9.8, 8.8; (4, 900, 900), 57 workgroups, 3.4, 4.6); more than four rows take eight
// columns to a wave where that leaves two workgroups to a unit (us, four and eight: (8, 4096, 4096) 17.0, 15.8; (12, 2048, 512) 4.9, 6.1).
struct DotShape {
  bool shared, wide;                                   // waves share K; eight columns to a wave
  int64_t grid;
};
DotShape dot_shape(int64_t M, int64_t K, int64_t N, int64_t units, bool may_be_wide) {
  const int64_t groups = (M + 7) / 8;
  auto blocks = [&](int64_t columns) { return (N + columns - 1) / columns; };
  DotShape s;
  s.shared = K >= tuning::kDotOwnColumnsBelow || blocks(M == 1 ? 8 : 16) * groups < units;
  s.wide = may_be_wide && M > 4 && K >= tuning::kDotOwnColumnsBelow && blocks(8) * groups >= 2 * units;
  s.grid = 8 * ((blocks((M == 1 ? 2 : s.wide ? 8 : 4) * (s.shared ? 1 : 4)) + 7) / 8) * groups;
  return s;
}

int32_t dense_few_rows_f32(DeviceState *st, hipStream_t stream, const DotShape &shape, const void *x, const void *w_nk, const void *bias, void *y, int64_t M, int64_t K,
                           int64_t N) {
  int32_t form = (shape.shared ? 1 : 0) | (M <= 8 && K * N > tuning::kWeightsPastBytes / 4 ? 2 : 0);
  void *args[] = {&x, &w_nk, &bias, &y, &M, &K, &N, &form};
  return launch(st, KernelName(M == 1 ? "mtrt_gemm_dense_rows1_f32" : M == 2 ? "mtrt_gemm_dense_rows2_f32" : M <= 4 ? "mtrt_gemm_dense_rows4_f32" :
                               shape.wide ? "mtrt_gemm_dense_rows8_wide_f32" : "mtrt_gemm_dense_rows8_f32"), uint32_t(shape.grid), kBlock, stream, args);
}
} // namespace

namespace {
// f32 products of more than 32 rows in 32 x 32 tiles whose K workgroups share: the parts with the shortest estimate, where it promises a twentieth
// against the same tiles unsplit; for tiles that have a ticket each, and at least one to an XCD.  Of fewer tiles parts would be the faster as well (us, whole and in
// parts, (64, 11072, 64) 57.3, 13.5; (64, 8192, 32) 43.1, 10.6; (50, 12288, 224) 63.5, 14.3; (33, 4096, 96) 22.6, 8.0; (65, 2048, 33) 13.0, 6.9; (33, 1024, 32) 7.9, 6.4): the line keeps
// products of six tiles, which a test holds to an unsplit kernel, where they are, and is not there for their time.
struct F32Split {
  FragSplit split;
  int64_t tiles = 0;
  double us = 0.0;
  int64_t workspace() const { return split.splits > 1 ? tiles * int64_t(split.splits) * 4096 : 0; }
};
F32Split make_f32_split(int64_t M, int64_t K, int64_t N, int64_t units) {
  F32Split best;
  best.tiles = ((M + 31) / 32) * ((N + 31) / 32);
  const int64_t steps = (K * 4 + 127) / 128;
  if (M <= 32 || best.tiles < 8 || best.tiles > int64_t(kTickets) || steps < 16)   // (eight slices to a part; the last one may have fewer)
    return best;
  const double alone = tuning::kF32FixedUs + (best.tiles <= units ? double(steps) * tuning::kF32FewTilesStepUs
                                                                  : (tuning::kF32TilesUs + double(steps) * tuning::kF32TilesStepUs) *
                                                                        std::max(1.0, double(best.tiles) / double(2 * units)));
  best.us = tuning::kF32SplitPromise * alone;
  for (int parts : {2, 3, 4, 6, 8}) {
    const FragSplit s = split_of(steps, parts);
    const double rounds = double((best.tiles * int64_t(s.splits) + units - 1) / units);
    const double us = tuning::kF32SplitUs + rounds * (tuning::kF32SplitRoundUs + tuning::kF32SplitStepUs * double(s.per));
    if (steps >= 8 * parts && us < best.us) {
      best.split = s;
      best.us = us;
    }
  }
  return best;
}
F32Split f32_split(int64_t M, int64_t K, int64_t N, int64_t units) {
  static thread_local LastPlan<F32Split> last;
  return last.of(M, N, K, units, true, [&] { return make_f32_split(M, K, N, units); });
}

int32_t linear_dense(mtrt_stream_t stream, const void *x, const void *w_nk, const void *bias, void *y, int32_t dtype, int64_t M, int64_t K, int64_t N,
                     void *workspace, int64_t workspace_bytes) {
  const char *xn = float_name(dtype);
  if (!xn)
    return set_error(MTRT_INVALID_ARGUMENT, "dense linear dtype %d is not one of f32/f16/bf16", dtype);
  if (M < 0 || K < 0 || N < 0)
    return set_error(MTRT_INVALID_ARGUMENT, "negative extent M=%lld K=%lld N=%lld", (long long)M, (long long)K,
                     (long long)N);
  if (M > kMaxMatrixExtent || K > kMaxMatrixExtent || N > kMaxMatrixExtent)
    return set_error(MTRT_INVALID_ARGUMENT, "matrix extents are limited to 2^31 - 1, got M=%lld K=%lld N=%lld", (long long)M,
                     (long long)K, (long long)N);
  if (M == 0 || N == 0)
    return MTRT_OK;
  if (!y || (K > 0 && (!x || !w_nk)))
    return set_error(MTRT_INVALID_ARGUMENT, "null operand");
  const int eb = float_bytes(dtype);
  if (!aligned(x, eb) || !aligned(w_nk, eb) || !aligned(y, eb) || !aligned(bias, eb))
    return set_error(MTRT_INVALID_ARGUMENT, "operand is not aligned to its element size");
  DeviceState *st = device_state();
  if (!st)
    return MTRT_RUNTIME_ERROR;
  const int64_t units = num_compute_units(st);
  const DotShape dot = dot_shape(M, K, N, units, true);
  const bool few = dtype == MTRT_F32 && M <= 32 && K >= 4 && K * N >= tuning::kDotMinWeights && launchable(dot.grid, kBlock);
  if (few && M <= 8)
    return dense_few_rows_f32(st, as_hip(stream), dot, x, w_nk, bias, y, M, K, N);
  const int64_t tiles32 = (N + 31) / 32, small_tiles = ((M + 31) / 32) * tiles32;
  F32Split split;
  if (dtype == MTRT_F32 && workspace && aligned(workspace, 16)) {
    split = f32_split(M, K, N, units);
    if (split.workspace() > workspace_bytes)
      split = F32Split();
  }
  // true: launched (or failed, in *rc) in parts, which take less than `us`
  const auto in_parts = [&](double us, bool ragged, int32_t *rc) {
    if (split.split.splits <= 1 || split.us >= us)
      return false;
    split.split.partial = workspace;
    split.split.tickets = split_tickets(st, as_hip(stream), uint32_t(split.tiles));
    if (!split.split.tickets)
      return false;
    void *sargs[] = {&x, &w_nk, &bias, &y, &M, &K, &N, &split.split};
    *rc = launch(st, KernelName(ragged ? "mtrt_gemm_dense_split_ragged_f32" : "mtrt_gemm_dense_split_f32"),
                 uint32_t(8 * ((split.tiles + 7) / 8) * int64_t(split.split.splits)), 512, as_hip(stream), sargs);
    return true;
  };
  int32_t rc;
  const bool whole_slices = K > 0 && (K * eb) % 128 == 0 && aligned(x, 16) && aligned(w_nk, 16);
  if (whole_slices && dtype == MTRT_F32) {
    // In 32 x 32 tiles, or up to 128 rows a column tile's rows together, or up to 32 on the vector units in groups of eight; in larger tiles where
    // they fill the chip.
    const double steps = double(K * eb / 128), rounds = double((tiles32 + units - 1) / units);
    const double rows_us = tuning::kF32FixedUs + rounds * steps * (M <= 32 ? tuning::kF32Rows32StepUs : M <= 64 ? tuning::kF32Rows64StepUs : tuning::kF32Rows128StepUs);
    if (M > 32) {
      const double tiles_us = tuning::kF32FixedUs + (small_tiles <= units ? steps * tuning::kF32FewTilesStepUs
                                                                          : (tuning::kF32TilesUs + steps * tuning::kF32TilesStepUs) * std::max(1.0, double(small_tiles) / double(2 * units)));
      const int64_t tiles128 = ((M + 127) / 128) * ((N + 127) / 128), rest128 = tiles128 % (2 * units), tiles256 = ((M + 255) / 256) * ((N + 127) / 128);
      const double one_us = tuning::kF32T128OneUs + steps * tuning::kF32T128OneStepUs, two_us = tuning::kF32T128TwoUs + steps * tuning::kF32T128TwoStepUs;
      const double t128_us = double(tiles128 / (2 * units)) * two_us + (rest128 == 0 ? 0.0 : rest128 <= units ? one_us : two_us);
      const double t256_us = double((tiles256 + units - 1) / units) * (tuning::kF32T256RoundUs + steps * tuning::kF32T256StepUs);
      const int64_t grid256 = 8 * ((tiles256 + 7) / 8);
      if (in_parts(std::min({t256_us, t128_us, tiles_us, M <= 128 && rounds <= tuning::kF32RowsRounds ? rows_us : tiles_us}), false, &rc))
        return rc;
      void *rargs[] = {&x, &w_nk, &bias, &y, &M, &K, &N};
      if (t256_us < std::min(t128_us, tiles_us) && M * K < (int64_t(1) << 30) && N * K < (int64_t(1) << 30) && launchable(grid256, kBlock))
        return launch(st, KernelName("mtrt_gemm_dense_t256x128_f32"), uint32_t(grid256), kBlock, as_hip(stream), rargs);
      if (t128_us < tiles_us)
        return launch(st, KernelName("mtrt_gemm_dense_t128x128_f32"), uint32_t(std::min<int64_t>(tiles128, kLoopGrid)), kBlock, as_hip(stream), rargs);
      // eight waves to a tile while there is a unit for each and (128 rows or more) K gives them slices; four beyond
      const bool tall = M <= 128 && rounds <= tuning::kF32RowsRounds && rows_us <= tiles_us, eight = small_tiles <= units && (M <= 128 || K >= 256);
      return launch(st, KernelName(tall ? (M <= 64 ? "mtrt_gemm_dense_rows64_tall_f32" : "mtrt_gemm_dense_rows128_tall_f32") :
                                   !eight ? "mtrt_gemm_dense_mfma_f32" : M <= 64 ? "mtrt_gemm_dense_rows64_f32" : "mtrt_gemm_dense_rows128_f32"),
                    uint32_t(std::min<int64_t>(tall ? tiles32 : 8 * ((small_tiles + 7) / 8), kLoopGrid)), tall ? (M <= 64 ? 512 : 256) : eight ? 512 : 256,
                    as_hip(stream), rargs);
    }
    const DotShape in_groups = dot_shape(M, K, N, units, false);
    int32_t as_tiles = !few || !launchable(in_groups.grid, kBlock) ||
                       rows_us < tuning::kF32FixedUs + double((M + 7) / 8) * 4.0 * double(K * N) / tuning::kDotGroupBytesPerUs;
    int32_t form = in_groups.shared;
    void *fargs[] = {&x, &w_nk, &bias, &y, &M, &K, &N, &as_tiles, &form};
    return launch(st, KernelName("mtrt_gemm_dense_rows32_f32"), uint32_t(as_tiles ? std::min<int64_t>(tiles32, kLoopGrid) : in_groups.grid),
                  as_tiles ? 512 : kBlock, as_hip(stream), fargs);
  }
  // 16-bit.  Decode-sized calls are bound by reading the weights once: up to 32 rows take one workgroup per 32 weight rows, its
  // eight waves splitting K (f16 M = 16, K = 4096, N = 11008: 55 us on the tile loop, 23.3 so, 3.9 TB/s of weights); 33 to 64 rows the form with two activation row tiles per weight fragment; the tile loop (about
  // 8 us + 6 ns per byte of a row, per round) only wins on very large weights.
  const double tile_us = (tuning::kTileFixedUs + tuning::kTileUsPerRowByte * double(K * eb)) *
                         double(((N + 255) / 256 + num_compute_units(st) - 1) / num_compute_units(st));
  const double small_us = tuning::kRowsFixedUs + double(N) * double(K * eb) / tuning::kRowsWideBytesPerUs;
  // 65 to 128 rows: four row tiles per weight fragment, rounds of one workgroup per compute unit (3.7 ns per byte of a row)
  const double mid_us = tuning::kRows128FixedUs + tuning::kRows128UsPerRowByte * double(K * eb) *
                                                      double((tiles32 + num_compute_units(st) - 1) / num_compute_units(st));
  if (whole_slices && (M <= 64 ? small_us < tile_us : M <= 128 && mid_us < tile_us)) {
    void *rargs[] = {&x, &w_nk, &bias, &y, &M, &K, &N};
    return launch(st, KernelName(M <= 32 ? "mtrt_gemm_dense_rows32_" : M <= 64 ? "mtrt_gemm_dense_rows64_" : "mtrt_gemm_dense_rows128_") + xn,
                  uint32_t(std::min<int64_t>(tiles32, kLoopGrid)), M <= 64 ? 512 : 256, as_hip(stream), rargs);
  }
  if (K > 0 && (K * eb) % 128 == 0 && aligned(x, 16) && aligned(w_nk, 16) && M * K * eb < (int64_t(1) << 32) &&
      N * K * eb < (int64_t(1) << 32)) {
    // operands in whole 128-byte slices of K: the matrix-core tile loop (tiles and rounds as in
    // mtrt_hip_gemm_w8a8; f16 [2048, 4096] x [11008, 4096]: 3654 us on the FMA kernel below)
    Panels panels = panels_of(M, N, units);
    if (panels.grid <= int64_t(kMaxGrid) * 1024) {
      void *margs[] = {&x, &w_nk, &bias, &y, &M, &K, &N, &panels.full};
      return launch(st, KernelName("mtrt_gemm_dense_mfma_") + xn, uint32_t(panels.grid), kBlock, as_hip(stream), margs);
    }
  }
  void *args[] = {&x, &w_nk, &bias, &y, &M, &K, &N};
  if (K > 0) {
    // any other K or alignment: element-aligned loads and a zero-padded last k-step, in 128 x 128 tiles
    // (f16 [2048, 4100] x [11008, 4100]: 3761 us on the FMA kernel below) or 32 x 32 ones whose K the waves share
    const int64_t edge_tiles = ((M + 127) / 128) * ((N + 127) / 128);
    const double steps = double((K * eb + 127) / 128);
    const double edge_us = tuning::kEdgeFixedUs + steps * (dtype == MTRT_F32 ? tuning::kEdgeF32StepUs : tuning::kEdge16StepUs) *
                                                      double((edge_tiles + units - 1) / units);
    const double small_us = tuning::kEdgeSmallFixedUs + steps * (small_tiles <= units ? tuning::kEdgeSmallFewStepUs
                                                                                      : tuning::kEdgeSmallStepUs * std::max(1.0, double(small_tiles) / double(2 * units)));
    // up to 32 rows of f32 may be read in groups of eight as well: us, 32 x 32 tiles and so, (9, 1192, 3456) 10.9, 9.4; (16, 1031, 260) 9.1,
    // 4.4; (16, 600, 8000) 9.1, 9.9; (32, 4097, 4096) 38.7, 40.5
    if (few && 3.0 + double((M + 7) / 8) * 4.0 * double(K * N) / tuning::kDotGroupBytesPerUs < std::min(small_us, edge_us))
      return dense_few_rows_f32(st, as_hip(stream), dot, x, w_nk, bias, y, M, K, N);
    if (in_parts(std::min(small_us, edge_us), true, &rc))
      return rc;
    int32_t waves = 0;
    if (K * eb >= 16 && small_us < edge_us)
      waves = dtype == MTRT_F32 && small_tiles <= units ? 8 : 4;
    void *eargs[] = {&x, &w_nk, &bias, &y, &M, &K, &N, &waves};
    return launch(st, KernelName("mtrt_gemm_dense_edge_") + xn, uint32_t(std::min<int64_t>(waves ? 8 * ((small_tiles + 7) / 8) : edge_tiles, kLoopGrid)),
                  waves ? uint32_t(64 * waves) : kBlock, as_hip(stream), eargs);
  }
  const int64_t tiles = ((M + 63) / 64) * ((N + 63) / 64);
  if (tiles > int64_t(kMaxGrid) * 1024)
    return set_error(MTRT_INVALID_ARGUMENT, "problem [%lld, %lld] needs too many tiles", (long long)M, (long long)N);
  return launch(st, KernelName("mtrt_gemm_dense_") + xn, uint32_t(tiles), kBlock, as_hip(stream), args);
}
} // namespace

int32_t mtrt_hip_linear_dense(mtrt_stream_t stream, const void *x, const void *w_nk, const void *bias, void *y, int32_t dtype, int64_t M, int64_t K,
                              int64_t N) {
  clear_error();
  return linear_dense(stream, x, w_nk, bias, y, dtype, M, K, N, nullptr, 0);
}

namespace {
// The re-laid weights hold two layouts back to back: fragment order for the 32 x 32 matrix-core tiles (per 32
// columns and 64 k: 64 lanes x 16 bytes) and, when K is a multiple of 128, strip order for the M <= 16 kernel
// (per 16 columns and 128 k: 64 lanes x 16 bytes).
int64_t w4_fragment_bytes(int64_t K, int64_t N) { return ((N + 31) / 32) * (K / 64) * 1024; }
int64_t w4_strip_bytes(int64_t K, int64_t N) { return K % 128 == 0 ? ((N + 15) / 16) * (K / 128) * 1024 : 0; }
} // namespace

int64_t mtrt_hip_gemm_w4a16_prepacked_bytes(int64_t K, int64_t N) {
  if (K <= 0 || N <= 0 || K % 64 != 0 || K > kMaxMatrixExtent || N > kMaxMatrixExtent)
    return 0;
  return w4_fragment_bytes(K, N) + w4_strip_bytes(K, N);
}

int32_t mtrt_hip_gemm_w4a16_prepack(mtrt_stream_t stream, const void *w_kn_packed, void *w_prepacked, int64_t K,
                                    int64_t N) {
  clear_error();
  if (K <= 0 || N <= 0 || K % 64 != 0 || K > kMaxMatrixExtent || N > kMaxMatrixExtent)
    return set_error(MTRT_INVALID_ARGUMENT, "prepack needs positive extents below 2^31 and K %% 64 == 0, got K=%lld N=%lld",
                     (long long)K, (long long)N);
  if (!w_kn_packed || !w_prepacked)
    return set_error(MTRT_INVALID_ARGUMENT, "null operand");
  if (!aligned(w_prepacked, 16))
    return set_error(MTRT_INVALID_ARGUMENT, "prepacked buffer must be 16-byte aligned");
  DeviceState *st = device_state();
  if (!st)
    return MTRT_RUNTIME_ERROR;
  const int64_t dwords = w4_fragment_bytes(K, N) / 4;
  void *args[] = {&w_kn_packed, &w_prepacked, &K, &N};
  const int32_t rc = launch(st, KernelName("mtrt_w4_prepack"), blocks_for(dwords, kBlock), kBlock, as_hip(stream), args);
  if (rc != MTRT_OK || w4_strip_bytes(K, N) == 0)
    return rc;
  void *strips = static_cast<char *>(w_prepacked) + w4_fragment_bytes(K, N);
  void *args2[] = {&w_kn_packed, &strips, &K, &N};
  return launch(st, KernelName("mtrt_w4_prepack_strips"), blocks_for(w4_strip_bytes(K, N) / 4, kBlock), kBlock, as_hip(stream), args2);
}

namespace {
bool w4_fast(const void *a, const void *w_prepacked, int64_t K, int64_t block) {
  return w_prepacked && K > 0 && K % 64 == 0 && block % 64 == 0 && aligned(a, 16) && aligned(w_prepacked, 16);
}

// Whether the strip kernel (16 rows by 16 columns over all of K, four waves) takes a product.  Up to 16 rows: blocks of 64 where each wave
// has a slice of 128 k; the kernel behind, with slices of 64, is as fast below that.
// 17 to 512 rows in groups of 16, where the 32-row kernel and the tiles leave most of the chip idle.  The lines are by the number of 16-column tiles that a
// workgroup has side by side when there is one to a compute unit (`each`), and by K, on which a workgroup walks alone.  How many times as long the
// others take (geometric means over 569 products, blocks of 64 and of 128 alike):
//                        K up to 255   511  1023  1407  2559  5000  6144  9000 12288 14336
//   one, more than 32 rows      1.14  1.35  1.71  2.05  1.92  1.95  1.86  1.67  1.44  1.41
//   one, up to 32 rows          1.12  1.14  1.19  1.29  1.31  1.48  1.65  1.72  1.79     -
//   two, more than 32 rows      1.01  1.18  1.39  1.69  1.62  1.71  1.52  1.39  1.13  1.00
//   two, up to 32 rows          0.98     -  1.03  1.07     -  1.10  1.23     -     -     -
//   three, more than 32 rows    0.93  1.04  1.17  1.47  1.45  1.35  1.37  1.15  0.97     -
//   three, up to 32 rows           -  0.91     -     -     -     -  1.04  1.02     -     -
//   four                        0.77  0.85  1.00  1.21  0.95  1.15  0.84  0.86  0.77     -
// us, the others and this: (119, 512, 384) 4.6, 3.0; (59, 1152, 302) 6.7, 3.2; (211, 6784, 384) 11.7, 7.9; (64, 8192, 96) 9.8, 6.1; (54, 5120, 4032), four, 12.0,
// 10.8; (186, 4224, 1664), five, 11.8, 12.8.
bool w4_strips(int64_t M, int64_t K, int64_t N, int64_t block, int64_t units) {
  if (K % 128 != 0 || (block != 64 && block % 128 != 0) || M > 512 || M * K > (int64_t(1) << 31))
    return false;
  if (M <= 16)
    return block != 64 || K >= 512;
  const int64_t groups = (M + 15) / 16, tiles = (N + 15) / 16, most = std::max<int64_t>(units / groups, 1), each = (tiles + most - 1) / most;
  if (M <= 32)
    return each == 1 || (each == 2 && K >= 1024);
  return each == 1 || (each == 2 && K >= 256 && K <= 12288) || (each == 3 && K >= 512 && K <= 9216);
}

// bias: f16 [N], added to the rounded product, or null (only with re-laid weights)
int32_t w4a16(hipStream_t stream, const void *a, const void *w_kn_packed, const void *w_prepacked, const void *scale, const void *bias, void *y,
              int64_t M, int64_t K, int64_t N, int64_t block, void *workspace, int64_t workspace_bytes) {
  if (M < 0 || K < 0 || N < 0)
    return set_error(MTRT_INVALID_ARGUMENT, "negative extent M=%lld K=%lld N=%lld", (long long)M, (long long)K,
                     (long long)N);
  if (M > kMaxMatrixExtent || K > kMaxMatrixExtent || N > kMaxMatrixExtent)
    return set_error(MTRT_INVALID_ARGUMENT, "matrix extents are limited to 2^31 - 1, got M=%lld K=%lld N=%lld", (long long)M,
                     (long long)K, (long long)N);
  if (M == 0 || N == 0)
    return MTRT_OK;
  if (block <= 0 || (K > 0 && K % block != 0))
    return set_error(MTRT_INVALID_ARGUMENT, "block size %lld does not divide K=%lld", (long long)block, (long long)K);
  if (!y || (K > 0 && (!a || !scale)) || (!w_kn_packed && !w_prepacked && K > 0))
    return set_error(MTRT_INVALID_ARGUMENT, "null operand");
  if (!aligned(a, 2) || !aligned(y, 2) || !aligned(scale, 2) || !aligned(bias, 2))
    return set_error(MTRT_INVALID_ARGUMENT, "operand is not aligned to its element size");
  DeviceState *st = device_state();
  if (!st)
    return MTRT_RUNTIME_ERROR;
  if (w4_fast(a, w_prepacked, K, block)) {
    const int64_t cus = num_compute_units(st);
    void *args[] = {&a, &w_prepacked, &scale, &y, &M, &K, &N, &block, &bias};
    // (rows of activations are addressed by 32-bit offsets below)
    if (w4_strips(M, K, N, block, cus)) {
      // 16-column tiles over all of K (weights in strip order).  One workgroup per compute unit; up to 16 rows two for more than three
      // tiles a unit, which a workgroup would take one after the other (K = 4096, M = 16: 768 tiles 9.0 against 10.6 us, 864 tiles
      // 12.3 against 11.9, 1024 tiles 12.9 against 12.3), and with up to four rows for more than one (M = 1: 320 tiles 5.6 against
      // 5.2 us, 688 tiles 7.4 against 7.1, 1024 tiles 10.2 against 9.8); more rows' groups share the units ((22, 13056, 2880) 12.9 against 17.0).
      const void *in_strips = static_cast<const char *>(w_prepacked) + w4_fragment_bytes(K, N);
      void *sargs[] = {&a, &in_strips, &scale, &y, &M, &K, &N, &block, &bias};
      const int64_t tiles = (N + 15) / 16, groups = (M + 15) / 16;
      const int64_t most = groups > 1 ? std::max<int64_t>(cus / groups, 1) : M <= 4 || tiles > 3 * cus ? 2 * cus : cus;
      return launch(st, KernelName(block == 64 ? "mtrt_gemm_w4a16_strips16_b64" : "mtrt_gemm_w4a16_strips16"),
                    uint32_t(std::min<int64_t>(tiles, most) * groups), kBlock, stream, sargs);
    }
    if (M <= 32 && M * K <= (int64_t(1) << 31)) {
      // one workgroup per 32-column tile; between one and two tiles per compute unit, one workgroup per
      // compute unit instead (the kernel then gives workgroup g the tiles g and g + grid, which share the
      // activations; measured: 6 % faster at M = 16, 21 % at M = 32, 3 % slower at M = 5)
      const int64_t tiles = (N + 31) / 32;
      const uint32_t grid = uint32_t(M > 8 && tiles > cus && tiles <= 2 * cus ? cus : tiles);
      return launch(st, KernelName(M <= 16 ? "mtrt_gemm_w4a16_skinny16" : "mtrt_gemm_w4a16_skinny"), grid, kBlock, stream, args);
    }
    if (M * K * 2 < (int64_t(1) << 32)) {
      W4Plan p = w4_plan(M, K, N, cus, true);
      if (!bind_split(st, stream, p, workspace, workspace_bytes))
        p = w4_plan(M, K, N, cus, false);
      if (p.tile) {
        KernelName name("mtrt_gemm_w4a16_");
        name + (p.narrow ? "t128x64" : p.tile->suffix) + (bias ? "_bias" : "");
        if (p.tile->rows == 256)
          return launch(st, name, p.grid(), p.tile->threads, stream, args);
        void *targs[] = {&a, &w_prepacked, &scale, &y, &M, &K, &N, &block, &bias, &p.split};
        return launch(st, name, p.grid(), p.narrow ? 256 : p.tile->threads, stream, targs);
      }
    }
  }
  if (!w_kn_packed || bias)
    return set_error(MTRT_INVALID_ARGUMENT, "this shape needs the original packed weights (K=%lld block=%lld)",
                     (long long)K, (long long)block);
  void *args[] = {&a, &w_kn_packed, &scale, &y, &M, &K, &N, &block};
  if (K > 0) {
    // any block, K, N and alignment from the original nibbles, still on the matrix cores: 128 x 128 tiles whose
    // weight stage is dequantised in the kernel (M = 256, K = N = 4096, block 32: 3660 us on the kernel below)
    const int64_t tiles = ((M + 127) / 128) * ((N + 127) / 128);
    return launch(st, KernelName("mtrt_gemm_w4a16_edge"), uint32_t(std::min<int64_t>(tiles, int64_t(kMaxGrid) * 1024)), kBlock,
                  stream, args);
  }
  return launch(st, KernelName("mtrt_gemm_w4a16_any"), blocks_for(M * N, kBlock), kBlock, stream, args);
}
} // namespace

int32_t mtrt_hip_gemm_w4a16(mtrt_stream_t stream, const void *a, const void *w_kn_packed, const void *w_prepacked,
                            const void *scale, void *y, int64_t M, int64_t K, int64_t N, int64_t block) {
  clear_error();
  return w4a16(as_hip(stream), a, w_kn_packed, w_prepacked, scale, nullptr, y, M, K, N, block, nullptr, 0);
}

int64_t mtrt_hip_gemm_w4a16_workspace(int64_t M, int64_t K, int64_t N, int64_t block) {
  if (M <= 32 || K <= 0 || N <= 0 || block <= 0 || K % 64 != 0 || block % 64 != 0 || M > kMaxMatrixExtent || K > kMaxMatrixExtent ||
      N > kMaxMatrixExtent || M * K * 2 >= (int64_t(1) << 32))
    return 0;
  DeviceState *st = device_state();
  if (!st)
    return 0;
  if (w4_strips(M, K, N, block, num_compute_units(st)))
    return 0;
  const W4Plan p = w4_plan(M, K, N, num_compute_units(st), true);
  return p.tile ? p.workspace() : 0;
}

int32_t mtrt_hip_gemm_w4a16_ws(mtrt_stream_t stream, const void *a, const void *w_kn_packed, const void *w_prepacked, const void *scale,
                               void *y, int64_t M, int64_t K, int64_t N, int64_t block, void *workspace, int64_t workspace_bytes) {
  clear_error();
  return w4a16(as_hip(stream), a, w_kn_packed, w_prepacked, scale, nullptr, y, M, K, N, block, workspace, workspace_bytes);
}

namespace {
// Dense GEMM on fragment-order 16-bit weights: x [M,K] (K % 64 == 0, 16-byte aligned).  Up to 64 rows by estimate either the
// wave-private kernel that reads the weights once or a tile; above, the tile and K split of frag_plan.
struct DensePlan {
  bool rows = false;
  FragPlan tile;
};
DensePlan dense_frag_plan(int64_t M, int64_t K, int64_t N, int64_t units, bool may_split) {
  DensePlan p;
  p.tile = frag_plan(M, N, K / 64, units, may_split);
  p.rows = M <= 64 && (!p.tile.tile || frag_rows_us(M, N, K / 64, units) < p.tile.us);
  return p;
}
// w_scale: of float8 codes (f32 [N]), null where w_frag holds the weights themselves
int32_t dense_fragments(DeviceState *st, hipStream_t stream, const void *x, const void *w_frag, const float *w_scale, const void *bias, void *y,
                        int32_t dtype, int64_t M, int64_t K, int64_t N, void *partial, int64_t partial_bytes) {
  DensePlan plan = dense_frag_plan(M, K, N, num_compute_units(st), true);
  if (!plan.rows && !bind_split(st, stream, plan.tile, partial, partial_bytes))
    plan = dense_frag_plan(M, K, N, num_compute_units(st), false);
  const char *xn = float_name(dtype);
  KernelName name("mtrt_gemm_dense_frag_");
  name + xn + (w_scale ? "_f8_" : "_") + (plan.rows ? (M <= 32 ? "rows32" : "rows64") : plan.tile.tile ? plan.tile.tile->suffix : "");
  if (!plan.rows && !plan.tile.tile)
    return set_error(MTRT_INVALID_ARGUMENT, "problem [%lld, %lld] needs too many tiles", (long long)M, (long long)N);
  const uint32_t grid = plan.rows ? uint32_t(std::min<int64_t>((N + 31) / 32, int64_t(kMaxGrid) * 1024)) : plan.tile.grid(), block = plan.rows ? 512 : 256;
  if (plan.rows || (plan.tile.tile->columns == 384 && plan.tile.tile->rows == 256)) {
    void *args[] = {&x, &w_frag, &bias, &y, &M, &K, &N, &w_scale};
    return launch(st, name, grid, block, stream, args);
  }
  void *args[] = {&x, &w_frag, &bias, &y, &M, &K, &N, &plan.tile.split, &w_scale};
  return launch(st, name, grid, block, stream, args);
}

int64_t round_up(int64_t v, int64_t step) { return (v + step - 1) / step * step; }

// How a plan's call runs: the row length its GEMM sees, whether x goes through the activation pass, and the two parts of the
// workspace (the pass's result, then the partial tiles).
// A decode step's Linear takes (and quantizes) its activations inside the GEMM, mtrt_linear_w8a8_decode and mtrt_gemm_dense_frag_*_rows16*,
// up to this many of them.
constexpr int64_t kDecodeElements = 16384;
struct LinearShape {
  bool fragments = false, pass = false, one_launch = false;
  int64_t Kp = 0, act_bytes = 0, partial_bytes = 0;
};
LinearShape linear_shape(const mtrt_hip_linear_plan &p, int64_t M, int64_t units) {
  LinearShape s;
  const bool quantized = p.q_dtype >= 0;
  const int eb = float_bytes(p.dtype);
  s.Kp = p.K;
  if (p.route == MTRT_LINEAR_W8A8) {
    s.fragments = p.w_frag != nullptr;
    s.Kp = s.fragments ? round_up(p.K, 128) : p.K;
    s.one_launch = s.fragments && M <= 16 && M * s.Kp <= kDecodeElements;
    s.pass = !s.one_launch;
    s.act_bytes = s.pass ? round_up(M * s.Kp, 256) : 0;
    if (s.fragments && M > 32) {
      const W8Plan w = w8_plan(M, s.Kp, p.N, units, true);
      s.partial_bytes = w.kind == W8Plan::kTile && w.tile.tile ? w.tile.workspace() : 0;
    }
  } else if (p.route == MTRT_LINEAR_DENSE || p.route == MTRT_LINEAR_DENSE_F8W) {
    // A K that is no whole number of slices costs an unquantized x a pass of its own (2.3 us and up), so small products
    // stay on the kernel that takes any K (about 15 us at a gigaflop).
    s.fragments = p.w_frag && eb == 2 && (p.K % 64 == 0 || !p.w || p.route == MTRT_LINEAR_DENSE_F8W || quantized || 2.0 * double(M) * double(p.K) * double(p.N) >= 1e9);
    s.Kp = s.fragments ? round_up(p.K, 64) : p.K;
    // Up to 16 rows in one launch.  Its 16-column workgroups each take x: where they are at most one to a compute unit, twice as many
    // elements (bf16, float8 inputs, us, two launches and one: (8, 4096, 4096) 11.3, 10.1, (2, 14336, 512) 18.5, 12.7; (16, 1536, 8192) 9.4, 11.5);
    // where they are more than two, half as many to quantize ((16, 1024, 16384) 10.1, 11.4; (8, 1024, 16384) 9.7, 8.5; (16, 1024, 8192) 7.2,
    // 6.8); and a plain x that needs no pass only saves the 32-column kernel's way to its rows, from 1024 elements a row (us, that and
    // this, bf16: (16, 512, 8192) 3.6, 4.2; (8, 768, 8192) 3.9, 4.1; (8, 1024, 8192) 4.2, 4.2; (4, 1024, 12000) 6.7, 5.2; (8, 2048, 8192) 5.1, 4.5.
    // Weights read from memory; where they lie in the Infinity Cache already two launches are the faster between two and three workgroups to
    // a unit, (1, 1024, 11008) 6.2, 6.9 against 8.8, 7.9.)
    const bool passes = quantized || s.Kp != p.K;
    const int64_t tiles16 = (p.N + 15) / 16, most = tiles16 <= units ? 2 * kDecodeElements : passes && tiles16 > 2 * units ? kDecodeElements / 2 : kDecodeElements;
    s.one_launch = s.fragments && M <= 16 && M * s.Kp <= most && launchable(tiles16, 512) && (passes || tiles16 <= units || s.Kp >= 1024);
    s.pass = !s.one_launch && passes;
    s.act_bytes = passes ? round_up(M * s.Kp * eb, 256) : 0;   // asked for, not used, where the GEMM takes x itself
    if (s.fragments) {
      const DensePlan d = dense_frag_plan(M, s.Kp, p.N, units, true);
      s.partial_bytes = !d.rows && d.tile.tile ? d.tile.workspace() : 0;
    } else if (eb == 4) {
      s.partial_bytes = f32_split(M, p.K, p.N, units).workspace();
    }
  }
  return s;
}

// Rows of one launch: the fragment kernels address the activations by 32-bit offsets, so more than 4 GiB of them go in parts.
int64_t linear_rows(const mtrt_hip_linear_plan &p, int64_t M) {
  const int64_t row = round_up(p.K, 128) * float_bytes(p.dtype);
  return M * row < (int64_t(1) << 32) ? M : std::max<int64_t>(1, ((int64_t(1) << 32) - 1) / row / 256 * 256);
}

// x [M,K] -> out [M,Kp]: codes (codes != 0), dequantized codes, or (q_dtype < 0) the values, padded with zeros
int32_t activation_pass(DeviceState *st, hipStream_t stream, bool codes, const void *x, int32_t dtype, int32_t q_dtype, const float *scale,
                        void *out, int64_t M, int64_t K, int64_t Kp) {
  if (Kp == K) {
    // no padding between the rows: one row of all elements, so that a short row does not leave most of a wave idle and a row
    // that is no whole number of groups needs none; the last group's padding lies in the workspace's own rounding
    K *= M;
    M = 1;
    Kp = round_up(K, 16);
  }
  const int group = dtype == MTRT_F32 ? 4 : 8;
  const int64_t chunks = (Kp / group + 127) / 128;
  KernelName name(q_dtype < 0 ? "mtrt_act_pad_b16" : codes ? "mtrt_act_codes_" : "mtrt_act_fake_");
  if (q_dtype >= 0)
    name + float_name(dtype) + "_" + code_name(q_dtype);
  void *args[] = {&x, &out, &scale, &M, &K, &Kp};
  return launch(st, name, blocks_for(M * chunks, kBlock / 64), kBlock, stream, args);
}

// What of a plan is wrong, or nullptr.
const char *linear_fault(const mtrt_hip_linear_plan *p, int64_t M) {
  if (!p)
    return "null plan";
  if (p->route < MTRT_LINEAR_W8A8 || p->route > MTRT_LINEAR_DENSE_F8W || !float_name(p->dtype))
    return "unknown route or dtype";
  if (M < 0 || p->K <= 0 || p->N <= 0 || M > kMaxMatrixExtent || p->K > kMaxMatrixExtent || p->N > kMaxMatrixExtent)
    return "extents must be positive and below 2^31";
  if (p->route < MTRT_LINEAR_DENSE && p->dtype != MTRT_F16)
    return "this route computes in f16";
  if (p->route == MTRT_LINEAR_DENSE_F8W && (float_bytes(p->dtype) != 2 || !p->w_frag || !p->w_scale || (p->q_dtype >= 0 && !p->x_scale)))
    return "float8 weights need a 16-bit type, their codes, their scales, and a scale where x is quantized";
  if (p->route == MTRT_LINEAR_DENSE_F8W && p->q_dtype >= 0 && p->q_dtype != MTRT_F8E4M3FN)
    return "float8 weights take an x that goes through f8E4M3FN codes, or a plain one";   // (no other kernel up to 16 rows reads codes)
  if (p->q_dtype >= 0 && p->q_dtype != MTRT_I8 && p->q_dtype != MTRT_F8E4M3FN && p->q_dtype != MTRT_I4)
    return "activations go through i8, f8E4M3FN or i4 codes";
  if (p->route == MTRT_LINEAR_W8A8 && (p->q_dtype != MTRT_I8 || !p->x_scale || !p->w_scale || (!p->w && !p->w_frag)))
    return "W8A8 needs int8 activations, both scales and weights";
  if (p->route == MTRT_LINEAR_W4A16 && (p->q_dtype >= 0 || !p->w_frag || !p->w_scale || p->K % 64 != 0))
    return "W4A16 needs plain activations, re-laid weights, their scales and K % 64 == 0";
  if (p->route == MTRT_LINEAR_DENSE && ((p->q_dtype >= 0 && !p->x_scale) || (!p->w && !(p->w_frag && float_bytes(p->dtype) == 2))))
    return "the dense route needs weights, and a scale where it quantizes";
  return nullptr;
}
} // namespace

int64_t mtrt_hip_linear_fragments_bytes(int32_t dtype, int64_t K, int64_t N) {
  const int eb = dtype == MTRT_I8 || dtype == MTRT_F8E4M3FN ? 1 : dtype == MTRT_F16 || dtype == MTRT_BF16 ? 2 : 0;
  if (!eb || K <= 0 || N <= 0 || K > kMaxMatrixExtent || N > kMaxMatrixExtent)
    return 0;
  return ((N + 31) / 32) * 32 * round_up(K * eb, dtype == MTRT_F8E4M3FN ? 64 : 128);
}

int32_t mtrt_hip_linear_prepack_fragments(mtrt_stream_t stream, const void *w_nk, int32_t dtype, void *w_frag, int64_t K, int64_t N) {
  clear_error();
  const int64_t bytes = mtrt_hip_linear_fragments_bytes(dtype, K, N);
  if (bytes == 0)
    return set_error(MTRT_INVALID_ARGUMENT, "fragment order holds i8, f8E4M3FN, f16 or bf16 weights of positive extents, got dtype %d [%lld, %lld]", dtype,
                     (long long)N, (long long)K);
  if (!w_nk || !w_frag)
    return set_error(MTRT_INVALID_ARGUMENT, "null operand");
  if (!aligned(w_frag, 16) || !aligned(w_nk, float_bytes(dtype) == 2 ? 2 : 1))
    return set_error(MTRT_INVALID_ARGUMENT, "the fragment buffer must be 16-byte aligned, the weights aligned to their elements");
  DeviceState *st = device_state();
  if (!st)
    return MTRT_RUNTIME_ERROR;
  int32_t is_nk = 1;
  void *args8[] = {&w_nk, &w_frag, &K, &N, &is_nk}, *args16[] = {&w_nk, &w_frag, &K, &N};
  if (dtype == MTRT_F8E4M3FN)
    return launch(st, KernelName("mtrt_wf8_prepack_frag"), blocks_for(bytes / 8, kBlock), kBlock, as_hip(stream), args16);
  return launch(st, KernelName(dtype == MTRT_I8 ? "mtrt_w8_prepack_frag" : "mtrt_w16_prepack_frag"), blocks_for(bytes / 16, kBlock), kBlock,
                as_hip(stream), dtype == MTRT_I8 ? args8 : args16);
}

int64_t mtrt_hip_linear_workspace(const mtrt_hip_linear_plan *plan, int64_t M) {
  if (M <= 0 || linear_fault(plan, M))
    return 0;
  DeviceState *st = device_state();
  if (!st)
    return 0;
  int64_t need = 0;
  const int64_t most = linear_rows(*plan, M), last = M % most;
  for (int64_t rows : {most, last}) {
    if (rows > 0) {
      if (plan->route == MTRT_LINEAR_W4A16) {
        need = std::max(need, mtrt_hip_gemm_w4a16_workspace(rows, plan->K, plan->N, plan->K));
        continue;
      }
      const LinearShape s = linear_shape(*plan, rows, num_compute_units(st));
      need = std::max(need, s.act_bytes + s.partial_bytes);
    }
  }
  return need;
}

int32_t mtrt_hip_linear(mtrt_stream_t stream, const mtrt_hip_linear_plan *plan, const void *x, void *y, int64_t M, void *workspace,
                        int64_t workspace_bytes) {
  clear_error();
  if (const char *fault = linear_fault(plan, M))
    return set_error(MTRT_INVALID_ARGUMENT, "linear plan: %s", fault);
  if (M == 0)
    return MTRT_OK;
  const mtrt_hip_linear_plan &p = *plan;
  const int eb = float_bytes(p.dtype);
  if (!x || !y)
    return set_error(MTRT_INVALID_ARGUMENT, "null operand");
  if (!aligned(x, eb) || !aligned(y, eb) || !aligned(p.bias, eb) || !aligned(p.w_frag, 16) ||
      (p.route == MTRT_LINEAR_DENSE_F8W && !aligned(p.w, 16)))
    return set_error(MTRT_INVALID_ARGUMENT, "x, y and bias must be aligned to their elements, w_frag to 16 bytes");
  DeviceState *st = device_state();
  if (!st)
    return MTRT_RUNTIME_ERROR;
  const int64_t most = linear_rows(p, M);
  if (most < M) {
    for (int64_t m0 = 0; m0 < M; m0 += most) {
      const int32_t rc = mtrt_hip_linear(stream, plan, static_cast<const char *>(x) + m0 * p.K * eb, static_cast<char *>(y) + m0 * p.N * eb,
                                         std::min(most, M - m0), workspace, workspace_bytes);
      if (rc != MTRT_OK)
        return rc;
    }
    return MTRT_OK;
  }
  if (p.route == MTRT_LINEAR_W4A16)
    return w4a16(as_hip(stream), x, nullptr, p.w_frag, p.w_scale, p.bias, y, M, p.K, p.N, p.K, workspace, workspace_bytes);
  const LinearShape s = linear_shape(p, M, num_compute_units(st));
  if (p.route >= MTRT_LINEAR_DENSE && s.fragments && p.q_dtype < 0 && s.Kp == p.K && !aligned(x, 16))
    return set_error(MTRT_INVALID_ARGUMENT, "x must be 16-byte aligned for these weights");
  // (an f32 product runs unsplit where the workspace has no room for its parts)
  const int64_t need = s.act_bytes + (eb == 4 ? 0 : s.partial_bytes);
  if (need > 0 && (!workspace || !aligned(workspace, 16) || workspace_bytes < need))
    return set_error(MTRT_INVALID_ARGUMENT, "workspace of %lld bytes, 16-byte aligned, needed", (long long)need);
  const float *codes_scale = p.route == MTRT_LINEAR_DENSE_F8W ? static_cast<const float *>(p.w_scale) : nullptr;
  if (s.one_launch && p.route >= MTRT_LINEAR_DENSE) {
    const float *x_scale = p.x_scale;
    const void *w_frag = p.w_frag, *bias = p.bias;
    int64_t K = p.K, Kp = s.Kp, N = p.N;
    int32_t past = Kp * N * (codes_scale ? 1 : eb) > tuning::kWeightsPastBytes;
    KernelName name("mtrt_gemm_dense_frag_");
    name + float_name(p.dtype) + (M * Kp <= kDecodeElements ? "_rows16" : "_rows16_long");
    if (p.q_dtype >= 0)
      name + "_" + code_name(p.q_dtype);
    void *args[] = {&x, &x_scale, &w_frag, &bias, &y, &M, &K, &Kp, &N, &past, &codes_scale};
    return launch(st, name, uint32_t((N + 15) / 16), 512, as_hip(stream), args);
  }
  if (s.one_launch) {
    const float *w_scale = static_cast<const float *>(p.w_scale), *x_scale = p.x_scale;
    const void *w_frag = p.w_frag, *bias = p.bias;
    int64_t K = p.K, Kp = s.Kp, N = p.N;
    void *args[] = {&x, &x_scale, &w_frag, &w_scale, &y, &M, &K, &Kp, &N, &bias};
    return launch(st, KernelName("mtrt_linear_w8a8_decode"), uint32_t((N + 15) / 16), 512, as_hip(stream), args);
  }
  char *ws = static_cast<char *>(workspace);
  const void *act = x;
  if (s.pass) {
    act = ws;
    const int32_t rc = activation_pass(st, as_hip(stream), p.route == MTRT_LINEAR_W8A8, x, p.dtype, p.q_dtype, p.x_scale, ws, M, p.K, s.Kp);
    if (rc != MTRT_OK)
      return rc;
  }
  void *partial = s.partial_bytes ? ws + s.act_bytes : nullptr;
  if (p.route == MTRT_LINEAR_W8A8) {
    const float *w_scale = static_cast<const float *>(p.w_scale), *x_scale = p.x_scale;
    if (s.fragments)
      return w8a8_fragments(as_hip(stream), act, p.w_frag, x_scale, 0, w_scale, p.bias, y, M, s.Kp, p.N, partial, s.partial_bytes);
    uint32_t a_step = 0;
    const void *w = p.w, *bias = p.bias;
    int64_t K = p.K, N = p.N;
    void *args[] = {&act, &w, &x_scale, &w_scale, &y, &M, &K, &N, &a_step, &bias};
    return launch(st, KernelName("mtrt_gemm_w8a8_nk_edge"), uint32_t(std::min<int64_t>(((M + 127) / 128) * ((N + 127) / 128), int64_t(kMaxGrid) * 1024)),
                  kBlock, as_hip(stream), args);
  }
  if (s.fragments)
    return dense_fragments(st, as_hip(stream), act, codes_scale && p.w ? p.w : p.w_frag, p.w ? nullptr : codes_scale, p.bias, y, p.dtype, M, s.Kp, p.N, partial, s.partial_bytes);
  return linear_dense(stream, act, p.w, p.bias, y, p.dtype, M, p.K, p.N, partial, workspace_bytes - s.act_bytes);
}

} // extern "C"
