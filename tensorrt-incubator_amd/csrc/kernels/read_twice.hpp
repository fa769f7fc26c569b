// The order in which two passes over one tensor take it, the second to find in the L2s what the first has left there; plain arithmetic,
// for the device and the host.
//
// Workgroups are dealt to the eight XCDs in turn, each with an L2 of its own (4 MiB) that keeps what a launch has READ there for the next
// one.  The second pass finds it if it takes the same bytes on the same XCD and begins where the first one ended.  The amax pass goes
// from the tensor's end to its front, in 32 KiB that a workgroup takes at a time; the passes that quantize by its maximum go
// forwards, as many neighbouring pieces of theirs on one XCD as make up 32 KiB, and so does the dequantize behind them, which finds their
// codes in the same way.  us, bf16 -> i8 of 8, 16, 24 and 48 Mi elements, with amax forwards, the quantizing pass from the end and the
// dequantize forwards piece by piece, and so: amax, then quantize and dequantize in one pass 12.6, 20.3, 30.5, 53.8 and 13.0, 20.6, 31.0, 54.0;
// a quantize and its dequantize 13.8, 23.7, 27.9, 51.7 and 10.7, 17.3, 24.7, 51.3 (the codes of the one lay in other L2s than the
// other read them through).  Pieces of 8 or 16 KiB to an XCD in all passes: amax of 33 MB from memory 9.0 -> 9.7.
#pragma once
#include <stdint.h>

namespace mtrt_dev {

// Larger tensors (bytes) and their results fill the Infinity Cache: nothing is left for the next pass, whose pieces go to the XCDs in turn
// (quantize and dequantize in one pass, f32 of 268 MB 90.6, and 94.0 in 32 KiB to an XCD).
constexpr int64_t kReadTwiceBelow = int64_t(192) << 20;
constexpr int64_t kReadTwiceKept = int64_t(32) << 20;     // what the eight L2s hold

// The amax pass: 256 lanes, turns of LOADS neighbouring vectors a lane; eight turns, one per XCD, to a group, the groups from the last to the
// first, then what is left at the tensor's end.
template <int LOADS>
struct AmaxTurns {
  static constexpr int64_t kTurn = LOADS * 256, kGroup = 8 * kTurn;
  int64_t groups, whole, turns;                       // groups of eight turns; turns in them; turns in all
  constexpr explicit AmaxTurns(int64_t nvec) : groups(nvec / kGroup), whole(8 * groups), turns(whole + (nvec - groups * kGroup + kTurn - 1) / kTurn) {}
  // The first turn whose vectors lie in the front `kept` vectors (whole groups of them).
  constexpr int64_t first_kept(int64_t kept) const { return groups > kept / kGroup ? 8 * (groups - kept / kGroup) : 0; }
  // A turn's first vector.
  constexpr int64_t first(int64_t turn) const { return turn < whole ? (groups - 1 - turn / 8) * kGroup + turn % 8 * kTurn : turn * kTurn; }
};

// Which of the launch's n pieces of 32 KiB / PER workgroup `id` takes: PER neighbouring ones on one XCD.  Any n: the last n % (8 PER) stay
// where they are.
template <uint32_t PER>
constexpr uint32_t piece_of(uint32_t id, uint32_t n, int64_t x_bytes) {
  if (id >= (n & ~(8 * PER - 1)) || uint32_t(x_bytes >> 20) >= uint32_t(kReadTwiceBelow >> 20)) return id;   // (in 32 bits: scalar comparisons)
  const uint32_t k = id >> 3;
  return k / PER * (8 * PER) + (id & 7) * PER + k % PER;
}

}  // namespace mtrt_dev
