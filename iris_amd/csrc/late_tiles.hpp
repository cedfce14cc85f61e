// Which workgroups of a kernel that reduces as it stores (gemm_skinny.hpp, REDUCE) wait for late peers.
//
// Ranks may share a device, and a workgroup that waits holds its LDS: a peer's workgroup, of whatever kernel, may need all
// of a CU's.  The hardware deals a launch's workgroups to the XCDs in turn and an XCD's to its four shader engines in turn (read
// from HW_ID and XCC_ID: 32 engines of eight CUs), whichever of them have room, so room is needed on every engine: three
// ranks with 15 workgroups waiting on each XCD, two CUs of it free, ran into the bound of their waits.  At most late_most(ws) workgroups of a
// launch wait on an engine: with all other ranks waiting and each of those workgroups on a CU of its own, one CU of the
// engine is left to the rank that they wait for.  A tile that finds as many waiting is left to them: they take the tiles that
// were left, one after the other, as they have reduced their own.  What they wait for is signalled by products, which wait
// for nothing, so the order is free.
//
// One word an engine holds both: the workgroups that wait in its low byte, above it the last tile left to them, plus one.  That
// tile's own word (its arrivals have been counted and taken back) holds the one left before it, plus one, or zero.  A word
// changes by compare-and-swap; a tile is left once a launch, so a word that compares equal is the same.  All are zero again
// when the last workgroup leaves.
#pragma once

#include <cstdint>

namespace iris_amd {

constexpr int LATE_ENGINES = 32, LATE_ENGINE_CUS = 8;

__host__ __device__ constexpr int late_most(int ws) { return ws > 1 ? (LATE_ENGINE_CUS - 1) / (ws - 1) : LATE_ENGINE_CUS - 1; }

// Whether a workgroup that comes upon a late tile waits for it itself, and the word it leaves.
__host__ __device__ constexpr bool late_waits(int32_t word, int most) { return (word & 0xFF) < most; }
__host__ __device__ constexpr int32_t late_join(int32_t word, int most, int tile) {
  return late_waits(word, most) ? word + 1 : (word & 0xFF) | (tile + 1) << 8;
}
// The tile left last (plus one, or zero), which goes with its word to a workgroup that is done with its own.
__host__ __device__ constexpr int late_left(int32_t word) { return word >> 8; }
// ... which leaves this word, `link` being that tile's, or waits for no more.
__host__ __device__ constexpr int32_t late_next(int32_t word, int32_t link) {
  return late_left(word) ? (word & 0xFF) | link << 8 : word - 1;
}

}  // namespace iris_amd
