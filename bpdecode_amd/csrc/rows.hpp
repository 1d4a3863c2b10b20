// Device helpers of the kernels that stream a [rows, vocab] batch: the block
// numbering over the XCDs and a row's state with queued pool writes.
#pragma once

#include "bpd_common.hpp"

namespace bpd {
namespace {

constexpr int kXcds = 8;

// Block index -> logical block, numbered so that consecutive logical blocks
// run on one XCD (workgroups are dealt round-robin to the 8 XCDs).
// gridDim.x is a multiple of kXcds.
__device__ __forceinline__ uint32_t logical_block() {
  const uint32_t nb = gridDim.x;
  const uint32_t hw = blockIdx.x;
  return (hw % kXcds) * (nb / kXcds) + hw / kXcds;
}

// Wave-uniform state of row r: the pool entry at its slot, or the value of a
// queued write to that slot (`pending` = num_pending slots, then as many
// values; slots are distinct).
__device__ __forceinline__ int32_t wave_row_state(const int32_t* states, const int64_t* slots,
                                                  const int64_t* pending, int32_t num_pending,
                                                  uint32_t r, int lane) {
  const int64_t slot = slots ? slots[r] : int64_t(r);
  int32_t s = __builtin_amdgcn_readfirstlane(states[slot]);
  for (int32_t base = 0; base < num_pending; base += 64) {
    const int32_t i = base + lane;
    const bool hit = i < num_pending && pending[i] == slot;
    const uint64_t m = __ballot(hit);
    if (m) {
      const int src = __builtin_ctzll(m);
      const int32_t v = hit ? int32_t(pending[num_pending + i]) : 0;
      s = __builtin_amdgcn_readlane(v, src);
    }
  }
  return s;
}

// Host-side checks of the queued pool writes that a launch applies.
inline int check_pending(const int64_t* pending, int64_t num_pending, const int64_t* slots, int64_t rows) {
  BPD_REQUIRE(num_pending >= 0 && num_pending <= BPD_MAX_FUSED_PENDING,
              "at most %d queued pool writes per launch (got %lld)", BPD_MAX_FUSED_PENDING,
              (long long)num_pending);
  BPD_REQUIRE(num_pending == 0 || (pending && slots), "queued writes need a slot map");
  BPD_REQUIRE(rows > 0 || num_pending == 0, "queued writes need at least one row");
  return BPD_OK;
}

}  // namespace
}  // namespace bpd
