// Device helpers of the kernels that stream a [rows, vocab] batch: the block
// numbering over the XCDs and a row's state with queued pool writes.
#pragma once

#include <cstring>

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

// Slot list and queued pool writes in a launch's arguments instead of an
// upload before it: `rows` slots, then `num_pending` slots and as many values.
// The launch also leaves the slots in device memory for those after it.
// N = 0: none (the launch takes pointers).
template <int N>
struct InlineRows {
  int32_t v[N];
};
template <>
struct InlineRows<0> {
  int32_t v[1];
};

// wave_row_state from the arguments.
__device__ __forceinline__ int32_t wave_row_state_inline(const int32_t* states, const int32_t* v, uint32_t rows,
                                                         int32_t num_pending, uint32_t r, int lane) {
  const int32_t slot = v[r];
  int32_t s = __builtin_amdgcn_readfirstlane(states[slot]);
  for (int32_t base = 0; base < num_pending; base += 64) {
    const int32_t i = base + lane;
    const bool hit = i < num_pending && v[rows + i] == slot;
    const uint64_t m = __ballot(hit);
    if (m) {
      const int32_t q = hit ? v[rows + num_pending + i] : 0;
      s = __builtin_amdgcn_readlane(q, __builtin_ctzll(m));
    }
  }
  return s;
}

// By one block of the launch: the queued writes, and the slots to slots_out.
__device__ __forceinline__ void store_inline_rows(const int32_t* v, uint32_t rows, int32_t num_pending,
                                                  int32_t* states, int64_t* slots_out) {
  for (uint32_t i = threadIdx.x; i < rows; i += blockDim.x) slots_out[i] = v[i];
  for (uint32_t i = threadIdx.x; i < uint32_t(num_pending); i += blockDim.x)
    states[v[rows + i]] = v[rows + uint32_t(num_pending) + i];
}

// Calls launch(InlineRows<N>) with the smallest N that holds the values.
template <class F>
inline int with_inline_rows(const int32_t* values, int64_t n, F launch) {
  if (n <= 64) {
    InlineRows<64> a;
    std::memcpy(a.v, values, size_t(n) * 4);
    return launch(a);
  }
  if (n <= 320) {
    InlineRows<320> a;
    std::memcpy(a.v, values, size_t(n) * 4);
    return launch(a);
  }
  InlineRows<BPD_MAX_INLINE_VALUES> a;
  std::memcpy(a.v, values, size_t(n) * 4);
  return launch(a);
}

inline int check_inline(const int32_t* values, int64_t rows, int64_t num_pending, const int32_t* states,
                        const int64_t* slots_out) {
  BPD_REQUIRE(rows > 0 && num_pending >= 0 && num_pending <= BPD_MAX_FUSED_PENDING &&
                  rows + 2 * num_pending <= BPD_MAX_INLINE_VALUES,
              "at most %d values in a launch's arguments", BPD_MAX_INLINE_VALUES);
  BPD_REQUIRE(values && states && slots_out, "null pointer argument");
  return BPD_OK;
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
