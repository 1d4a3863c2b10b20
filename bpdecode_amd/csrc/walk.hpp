// Token walks through a symbol-class DFA staged in LDS, for the kernels that
// walk many tokens from many states (the dense table builder and the packed
// masks of bundles without a dense table).
//
// The staged table is absorbing, so a walk step has no test: entry
// T[row + symbol] is the LDS offset of the next state's row.  Row S is the
// failed walk.  Of a row's M + 3 columns the first M are the symbol classes,
// column M takes every symbol id at or above M (a failed walk), column M + 1
// keeps the state (the padding of short tokens) and column M + 2 holds the
// walk's result (the state, or kWalkNone where the state is not live).
// A step is then one byte extract, one add and one LDS read; a token's first
// 16 symbols sit in four registers, and a wave leaves the walk at the first
// four symbols after which all its lanes have failed or ended.
#pragma once

#include "bpd_common.hpp"

namespace bpd {
namespace {

constexpr uint32_t kWalkNone = 0xFFFFu;
constexpr int kWalkRows = 4;  // states walked side by side (their LDS reads overlap)

// 16-bit offsets and 8-bit symbols bound the tables that can be staged.
inline bool walk_table_fits(int64_t S, int64_t M, size_t max_bytes) {
  return M <= 253 && (S + 1) * (M + 3) <= 65536 && size_t((S + 1) * (M + 3)) * 2 <= max_bytes;
}
inline size_t walk_table_bytes(int64_t S, int64_t M) { return size_t((S + 1) * (M + 3)) * 2; }

// Stages the table; every thread of the block takes part, and a barrier must
// follow.  DeadEnds: a step into `dead` ends the walk with `dead`'s own
// liveness, as does a walk that starts there (the dense builder's rule);
// otherwise a step into `dead` fails and a walk that starts there goes on.
// Loads go out eight entries at a time: one
// entry per iteration made the staging a chain of memory round trips (the
// dense builder's 2,400 entries per block took 10 of its 38 us).
template <bool DeadEnds>
__device__ __forceinline__ void stage_walk_table(uint16_t* T, const int32_t* __restrict__ trans, int32_t S,
                                                 int32_t M, int32_t dead, const uint8_t* __restrict__ live) {
  constexpr int kBatch = 8;
  const uint32_t W = uint32_t(M) + 3, n = uint32_t(S + 1) * W, nt = blockDim.x;
  const uint32_t magic = uint32_t((0x100000000ull + W - 1) / W);  // i / W = hi32(i * magic) for i < 65536
  const uint32_t fail = uint32_t(S) * W;
  const uint32_t dead_row = DeadEnds && live[dead] ? uint32_t(dead) * W : fail;
  for (uint32_t i0 = threadIdx.x; i0 < n; i0 += kBatch * nt) {
    int32_t d[kBatch];
#pragma unroll
    for (int k = 0; k < kBatch; ++k) {
      const uint32_t i = i0 + k * nt;
      const uint32_t s = __umulhi(i, magic), c = i - s * W;
      d[k] = s < uint32_t(S) && c < uint32_t(M) ? trans[s * uint32_t(M) + c] : -1;
    }
#pragma unroll
    for (int k = 0; k < kBatch; ++k) {
      const uint32_t i = i0 + k * nt;
      const uint32_t s = __umulhi(i, magic), c = i - s * W;
      if (i < n && c != uint32_t(M) + 2) {
        uint32_t v = uint32_t(d[k]) < uint32_t(S) ? uint32_t(d[k]) * W : fail;
        if (c == uint32_t(M) + 1) v = s * W;
        if (d[k] == dead || (DeadEnds && s == uint32_t(dead))) v = dead_row;
        T[i] = uint16_t(v);
      }
    }
  }
  for (uint32_t s = threadIdx.x; s <= uint32_t(S); s += nt)
    T[s * W + M + 2] = s < uint32_t(S) && live[s] ? uint16_t(s) : uint16_t(kWalkNone);
}

// One token's symbols: the first 16 as columns of the table (ids at or above
// M as M, padding as M + 1), the rest where they lie.
struct WalkToken {
  uint32_t w[4];
  int32_t len;
  const uint8_t* rest;
};

typedef uint32_t U4b __attribute__((ext_vector_type(4), aligned(1)));

// `total`: symbols in the array (a 16-byte read must not pass its end).  A
// token of no symbols is all padding.
__device__ __forceinline__ WalkToken load_walk_token(const uint8_t* __restrict__ syms, int64_t begin,
                                                     int32_t len, int64_t total, int32_t M) {
  WalkToken t;
  if (len <= 0) begin = len = 0;
  t.len = len;
  t.rest = syms + begin;
  if (begin + 16 <= total) {
    const U4b v = *reinterpret_cast<const U4b*>(syms + begin);
#pragma unroll
    for (int i = 0; i < 4; ++i) t.w[i] = v[i];
  } else {
#pragma unroll
    for (int i = 0; i < 4; ++i) t.w[i] = 0;
#pragma unroll
    for (int i = 0; i < 16; ++i)
      if (i < len) t.w[i >> 2] |= uint32_t(t.rest[i]) << (8 * (i & 3));
  }
#pragma unroll
  for (int i = 0; i < 16; ++i) {
    uint32_t c = (t.w[i >> 2] >> (8 * (i & 3))) & 0xFFu;
    c = i < len ? (c < uint32_t(M) ? c : uint32_t(M)) : uint32_t(M) + 1;
    t.w[i >> 2] = (t.w[i >> 2] & ~(0xFFu << (8 * (i & 3)))) | (c << (8 * (i & 3)));
  }
  return t;
}

// Walks the token from the kWalkRows rows in cur (LDS offsets, changed in
// place).  Every lane of the wave calls it.
__device__ __forceinline__ void walk_rows(const uint16_t* T, int32_t M, uint32_t fail, const WalkToken& t,
                                          uint32_t (&cur)[kWalkRows]) {
  static_assert(kWalkRows == 4, "the failed test below takes four rows");
  // `fail` is the largest row offset, so the minimum tells whether all failed
  auto walking = [&](int done) {
    const uint32_t a = cur[0] < cur[1] ? cur[0] : cur[1], b = cur[2] < cur[3] ? cur[2] : cur[3];
    return __any(t.len > done && (a < b ? a : b) != fail) != 0;
  };
  bool on = true;
#pragma unroll
  for (int w = 0; w < 4; ++w) {
    if (w > 0) on = on && walking(4 * w);
    if (on) {
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        const uint32_t c = (t.w[w] >> (8 * i)) & 0xFFu;
#pragma unroll
        for (int q = 0; q < kWalkRows; ++q) cur[q] = T[cur[q] + c];
      }
    }
  }
  if (on && walking(16)) {
    for (int32_t i = 16; i < t.len; ++i) {
      const uint32_t k = t.rest[i];
      const uint32_t c = k < uint32_t(M) ? k : uint32_t(M);
#pragma unroll
      for (int q = 0; q < kWalkRows; ++q) cur[q] = T[cur[q] + c];
    }
  }
}

}  // namespace
}  // namespace bpd
