// Dense tok_next path for gfx950: the mask over a [rows, vocab] logits batch
// (from the packed allow-bit table or from tok_next itself), the commit
// gather/advance/scatter, the packed allow-bit kernel and the device-side
// table builder.
//
// The mask is HBM-bound byte work that writes only what it must: the
// rejected logits.  A wave owns one row and 2048 columns; for each group of
// 64 columns the allowed/rejected verdicts select the lanes that store the
// fill value, one element per lane, so a group is one store instruction over
// 64 consecutive elements and allowed logits are neither read nor written.
// Measured on MI355X (B = 256, V = 151,936 bf16, email DFA) this matches a
// plain copy of the logits: with ~5 % of the tokens allowed and scattered,
// nearly every 128-byte line mixes kept and filled elements, so the memory
// side merges each partial line (a read and a write per line), the same
// traffic a kernel that reads, blends and rewrites the logits produces --
// but without the round trip through the CUs.  Non-temporal stores were
// slower (33 against 27 us).
//
// The queued state-pool writes of ConstraintBatch.add/evict/reset ride in
// the mask and commit launches (`pending`): rows read the queued value of
// their slot and one wave stores the queued values, so continuous batching
// costs no launch of its own.
#include <algorithm>

#include "bpd_common.hpp"
#include "rows.hpp"
#include "walk.hpp"

namespace bpd {
namespace {

constexpr int kFillWaves = 4;                 // waves per block: one row, 4 chunks
constexpr int kFillThreads = 64 * kFillWaves;
constexpr int kFillGroups = 32;               // 64-column groups per chunk (one wave)
constexpr int64_t kChunkCols = int64_t(kFillGroups) * 64;

template <int E> struct Elem;
template <> struct Elem<2> { using T = uint16_t; };
template <> struct Elem<4> { using T = uint32_t; };
template <> struct Elem<8> { using T = uint64_t; };

// Dense mask, write-only.  A wave owns one row and a chunk of 2048 columns
// (32 groups of 64); for each group the 64 verdicts of its columns decide
// which lanes store the fill value (one 2/4/8-byte store per lane, the
// group's store instruction covering 64 consecutive elements); allowed
// elements are never read or written.  Kernel `Bits`: the verdicts come from
// the packed allow-bit table, one uint32 word per lane holding the chunk's
// 64 words, broadcast per group with readlane; otherwise from the int32
// tok_next row (one coalesced load per group and lane).  A block holds one
// row and 4 consecutive chunks; logical blocks are numbered column-group
// major, so one XCD's L2 serves a contiguous band of table columns to every
// row.  The block with logical index 0 also applies the queued pool writes.
// The columns of `vocab` past `tokens` (a padded lm_head) are rejected in
// every row, whatever the bits past `tokens` in a row's last word.
// N: slots and queued writes come in the arguments (rows.hpp), and block 0
// leaves the slots in slots_out: [33, 100003] fp16 and two requests turning
// over: a step of 16.1 us, 18.5 with an upload before the launch (256 rows of
// V = 151,936 bf16: 28.1 and 30.4).
template <int E, bool Bits, int N>
__global__ __launch_bounds__(kFillThreads) void dense_fill_kernel(
    uint8_t* __restrict__ logits, int64_t ld_bytes, const void* __restrict__ table,
    int64_t table_ld, int64_t vocab, int64_t tokens, int32_t num_states, int32_t* states,
    const int64_t* __restrict__ slots, const int64_t* __restrict__ pending, int32_t num_pending,
    uint32_t rows, uint32_t chunks, uint64_t fill, int32_t* __restrict__ err, InlineRows<N> inl,
    int64_t* __restrict__ slots_out) {
  using T = typename Elem<E>::T;
  const uint32_t lb = logical_block();
  const uint32_t wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int lane = threadIdx.x & 63;
  const uint32_t cg = lb / rows;
  const uint32_t r = lb - cg * rows;
  const uint32_t chunk = cg * kFillWaves + wave;
  if (N > 0 && lb == 0) store_inline_rows(inl.v, rows, num_pending, states, slots_out);
  if (N == 0 && lb == 0 && wave == 0)
    for (int32_t i = lane; i < num_pending; i += 64) states[pending[i]] = int32_t(pending[num_pending + i]);
  if (chunk >= chunks) return;
  const int32_t s = N > 0 ? wave_row_state_inline(states, inl.v, rows, num_pending, r, lane)
                          : wave_row_state(states, slots, pending, num_pending, r, lane);
  const bool live = s >= 0 && s < num_states;
  if (s >= num_states && err && lane == 0 && chunk == 0) atomicOr(err, BPD_FLAG_STATE_RANGE);
  const int64_t c0 = int64_t(chunk) * kChunkCols;
  const bool tail = c0 + kChunkCols > vocab;
  const int64_t lim = vocab - c0 - lane;  // columns left for this lane
  T* p = reinterpret_cast<T*>(logits + int64_t(r) * ld_bytes) + c0 + lane;
  const T f = T(fill);
  if (Bits) {
    const uint32_t* bw = static_cast<const uint32_t*>(table);
    const int64_t w = c0 / 32 + lane;
    uint32_t mine = (live && w < table_ld) ? bw[int64_t(s) * table_ld + w] : 0u;
    if (w == tokens >> 5) mine &= (1u << (tokens & 31)) - 1;  // a caller's table may have bits there
    const uint32_t lanebit = 1u << (lane & 31);
#pragma unroll
    for (int j = 0; j < kFillGroups; ++j) {
      const uint32_t lo = __builtin_amdgcn_readlane(mine, 2 * j);
      const uint32_t hi = __builtin_amdgcn_readlane(mine, 2 * j + 1);
      const uint32_t word = lane < 32 ? lo : hi;
      const int c = j * 64;
      if (!(word & lanebit) && (!tail || c < lim)) p[c] = f;
    }
  } else {
    const int32_t* tn = static_cast<const int32_t*>(table) + (live ? int64_t(s) * table_ld : 0) + c0 + lane;
    int32_t v[kFillGroups];
#pragma unroll
    for (int j = 0; j < kFillGroups; ++j) v[j] = (live && (!tail || j * 64 < lim)) ? tn[j * 64] : -1;
#pragma unroll
    for (int j = 0; j < kFillGroups; ++j) {
      const int c = j * 64;
      if (v[j] == -1 && (!tail || c < lim)) p[c] = f;
    }
  }
}

// Token id of row b: int32, int64, or int64 read as its low 32 bits (what
// tensor.to(torch.int32) keeps); a negative id indexes from the end, as
// torch advanced indexing does.  False when the id is out of range.
__device__ __forceinline__ int32_t row_state(const int32_t* __restrict__ states,
                                             const int64_t* __restrict__ slots, int64_t r) {
  if (!states) return int32_t(r);  // every state's row
  return states[slots ? slots[r] : r];
}

__device__ __forceinline__ bool token_index(const void* tokens, int tok_dtype, int64_t b,
                                            int64_t vocab, int64_t* out) {
  int64_t t = read_token(tokens, tok_dtype, b);
  if (t < 0) t += vocab;
  *out = t;
  return t >= 0 && t < vocab;
}

__device__ __forceinline__ int32_t advance_one(const int32_t* __restrict__ tok_next,
                                               int32_t num_states, int64_t vocab, int32_t s,
                                               const void* tokens, int tok_dtype, int64_t b,
                                               int32_t* __restrict__ err) {
  int64_t t;
  const bool t_ok = token_index(tokens, tok_dtype, b, vocab, &t);
  if (!t_ok) {
    if (err) atomicOr(err, BPD_FLAG_TOKEN_RANGE);
    return -1;
  }
  if (s >= num_states) {
    if (err) atomicOr(err, BPD_FLAG_STATE_RANGE);
    return -1;
  }
  if (s < 0) return -1;
  return tok_next[int64_t(s) * vocab + t];
}

// advance_one with the token id already read (raw: negative ids index from
// the end)
__device__ __forceinline__ int32_t advance_tok(const int32_t* __restrict__ tok_next, int32_t num_states,
                                               int64_t vocab, int32_t s, int64_t t, int32_t* __restrict__ err) {
  if (t < 0) t += vocab;
  if (t < 0 || t >= vocab) {
    if (err) atomicOr(err, BPD_FLAG_TOKEN_RANGE);
    return -1;
  }
  if (s >= num_states) {
    if (err) atomicOr(err, BPD_FLAG_STATE_RANGE);
    return -1;
  }
  if (s < 0) return -1;
  return tok_next[int64_t(s) * vocab + t];
}

constexpr int kAdvThreads = 1024;
constexpr int kAdvPerThread = 4;

// rows <= kAdvThreads * kAdvPerThread: one block.  The queued pool writes are
// staged in LDS.  Every pool read happens before the second barrier, the
// queued writes land between the second and third and the rows' write-backs
// after the third -- the order of the calls: the queued writes were made
// before the commit, and a row reads the queued value of its slot.
__global__ __launch_bounds__(kAdvThreads) void dense_advance_block_kernel(
    const int32_t* __restrict__ tok_next, int32_t num_states, int64_t vocab,
    int32_t* __restrict__ states, const int64_t* __restrict__ slots,
    const int64_t* __restrict__ pending, int32_t num_pending, const void* __restrict__ tokens,
    int tok_dtype, int64_t tok_stride, int64_t rows, int32_t* __restrict__ next_out, int write_back,
    int32_t* __restrict__ err) {
  __shared__ int64_t pslot[BPD_MAX_FUSED_PENDING];
  __shared__ int32_t pval[BPD_MAX_FUSED_PENDING];
  // every load that does not need the queued writes is issued before they
  // are staged: each row's slot and token, then the slot's state (one chain
  // of two dependent loads beside the staging instead of after it)
  int64_t slot[kAdvPerThread], tk[kAdvPerThread];
#pragma unroll
  for (int i = 0; i < kAdvPerThread; ++i) {
    const int64_t b = int64_t(i) * kAdvThreads + threadIdx.x;
    slot[i] = b < rows ? (slots ? slots[b] : b) : -1;
    tk[i] = b < rows ? read_token(tokens, tok_dtype, b * tok_stride) : 0;
  }
  int32_t st[kAdvPerThread];
#pragma unroll
  for (int i = 0; i < kAdvPerThread; ++i) st[i] = slot[i] >= 0 ? states[slot[i]] : 0;
  for (int32_t i = threadIdx.x; i < num_pending; i += kAdvThreads) {
    pslot[i] = pending[i];
    pval[i] = int32_t(pending[num_pending + i]);
  }
  __syncthreads();
  int32_t nxt[kAdvPerThread];
#pragma unroll
  for (int i = 0; i < kAdvPerThread; ++i) {
    const int64_t b = int64_t(i) * kAdvThreads + threadIdx.x;
    nxt[i] = -1;
    if (b < rows) {
      int32_t s = st[i];
      for (int32_t k = 0; k < num_pending; ++k)
        if (pslot[k] == slot[i]) s = pval[k];
      nxt[i] = advance_tok(tok_next, num_states, vocab, s, tk[i], err);
      if (next_out) next_out[b] = nxt[i];
    }
  }
  __syncthreads();
  for (int32_t i = threadIdx.x; i < num_pending; i += kAdvThreads) states[pslot[i]] = pval[i];
  if (!write_back) return;
  __syncthreads();
#pragma unroll
  for (int i = 0; i < kAdvPerThread; ++i)
    if (slot[i] >= 0) states[slot[i]] = nxt[i];
}

__global__ void dense_advance_gather_kernel(const int32_t* __restrict__ tok_next,
                                            int32_t num_states, int64_t vocab,
                                            const int32_t* __restrict__ states,
                                            const int64_t* __restrict__ slots,
                                            const void* __restrict__ tokens, int tok_dtype,
                                            int64_t tok_stride, int64_t rows,
                                            int32_t* __restrict__ next_out, int32_t* __restrict__ err) {
  const int64_t b = int64_t(blockIdx.x) * blockDim.x + threadIdx.x;
  if (b >= rows) return;
  const int64_t slot = slots ? slots[b] : b;
  next_out[b] = advance_one(tok_next, num_states, vocab, states[slot], tokens, tok_dtype, b * tok_stride, err);
}

__global__ void dense_scatter_kernel(int32_t* __restrict__ states, const int64_t* __restrict__ slots,
                                     const int32_t* __restrict__ next, int64_t rows) {
  const int64_t b = int64_t(blockIdx.x) * blockDim.x + threadIdx.x;
  if (b >= rows) return;
  states[slots ? slots[b] : b] = next[b];
}

// Packed allow bits of the rows' table rows, grid (ceil(vocab / 4096), rows).
// Bound by the read of the int32 rows, so each lane has four 16-byte loads in
// flight (a row starts at any 4-byte boundary).  A lane's four verdicts are a
// nibble of its word; the eight lanes of a word are combined by DPP
// exchanges, and lane u of the eight writes the word of load u (LSB-first).
// 71 rows of V = 151,936: 22.4 us with one load per thread, 8.2 now.
constexpr int kBitsThreads = 256;
constexpr int kBitsLoads = 4;
constexpr int64_t kBitsTokens = int64_t(kBitsThreads) * 4 * kBitsLoads;
typedef int32_t I4u __attribute__((ext_vector_type(4), aligned(4)));

template <int Ctrl>
__device__ __forceinline__ uint32_t or_lane(uint32_t v) {
  return v | uint32_t(__builtin_amdgcn_update_dpp(0, int(v), Ctrl, 0xF, 0xF, false));
}

__global__ __launch_bounds__(kBitsThreads) void dense_bits_kernel(
    const int32_t* __restrict__ tok_next, int32_t num_states, int64_t vocab,
    const int32_t* __restrict__ states, const int64_t* __restrict__ slots, int64_t rows,
    uint32_t* __restrict__ bits, int64_t words, int32_t* __restrict__ err) {
  const int64_t r = blockIdx.y;
  const int sub = threadIdx.x & 7;
  const int64_t t0 = int64_t(blockIdx.x) * kBitsTokens + threadIdx.x * 4;
  const int32_t s = row_state(states, slots, r);
  const bool live_row = s >= 0 && s < num_states;
  if (s >= num_states && err && t0 == 0) atomicOr(err, BPD_FLAG_STATE_RANGE);
  const int32_t* row = tok_next + (live_row ? int64_t(s) * vocab : 0);
  I4u v[kBitsLoads];
#pragma unroll
  for (int u = 0; u < kBitsLoads; ++u) {
    const int64_t t = t0 + int64_t(u) * kBitsThreads * 4;
    v[u] = I4u{-1, -1, -1, -1};
    if (live_row && t + 4 <= vocab) {
      v[u] = *reinterpret_cast<const I4u*>(row + t);
    } else if (live_row) {
#pragma unroll
      for (int q = 0; q < 4; ++q)
        if (t + q < vocab) v[u][q] = row[t + q];
    }
  }
  uint32_t mine = 0;
#pragma unroll
  for (int u = 0; u < kBitsLoads; ++u) {
    uint32_t w = 0;
#pragma unroll
    for (int q = 0; q < 4; ++q) w |= v[u][q] != -1 ? 1u << q : 0u;
    w <<= 4 * sub;
    w = or_lane<0xB1>(w);   // lane ^ 1
    w = or_lane<0x4E>(w);   // lane ^ 2
    w = or_lane<0x141>(w);  // the other four of the eight
    if (sub == u) mine = w;
  }
  const int64_t at = (t0 - 4 * sub) / 32 + int64_t(sub) * (kBitsThreads / 8);
  if (sub < kBitsLoads && at < words) bits[r * words + at] = mine;
}

// The rows' words of a packed allow-bit table, grid (ceil(words / 2048), rows);
// zeros for a negative state or one outside the table (flagged).  A copy of
// words 4-byte aligned at best (odd row lengths), 16 bytes per access.
// 256 rows of V = 151,936: 4.9 MB in 3.3 us, where walking the tokens of 826
// states' table takes 67 us.
constexpr int kBitRowLoads = 2;

__global__ __launch_bounds__(kBitsThreads) void bit_rows_kernel(
    const uint32_t* __restrict__ table, int64_t words, int32_t num_states, const int32_t* __restrict__ states,
    uint32_t* __restrict__ out, int32_t* __restrict__ err) {
  const int64_t r = blockIdx.y;
  const int32_t s = states[r];
  const bool live_row = s >= 0 && s < num_states;
  if (s >= num_states && err && blockIdx.x == 0 && threadIdx.x == 0) atomicOr(err, BPD_FLAG_STATE_RANGE);
  const uint32_t* from = table + (live_row ? int64_t(s) * words : 0);
  uint32_t* to = out + r * words;
  I4u v[kBitRowLoads];
#pragma unroll
  for (int u = 0; u < kBitRowLoads; ++u) {
    const int64_t w = ((int64_t(blockIdx.x) * kBitRowLoads + u) * kBitsThreads + threadIdx.x) * 4;
    v[u] = I4u{0, 0, 0, 0};
    if (live_row && w + 4 <= words) v[u] = *reinterpret_cast<const I4u*>(from + w);
  }
#pragma unroll
  for (int u = 0; u < kBitRowLoads; ++u) {
    const int64_t w = ((int64_t(blockIdx.x) * kBitRowLoads + u) * kBitsThreads + threadIdx.x) * 4;
    if (w + 4 <= words) {
      *reinterpret_cast<I4u*>(to + w) = v[u];
    } else {
      for (int64_t i = w; i < words; ++i) to[i] = live_row ? from[i] : 0u;
    }
  }
}

// tok_next builder over the staged walk table (walk.hpp), grid (tokens, rows /
// rows_per_block): a thread holds one token's symbols and walks them from the
// block's rows, four at a time; each row's results go out as one coalesced
// store per wave.  Bound by the walk's instructions and LDS reads.  71 states
// x 151,936 tokens: 68.2 us with one thread per (row, token) reading symbols
// and table from memory, 21.1 us now (19 without the stores).
__global__ __launch_bounds__(1024) void build_walk_kernel(
    const int32_t* __restrict__ trans, int32_t S, int32_t M, int32_t dead,
    const uint8_t* __restrict__ accept, const uint8_t* __restrict__ live,
    const int32_t* __restrict__ offsets, const uint8_t* __restrict__ syms, int64_t vocab,
    int32_t eos_id, const int32_t* __restrict__ row_states, int32_t num_rows, int32_t rows_per_block,
    int32_t* __restrict__ out) {
  extern __shared__ __align__(16) uint16_t walk_tab[];
  const int64_t t = int64_t(blockIdx.x) * blockDim.x + threadIdx.x;
  const bool on = t < vocab;
  int32_t b = 0, e = 0;
  if (on && t != eos_id) {
    b = offsets[t];
    e = offsets[t + 1];
  }
  const WalkToken tok = load_walk_token(syms, b, e - b, offsets[vocab], M);
  stage_walk_table<true>(walk_tab, trans, S, M, dead, live);
  __syncthreads();
  const uint32_t W = uint32_t(M) + 3, fail = uint32_t(S) * W;
  const int32_t r0 = int32_t(blockIdx.y) * rows_per_block;
  const int32_t r1 = r0 + rows_per_block < num_rows ? r0 + rows_per_block : num_rows;
  const bool has_eos = __any(t == eos_id) != 0;  // only this wave needs the accepting flags
  int32_t* o = out + int64_t(r0) * vocab + t;
  for (int32_t r = r0; r < r1; r += kWalkRows) {
    uint32_t cur[kWalkRows];
    int32_t st[kWalkRows];
#pragma unroll
    for (int q = 0; q < kWalkRows; ++q) {
      st[q] = r + q;
      if (row_states) st[q] = r + q < r1 ? row_states[r + q] : -1;
      cur[q] = uint32_t(st[q]) < uint32_t(S) ? uint32_t(st[q]) * W : fail;
    }
    walk_rows(walk_tab, M, fail, tok, cur);
    int32_t res[kWalkRows];
#pragma unroll
    for (int q = 0; q < kWalkRows; ++q) {
      const uint32_t v = walk_tab[cur[q] + M + 2];
      res[q] = v == kWalkNone ? -1 : int32_t(v);
    }
    if (has_eos) {
#pragma unroll
      for (int q = 0; q < kWalkRows; ++q)
        if (t == eos_id) res[q] = uint32_t(st[q]) < uint32_t(S) && accept[st[q]] ? st[q] : -1;
    }
#pragma unroll
    for (int q = 0; q < kWalkRows; ++q)
      if (on && r + q < r1) o[int64_t(q) * vocab] = res[q];
    o += int64_t(kWalkRows) * vocab;
  }
}

// The builder for tables too large to stage: one thread per (row, token),
// symbols and table read through the caches.
__global__ __launch_bounds__(256) void build_tok_next_kernel(
    const int32_t* __restrict__ trans, int32_t num_states, int32_t num_symbols, int32_t dead,
    const uint8_t* __restrict__ accept, const uint8_t* __restrict__ live,
    const int32_t* __restrict__ offsets, const uint8_t* __restrict__ syms, int64_t vocab,
    int32_t eos_id, const int32_t* __restrict__ row_states, int32_t num_rows,
    int32_t* __restrict__ out) {
  const int64_t t = int64_t(blockIdx.x) * blockDim.x + threadIdx.x;
  const int32_t r = blockIdx.y;
  if (t >= vocab || r >= num_rows) return;
  const int32_t s0 = row_states ? row_states[r] : r;
  int32_t res = -1;
  if (s0 < 0 || s0 >= num_states) {
    res = -1;
  } else if (t == eos_id) {
    res = accept[s0] ? s0 : -1;
  } else {
    int32_t cur = s0;
    const int32_t b = offsets[t], e = offsets[t + 1];
    bool ok = true;
    for (int32_t i = b; i < e && cur != dead; ++i) {
      const int32_t k = syms[i];
      if (k >= num_symbols) {
        ok = false;
        break;
      }
      cur = trans[int64_t(cur) * num_symbols + k];
      if (cur < 0 || cur >= num_states) {
        ok = false;
        break;
      }
    }
    res = (ok && live[cur]) ? cur : -1;
  }
  out[int64_t(r) * vocab + t] = res;
}

// int32 symbol ids to bytes, and *bad = 1 where one lies outside [0, 255]
// (a plain store: `bad` may be host memory).
__global__ __launch_bounds__(256) void narrow_symbols_kernel(const int32_t* __restrict__ sym, int64_t n,
                                                             uint8_t* __restrict__ out,
                                                             int32_t* __restrict__ bad) {
  const int64_t i = int64_t(blockIdx.x) * blockDim.x + threadIdx.x;
  const int32_t v = i < n ? sym[i] : 0;
  if (i < n) out[i] = uint8_t(v);
  if (__any(v < 0 || v > 255) && (threadIdx.x & 63) == 0) *bad = 1;
}

// Reachability (the live set of a DFA): live[s] = 1 iff an accepting state
// is reachable from s.  One workgroup sweeps the states in place over LDS
// flags until a sweep changes nothing (monotone, so at most num_states + 1
// sweeps); the flag is read by every thread between two barriers, so every
// wave takes the same exit.
constexpr int kReachThreads = 1024;
constexpr int kReachMaxStates = 65536;  // LDS flags

__global__ __launch_bounds__(kReachThreads) void reachability_kernel(
    const int32_t* __restrict__ trans, int32_t num_states, int32_t num_symbols,
    const uint8_t* __restrict__ accept, uint8_t* __restrict__ live_out) {
  __shared__ uint8_t live[kReachMaxStates];
  __shared__ int changed;
  const int tid = threadIdx.x;
  for (int32_t s = tid; s < num_states; s += kReachThreads) live[s] = accept[s] ? 1 : 0;
  for (int32_t sweep = 0; sweep <= num_states; ++sweep) {
    if (tid == 0) changed = 0;
    __syncthreads();
    for (int32_t s = tid; s < num_states; s += kReachThreads) {
      if (live[s]) continue;
      const int32_t* row = trans + int64_t(s) * num_symbols;
      for (int32_t k = 0; k < num_symbols; ++k) {
        const int32_t t = row[k];
        if (t >= 0 && t < num_states && live[t]) {
          live[s] = 1;
          changed = 1;
          break;
        }
      }
    }
    __syncthreads();
    const int more = changed;
    __syncthreads();  // every thread has read the flag before it is reset
    if (!more) break;
  }
  for (int32_t s = tid; s < num_states; s += kReachThreads) live_out[s] = live[s];
}

}  // namespace
}  // namespace bpd

using namespace bpd;

namespace {

// Shared launch of the write-only mask (both table forms): `vocab` columns,
// of which the first `tokens` have verdicts in the table.
int launch_fill(void* logits, int dtype, int64_t rows, int64_t vocab, int64_t tokens, int64_t ld, const void* table,
                int64_t table_ld, bool bits, int32_t num_states, int32_t* states,
                const int64_t* slots, const int64_t* pending, int64_t num_pending, double neg_inf,
                int32_t* err, void* stream, const int32_t* inline_values = nullptr,
                int64_t* slots_out = nullptr) {
  const int E = dense_elem_bytes(dtype);
  BPD_REQUIRE(E != 0, "unknown logits dtype code %d", dtype);
  BPD_REQUIRE(rows >= 0 && vocab >= 0 && ld >= vocab, "bad logits shape rows=%lld vocab=%lld ld=%lld",
              (long long)rows, (long long)vocab, (long long)ld);
  BPD_REQUIRE(num_states > 0, "empty grammar table");
  if (!inline_values)
    if (int rc = check_pending(pending, num_pending, slots, rows)) return rc;
  uint64_t fill = 0;
  if (int rc = fill_bits64(dtype, neg_inf, &fill)) return rc;
  if (rows == 0) return BPD_OK;
  BPD_REQUIRE(logits && table && states, "null pointer argument");
  BPD_REQUIRE(reinterpret_cast<uintptr_t>(logits) % E == 0, "logits are not aligned to their element size");
  BPD_REQUIRE(rows < (int64_t(1) << 31), "too many rows for one launch");
  const int64_t chunks = vocab == 0 ? 1 : (vocab + kChunkCols - 1) / kChunkCols;
  int64_t blocks = (chunks + kFillWaves - 1) / kFillWaves * rows;
  blocks = (blocks + kXcds - 1) / kXcds * kXcds;
  BPD_REQUIRE(blocks < (int64_t(1) << 31), "batch too large for one launch");
  hipStream_t s = as_stream(stream);
  uint8_t* lg = static_cast<uint8_t*>(logits);
  const int32_t np = int32_t(num_pending);
#define BPD_FILL(EB, BITS, N, INL)                                                              \
  dense_fill_kernel<EB, BITS, N><<<dim3(unsigned(blocks)), dim3(kFillThreads), 0, s>>>(         \
      lg, ld * EB, table, table_ld, vocab, tokens, num_states, states, slots, pending, np,      \
      uint32_t(rows), uint32_t(chunks), fill, err, INL, slots_out)
  if (inline_values) {
    return with_inline_rows(inline_values, rows + 2 * num_pending, [&](const auto& inl) -> int {
      constexpr int N = int(sizeof(inl.v) / sizeof(inl.v[0]));
      if (E == 2) BPD_FILL(2, true, N, inl);
      else if (E == 4) BPD_FILL(4, true, N, inl);
      else BPD_FILL(8, true, N, inl);
      BPD_LAUNCHED();
      return BPD_OK;
    });
  }
  const InlineRows<0> none{};
  if (bits) {
    if (E == 2) BPD_FILL(2, true, 0, none);
    else if (E == 4) BPD_FILL(4, true, 0, none);
    else BPD_FILL(8, true, 0, none);
  } else {
    if (E == 2) BPD_FILL(2, false, 0, none);
    else if (E == 4) BPD_FILL(4, false, 0, none);
    else BPD_FILL(8, false, 0, none);
  }
#undef BPD_FILL
  BPD_LAUNCHED();
  return BPD_OK;
}

}  // namespace

extern "C" int bpd_dense_apply_mask(void* logits, int dtype, int64_t rows, int64_t vocab,
                                    int64_t ld, const int32_t* tok_next, int32_t num_states,
                                    int32_t* states, const int64_t* slots,
                                    const int64_t* pending, int64_t num_pending, double neg_inf,
                                    int32_t* err, void* stream) {
  return launch_fill(logits, dtype, rows, vocab, vocab, ld, tok_next, vocab, false, num_states, states,
                     slots, pending, num_pending, neg_inf, err, stream);
}

extern "C" int bpd_dense_apply_mask_bits(void* logits, int dtype, int64_t rows, int64_t vocab,
                                         int64_t ld, const uint32_t* allow_bits, int64_t words,
                                         int32_t num_states, int32_t* states,
                                         const int64_t* slots, const int64_t* pending,
                                         int64_t num_pending, double neg_inf, int32_t* err,
                                         void* stream) {
  BPD_REQUIRE(words == (vocab + 31) / 32, "allow-bit rows must hold ceil(vocab/32) words");
  return launch_fill(logits, dtype, rows, vocab, vocab, ld, allow_bits, words, true, num_states, states,
                     slots, pending, num_pending, neg_inf, err, stream);
}

extern "C" int bpd_dense_apply_mask_padded(void* logits, int dtype, int64_t rows, int64_t vocab, int64_t cols,
                                           int64_t ld, const uint32_t* allow_bits, int64_t words,
                                           int32_t num_states, int32_t* states, const int64_t* slots,
                                           const int64_t* pending, int64_t num_pending, double neg_inf,
                                           int32_t* err, void* stream) {
  BPD_REQUIRE(words == (vocab + 31) / 32, "allow-bit rows must hold ceil(vocab/32) words");
  BPD_REQUIRE(cols >= vocab, "fewer columns than tokens");
  return launch_fill(logits, dtype, rows, cols, vocab, ld, allow_bits, words, true, num_states, states,
                     slots, pending, num_pending, neg_inf, err, stream);
}

extern "C" int bpd_dense_apply_mask_inline(void* logits, int dtype, int64_t rows, int64_t vocab, int64_t cols,
                                           int64_t ld, const uint32_t* allow_bits, int64_t words,
                                           int32_t num_states, int32_t* states, const int32_t* values,
                                           int64_t num_pending, int64_t* slots_out, double neg_inf,
                                           int32_t* err, void* stream) {
  BPD_REQUIRE(words == (vocab + 31) / 32, "allow-bit rows must hold ceil(vocab/32) words");
  BPD_REQUIRE(cols >= vocab, "fewer columns than tokens");
  if (int rc = check_inline(values, rows, num_pending, states, slots_out)) return rc;
  return launch_fill(logits, dtype, rows, cols, vocab, ld, allow_bits, words, true, num_states, states, nullptr,
                     nullptr, num_pending, neg_inf, err, stream, values, slots_out);
}

extern "C" int bpd_dense_advance(const int32_t* tok_next, int32_t num_states, int64_t vocab,
                                 int32_t* states, const int64_t* slots, const int64_t* pending,
                                 int64_t num_pending, const void* tokens, int token_dtype,
                                 int64_t rows, int32_t* next_out, int write_back, int32_t* err,
                                 void* stream) {
  return bpd_dense_advance_strided(tok_next, num_states, vocab, states, slots, pending, num_pending, tokens,
                                   token_dtype, 1, rows, next_out, write_back, err, stream);
}

extern "C" int bpd_dense_advance_strided(const int32_t* tok_next, int32_t num_states, int64_t vocab,
                                         int32_t* states, const int64_t* slots, const int64_t* pending,
                                         int64_t num_pending, const void* tokens, int token_dtype,
                                         int64_t token_stride, int64_t rows, int32_t* next_out,
                                         int write_back, int32_t* err, void* stream) {
  BPD_REQUIRE(token_dtype_ok(token_dtype), "unknown token dtype code %d", token_dtype);
  BPD_REQUIRE(num_states > 0 && vocab > 0, "empty tok_next table");
  BPD_REQUIRE(rows >= 0, "negative row count");
  BPD_REQUIRE(num_pending >= 0 && num_pending <= BPD_MAX_FUSED_PENDING,
              "at most %d queued pool writes per launch (got %lld)", BPD_MAX_FUSED_PENDING,
              (long long)num_pending);
  BPD_REQUIRE(num_pending == 0 || (pending && slots && write_back),
              "queued writes need a slot map and write_back");
  BPD_REQUIRE(rows > 0 || num_pending == 0, "queued writes need at least one row");
  if (rows == 0) return BPD_OK;
  BPD_REQUIRE(tok_next && states && tokens, "null pointer argument");
  BPD_REQUIRE(next_out || write_back, "advance with neither next_out nor write_back");
  hipStream_t s = as_stream(stream);
  if (rows <= int64_t(kAdvThreads) * kAdvPerThread) {
    dense_advance_block_kernel<<<1, kAdvThreads, 0, s>>>(tok_next, num_states, vocab, states,
                                                         slots, pending, int32_t(num_pending),
                                                         tokens, token_dtype, token_stride, rows,
                                                         next_out, write_back, err);
    BPD_LAUNCHED();
    return BPD_OK;
  }
  BPD_REQUIRE(next_out, "batches above %d rows need next_out", kAdvThreads * kAdvPerThread);
  BPD_REQUIRE(num_pending == 0, "batches above %d rows take no queued writes",
              kAdvThreads * kAdvPerThread);
  const unsigned g = unsigned((rows + 255) / 256);
  dense_advance_gather_kernel<<<g, 256, 0, s>>>(tok_next, num_states, vocab, states, slots,
                                                tokens, token_dtype, token_stride, rows, next_out, err);
  BPD_LAUNCHED();
  if (write_back) {
    dense_scatter_kernel<<<g, 256, 0, s>>>(states, slots, next_out, rows);
    BPD_LAUNCHED();
  }
  return BPD_OK;
}

extern "C" int bpd_dense_compute_mask(const int32_t* tok_next, int32_t num_states, int64_t vocab,
                                      const int32_t* states, const int64_t* slots, int64_t rows,
                                      uint32_t* bits, int32_t* err, void* stream) {
  BPD_REQUIRE(num_states > 0 && vocab >= 0 && rows >= 0, "bad shape");
  const int64_t words = (vocab + 31) / 32;
  if (rows == 0 || words == 0) return BPD_OK;
  BPD_REQUIRE(rows < 65536, "at most 65535 rows");
  BPD_REQUIRE(tok_next && states && bits, "null pointer argument");
  const dim3 grid = dim3(unsigned((vocab + kBitsTokens - 1) / kBitsTokens), unsigned(rows));
  dense_bits_kernel<<<grid, kBitsThreads, 0, as_stream(stream)>>>(tok_next, num_states, vocab, states,
                                                          slots, rows, bits, words, err);
  BPD_LAUNCHED();
  return BPD_OK;
}

extern "C" int bpd_bit_rows(const uint32_t* allow_bits, int64_t words, int32_t num_states,
                            const int32_t* states, int64_t rows, uint32_t* out, int32_t* err, void* stream) {
  BPD_REQUIRE(num_states > 0 && words >= 0 && rows >= 0, "bad shape");
  if (rows == 0 || words == 0) return BPD_OK;
  BPD_REQUIRE(allow_bits && states && out, "null pointer argument");
  const unsigned gx = unsigned((words + 4 * kBitsThreads * kBitRowLoads - 1) / (4 * kBitsThreads * kBitRowLoads));
  for (int64_t r0 = 0; r0 < rows; r0 += 65535) {  // the grid's second dimension
    const int64_t n = rows - r0 < 65535 ? rows - r0 : 65535;
    bit_rows_kernel<<<dim3(gx, unsigned(n)), kBitsThreads, 0, as_stream(stream)>>>(
        allow_bits, words, num_states, states + r0, out + r0 * words, err);
    BPD_LAUNCHED();
  }
  return BPD_OK;
}

extern "C" int bpd_dense_table_bits(const int32_t* tok_next, int32_t num_states, int64_t vocab, uint32_t* bits,
                                    void* stream) {
  BPD_REQUIRE(num_states > 0 && vocab >= 0, "bad shape");
  const int64_t words = (vocab + 31) / 32;
  if (words == 0) return BPD_OK;
  BPD_REQUIRE(tok_next && bits, "null pointer argument");
  hipStream_t st = as_stream(stream);
  // the grid's second dimension takes 65535 rows
  for (int32_t s0 = 0; s0 < num_states; s0 += 65535) {
    const int32_t n = num_states - s0 < 65535 ? num_states - s0 : 65535;
    const dim3 grid = dim3(unsigned((vocab + kBitsTokens - 1) / kBitsTokens), unsigned(n));
    dense_bits_kernel<<<grid, kBitsThreads, 0, st>>>(tok_next + int64_t(s0) * vocab, n, vocab, nullptr, nullptr, n,
                                            bits + int64_t(s0) * words, words, nullptr);
    BPD_LAUNCHED();
  }
  return BPD_OK;
}

extern "C" int bpd_build_tok_next(const int32_t* trans, int32_t num_states, int32_t num_symbols,
                                  int32_t dead, const uint8_t* accept, const uint8_t* live,
                                  const int32_t* tok_offsets, const uint8_t* tok_symbols,
                                  int64_t vocab, int32_t eos_id, const int32_t* row_states,
                                  int32_t num_rows, int32_t* out, void* stream) {
  BPD_REQUIRE(num_states > 0 && num_symbols > 0 && vocab >= 0 && num_rows >= 0, "bad shape");
  BPD_REQUIRE(dead >= 0 && dead < num_states, "dead state out of range");
  if (vocab == 0 || num_rows == 0) return BPD_OK;
  BPD_REQUIRE(num_rows < 65536, "at most 65535 table rows per launch");
  // A staged table up to 16 KB leaves a CU its four blocks of 512 threads
  // (71 states: 21.6 us; 256 threads 23.6, 1024 22.9); a larger one is shared
  // by a block of 1024 threads (two on a CU).
  if (walk_table_fits(num_states, num_symbols, 79 * 1024)) {
    const size_t lds = walk_table_bytes(num_states, num_symbols);
    const int threads = lds <= 16 * 1024 ? 512 : 1024;
    const int64_t tiles = (vocab + threads - 1) / threads;
    // as many waves as the chip holds (8192), so that each staging serves as
    // many rows as that allows (half as many: 23.9 us, twice as many: 26.5)
    int64_t split = (8192 * 64 + tiles * threads - 1) / (tiles * threads);
    const int64_t groups = (num_rows + kWalkRows - 1) / kWalkRows;
    if (split > groups) split = groups;
    const int64_t per = (groups + split - 1) / split * kWalkRows;
    const dim3 grid = dim3(unsigned(tiles), unsigned((num_rows + per - 1) / per));
    build_walk_kernel<<<grid, threads, lds, as_stream(stream)>>>(
        trans, num_states, num_symbols, dead, accept, live, tok_offsets, tok_symbols, vocab, eos_id,
        row_states, num_rows, int32_t(per), out);
    BPD_LAUNCHED();
    return BPD_OK;
  }
  const dim3 grid = dim3(unsigned((vocab + 255) / 256), unsigned(num_rows));
  build_tok_next_kernel<<<grid, 256, 0, as_stream(stream)>>>(
      trans, num_states, num_symbols, dead, accept, live, tok_offsets, tok_symbols, vocab,
      eos_id, row_states, num_rows, out);
  BPD_LAUNCHED();
  return BPD_OK;
}

extern "C" int bpd_narrow_symbols(const int32_t* symbols, int64_t n, uint8_t* out, int32_t* bad, void* stream) {
  BPD_REQUIRE(n >= 0 && n < (int64_t(1) << 31), "bad symbol count");
  if (n == 0) return BPD_OK;
  BPD_REQUIRE(symbols && out && bad, "null pointer argument");
  narrow_symbols_kernel<<<unsigned((n + 255) / 256), 256, 0, as_stream(stream)>>>(symbols, n, out, bad);
  BPD_LAUNCHED();
  return BPD_OK;
}

extern "C" int bpd_build_reachability(const int32_t* trans, int32_t num_states, int32_t num_symbols,
                                      const uint8_t* accept, uint8_t* live, void* stream) {
  BPD_REQUIRE(num_states >= 0 && num_symbols > 0, "bad table shape");
  BPD_REQUIRE(num_states <= kReachMaxStates, "at most %d states on the device", kReachMaxStates);
  if (num_states == 0) return BPD_OK;
  BPD_REQUIRE(trans && accept && live, "null pointer argument");
  reachability_kernel<<<1, kReachThreads, 0, as_stream(stream)>>>(trans, num_states, num_symbols,
                                                                   accept, live);
  BPD_LAUNCHED();
  return BPD_OK;
}
