// Pieces of the GDN chunk-64 prefill kernels, some of them shared with KDA's: operand tiles, asynchronous copies, the
// device-side chunk tables, the split of long sequences, the plans made on the host.
#pragma once

#include <mutex>

#include "common.h"
#include "mfma_bf16.h"

namespace pla {

constexpr int CHUNK = 64;

typedef short i16x4_t __attribute__((ext_vector_type(4)));

// One transposing read: lane i of a group of 16 receives column i of the four rows the group addresses (lane t
// addresses columns 4 (t % 4) .. + 3 of row t / 4), packed as 16-bit (row 0, row 1), (row 2, row 3).
__device__ __forceinline__ uint2 read_tr4(const uint16_t* at) {
  const i16x4_t v = __builtin_amdgcn_ds_read_tr16_b64_v4i16((__attribute__((address_space(3))) i16x4_t*)at);
  return __builtin_bit_cast(uint2, v);
}

// A lower triangular 64 x 64 tile as the A (or B) operands of the products that contract over its columns: only six
// of the eight 16 x 32 operand blocks hold anything (row block m, column half s: s = 0 for every m, s = 1 for
// m = 2, 3).  Block b is 1 KiB: lane (r, kb) owns 16 bytes, columns 32 s + 4 kb .. + 3 and 32 s + 16 + 4 kb .. + 3 of
// row 16 m + r, which is the contraction order in which a pair of accumulator tiles presents its rows.  A consumer
// copies the blocks to LDS as they are and reads an operand with one 16-byte access per lane.
constexpr int TRI_BLOCKS = 6;
__device__ __forceinline__ constexpr int tri_block_m(int b) { return b < 4 ? b : b - 2; }
__device__ __forceinline__ constexpr int tri_block_s(int b) { return b < 4 ? 0 : 1; }

// ---------------------------------------------------------------------------------------------
// Asynchronous global -> LDS tile copies (global_load_lds_dwordx4: no registers, no LDS store
// instructions).  Lane i of a wavefront writes its 16 bytes at (wave-uniform LDS base) + 16 i.
//
// The copy is issued from inline assembly so that the compiler's wait-count bookkeeping does not
// see it (it would drain every outstanding copy before each LDS read).  Kernels wait by hand with
// wait_vmcnt<N>(), N = number of copies this wavefront issued after the one it needs: vector
// memory operations complete in issue order, and other memory operations issued in between only
// make such a wait longer than necessary, never shorter.
__device__ __forceinline__ void dma16(const char* gbase, uint32_t byte_offset, uint32_t lds_wave_base) {
  asm volatile("s_mov_b32 m0, %0\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %1, %2"
               :: "s"(lds_wave_base), "v"(byte_offset), "s"(gbase) : "memory", "m0");
}
// A pointer whose value is the same in every lane, as a scalar: where the compiler holds such a value in vector
// registers (a value merged from two branches of one kernel, say) dma16 cannot take it as its base.
template <typename T>
__device__ __forceinline__ T* uniform_pointer(T* p) {
  const uint64_t a = reinterpret_cast<uint64_t>(p);
  const uint32_t lo = __builtin_amdgcn_readfirstlane((uint32_t)a), hi = __builtin_amdgcn_readfirstlane((uint32_t)(a >> 32));
  return reinterpret_cast<T*>(((uint64_t)hi << 32) | lo);
}
template <int N>
__device__ __forceinline__ void wait_vmcnt() {
  static_assert(N >= 0 && N < 64, "vmcnt is a 6-bit counter");
  __builtin_amdgcn_s_waitcnt((N & 15) | ((N >> 4) << 14) | (7 << 4) | (15 << 8));
}
// Workgroup barrier that orders LDS traffic only: this wavefront's LDS operations are complete before it arrives
// and the compiler moves no memory access across it, but vector memory operations (copies, loads, stores that
// nobody in the workgroup waits for) stay in flight.
__device__ __forceinline__ void lds_barrier() {
  asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory");
}
__device__ __forceinline__ uint32_t lds_address(const void* ptr) {
  return (uint32_t)(uintptr_t)(const __attribute__((address_space(3))) void*)ptr;
}

// ---------------------------------------------------------------------------------------------
// Unpadded, swizzled 64 x 128 tiles of 16-bit values (16 KiB).  A row is sixteen 16-byte granules; granule g of row i
// lies at granule g ^ (2 (i & 7)) of that row's 256 bytes.  Measured on gfx950 with all eight wavefronts of a workgroup
// reading: 16-byte operand reads (sixteen consecutive rows, one granule index) run at the LDS peak of 256 bytes per
// cycle and the transposing 8-byte reads (four rows x four 8-byte pieces per group of sixteen lanes) at the 128 bytes
// per cycle of 8-byte reads, where rows padded to 272 bytes give 85 (two 8-byte reads per operand) and 128.
//
// Operand tiles (K, Q) also permute the columns inside each group of 32 so that the eight contraction elements a lane
// feeds to one MFMA step - columns 32 s + 4 kb .. + 3 and 32 s + 16 + 4 kb .. + 3, the order in which a pair of
// accumulator tiles presents its rows - are the two halves of ONE granule, index 4 s + kb.
constexpr int TILE128_HALVES = CHUNK * 128;
__device__ __forceinline__ int swizzled_granule(int row, int g) { return g ^ (2 * (row & 7)); }
// offset (in 16-bit elements) of granule g of row `row`
__device__ __forceinline__ int tile_offset(int row, int g) { return row * 128 + 8 * swizzled_granule(row, g); }
// A (or B) operand of contraction step s for row `row` of an operand tile: one 16-byte read
__device__ __forceinline__ bf16x8_t operand_granule(const uint16_t* tile, int row, int s, int kb) {
  return __builtin_bit_cast(bf16x8_t, *reinterpret_cast<const uint4*>(tile + tile_offset(row, 4 * s + kb)));
}
// The same operand from the TRANSPOSE of an operand tile: lane (r, kb) takes rows [32 s + 4 kb, + 4) and
// [32 s + 16 + 4 kb, + 4) of original column 16 m + r.  Lane t of a group of 16 addresses the four columns
// 16 m + 4 (t % 4) .. + 3 of row base + t / 4, which are half (m & 1) of granule 4 (m / 2) + t % 4.
__device__ __forceinline__ bf16x8_t operand_granule_transposed(const uint16_t* tile, int s, int m, int kb, int r) {
  const int row = 32 * s + 4 * kb + (r >> 2);                  // (row + 16) & 7 == row & 7: both reads share the swizzle
  const uint16_t* at = tile + tile_offset(row, 4 * (m >> 1) + (r & 3)) + 4 * (m & 1);
  const i16x4_t p0 = __builtin_amdgcn_ds_read_tr16_b64_v4i16((__attribute__((address_space(3))) i16x4_t*)at);
  const i16x4_t p1 = __builtin_amdgcn_ds_read_tr16_b64_v4i16((__attribute__((address_space(3))) i16x4_t*)(at + 16 * 128));
  typedef short i16x8_t __attribute__((ext_vector_type(8)));
  const i16x8_t u = {p0[0], p0[1], p0[2], p0[3], p1[0], p1[1], p1[2], p1[3]};
  return __builtin_bit_cast(bf16x8_t, u);
}
// Copy plan for a swizzled 64 x 128 tile whose columns keep their order (V): a 1 KiB piece is four rows, lane i of
// the issuing wavefront fills physical granule i % 16 of row 4 piece + i / 16, which holds granule
// (i % 16) ^ swizzle of that row.  Rows beyond `last_row` re-read that row.
template <int WAVES>
struct SwizzledTileCopy {
  static constexpr int PIECES = TILE128_HALVES * 2 / 1024;
  static_assert(PIECES % WAVES == 0, "every wavefront issues the same number of copies");
  static constexpr int EACH = PIECES / WAVES;
  uint32_t off[EACH];
  __device__ __forceinline__ void plan(uint32_t row_pitch_b, int last_row, int wave, int lane) {
#pragma unroll
    for (int j = 0; j < EACH; ++j) {
      const int row = 4 * (WAVES * j + wave) + (lane >> 4);
      off[j] = (uint32_t)min(row, last_row) * row_pitch_b + 16u * (uint32_t)swizzled_granule(row, lane & 15);
    }
  }
  __device__ __forceinline__ void issue(const void* tile, const char* gbase, int wave) const {
    const uint32_t base = lds_address(tile) + 1024u * wave;
#pragma unroll
    for (int j = 0; j < EACH; ++j) dma16(gbase, off[j], base + 1024u * WAVES * j);
  }
};

// Chunk table from cu_seqlens, built on the device so that no call reads offsets back to the host.
// Single workgroup.  seq_chunk_off[n] = first chunk of sequence n (seq_chunk_off[N] = total).
__device__ __forceinline__ void chunk_map(const int32_t* cu_seqlens, int N, int NC_max, int32_t* seq_chunk_off,
                                          int32_t* chunk_seq, int32_t* chunk_tok, int32_t* chunk_len) {
  // exclusive scan of the chunk counts by the first wavefront, 64 sequences per trip to memory (a serial loop
  // over the sequences would pay one memory latency per sequence)
  if (threadIdx.x < 64) {
    const int lane0 = threadIdx.x;
    int carry = 0;
    for (int base = 0; base < N; base += 64) {
      const int n = base + lane0;
      int nc = 0;
      if (n < N) nc = (max(cu_seqlens[n + 1] - cu_seqlens[n], 0) + CHUNK - 1) / CHUNK;
      int incl = nc;
#pragma unroll
      for (int d = 1; d < 64; d <<= 1) {
        const int up = __shfl_up(incl, d, 64);
        if (lane0 >= d) incl += up;
      }
      if (n < N) seq_chunk_off[n] = carry + incl - nc;
      carry += __shfl(incl, 63, 64);
    }
    if (lane0 == 0) seq_chunk_off[N] = carry;
  }
  __syncthreads();
  // one wavefront per sequence, its lanes stride over the chunks
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6, waves = blockDim.x >> 6;
  for (int n = wave; n < N; n += waves) {
    const int start = cu_seqlens[n];
    const int len = max(cu_seqlens[n + 1] - start, 0);
    const int c0 = seq_chunk_off[n];
    const int nc = (len + CHUNK - 1) / CHUNK;
    for (int c = lane; c < nc && c0 + c < NC_max; c += 64) {
      chunk_seq[c0 + c] = n;
      chunk_tok[c0 + c] = start + c * CHUNK;
      chunk_len[c0 + c] = min(CHUNK, len - c * CHUNK);
    }
  }
}

// ---------------------------------------------------------------------------------------------
// Splitting long sequences into segments, for calls with too few (sequence, head) chains to fill the
// chip.  The per-token recurrence is affine in the state, S_out = S_in M + B, where for one segment
// B is the state the segment produces from a zero state and M (K x K) is what it produces from the
// identity with all values v = 0 (rows of the k-last state transform independently).  So:
//   pass 1   A first segment runs from the caller's state, with output: it is done with, and the state it ends in is
//            its B (or, where it is the whole sequence, the final state; KDA leaves such a one to pass 2); every segment between the first and the last
//            of its sequence runs twice without output, from zero (-> B) and from the identity with v = 0 (-> M); the
//            last segment does not run: nothing needs its summary
//   combine  per (sequence, head): the state each middle segment ends in, S <- S M + B in FP32, in the place of its B
//   pass 2   every later segment runs from the state its predecessor ends in and writes o; the last one delivers the
//            final state
// which costs three sweeps over a middle segment instead of one but runs them all concurrently.  Both passes run
// one workgroup less per sequence and head than there are segments: a chip of 256 CUs takes nine segments of 32 heads.
struct SegmentTable {
  int32_t* seq_seg_off;   // [N + 1] first segment of each sequence (KDA's kernels count them: count_segments)
  int32_t* seg_c0;        // [segments] first chunk (global chunk index)
  int32_t* seg_nc;        // number of chunks
  float* M;               // [segment, head, 128, 128] transition matrices
  float* B;               // [segment, head, V, K] zero-state results, then the state the segment ends in (first segments: at once)
  float* identity;        // [128, 128]
  int seg_chunks;         // chunks per segment (0: sequences are not split)
  int split_from;         // GDN: with a longest sequence of fewer chunks none is split (KDA's kernels: count_segments)
  int max_segments;
};

// ---------------------------------------------------------------------------------------------
// Stages: with enough chains to fill the chip the per-chunk preparation (which every CU works on) and
// the sequential sweep (one workgroup per chain, most of a CU idle) are pipelined.  Each sequence is cut
// into `stages` consecutive parts; stage s of the sweep needs only the preparation of stage s, so the
// preparation of stage s + 1 runs on a second stream underneath the sweep of stage s.  The state is
// carried from stage to stage through one [V, K] tile per chain.
struct StageTable {
  int32_t* order;         // [chunks] global chunk ids, all of stage 0 first, then stage 1, ...
  int32_t* stage_begin;   // [MAX_STAGES + 2]: offsets into `order` per stage, then (last word) the number of stages in effect
  float* carry;           // [N, heads, V, K]
  int stages;             // 0: not staged
};
constexpr int MAX_STAGES = 2;
// Chunks [stage_cut(nc, s, S), stage_cut(nc, s + 1, S)) of an item of `nc` chunks belong to stage s of the S stages in
// effect (stages beyond S are empty).
// The cut is described by a plan word: the number of stages in effect in its low byte and, above it, the sixteenths of
// an item's chunks that the first of TWO stages takes.  Whoever sees the lengths on the device makes the plan
// (stage_plan): one stage when the chains are of nearly equal length (their chunks fill 80 % or more of `items x
// longest chain`: no CU falls idle before a sweep ends, so a later preparation would not run underneath it); else
// the stages the host allowed, the first of two stages taking 3/8 of every chain when the chains fill less than
// 5/8 of that rectangle and half otherwise: the preparation of the first stage is exposed, that of the second hides
// under the first sweep only as far as chains that have ended leave CUs to it (measured, ms per call, first stage of
// 8 / 7 / 6 / 5 / 4 sixteenths: 0.440 / 0.434 / 0.428 / 0.434 / 0.443 at a fill of 0.57; at fills of 0.66 half is the
// better cut by 0.4-1.1 %, at 0.31 and 0.61 three eighths by 1.4-1.9 %).
__host__ __device__ __forceinline__ int stage_plan(int64_t total, int n_items, int longest, int S) {
  const int64_t rectangle = (int64_t)n_items * longest;
  if (S <= 0 || 5 * total >= 4 * rectangle) return 1 | (8 << 8);
  return S | ((S == 2 && 8 * total < 5 * rectangle ? 6 : 8) << 8);
}
__host__ __device__ __forceinline__ int plan_stages(int plan) { return plan & 0xff; }
__host__ __device__ __forceinline__ int stage_cut(int nc, int s, int plan) {
  const int S = plan & 0xff;
  if (S == 2 && s == 1) return (int)((int64_t)nc * (plan >> 8) / 16);
  return (int)((int64_t)nc * (s < S ? s : S) / S);
}

// Single workgroup of 256 threads with (stages + 1) * N + 1 words of LDS at `pair_begin`.  Sequence i holds chunks starts[i] ..
// starts[i + 1].  (Stage, sequence) pairs count their chunks, a serial prefix places them, then every pair
// writes its own chunk ids.
__device__ __forceinline__ void stage_map(const int32_t* starts, int N, int NC_max, StageTable t, int32_t* pair_begin) {
  // pair_begin: [stages * N + 1], then N chunk counts
  const int S = t.stages;
  int32_t* const count = pair_begin + S * N + 1;
  __shared__ int stages_in_effect;
  for (int i = threadIdx.x; i < N; i += blockDim.x) count[i] = starts[i + 1] - starts[i];
  __syncthreads();
  auto count_of = [&](int i) { return count[i]; };
  if (threadIdx.x == 0) {
    // The stages pay where chains of unequal length leave CUs idle for the later preparation to run on: with
    // chains of (nearly) equal length the chip stays full to the end of a sweep, the preparation of the next stage
    // runs after it either way, and the second pair of launches is pure overhead (measured on 8 x 2048 tokens:
    // 0.24 ms in one stage, 0.27 ms in two; on eight ragged sequences of 32 810 tokens 0.50 against 0.48 ms).
    // One stage then takes everything, the others stay empty.
    int64_t total = 0;
    int longest = 0;
    for (int i = 0; i < N; ++i) { total += count_of(i); longest = max(longest, count_of(i)); }
    const int E = stage_plan(total, N, longest, S);                  // the plan word: stages in effect and the cut
    stages_in_effect = E;
    t.stage_begin[MAX_STAGES + 1] = E;
    int k = 0;
    for (int s = 0; s < S; ++s) {
      t.stage_begin[s] = k;
      for (int i = 0; i < N; ++i) {
        const int nc = count_of(i);
        pair_begin[s * N + i] = k;
        k += stage_cut(nc, s + 1, E) - stage_cut(nc, s, E);
      }
    }
    t.stage_begin[S] = k;
  }
  __syncthreads();
  const int E = stages_in_effect;
  for (int pair = threadIdx.x >> 3; pair < S * N; pair += blockDim.x >> 3) {      // eight threads per pair
    const int s = pair / N, i = pair - s * N;
    const int nc = count_of(i), lo = stage_cut(nc, s, E), hi = stage_cut(nc, s + 1, E);
    const int base = pair_begin[pair];
    for (int cc = lo + (threadIdx.x & 7); cc < hi; cc += 8)
      if (base + cc - lo < NC_max) t.order[base + cc - lo] = starts[i] + cc;
  }
}
// Chunk handled by workgroup `index` of a per-chunk kernel: all chunks in order, or those of one stage.
__device__ __forceinline__ int staged_chunk(const StageTable& t, int stage, int index, int total_chunks) {
  if (t.stages == 0) return index < total_chunks ? index : -1;
  const int begin = t.stage_begin[stage], end = t.stage_begin[stage + 1];
  return begin + index < end ? t.order[begin + index] : -1;
}

// Workgroups are handed to the eight XCDs (each with an L2 of its own) round robin by index.  Workgroups that read
// the same tiles at the same time - the `group` value heads of one q/k head sweep the same K and Q - fetch them
// from memory once if they share an L2: this maps the hardware index onto a logical one such that the members
// of a group get indices that are equal modulo 8.  The grid must be xcd_grouped_grid(total, group); indices
// beyond `total` come back as -1.
constexpr int XCDS = 8;
inline unsigned xcd_grouped_grid(unsigned total, unsigned group) {
  const unsigned groups = (total + group - 1) / group;
  return (groups + XCDS - 1) / XCDS * XCDS * group;
}
// Workgroups, a CU each, that the chip takes at once under this map: whole groups only on an XCD.
constexpr int CUS = 256;
inline int xcd_grouped_capacity(int group) {
  const int cus = CUS / XCDS;
  return group > cus ? CUS : XCDS * (cus / group) * group;
}
__device__ __forceinline__ int xcd_grouped_index(int hw_index, int group, int total) {
  const int xcd = hw_index % XCDS, t = hw_index / XCDS;
  const int member = t % group, g = (t / group) * XCDS + xcd;
  const int logical = g * group + member;
  return logical < total ? logical : -1;
}

// What one workgroup of a GDN sweep runs through: a whole sequence (with stages only the part of it that belongs to
// `stage`, which may hold no chunk at all, the state being carried from stage to stage in a tile), or one segment of a split
// call in one of the roles above.
struct SweepRole {
  int n, head, c_begin, c_end;
  const float* init;      // [V, K] tile the state starts from (nullptr: zero)
  float* fin;             // [V, K] tile that receives the state at the end (nullptr: none)
  bool zero_v, active;
};
struct SweepStates { const float* h0; const int32_t* h0_indices; int64_t h0_slot_stride; float* ht; const int32_t* ht_indices; int64_t ht_slot_stride; };
__device__ __forceinline__ const float* state_in(const SweepStates& x, int n, int head) {
  const int slot = (x.h0 != nullptr) ? (x.h0_indices ? x.h0_indices[n] : n) : -1;
  return slot >= 0 ? x.h0 + (int64_t)slot * x.h0_slot_stride + (int64_t)head * 16384 : nullptr;
}
__device__ __forceinline__ float* state_out(const SweepStates& x, int n, int head) {
  const int slot = (x.ht != nullptr) ? (x.ht_indices ? x.ht_indices[n] : n) : -1;
  return slot >= 0 ? x.ht + (int64_t)slot * x.ht_slot_stride + (int64_t)head * 16384 : nullptr;
}
// block: logical index of the (sequence, head).  inline_chunks (x >= 0): (first chunk, end chunk, stages in effect) of its sequence
// worked out by the caller (inline_sequences) instead of read from the tables.
__device__ __forceinline__ SweepRole sequence_role(int block, int heads, const int32_t* seq_chunk_off, const StageTable& stg, int stage,
                                                   const SweepStates& states, const int3 inline_chunks) {
  SweepRole r{};
  r.n = block / heads;
  r.head = block - r.n * heads;
  r.c_begin = inline_chunks.x >= 0 ? inline_chunks.x : seq_chunk_off[r.n];
  r.c_end = inline_chunks.x >= 0 ? inline_chunks.y : seq_chunk_off[r.n + 1];
  if (r.c_begin >= r.c_end) return r;              // empty sequence: state untouched, no output
  r.init = state_in(states, r.n, r.head);
  r.fin = state_out(states, r.n, r.head);
  if (stg.stages > 0) {
    const int E = inline_chunks.x >= 0 ? inline_chunks.z : stg.stage_begin[MAX_STAGES + 1];   // the plan word (stage_plan)
    if (stage >= plan_stages(E)) return r;                                      // an empty stage: the one before it delivered the state
    float* const carry = stg.carry + ((int64_t)r.n * heads + r.head) * 16384;
    const int nc = r.c_end - r.c_begin, c0 = r.c_begin;
    r.c_begin = c0 + stage_cut(nc, stage, E);
    r.c_end = c0 + stage_cut(nc, stage + 1, E);
    if (stage > 0) r.init = carry;
    if (stage < plan_stages(E) - 1) r.fin = carry;
  }
  r.active = true;
  return r;
}

// ---------------------------------------------------------------------------------------------
// The same tables worked out by ONE wavefront in registers, for calls of whole sequences with at most 64
// sequences: lane n holds sequence n, prefix sums run over the lanes.  A kernel that does this at its start needs no
// table kernel before it (one launch and its gap less on the critical path of a call) and no dependent trips to
// memory for its tile: one load of cu_seqlens per lane.  The results equal chunk_map / stage_map / staged_chunk /
// sequence_role for the same offsets, including the rule that keeps a single stage for chains of nearly equal
// length.  All 64 lanes of the wavefront must call these functions together.
constexpr int INLINE_TABLE_SEQUENCES = 64;
// Inclusive scan over the 64 lanes by DPP: six moves in the vector pipe instead of six dependent LDS permutes, which
// stood at the head of every workgroup (three prompts of 24 to 200 tokens: preparation 9.5 -> 8.8 us, sweep 15.8 -> 15.2).
// `identity` is the operation's.
template <typename Op>
__device__ __forceinline__ int wave_scan(int x, int identity, Op op) {
  x = op(x, __builtin_amdgcn_update_dpp(identity, x, 0x111, 0xF, 0xF, false));     // row_shr:1, 2, 4, 8
  x = op(x, __builtin_amdgcn_update_dpp(identity, x, 0x112, 0xF, 0xF, false));
  x = op(x, __builtin_amdgcn_update_dpp(identity, x, 0x114, 0xF, 0xF, false));
  x = op(x, __builtin_amdgcn_update_dpp(identity, x, 0x118, 0xF, 0xF, false));
  x = op(x, __builtin_amdgcn_update_dpp(identity, x, 0x142, 0xA, 0xF, false));     // row_bcast:15 into rows 1 and 3
  return op(x, __builtin_amdgcn_update_dpp(identity, x, 0x143, 0xC, 0xF, false));  // row_bcast:31 into rows 2 and 3
}
__device__ __forceinline__ int wave_inclusive_scan(int x) {
  return wave_scan(x, 0, [](int a, int b) { return a + b; });
}
struct InlineSequences {
  int start, len, nc, off;      // this lane's sequence: first token, tokens, chunks, first chunk (global index)
  int total, E;                 // chunks of the call; the plan word (stage_plan)
};
__device__ __forceinline__ InlineSequences inline_sequences(const int32_t* cu_seqlens, int N, int stages, int lane) {
  InlineSequences q;
  const int a = lane < N ? cu_seqlens[lane] : 0, b = lane < N ? cu_seqlens[lane + 1] : 0;
  q.start = a;
  q.len = max(b - a, 0);
  q.nc = (q.len + CHUNK - 1) / CHUNK;
  const int incl = wave_inclusive_scan(q.nc);
  q.off = incl - q.nc;
  q.total = __builtin_amdgcn_readlane(incl, 63);
  const int longest = __builtin_amdgcn_readlane(wave_scan(q.nc, 0, [](int a, int b) { return max(a, b); }), 63);
  q.E = stage_plan(q.total, N, longest, stages);
  return q;
}
// Chunk `index` of stage `stage` (all chunks in order when the call is not staged): its global chunk id, first token
// and length, or id -1 when the stage holds fewer chunks.
struct InlineTile { int cb, t0, len; };
__device__ __forceinline__ InlineTile inline_tile(const InlineSequences& q, int stage, int index, int NC_max) {
  InlineTile t{-1, 0, 0};
  if (stage >= plan_stages(q.E)) return t;
  const int lo = stage_cut(q.nc, stage, q.E), hi = stage_cut(q.nc, stage + 1, q.E);
  const int cnt = hi - lo;
  const int before = wave_inclusive_scan(cnt) - cnt;
  const unsigned long long owner = __ballot(index >= before && index < before + cnt);
  if (owner == 0) return t;
  const int n = __builtin_amdgcn_readfirstlane(__ffsll((long long)owner) - 1);
  const int cc = __builtin_amdgcn_readlane(lo, n) + index - __builtin_amdgcn_readlane(before, n);
  const int cb = __builtin_amdgcn_readlane(q.off, n) + cc;
  if (cb >= NC_max) return t;                   // offsets that do not fit the workspace: the tile is skipped
  t.cb = cb;
  t.t0 = __builtin_amdgcn_readlane(q.start, n) + cc * CHUNK;
  t.len = min(CHUNK, __builtin_amdgcn_readlane(q.len, n) - cc * CHUNK);
  return t;
}

// The tokens of sequence n, whatever the offsets hold, inside the call's T tokens: (first token, tokens).
__device__ __forceinline__ int2 sequence_tokens(const int32_t* cu_seqlens, int n, int T) {
  const int a = min(max(cu_seqlens[n], 0), T), b = min(max(cu_seqlens[n + 1], a), T);
  return make_int2(a, b - a);
}
// The segments of a split call (at most 64 sequences), counted by one wavefront: lane n counts those of sequence n.  With a longest
// sequence of less than `split_from` chunks none is split.  The sweeps and the combine step between them take the same counts from
// here, so that they agree on every tile whatever the offsets hold.
struct SegmentCounts { int2 tokens; int chunks, count, before; };      // chunks: of a segment; the others: of this lane's sequence
__device__ __forceinline__ SegmentCounts count_segments(const int32_t* cu_seqlens, int N, int T, int seg_chunks, int split_from, int lane) {
  SegmentCounts r;
  r.tokens = lane < N ? sequence_tokens(cu_seqlens, lane, T) : make_int2(0, 0);
  const int nc = (r.tokens.y + CHUNK - 1) / CHUNK;
  const int longest = __builtin_amdgcn_readlane(wave_scan(nc, 0, [](int a, int b) { return max(a, b); }), 63);
  r.chunks = longest < split_from ? max(longest, 1) : seg_chunks;
  r.count = (nc + r.chunks - 1) / r.chunks;
  r.before = wave_inclusive_scan(r.count) - r.count;
  return r;
}

// Segment `i` of those that one of the sweeps over segments runs: the first one all but the last of each sequence (`second`: all
// but the first), a sequence of one segment belonging to the sweep that names it (`singles`).  `count` is that of the lane's sequence.
// Counted like this, the workgroups of segments that a sweep does not run are all behind the others in its grid.  Among them each
// takes its turn on a CU, and as workgroups go to the XCDs and their engines in turn, full or not, 228 that swept could take two rounds
// on 256 CUs (first sweep, us, among them / behind: KDA, 2245 + 1173 + 1657 + 1355 tokens of 12 heads 84.0 / 48.6; GDN, three of 4200 to
// 4500 tokens, 16 value heads 87.0 / 53.8; 16 384 tokens, 32 value heads, where it is the last 32 of 288, 128 / 105.6).
struct SweptSegment { int sequence, index, count, number; };      // sequence < 0: none; number: among all segments of the call
struct SweptSegments { int before, swept; unsigned long long left_out; };
__device__ __forceinline__ SweptSegments swept_segments(int count, bool singles) {      // lane n: of sequence n
  SweptSegments r;
  r.swept = count > 1 ? count - 1 : singles ? count : 0;
  r.before = wave_inclusive_scan(r.swept) - r.swept;
  r.left_out = __ballot(count > r.swept);
  return r;
}
__device__ __forceinline__ SweptSegment swept_segment(const SweptSegments& s, int count, bool second, int i) {
  const unsigned long long owner = __ballot(i >= s.before && i < s.before + s.swept);
  if (owner == 0) return SweptSegment{-1, 0, 0, 0};
  SweptSegment r;
  r.sequence = __builtin_amdgcn_readfirstlane(__ffsll((long long)owner) - 1);
  r.count = __builtin_amdgcn_readlane(count, r.sequence);
  const int before = __builtin_amdgcn_readlane(s.before, r.sequence);
  r.index = i - before + (second && r.count > 1 ? 1 : 0);
  r.number = before + __popcll(s.left_out & ((1ull << r.sequence) - 1)) + r.index;
  return r;
}
// The role of (segment, head) in a sweep of a GDN call.
//   FIRST_OUT  first sweep, a first segment: with output from the caller's state
//   ZERO, IDENTITY  first sweep, a segment between the first and the last: for its summaries B and M
//   LATER      second sweep: with output from the state that the combine step left in its predecessor's B
enum class SegmentSweep { FIRST_OUT, ZERO, IDENTITY, LATER };
__device__ __forceinline__ SweepRole segment_role(SegmentSweep sweep, const SweptSegment& s, int head, int heads, const SegmentTable& seg,
                                                  const SweepStates& states) {
  SweepRole r{};
  if (s.sequence < 0 || s.number >= seg.max_segments) return r;      // (number: offsets that do not fit the workspace)
  r.active = true;
  r.n = s.sequence;
  r.head = head;
  r.c_begin = seg.seg_c0[s.number];
  r.c_end = r.c_begin + seg.seg_nc[s.number];
  const int64_t tile = ((int64_t)s.number * heads + head) * 16384;
  if (sweep == SegmentSweep::FIRST_OUT) r.init = state_in(states, r.n, head);
  if (sweep == SegmentSweep::IDENTITY) { r.init = seg.identity; r.zero_v = true; }
  if (sweep == SegmentSweep::LATER) r.init = seg.B + tile - (int64_t)heads * 16384;
  if (sweep == SegmentSweep::IDENTITY) r.fin = seg.M + tile;
  else if (s.index + 1 == s.count) r.fin = state_out(states, r.n, head);
  else if (sweep != SegmentSweep::LATER) r.fin = seg.B + tile;
  return r;
}

// The tables of a split call (at most 64 sequences): chunks and segments per sequence, the segments, the 128 x 128 identity.  Single
// workgroup; every wavefront counts for itself from one load of the offsets, as every trip to memory more stands at the end of the
// preparation (32 sequences of 65 tokens, 2 value heads, 26.7 -> 23.6 us against tables made one from another).
__device__ __forceinline__ void segment_map(const int32_t* cu_seqlens, int N, int32_t* seq_chunk_off, SegmentTable t) {
  const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int nc = lane < N ? (max(cu_seqlens[lane + 1] - cu_seqlens[lane], 0) + CHUNK - 1) / CHUNK : 0;
  const int longest = __builtin_amdgcn_readlane(wave_scan(nc, 0, [](int a, int b) { return max(a, b); }), 63);
  const int chunks = longest < t.split_from ? max(longest, 1) : t.seg_chunks;
  const int ns = (nc + chunks - 1) / chunks;
  const int c0 = wave_inclusive_scan(nc) - nc, s0 = wave_inclusive_scan(ns) - ns;
  if (wave == 0 && lane <= N) {                // (lane N, or lane 63 for 64 sequences, holds the totals)
    seq_chunk_off[lane] = c0;
    t.seq_seg_off[lane] = s0;
  }
  if (N == 64 && threadIdx.x == 63) {
    seq_chunk_off[64] = c0 + nc;
    t.seq_seg_off[64] = s0 + ns;
  }
  for (int n = wave; n < N; n += blockDim.x >> 6) {
    const int first = __builtin_amdgcn_readlane(c0, n), count = __builtin_amdgcn_readlane(ns, n), at = __builtin_amdgcn_readlane(s0, n);
    const int all = __builtin_amdgcn_readlane(nc, n);
    for (int i = lane; i < count && at + i < t.max_segments; i += 64) {
      t.seg_c0[at + i] = first + i * chunks;
      t.seg_nc[at + i] = min(chunks, all - i * chunks);
    }
  }
  for (int i = threadIdx.x; i < 128 * 128; i += blockDim.x) t.identity[i] = (i >> 7) == (i & 127) ? 1.f : 0.f;
}

// Eight workgroups of 256 threads per (sequence, head), each owning 16 rows of the state (rows transform
// independently): walks the sequence's middle segments and leaves the state each of them ends in - the one that enters
// the next - in the place of its B.  A step S <- S M + B is a 16 x 128 x 128 product per workgroup on the FP32 MFMA
// (v_mfma_f32_16x16x4_f32, exact products, FP32 accumulation): wavefront w owns columns 32 w .. 32 w + 31 as two
// accumulator tiles that start from B; the A operand is the workgroup's 16 rows of S from LDS (lane (r, kb) takes
// S[r][16 s + 4 kb + e] for step (s, e)), the B operand the matching row of M straight from memory (lane (c, kb): columns 2 c
// and 2 c + 1 of the wavefront's in the two tiles, eight bytes of row 16 s + 4 kb + e, 128 contiguous bytes per group of 16
// lanes).  M and B do not depend on the state, so those of the next segment are requested during the products of this one, whose 64
// MFMAs (32 cycles each) are what bounds a step: 1.28 us.  A wavefront issues in order, so requests ahead of the products
// delay them, and the compiler waits by a count of those still out, of which the hardware counts 63.  17 858 + 20 774 tokens of 3 heads, 46
// segments: 67.7 us with M requested where it is used, 70.9 with 72 requests of four bytes ahead of the products, left out at the
// end (every other step then waited for all of them), 81 with 36 of eight bytes, 59.5 with one of those at every second MFMA.
constexpr int COMBINE_SPLIT = 8;
template <bool TABLE>
static __global__ __launch_bounds__(256, 1) void segment_combine_kernel(SegmentTable t, const int32_t* cu_seqlens, int N, int T, int heads, int split_from) {
  // the eight workgroups of a chain read the same M tiles: on one XCD they come from memory once (xcd_grouped_index)
  const int logical = xcd_grouped_index(blockIdx.x, COMBINE_SPLIT, N * heads * COMBINE_SPLIT);
  if (logical < 0) return;
  const int part = logical % COMBINE_SPLIT;
  const int chain = logical / COMBINE_SPLIT;
  const int n = chain / heads, h = chain - n * heads;
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  // the sequence's segments as the sweeps have them: from the table (GDN), or counted by every wavefront for itself; offsets
  // of overlapping sequences may give more of them than there are tiles.  (Counting them for GDN too: 2915 tokens of 16 heads 110.3 ->
  // 110.9 us, 8192 of 8 122.1 -> 123.2.)
  int first, end;
  if constexpr (TABLE) {
    first = t.seq_seg_off[n];
    end = t.seq_seg_off[n + 1];
  } else {
    const SegmentCounts s = count_segments(cu_seqlens, N, T, t.seg_chunks, split_from, lane);
    first = __builtin_amdgcn_readlane(s.before, n);
    end = first + __builtin_amdgcn_readlane(s.count, n);
  }
  end = min(end, t.max_segments);
  if (end - first < 3) return;                 // no middle segment: the second one starts from the first one's B
  __shared__ __align__(16) float S[2][16][132];
  const int c = lane & 15, kb = lane >> 4;
  const int col0 = 32 * wave + 2 * c;          // this lane's column of accumulator tile 0 (tile 1: + 1)
  // place of accumulator elements (tile 0 and 1, row v) inside a [128, 128] tile
  auto at = [&](int v) { return (int64_t)(16 * part + 4 * kb + v) * 128 + col0; };
  auto tile_of = [&](int seg) { return ((int64_t)seg * heads + h) * 16384; };
  struct Operands { float2 m[32], b[4]; };
  auto request_b = [&](int seg, Operands& x) {
#pragma unroll
    for (int v = 0; v < 4; ++v) x.b[v] = *reinterpret_cast<const float2*>(t.B + tile_of(seg) + at(v));
  };
  const float* const M_lane = t.M + 4 * kb * 128 + col0;
  auto request_m = [&](int seg, Operands& x, int i) {          // row 16 (i / 4) + 4 kb + i % 4
    x.m[i] = *reinterpret_cast<const float2*>(M_lane + tile_of(seg) + (16 * (i >> 2) + (i & 3)) * 128);
  };
  f32x4_t acc[2];
#pragma unroll
  for (int v = 0; v < 4; ++v) {
    const float2 b = *reinterpret_cast<const float2*>(t.B + tile_of(first) + at(v));
    acc[0][v] = b.x;
    acc[1][v] = b.y;
  }
  const int last = end - 1;                    // the last segment has no summary (its tiles may be requested, and are not used)
  // S in LDS is double buffered by the parity of the step: one barrier a step
  auto step = [&](int seg, const Operands& x, Operands& next, float (&Sp)[16][132]) {
#pragma unroll
    for (int v = 0; v < 4; ++v) *reinterpret_cast<float2*>(&Sp[4 * kb + v][col0]) = make_float2(acc[0][v], acc[1][v]);
    lds_barrier();
    float4 a[8];
#pragma unroll
    for (int s8 = 0; s8 < 8; ++s8) a[s8] = *reinterpret_cast<const float4*>(&Sp[c][16 * s8 + 4 * kb]);
#pragma unroll
    for (int v = 0; v < 4; ++v) {
      acc[0][v] = x.b[v].x;
      acc[1][v] = x.b[v].y;
      asm volatile("" : "+v"(acc[0][v]), "+v"(acc[1][v]));      // (here: the compiler would wait for them in the step before)
    }
    request_b(seg + 1, next);
#pragma unroll
    for (int i = 0; i < 32; ++i) {
      const float4 q = a[i >> 2];
      const float av = (i & 3) == 0 ? q.x : (i & 3) == 1 ? q.y : (i & 3) == 2 ? q.z : q.w;
      request_m(seg + 1, next, i);
      acc[0] = __builtin_amdgcn_mfma_f32_16x16x4f32(av, x.m[i].x, acc[0], 0, 0, 0);
      acc[1] = __builtin_amdgcn_mfma_f32_16x16x4f32(av, x.m[i].y, acc[1], 0, 0, 0);
      __builtin_amdgcn_sched_barrier(0);
    }
    float* const dst = t.B + tile_of(seg);
#pragma unroll
    for (int v = 0; v < 4; ++v) *reinterpret_cast<float2*>(dst + at(v)) = make_float2(acc[0][v], acc[1][v]);
  };
  Operands even, odd;
  request_b(first + 1, even);
#pragma unroll
  for (int i = 0; i < 32; ++i) request_m(first + 1, even, i);
  int seg = first + 1;
  for (; seg + 1 < last; seg += 2) {
    step(seg, even, odd, S[0]);
    step(seg + 1, odd, even, S[1]);
  }
  if (seg < last) step(seg, even, odd, S[0]);
}

// Zero the rows of a dense [T, heads, 128] 16-bit output that lie beyond the last sequence (workgroup `block` of `blocks`).
__device__ __forceinline__ void zero_tail(uint16_t* o, const int32_t* cu_seqlens, int N, int T, int heads, int block, int blocks) {
  const int64_t first = (int64_t)max(cu_seqlens[N], 0) * heads * 128;
  const int64_t total = (int64_t)T * heads * 128;
  for (int64_t i = first + (int64_t)block * blockDim.x + threadIdx.x; i < total; i += (int64_t)blocks * blockDim.x)
    o[i] = 0;
}

// The tables of a call of more than 64 sequences in one launch.  Workgroup 0 builds the chunk table, then (pipelined calls) the
// stage table from it, through memory, after a device-scope fence and a barrier of that one workgroup.  The other workgroups zero the
// output rows beyond the last sequence.  Dynamic LDS: (stages + 1) * N + 1 words.
constexpr int TABLE_WORKGROUPS = 1 + 64;
static __global__ __launch_bounds__(256) void prefill_tables_kernel(
    const int32_t* cu_seqlens, int N, int T, int NC_max, int32_t* seq_chunk_off, int32_t* chunk_seq,
    int32_t* chunk_tok, int32_t* chunk_len, StageTable stg, uint16_t* o, int heads) {
  extern __shared__ int32_t table_lds[];
  if (blockIdx.x > 0) {
    zero_tail(o, cu_seqlens, N, T, heads, blockIdx.x - 1, gridDim.x - 1);
    return;
  }
  chunk_map(cu_seqlens, N, NC_max, seq_chunk_off, chunk_seq, chunk_tok, chunk_len);
  if (stg.stages > 0) {
    __threadfence();
    __syncthreads();
    stage_map(seq_chunk_off, N, NC_max, stg, table_lds);
  }
}
inline void launch_tables(hipStream_t s, const int32_t* cu_seqlens, int N, int T, int NC_max, int32_t* seq_chunk_off,
                          int32_t* chunk_seq, int32_t* chunk_tok, int32_t* chunk_len, const StageTable& stg, void* o, int heads) {
  const size_t lds = stg.stages > 0 ? (size_t)((stg.stages + 1) * N + 1) * 4 : 0;
  hipLaunchKernelGGL(prefill_tables_kernel, dim3(TABLE_WORKGROUPS), dim3(256), lds, s, cu_seqlens, N, T, NC_max,
                     seq_chunk_off, chunk_seq, chunk_tok, chunk_len, stg, reinterpret_cast<uint16_t*>(o), heads);
}

inline size_t align_up256(size_t x) { return (x + 255) & ~(size_t)255; }

// Side streams (default priority, non-blocking), each with its own fork / ready events.  A call takes one from
// its device's pool for the time it enqueues its launches and puts it back before it returns, so calls that
// are enqueued concurrently (host threads launching on different streams) never share a stream or an event,
// while consecutive calls reuse the same few objects: an event wait binds to the record that precedes it in
// the calling thread, and work queued on a reused side stream simply runs after the previous call's.  A side
// stream that has joined a graph capture stays part of it until the capture ends: only calls of that same
// capture may take it again (every staged call of one capture then shares one side stream), any other call
// passes it over.  Streams and events are created on first need and kept for the life of the process.  A call
// that finds no side stream (the pool is exhausted, or creation failed) is not staged: the lease is taken
// before the first launch, so nothing has been enqueued by then.
struct SideStream {
  hipStream_t stream;
  hipEvent_t fork;
  hipEvent_t ready[MAX_STAGES];
  bool busy;
};
class SideStreamLease {
 public:
  // caller: the stream the call launches on; wanted: false leaves the lease empty
  SideStreamLease(hipStream_t caller, bool wanted) : taken_(nullptr) {
    int dev = 0;
    if (!wanted || hipGetDevice(&dev) != hipSuccess || dev < 0 || dev >= MAX_DEVICES) return;
    unsigned long long caller_capture = 0;
    const bool caller_capturing = capture_of(caller, &caller_capture);
    std::lock_guard<std::mutex> lock(guard());
    SideStream* const pool = pools()[dev];
    SideStream* idle = nullptr;
    for (int i = 0; i < POOL && taken_ == nullptr; ++i) {
      if (pool[i].stream == nullptr || pool[i].busy) continue;
      unsigned long long id = 0;
      if (!capture_of(pool[i].stream, &id)) { if (idle == nullptr) idle = &pool[i]; }
      else if (caller_capturing && id == caller_capture) taken_ = &pool[i];      // already part of the caller's capture
    }
    if (taken_ == nullptr) taken_ = idle;
    if (taken_ == nullptr)
      for (int i = 0; i < POOL; ++i)
        if (pool[i].stream == nullptr) {
          if (create(pool[i])) taken_ = &pool[i];
          break;
        }
    if (taken_ != nullptr) taken_->busy = true;
  }
  ~SideStreamLease() {
    if (taken_ == nullptr) return;
    std::lock_guard<std::mutex> lock(guard());
    taken_->busy = false;
  }
  SideStreamLease(const SideStreamLease&) = delete;
  SideStreamLease& operator=(const SideStreamLease&) = delete;
  SideStream* get() const { return taken_; }     // nullptr: not wanted, none could be created, or the pool is in use

 private:
  static constexpr int MAX_DEVICES = 64, POOL = 16;
  static std::mutex& guard() { static std::mutex m; return m; }
  static SideStream (*pools())[POOL] { static SideStream table[MAX_DEVICES][POOL] = {}; return table; }
  // true (and the capture's id) while the stream is part of an unfinished graph capture; a stream whose state
  // cannot be read counts as capturing with an id no caller has
  static bool capture_of(hipStream_t stream, unsigned long long* id) {
    hipStreamCaptureStatus status = hipStreamCaptureStatusNone;
    if (hipStreamGetCaptureInfo(stream, &status, id) != hipSuccess) { *id = ~0ull; return true; }
    return status != hipStreamCaptureStatusNone;
  }
  static bool create(SideStream& t) {
    SideStream made{};
    if (hipStreamCreateWithFlags(&made.stream, hipStreamNonBlocking) != hipSuccess) return false;
    bool ok = hipEventCreateWithFlags(&made.fork, hipEventDisableTiming) == hipSuccess;
    for (int i = 0; i < MAX_STAGES && ok; ++i) ok = hipEventCreateWithFlags(&made.ready[i], hipEventDisableTiming) == hipSuccess;
    if (!ok) {                                   // give back what was created
      for (int i = 0; i < MAX_STAGES; ++i)
        if (made.ready[i] != nullptr) (void)hipEventDestroy(made.ready[i]);
      if (made.fork != nullptr) (void)hipEventDestroy(made.fork);
      (void)hipStreamDestroy(made.stream);
      return false;
    }
    t = made;
    return true;
  }
  SideStream* taken_;
};

// Plan of a mixed sweep (gdn_fused_sweep_mixed_kernel, kda_sweep_mixed_kernel: the chains of the longest sequences as
// two workgroups of 64 V columns each, first in the grid, the others whole, longest first, in one launch) for sequences that sweep `r[n]` chunks in one launch:
// order[] receives the sequences longest first, the return value is the number of leading ones whose chains are swept
// as two halves (0: sweep all chains whole).  The launch is priced in chunk times of a whole chain on an idle chip:
// a half takes `half_cost` (0.9 measured for GDN) of that, the launch lasts as long as its longest chain (or as the whole chains need on the CUs the
// halves leave them, or as all the work needs on all CUs), and a chunk takes up to `fill_cost` (17 % for GDN) longer as the chip fills (3.0
// us with a third of the CUs busy, 3.5 us with all of them: the sweeps share the memory system).  The split is taken
// where the price falls by 5 % or more.
inline int mixed_sweep_plan(const int* r, int N, int HV, unsigned char* order, double half_cost = 0.9, double fill_cost = 0.17) {
  for (int n = 0; n < N; ++n) {
    int at = n;
    for (; at > 0 && r[order[at - 1]] < r[n]; --at) order[at] = order[at - 1];
    order[at] = (unsigned char)n;
  }
  double rest = 0, halves = 0;
  for (int n = 0; n < N; ++n) rest += r[n];
  if (rest == 0) return 0;
  double whole_price = 0, best = 0;
  int best_k = 0;
  for (int k = 0; k <= N && 2 * k * HV <= CUS; ++k) {
    if (k > 0) { halves += r[order[k - 1]]; rest -= r[order[k - 1]]; }
    const double work = (2 * half_cost * halves + rest) * HV;
    double span = std::max(k > 0 ? half_cost * r[order[0]] : 0.0, work / CUS);
    if (k < N) {
      span = std::max(span, (double)r[order[k]]);
      if ((int64_t)(N + k) * HV > CUS) {          // whole chains wait for CUs: longest first on those the halves leave
        const int free_cus = CUS - 2 * k * HV;
        if (free_cus <= 0) break;
        span = std::max(span, rest * HV / free_cus + 0.5 * r[order[N - 1]]);
      }
    }
    const double price = span * (1.0 + fill_cost * std::min(1.0, work / (CUS * span)));
    if (k == 0) whole_price = best = price;
    else if (price < best) { best = price; best_k = k; }
  }
  return best <= 0.95 * whole_price ? best_k : 0;
}

// Stages for a call of whole sequences: two, where there are enough chains to fill the chip and 16 chunks per
// sequence on average; the table kernel then keeps both only for chains of unequal length (stage_map).  Measured on
// GDN, eight ragged sequences of 32 810 tokens: 0.50 ms in one stage, 0.48 in two, 0.52 in four - every further stage
// costs about 25 us (two more launches, an event between two streams, the state through memory, a pipeline that
// fills again), and the preparation only hides under a sweep on CUs that chains which ended early have left.
// (Segmented calls already keep every CU busy with sweeps - staging them was measured for GDN: 0.57 -> 0.66 ms for
// one sequence of 16 384 tokens -; the KDA path has no stages: its sweeps form their operands themselves.)
inline int pick_stages(int T, int N, int heads) {
  // (the stage map keeps (stages + 1) counters per sequence in LDS: at most 2048 sequences)
  return ((int64_t)N * heads >= 128 && T / CHUNK >= 16 * N && N <= 2048) ? MAX_STAGES : 0;
}

// Launch order of a prefill call, shared by both paths.  `prepare(stream)` launches the per-chunk
// kernels of stage *stage_field, `sweep()` the sequential kernel of that stage.
// Stage 0 is prepared on the caller's stream, alone; the side stream (a SideStreamLease the caller holds for the
// time of the call) prepares the other stages underneath the sweeps and is joined before the last sweep starts.
template <typename Prepare, typename Sweep>
inline bool launch_pipeline(hipStream_t s, int stages, SideStream* side, int* stage_field, Prepare prepare, Sweep sweep) {
  if (stages == 0) {
    *stage_field = 0;
    prepare(s);
    sweep();
    return true;
  }
  if (side == nullptr) return false;             // (callers stage a call only with a side stream in hand)
  bool ok = true;
  for (int st = 0; st < stages; ++st) {
    *stage_field = st;
    prepare(st == 0 ? s : side->stream);
    if (st == 0) {
      ok = ok && hipEventRecord(side->fork, s) == hipSuccess;
      ok = ok && hipStreamWaitEvent(side->stream, side->fork, 0) == hipSuccess;
    } else {
      ok = ok && hipEventRecord(side->ready[st], side->stream) == hipSuccess;
    }
  }
  for (int st = 0; st < stages; ++st) {
    *stage_field = st;
    if (st > 0) ok = ok && hipStreamWaitEvent(s, side->ready[st], 0) == hipSuccess;
    sweep();
  }
  return ok;
}

}  // namespace pla
