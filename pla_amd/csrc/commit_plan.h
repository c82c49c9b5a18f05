// Device-side commit plan of the request-row KDA replay (vLLM-style runner).  From the sampled-token counts,
// the source checkpoints and, in align mode, the block table, every request gets four integers
//     commit length, final slot, boundary slot, boundary length
// without any value leaving the device, so a commit can be captured in a graph.  The plan must equal the one
// the reference computes (src/decode/kda_replayssm_vllm/commit_plan.cu:19-117; expected values
// tests/test_kda_replayssm_vllm.py:148-178); the rules, as a specification:
//
//   live       a request whose source slot is valid (> null_block_id, >= 0, < slots) and whose query interval
//              [offsets[b], offsets[b + 1]) is well formed (0 <= begin < end <= token_capacity, length <= Q).
//   commits    a live request with offsets[0] == 0 and a sampler row (mapping[b], or b) inside the table commits
//              n = min(max(sampled[row], 0), length) tokens into its source slot.
//   align      with a block table (block_size > 0) and p = computed[row] tokens already in the cache, the state
//              after n tokens belongs to the block holding token p + n - 1 (the last column when beyond the
//              table), and when the window reaches the next block boundary (n >= block_size - p % block_size)
//              the state after that many tokens also belongs to the block of position p.  A row outside the
//              block table, a negative p, an invalid destination, a boundary column beyond the table, or a
//              boundary block equal to the final block with a different length cancels the request.
//   exclusive  every slot a request writes (final, boundary) must be touched by no other request, where a
//              live request touches its source and a committing one also its destinations; and the source of a
//              committing request must be no other request's destination.  Both sides of a clash are cancelled.

#pragma once

#include "decode_common.h"

namespace pla {

struct PlanInputs {
  const void* sampled; const void* source; const void* offsets; const void* mapping; const void* computed;
  const void* blocks;
  int sampled_wide, source_wide, offsets_wide, mapping_wide, computed_wide, blocks_wide;
  int batch, capacity, sampler_rows, block_rows, block_cols, slots, Q, null_id, token_capacity;
  int64_t block_row_stride, block_col_stride, block_size;

  __device__ int64_t at(const void* base, int wide, int64_t i) const {
    return wide ? static_cast<const int64_t*>(base)[i] : (int64_t) static_cast<const int32_t*>(base)[i];
  }
  __device__ bool slot_ok(int64_t slot) const { return slot > null_id && slot >= 0 && slot < slots; }
  __device__ int64_t block_of(int64_t row, int64_t col) const {
    return at(blocks, blocks_wide, row * block_row_stride + col * block_col_stride);
  }
};

constexpr int32_t NO_CLAIM = -1;        // an absent claim of another request: equals no valid slot
constexpr int32_t NO_SLOT = -2;         // an absent slot of the examined request: equals no claim at all

struct Request {
  int32_t reads;                        // source slot of a live request, else NO_CLAIM
  int32_t tokens, final_slot, boundary_slot, boundary_tokens;     // zeroes unless it commits
};

__device__ inline Request classify(const PlanInputs& in, int b) {
  Request r{NO_CLAIM, 0, 0, 0, 0};
  if (b >= in.batch) return r;
  // Every value is read before any is judged: one trip to memory, two with a mapping.
  const int64_t source = in.at(in.source, in.source_wide, b), first = in.at(in.offsets, in.offsets_wide, 0);
  const int64_t begin = in.at(in.offsets, in.offsets_wide, b), end = in.at(in.offsets, in.offsets_wide, b + 1);
  const int64_t row = in.mapping ? in.at(in.mapping, in.mapping_wide, b) : (int64_t)b;
  const bool sampler_row = row >= 0 && row < in.sampler_rows;
  const int64_t sampled = sampler_row ? in.at(in.sampled, in.sampled_wide, row) : 0;
  const int64_t length = end - begin;
  if (!in.slot_ok(source) || begin < 0 || length <= 0 || end > in.token_capacity || length > in.Q) return r;
  r.reads = (int32_t)source;
  if (first != 0 || !sampler_row || sampled <= 0) return r;
  const int64_t n = sampled < length ? sampled : length;
  int64_t final_slot = source, boundary_slot = 0, boundary_tokens = 0;
  bool ok = true;
  if (in.block_size != 0) {             // align mode: destinations come from the block table
    ok = row < in.block_rows;
    const int64_t cached = ok ? in.at(in.computed, in.computed_wide, row) : -1;
    ok = ok && cached >= 0 && cached <= INT64_MAX - in.Q;
    if (ok) {
      int64_t last_col = (cached + n - 1) / in.block_size;
      if (last_col > in.block_cols - 1) last_col = in.block_cols - 1;
      final_slot = in.block_of(row, last_col);
      ok = in.slot_ok(final_slot);
      const int64_t to_boundary = in.block_size - cached % in.block_size;
      if (ok && n >= to_boundary) {     // the window reaches the end of the block that holds position `cached`
        const int64_t col = cached / in.block_size;
        ok = col < in.block_cols;
        if (ok) {
          boundary_slot = in.block_of(row, col);
          // one block cannot hold two different states
          ok = in.slot_ok(boundary_slot) && !(boundary_slot == final_slot && to_boundary != n);
          boundary_tokens = to_boundary;
        }
      }
    }
  }
  if (!ok) return r;
  r.tokens = (int32_t)n;
  r.final_slot = (int32_t)final_slot;
  r.boundary_slot = (int32_t)boundary_slot;
  r.boundary_tokens = (int32_t)boundary_tokens;
  return r;
}

// The slots a request touches, and whether two requests may not commit together (see "exclusive").
struct Claims {
  int32_t reads, final_slot, boundary_slot;        // NO_CLAIM where there is none
};
__device__ inline Claims claims_of(const Request& r) {
  return {r.reads, r.tokens > 0 ? r.final_slot : NO_CLAIM, r.boundary_tokens > 0 ? r.boundary_slot : NO_CLAIM};
}
__device__ inline bool claims_clash(const Claims& mine, const Claims& other) {     // mine commits: it reads and writes
  const int32_t boundary = mine.boundary_slot == NO_CLAIM ? NO_SLOT : mine.boundary_slot;
  const bool written_slot_taken = mine.final_slot == other.reads || mine.final_slot == other.final_slot ||
                                  mine.final_slot == other.boundary_slot || boundary == other.reads ||
                                  boundary == other.final_slot || boundary == other.boundary_slot;
  const bool source_overwritten = mine.reads == other.final_slot || mine.reads == other.boundary_slot;
  return written_slot_taken || source_overwritten;
}

// The plan of request b alone, worked out by a whole workgroup (every thread calls it and gets the same answer): a
// thread classifies every blockDim.x-th of the other requests and holds its claims against those of b.
__device__ inline Request commit_decision(const PlanInputs& in, int b) {
  const Request mine = classify(in, b);
  const Claims claims = claims_of(mine);
  bool clash = false;
  for (int other = threadIdx.x; other < in.batch; other += blockDim.x)
    clash = clash || (other != b && claims_clash(claims, claims_of(classify(in, other))));
  if (!__syncthreads_or(clash && mine.tokens > 0)) return mine;
  return Request{mine.reads, 0, 0, 0, 0};
}

// One channel of the conv windows of record row `row` into the paged conv history of a layer (`entry`: its row of the layer
// table): the window after the boundary, if there is one, then the window after the last committed token.
__device__ inline void copy_conv_window(const int64_t* entry, int row, int channel, const Request& r) {
  const auto conv = as_global(reinterpret_cast<uint16_t*>(entry[6]));
  const auto windows = as_global(reinterpret_cast<const uint16_t*>(entry[10]));
  const int count[2] = {r.boundary_tokens, r.tokens}, slot[2] = {r.boundary_slot, r.final_slot};
#pragma unroll
  for (int i = 0; i < 2; ++i) {
    if (count[i] <= 0) continue;
    const auto src = windows + row * entry[11] + (count[i] - 1) * entry[12] + channel * entry[13];
    const auto dst = conv + slot[i] * entry[7] + channel * entry[8];
#pragma unroll
    for (int w = 0; w < 3; ++w) dst[w * entry[9]] = src[w * entry[14]];
  }
}

// The host's checks of the plan's arguments; 0 or the error code.
inline int check_plan_inputs(const PlanInputs& in) {
  PLA_REQUIRE(in.sampled && in.source && in.offsets, "null tensor pointer");
  PLA_REQUIRE(in.batch >= 0 && in.batch <= in.capacity && in.capacity > 0, "commit query count exceeds capacity");
  PLA_REQUIRE(in.Q >= 1 && in.Q <= 32 && in.slots > 0, "invalid commit plan dimensions");
  PLA_REQUIRE(in.null_id == -1 || in.null_id == 0, "null_block_id must be -1 or 0");
  PLA_REQUIRE(in.token_capacity >= 0, "token_capacity must be between 0 and INT32_MAX");
  PLA_REQUIRE((in.blocks != nullptr) == (in.computed != nullptr) && (in.blocks != nullptr) == (in.block_size != 0),
              "align arguments must be supplied together");
  PLA_REQUIRE(in.blocks == nullptr || (in.block_size >= in.Q && in.block_cols > 0 && in.block_rows >= 0),
              "invalid align table/count/block size");
  return 0;
}

// Whether the plan's rows ([4, capacity]) share no byte with its inputs, which other workgroups may read at any time.
inline bool plan_apart(const PlanInputs& in, const int32_t* plan) {
  const uintptr_t plan_begin = reinterpret_cast<uintptr_t>(plan), plan_end = plan_begin + (uintptr_t)in.capacity * 16;
  auto apart = [&](const void* base, int wide, int64_t items) {
    const uintptr_t begin = reinterpret_cast<uintptr_t>(base);
    return base == nullptr || items <= 0 || begin >= plan_end || begin + (uintptr_t)items * (wide ? 8 : 4) <= plan_begin;
  };
  const int64_t blocks = in.block_rows > 0 ? (in.block_rows - 1) * in.block_row_stride + (in.block_cols - 1) * in.block_col_stride + 1 : 0;
  return apart(in.sampled, in.sampled_wide, in.sampler_rows) && apart(in.source, in.source_wide, in.batch) &&
         apart(in.offsets, in.offsets_wide, in.batch + 1) && apart(in.mapping, in.mapping_wide, in.batch) &&
         apart(in.computed, in.computed_wide, in.sampler_rows) && apart(in.blocks, in.blocks_wide, blocks);
}

}  // namespace pla
