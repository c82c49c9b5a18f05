// The plan of a whole commit (commit_plan.h) in a launch of its own.  Every workgroup turns all requests into three claims
// - the slot a request reads and the up to two slots it writes, -1 for none - and then decides on its share of them: a
// wavefront per committing request, lanes striding over the other requests, looks its slots up among everybody else's
// claims; the claims are never modified, so a clash cancels both sides whichever is examined first.  The claims live in
// LDS, or in the caller's scratch rows (to which all workgroups write the same values) when the batch exceeds
// what LDS holds.  Workgroups behind the batch only clear their plan rows (64 requests of a capacity of 16 384: 32.9 us
// when they classified the batch as well, 4.6 now).
//
// Bound by latency: the trips to memory of a classification, then batch / 64 steps of look-up per request.  One workgroup
// doing all look-ups takes the square of the batch: a commit of 768 requests (4 heads, 1 layer) took 235 us with it and
// takes 93 with a request per wavefront, 512 requests (6 heads, 4 layers) 378 and 314 us, 21 requests the same.

#include "commit_plan.h"

namespace pla {

constexpr int PLAN_THREADS = 256;
constexpr int PLAN_SHARE = 4;           // requests a workgroup decides on
// Up to this many requests the claims lie in LDS: 36 KB, four workgroups a CU.  us of the plan, LDS / scratch: 64 requests 4.7 / 4.3,
// 512 4.9 / 5.3, 1024 8.1 / 8.6, 2048 15.4 / 18.8, 3072 23.4 / 27.3; 4096 (three workgroups a CU, so a second round) 53.0 / 37.4.
constexpr int PLAN_LDS_BATCH = 3072;

template <bool IN_LDS>
__global__ __launch_bounds__(PLAN_THREADS) void commit_plan_kernel(const PlanInputs in, int share, int32_t* spill, int32_t* plan) {
  extern __shared__ int32_t claims_lds[];
  int32_t* const reads = IN_LDS ? claims_lds : spill;
  int32_t* const writes_final = reads + in.batch;
  int32_t* const writes_boundary = writes_final + in.batch;
  const int cap = in.capacity, first = blockIdx.x * share, last = min(first + share, cap);
  if (first >= in.batch) {
    for (int i = threadIdx.x; i < 4 * (last - first); i += PLAN_THREADS) plan[(i & 3) * cap + first + (i >> 2)] = 0;
    return;
  }

  for (int b = threadIdx.x; b < max(in.batch, last); b += PLAN_THREADS) {
    const Request r = classify(in, b);
    if (b < in.batch) {
      const Claims claims = claims_of(r);
      reads[b] = claims.reads;
      writes_final[b] = claims.final_slot;
      writes_boundary[b] = claims.boundary_slot;
    }
    if (b < first || b >= last) continue;
    plan[b] = r.tokens;
    plan[cap + b] = r.final_slot;
    plan[2 * cap + b] = r.boundary_slot;
    plan[3 * cap + b] = r.boundary_tokens;
  }
  __syncthreads();

  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  for (int b = first + wave; b < min(last, in.batch); b += PLAN_THREADS / 64) {
    const Claims mine{reads[b], writes_final[b], writes_boundary[b]};
    if (mine.final_slot == NO_CLAIM) continue;                 // wave-uniform: b commits nothing
    bool clash = false;
    for (int other = lane; other < in.batch; other += 64) {
      const Claims theirs{reads[other], writes_final[other], writes_boundary[other]};
      clash = clash || (other != b && claims_clash(mine, theirs));
    }
    if (__ballot(clash) != 0 && lane < 4) plan[lane * cap + b] = 0;
  }
}

}  // namespace pla

extern "C" int pla_kda_commit_plan_launch(
    const void* sampled, int sampled_wide, const void* source, int source_wide, const void* offsets, int offsets_wide,
    const void* mapping, int mapping_wide, const void* computed, int computed_wide, const void* blocks, int blocks_wide,
    int batch, int capacity, int sampler_rows, int block_rows, int block_cols, int slots, int Q, int null_block_id,
    int token_capacity, int64_t block_row_stride, int64_t block_col_stride, int64_t block_size,
    int32_t* candidate, int32_t* plan, void* stream) {
  using namespace pla;
  if (capacity == 0) return 0;
  PLA_REQUIRE(candidate && plan, "null tensor pointer");
  const PlanInputs in{sampled, source, offsets, mapping, computed, blocks,
                      sampled_wide, source_wide, offsets_wide, mapping_wide, computed_wide, blocks_wide,
                      batch, capacity, sampler_rows, block_rows, block_cols, slots, Q, null_block_id, token_capacity,
                      block_row_stride, block_col_stride, block_size};
  if (const int bad = check_plan_inputs(in)) return bad;
  // inputs among the plan's rows: one workgroup, so that no other one overwrites what it has yet to read
  const int share = plan_apart(in, plan) ? PLAN_SHARE : capacity;
  const dim3 grid((unsigned)((capacity + share - 1) / share)), block(PLAN_THREADS);
  const hipStream_t s = static_cast<hipStream_t>(stream);
  if (batch <= PLAN_LDS_BATCH)
    commit_plan_kernel<true><<<grid, block, (size_t)batch * 3 * sizeof(int32_t), s>>>(in, share, candidate, plan);
  else
    commit_plan_kernel<false><<<grid, block, 0, s>>>(in, share, candidate, plan);
  return check_launch("commit_plan_kernel");
}
