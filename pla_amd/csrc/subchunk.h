// Pieces of the one-pass prefill sweeps over sub-chunks of 16 tokens: the operand layouts that producing and computing
// wavefronts share through LDS, the inverse of a 16 x 16 unit triangle, the token range of a chain.
//
// Layout.  A token row of 128 channels is a row operand of the 16x16x32 MFMA in four contraction steps: lane (t, g) =
// (lane % 16, lane / 16) holds channels 32 s + 8 g .. + 7 of token t, one 16-byte piece a step, which is also how the
// rows lie in memory.  The state follows that order: accumulator block b = 2 s + h of S^T holds channel
// 32 s + 8 (rho / 4) + 4 h + rho % 4 in row rho, so that blocks 2 s and 2 s + 1 of a lane, side by side, are its column
// operand of step s.
//   row tile      4 KiB, the pieces in the order (s, lane): written and read 16 bytes per lane at consecutive addresses
//   turned tile   the same with token t ^ 4 g in the place of t: read through the transposing LDS read (tokens as
//                 contraction), which then touches every bank once
//   W             16 bytes per lane (i, g): W[i][4 g .. + 3] as fp16, hi then lo; against [X, X] one MFMA multiplies both
//   P             8 bytes per lane (i, g): P[i][4 g .. + 3] as fp16
// Products go to the 16x16x32 MFMA alone.  (An accumulator that v_mfma_f32_16x16x16_f16 had written and 16x16x32 read one or two
// instructions later was seen to lack the first product in half of its registers, depending on what else ran: the compiler
// puts no wait between the two.)
#pragma once

#include "prefill_common.h"

namespace pla {

constexpr int SUB = 16;                          // tokens of a sub-chunk

__device__ __forceinline__ bf16x8_t pair_of(uint2 a, uint2 b) { return __builtin_bit_cast(bf16x8_t, make_uint4(a.x, a.y, b.x, b.y)); }
__device__ __forceinline__ bf16x8_t lds_granule(const char* at) { return __builtin_bit_cast(bf16x8_t, *reinterpret_cast<const uint4*>(at)); }
__device__ __forceinline__ uint2 lds_turned(const char* at) { return read_tr4(reinterpret_cast<const uint16_t*>(at)); }

// Bytes from the start of a turned tile to what lane `lane` addresses for block (s = 0, h = 0); block (s, h): + 1024 s + 8 h.
// Lane i of a group of sixteen addresses columns 4 (i % 4) .. + 3 of row i / 4 (read_tr4).
__device__ __forceinline__ int turned_offset(int lane) {
  const int g = lane >> 4, row = 4 * g + ((lane >> 2) & 3), quad = lane & 3;
  return 16 * (16 * quad + (row ^ (4 * quad)));
}
// The place of lane (t, g)'s piece in a turned tile (step s: + 1024 s).
__device__ __forceinline__ int turned_piece(int lane) {
  const int t = lane & 15, g = lane >> 4;
  return 16 * (16 * g + (t ^ (4 * g)));
}

// Eight FP32 values as a bf16 pair each: round_bf16 is hi, to nearest, rest_bf16 is lo = bf16(x - hi) (v_dot2 forms x - hi in place:
// x is used up).
__device__ __forceinline__ bf16x8_t round_bf16(const float (&x)[8]) {
  return __builtin_bit_cast(bf16x8_t, make_uint4(pack2<bf16_t>(x[0], x[1]), pack2<bf16_t>(x[2], x[3]), pack2<bf16_t>(x[4], x[5]),
                                                 pack2<bf16_t>(x[6], x[7])));
}
__device__ __forceinline__ bf16x8_t rest_bf16(const float (&x)[8], bf16x8_t hi) {
  const uint4 h = __builtin_bit_cast(uint4, hi);
  // (-1, 0) and (0, -1), from registers: as an operand of this instruction the compiler writes 0x0000BF80 as the inline constant
  // -1.0, whose 32 bits are the other pair
  uint32_t LO, HI;
  asm("s_mov_b32 %0, 0xbf80" : "=s"(LO));
  asm("s_mov_b32 %0, 0xbf800000" : "=s"(HI));
  const float r[8] = {dot2<bf16_t>(h.x, LO, x[0]), dot2<bf16_t>(h.x, HI, x[1]), dot2<bf16_t>(h.y, LO, x[2]), dot2<bf16_t>(h.y, HI, x[3]),
                      dot2<bf16_t>(h.z, LO, x[4]), dot2<bf16_t>(h.z, HI, x[5]), dot2<bf16_t>(h.w, LO, x[6]), dot2<bf16_t>(h.w, HI, x[7])};
  return round_bf16(r);
}

// From here on this wavefront's conversions to fp16 round a finite value beyond the range to the largest finite fp16 (MODE bit
// 23, FP16_OVFL; infinities stay): to nearest with the saturation that otherwise only rounding toward zero gives.
__device__ __forceinline__ void fp16_saturates() { __builtin_amdgcn_s_setreg(1 | (23 << 6), 1); }

// Four FP32 values as an fp16 pair each: hi to nearest after a clamp (SATURATES: of a wavefront whose conversions do that, see
// fp16_saturates), the rest toward zero (as half8_pair).  x - hi is one v_fma_mix_f32, which takes a half of hi as it is, in the
// place of x (in registers of its own the mixed sweep spills eight more); the compiler forms a conversion and a subtraction.  Both
// halves of hi come from x, so that an MFMA that wrote x has been waited for.
struct QuadPair { uint2 hi, lo; };
template <bool SATURATES>
__device__ __forceinline__ QuadPair quad_pair(f32x4_t x) {
  QuadPair r;
  auto c = [](float v) { return SATURATES ? v : __builtin_amdgcn_fmed3f(v, -65504.f, 65504.f); };
  auto two = [&](float a, float b, uint32_t& hi, uint32_t& lo) {
    const f32x2_t v = {c(a), c(b)};
    hi = __builtin_bit_cast(uint32_t, __builtin_convertvector(v, f16x2_t));
    asm("v_fma_mix_f32 %0, %1, -1.0, %0 op_sel_hi:[1,0,0]" : "+v"(a) : "v"(hi));
    asm("v_fma_mix_f32 %0, %1, -1.0, %0 op_sel:[1,0,0] op_sel_hi:[1,0,0]" : "+v"(b) : "v"(hi));
    lo = pack2_rtz(a, b);
  };
  two(x[0], x[1], r.hi.x, r.lo.x);
  two(x[2], x[3], r.hi.y, r.lo.y);
  return r;
}

// Sum over the lanes from this one to the last of a DPP row (the tokens of a sub-chunk).
__device__ __forceinline__ float row16_suffix(float x) {
  x += dpp_mov<0x101>(x);     // row_shl:1, 2, 4, 8; lanes outside the row count as zero
  x += dpp_mov<0x102>(x);
  x += dpp_mov<0x104>(x);
  x += dpp_mov<0x108>(x);
  return x;
}
// The value of the next lane of the row, zero in its last lane.
__device__ __forceinline__ float row16_next(float x) { return dpp_mov<0x101>(x); }
// x[e] *= f[e] of the next lane of the row, unchanged in its last lane (a lane that a DPP operand leaves out is not written; the
// compiler would form the factor 1 of that lane first), or of the row's first lane (the compiler would move it first where it
// is used twice).  The s_nop covers the wait states behind the last write before the block.
#define PLA_MUL(X, F, FROM) "v_mul_f32_dpp " X ", " F ", " X " " FROM " row_mask:0xf bank_mask:0xf\n\t"
#define PLA_TIMES(FROM)                                                                                                   \
  asm("s_nop 1\n\t" PLA_MUL("%0", "%8", FROM) PLA_MUL("%1", "%9", FROM) PLA_MUL("%2", "%10", FROM)                        \
      PLA_MUL("%3", "%11", FROM) PLA_MUL("%4", "%12", FROM) PLA_MUL("%5", "%13", FROM) PLA_MUL("%6", "%14", FROM)         \
      PLA_MUL("%7", "%15", FROM)                                                                                          \
      : "+&v"(x[0]), "+&v"(x[1]), "+&v"(x[2]), "+&v"(x[3]), "+&v"(x[4]), "+&v"(x[5]), "+&v"(x[6]), "+&v"(x[7])            \
      : "v"(f[0]), "v"(f[1]), "v"(f[2]), "v"(f[3]), "v"(f[4]), "v"(f[5]), "v"(f[6]), "v"(f[7]))
__device__ __forceinline__ void times_next(float (&x)[8], const float (&f)[8]) { PLA_TIMES("row_shl:1"); }
__device__ __forceinline__ void times_first(float (&x)[8], const float (&f)[8]) { PLA_TIMES("row_newbcast:0"); }
#undef PLA_TIMES
#undef PLA_MUL
// Sum over the four lanes (t, 0 .. 3) of a token.
__device__ __forceinline__ float token_sum(float x) {
  const LanePair a = swap_rows16(x);
  const float y = a.lo + a.hi;
  const LanePair b = swap_halves(y);
  return b.lo + b.hi;
}

// Rows that a buffer access may reach: `rows` of them, `pitch` bytes apart, 256 bytes of each; reads beyond return zero, writes
// are dropped.
__device__ __forceinline__ __amdgpu_buffer_rsrc_t rows_resource(const void* base, int rows, uint32_t pitch) {
  const uint32_t bytes = rows > 0 ? (uint32_t)(min(rows, SUB) - 1) * pitch + 256u : 0u;
  return __builtin_amdgcn_make_buffer_rsrc(const_cast<void*>(base), 0, bytes, 0x00020000);
}

// Order of this wavefront's own LDS accesses on both sides (the LDS serves one wavefront in order; this keeps the compiler
// from moving them).
__device__ __forceinline__ void own_lds_order() {
  __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
  __builtin_amdgcn_wave_barrier();
  __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
}

// Lane `LANE` of the row, in every lane of it.
template <int LANE>
__device__ __forceinline__ float row16_lane(float x) { return dpp_mov<0x150 + LANE>(x); }   // row_newbcast

// W = (I + L)^-1 diag(beta) of one sub-chunk on one wavefront, from (I + L) W = diag(beta): lane (t, g) holds W[t][4 g .. + 3],
// and with row l known every lane subtracts L[t][l] W[l][.], row l being lane l's registers, a DPP operand: four instructions
// a step and no wait between them, as three others stand between a register's last write and its next use by DPP.
// (Row t of the inverse solved in every group of sixteen lanes, last column first, took 120 such instructions for these 60, a
// wait with every four, and 44 more for the factors beta and the choice of a group's columns: 18 ragged sequences of 12 heads
// 98.4 -> 95.5 us, 65 536 tokens of 32 heads 1795 -> 1757, eight sequences of 2048 tokens 236.5 -> 231.4.)
// `m`: lane (t, g) holds M[t][4 g + r], of which only j < t is read; L_ij = beta_i M_ij, `beta` the lane's token's.  `scratch`: 1
// KiB of LDS (W may replace it).
__device__ __forceinline__ void store_row(f32x4_t m, float beta, char* scratch, int lane) {
  const int t = lane & 15, g = lane >> 4;
  float4 x;                                        // row t of -L, zero from the diagonal on
  x.x = 4 * g < t ? -beta * m[0] : 0.f;
  x.y = 4 * g + 1 < t ? -beta * m[1] : 0.f;
  x.z = 4 * g + 2 < t ? -beta * m[2] : 0.f;
  x.w = 4 * g + 3 < t ? -beta * m[3] : 0.f;
  *reinterpret_cast<float4*>(scratch + 64 * t + 16 * g) = x;
}
// x[c] += row[l] * x[c] of lane l, for l = 0 .. 14.  One block: nothing may come between a write and its use by DPP.  (v_fmac_f32
// with a DPP operand is not formed by the compiler; the s_nop covers the wait states behind the last write before the block.)
#define PLA_STEP(ROW, LANE)                                                             \
  "v_fmac_f32_dpp %0, %0, " ROW " row_newbcast:" LANE " row_mask:0xf bank_mask:0xf\n\t" \
  "v_fmac_f32_dpp %1, %1, " ROW " row_newbcast:" LANE " row_mask:0xf bank_mask:0xf\n\t" \
  "v_fmac_f32_dpp %2, %2, " ROW " row_newbcast:" LANE " row_mask:0xf bank_mask:0xf\n\t" \
  "v_fmac_f32_dpp %3, %3, " ROW " row_newbcast:" LANE " row_mask:0xf bank_mask:0xf\n\t"
__device__ __forceinline__ void eliminate(const float (&row)[SUB], float (&x)[4]) {
  asm("s_nop 1\n\t" PLA_STEP("%4", "0") PLA_STEP("%5", "1") PLA_STEP("%6", "2") PLA_STEP("%7", "3") PLA_STEP("%8", "4")
      PLA_STEP("%9", "5") PLA_STEP("%10", "6") PLA_STEP("%11", "7") PLA_STEP("%12", "8") PLA_STEP("%13", "9")
      PLA_STEP("%14", "10") PLA_STEP("%15", "11") PLA_STEP("%16", "12") PLA_STEP("%17", "13") PLA_STEP("%18", "14")
      : "+&v"(x[0]), "+&v"(x[1]), "+&v"(x[2]), "+&v"(x[3])
      : "v"(row[0]), "v"(row[1]), "v"(row[2]), "v"(row[3]), "v"(row[4]), "v"(row[5]), "v"(row[6]), "v"(row[7]), "v"(row[8]),
        "v"(row[9]), "v"(row[10]), "v"(row[11]), "v"(row[12]), "v"(row[13]), "v"(row[14]));
}
#undef PLA_STEP
__device__ __forceinline__ void solve_and_store_w(float beta, const char* scratch, char* w_tile, int lane) {
  const int t = lane & 15, g = lane >> 4;
  float row[SUB], x[4];
#pragma unroll
  for (int q = 0; q < 4; ++q) {
    const float4 c = *reinterpret_cast<const float4*>(scratch + 64 * t + 16 * q);
    row[4 * q] = c.x; row[4 * q + 1] = c.y; row[4 * q + 2] = c.z; row[4 * q + 3] = c.w;
  }
#pragma unroll
  for (int r = 0; r < 4; ++r) x[r] = t == 4 * g + r ? beta : 0.f;
  eliminate(row, x);
  own_lds_order();
  const QuadPair pair = quad_pair<false>(f32x4_t{x[0], x[1], x[2], x[3]});
  *reinterpret_cast<uint4*>(w_tile + 16 * lane) = make_uint4(pair.hi.x, pair.hi.y, pair.lo.x, pair.lo.y);
}

// The ring of sub-chunks between producing and computing wavefronts.  Sub-chunk i lives in slot i % RING; full[slot] counts
// its productions, done[slot] the computing wavefronts that have finished with it.  A wavefront's LDS operations happen in
// order, so a count raised after the accesses it stands for needs no more than the compiler to keep the order.
constexpr int RING = 8;
struct RingFlags { uint32_t full[RING], done[RING]; };
typedef __attribute__((address_space(3))) uint32_t lds_word_t;
// (Through an LDS pointer: a generic one would be read as memory, behind every load and store in flight.)
__device__ __forceinline__ uint32_t read_count(const uint32_t* count) {
  return __hip_atomic_load((lds_word_t*)const_cast<uint32_t*>(count), __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
}
__device__ __forceinline__ bool count_reached(uint32_t now, uint32_t target) {
  return (int32_t)(__builtin_amdgcn_readfirstlane(now) - target) >= 0;
}
__device__ __forceinline__ void ring_reset(RingFlags* f) {      // by the whole workgroup, before any of it uses the ring
  if (threadIdx.x < 2 * RING) reinterpret_cast<uint32_t*>(f)[threadIdx.x] = 0u;
  __syncthreads();
}
__device__ __forceinline__ void wait_count(const uint32_t* count, uint32_t target) {
  while (!count_reached(read_count(count), target)) __builtin_amdgcn_s_sleep(1);
  asm volatile("" ::: "memory");
}
__device__ __forceinline__ void slot_filled(RingFlags* f, int i, int lane) {
  asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
  if (lane == 0)
    __hip_atomic_store((lds_word_t*)&f->full[i % RING], (uint32_t)(i / RING) + 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
  asm volatile("" ::: "memory");
}
__device__ __forceinline__ void slot_done(RingFlags* f, int i, int lane) {
  asm volatile("" ::: "memory");
  if (lane == 0) __hip_atomic_fetch_add((lds_word_t*)&f->done[i % RING], 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
  asm volatile("" ::: "memory");
}

// Tokens and states of one chain: a (sequence, head), or a (segment, head) of a call whose sequences are split.
struct Chain {
  int64_t token;          // first token
  int tokens, head;       // tokens (0: nothing to do)
  int64_t slot;           // number of its first sub-chunk among prepared ones
  const float* init;      // [V, K] tile the state starts from (nullptr: zero)
  float* fin;             // [V, K] tile that receives the state at the end (nullptr: none)
  bool identity;          // the state starts from the identity and v is zero: the segment's transition matrix
};
// Sub-chunk i of sequence n is number first_slot + i among the prepared ones of a call: sequences do not overlap in it, whatever
// their lengths, and no table is needed.
__device__ __forceinline__ int64_t first_slot(int n, int token) { return token / SUB + n; }
// Segment `i` of those that a sweep over the segments of a split call runs (swept_segment).  sequence < 0: it runs fewer.
struct Segment { int sequence, index, count, number, token, tokens; int64_t slot; };
__device__ __forceinline__ Segment inline_segment(const int32_t* cu_seqlens, int N, int T, const SegmentTable& t, int split_from, bool second, int i, int lane) {
  const SegmentCounts c = count_segments(cu_seqlens, N, T, t.seg_chunks, split_from, lane);
  const SweptSegment s = swept_segment(swept_segments(c.count, second), c.count, second, i);
  Segment r{-1, 0, 0, 0, 0, 0, 0};
  if (s.sequence < 0 || s.number >= t.max_segments) return r;      // (number: offsets that do not fit the workspace)
  r.sequence = s.sequence;
  r.index = s.index;
  r.count = s.count;
  r.number = s.number;
  const int skipped = r.index * c.chunks * CHUNK;
  r.token = __builtin_amdgcn_readlane(c.tokens.x, r.sequence) + skipped;
  r.slot = first_slot(r.sequence, r.token - skipped) + skipped / SUB;
  r.tokens = min(c.chunks * CHUNK, __builtin_amdgcn_readlane(c.tokens.y, r.sequence) - skipped);
  return r;
}

}  // namespace pla
