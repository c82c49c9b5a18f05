// Gated delta-rule prefill for KDA (per-channel gate) on gfx950: one pass over the tokens in sub-chunks of 16.
//
// Per sub-chunk, with G_i[c] the inclusive cumulative log-decay of channel c inside it (g <= 0, so G decreases along
// the tokens) and S the FP32 k-last state:
//     M_ij = sum_c k_i[c] k_j[c] e^{G_i[c] - G_j[c]}   (i > j)      L = I + diag(beta) M
//     P_ij = sum_c q_i[c] k_j[c] e^{G_i[c] - G_j[c]}   (i >= j)
//     W    = L^-1 diag(beta)
//     X    = V - (K (.) e^{G}) S^T            U = W X
//     O    = scale ((Q (.) e^{G}) S^T + P U)
//     S^T  = e^{G_last} (.) S^T + (K (.) e^{G_last - G})^T U
// (reference pipeline: src/prefill/flashkdapro/tc01/fla/runtime.cc:474-545 - gate, token, inter,
// recompute, recurrence, output; public contract pla/prefill/flashkdapro/ops.py:68-219).
//
// One workgroup per (sequence, head).  Four wavefronts carry the state (32 V columns each) through the sub-chunks; four
// others, one per SIMD beside them, form the operands of the next sub-chunks in LDS from the raw rows, each every fourth one.
// A ring of eight slots with counters stands between them (subchunk.h); there is no barrier in the loop.
// Nothing but the tokens, the outputs and the states crosses memory, and a call of many chains is one launch.  What bounds it is
// issue: a sub-chunk costs a SIMD about 300 vector instructions of its producing wavefront (a quarter of a sub-chunk) and 210
// of its computing one, with 59 MFMAs that overlap little of it (with 245: 3600 cycles, of which each of the two sides alone took 2440; the
// 35 were clamps that the saturating conversions repeat and the subtractions of quad_pair: 18 ragged sequences of 12 heads 102.3 ->
// 99.3 us, 65 536 tokens of 32 heads 1737 -> 1684).  Eight
// producing wavefronts instead of four gain nothing (168 registers: the computing ones spill), nor do eight computing ones of 16
// columns (246 against 228 us, eight sequences of 2048 tokens, 32 heads: twice the LDS reads).  Sixteen tokens decay
// by at most 16 x |lower_bound| <= 80, so a factor and its inverse are FP32 numbers and M and P one product each; a longer chunk needs
// a reference row, and its exponentials again, for every block of 16 x 16.
//
// The decay is summed from the sub-chunk's end: R_j = G_last - G_j is what the tokens behind j decay.  e^{R_j} is the factor of the
// state's update, the factors of M and P are k e^{R_j} against k e^{-R_i} and q e^{-R_i}, and e^{G_i} = e^{G_last} e^{-R_i} goes to
// operands that fp16 rounds anyway.  Summed from the front, e^{G_last - G_j} has the roundings of sums of up to 115 (base 2) also
// where it stands for one token: final states of 15 tokens under a strong gate 1.6e-6 to 3.2e-6 from 64 bits, now 2.9e-7 to 5.5e-7;
// the time is the same (18 ragged sequences 102.1 / 101.5 us, 65 536 tokens 1778 / 1769).  M takes both factors as bf16 hi + lo pairs, P its key
// factor: with that rounded once too the output is 1.14 x as far from 64 bits (44 calls), for the same time.
//
// The operands of the products with the state (k e^{G}, q e^{G}, k e^{G_last - G}, W, P, S, X, U) go to the MFMA as fp16,
// rounded once or (W, k e^{G_last - G}, X, U) as hi + lo pairs: the pairs keep keys that repeat within a few tokens
// inside the state's bound of 1e-3 (a single rounding of k e^{G_last - G} leaves 1.7e-3), and that of X takes the state's error
// against 64 bits from 2.5e-4 to 1.1e-4 (ragged prompts of 121 to 999 tokens) for 1-2 % of the time.  One product takes [hi, lo]
// against [U, U], sixteen tokens of each filling its contraction of 32.
//
// (A chunk of 64 tokens with its operands prepared in memory, 82 KB written and 76 and 98 KB read back per chunk and head, took 160
// us for 18 ragged sequences of 12 heads and 2160 us for 65 536 tokens of 32 heads; this form takes 99 and 1690.  Chains with a CU
// to themselves are where the longer chunk was the faster: 2.0-2.2 us for its 64 tokens against 2.45-2.7 for four dependent steps here,
// which one sequence of 700 to 1000 tokens of 8 to 16 heads still shows, 870 of 16 heads 51.5 and 53.0.)
//
// Kernels:
//   kda_prepare_kernel      calls of at most 128 chains: the operands of all sub-chunks, formed on every CU ahead of the sweep
//   kda_sweep_kernel        a whole sequence, or a segment in the second sweep; NB = 1: two workgroups per chain, 64 V
//                           columns each (calls of at most 128 chains)
//   kda_sweep_mixed_kernel  ragged whole sequences: the chains of the longest sequences as two halves, the others whole, in one
//                           launch (plan from the host offsets)
//   kda_first_sweep_kernel  first sweep over segments: first segments with output, of every other but the last one the zero-state
//                           sweep and the transition-matrix sweep in one workgroup that forms the operands once for both

#include "subchunk.h"

namespace pla {

struct KdaPrefillParams {
  const void* q; const void* k; const void* v; const void* g; const void* beta;   // bf16
  int64_t stride_q, stride_k, stride_v, stride_g, stride_beta;                    // token pitches (elements)
  const float* A_log; const float* dt_bias;                                       // [H], [H*128]
  float lower_bound, scale;
  const int32_t* cu_seqlens; int N; int T;
  const float* h0; const int32_t* h0_indices; int64_t h0_slot_stride;
  float* ht; const int32_t* ht_indices; int64_t ht_slot_stride;
  void* o;
  char* prepared;                                  // sub-chunks prepared by kda_prepare_kernel (null: the sweeps form them)
  SegmentTable seg;                                // split long sequences (seg.seg_chunks > 0)
  int pass;                                        // 0: whole sequences; 1, 2: the two sweeps over segments
  int split_from;                                  // chunks of the longest sequence from which on any is split
  int H;
  int empty_states;                                // also write the final states of empty sequences
  // kda_sweep_mixed_kernel: the first `split_grid` workgroups sweep the chains of sequences seq_order[0 .. n_long) as
  // two halves, the others those of seq_order[n_long .. N) whole
  unsigned split_grid; int n_long;
  unsigned char seq_order[INLINE_TABLE_SEQUENCES];
};

constexpr float LOG2E = 1.4426950408889634f;

// A sub-chunk's operands (bytes), in LDS or in the workspace: the row tile k e^{G}, the turned tiles of k e^{G_last - G} (hi, lo),
// W, e^{G_last}; with output P and the row tile q e^{G}.  A sweep without output takes the first 13.5 KiB.
struct KdaSlot {
  static constexpr int K = 0, TH = 4096, TL = 8192, W = 12288, F = 13312, P = 13824, Q = 14336, BYTES = 18432;
};
template <bool OUT>
constexpr int KDA_SLOT_BYTES = OUT ? KdaSlot::BYTES : KdaSlot::P;
template <bool OUT>
struct KdaLds {
  __align__(16) char slots[RING * KDA_SLOT_BYTES<OUT>];         // 147 KiB with output, 111 KiB without
  float bias[128];          // -e^{A_log} log2 e dt_bias
  RingFlags flags;
};

// The raw rows of a lane: token t = lane % 16 of a sub-chunk, channels 32 s + 8 g .. + 7.
template <bool OUT>
struct KdaRows {
  const uint16_t *kp, *gp, *qp, *bp;
  uint4 k[4], g[4], q[4];
  uint16_t beta;
  // sub-chunk i of the chain (rows past the sequence re-read its last row)
  __device__ __forceinline__ void seek(const KdaPrefillParams& p, const Chain& chain, int i, int lane) {
    const int64_t row = chain.token + min(SUB * i + (lane & 15), chain.tokens - 1), col = (int64_t)chain.head * 128 + 8 * (lane >> 4);
    kp = reinterpret_cast<const uint16_t*>(p.k) + row * p.stride_k + col;
    gp = reinterpret_cast<const uint16_t*>(p.g) + row * p.stride_g + col;
    if constexpr (OUT) qp = reinterpret_cast<const uint16_t*>(p.q) + row * p.stride_q + col;
    bp = reinterpret_cast<const uint16_t*>(p.beta) + row * p.stride_beta + chain.head;
  }
  __device__ __forceinline__ void advance(const KdaPrefillParams& p, const Chain& chain, int i, int step, int lane) {      // from i - step to i
    if (SUB * (i + 1) > chain.tokens) { seek(p, chain, i, lane); return; }
    kp += step * SUB * p.stride_k;
    gp += step * SUB * p.stride_g;
    if constexpr (OUT) qp += step * SUB * p.stride_q;
    bp += step * SUB * p.stride_beta;
  }
  __device__ __forceinline__ void load() {
#pragma unroll
    for (int s = 0; s < 4; ++s) g[s] = *reinterpret_cast<const uint4*>(gp + 32 * s);
#pragma unroll
    for (int s = 0; s < 4; ++s) k[s] = *reinterpret_cast<const uint4*>(kp + 32 * s);
    beta = *bp;
    if constexpr (OUT) {
#pragma unroll
      for (int s = 0; s < 4; ++s) q[s] = *reinterpret_cast<const uint4*>(qp + 32 * s);
    }
  }
};
// A head's gate: bound / (1 + 2^{slope (g + dt_bias)}) in base 2, as 1 / fma(2^., 1 / bound, 1 / bound).  `bias`: slope dt_bias,
// 128 values in LDS (there they cost no registers); every wavefront that uses them writes them all and reads its own.
struct KdaGate {
  float slope, inv_bound;
  const float* bias;
  __device__ __forceinline__ KdaGate(const KdaPrefillParams& p, int head, float* lds_bias, int lane) : bias(lds_bias) {
    const float bound = p.lower_bound * LOG2E;
    slope = -expf(p.A_log[head]) * LOG2E;
    inv_bound = bound < -1e-30f ? 1.f / bound : -1e30f;       // (nearer to zero it decays nothing; 0 x 1 / bound has to stay a number)
#pragma unroll
    for (int i = 0; i < 2; ++i) lds_bias[lane + 64 * i] = slope * p.dt_bias[head * 128 + lane + 64 * i];
    own_lds_order();
  }
};

// One sub-chunk on one wavefront, from its raw rows to `slot` (LDS or workspace); `scratch`: 1 KiB of LDS.  `loaded` runs when the
// raw rows have been used.  What bounds it are its vector instructions, about 1200 with 128 exponentials and reciprocals
// among them, so it counts those: eight channels at a time go through gate, sum over the tokens, norm and decay to
// their places; the sum over the tokens, the broadcast of the last one and the rows of the triangular solve are DPP operands,
// the gate's bound is folded into the reciprocal of its sigmoid.  M takes its operands as bf16 pairs (e^{-G} leaves the range
// of fp16), P its key factor as such a pair: the FP32 MFMA would take them as they are, but no vector instruction of the SIMD
// runs beside it (64 of them a sub-chunk: 130 sequences-and-heads of 2048 tokens 224 -> 198 us without).
template <bool OUT, typename Loaded>
__device__ __forceinline__ void kda_sub_chunk(const KdaGate& gate, KdaRows<OUT>& rows, bool valid, char* slot, char* scratch, int lane,
                                              Loaded loaded) {
  using Slot = KdaSlot;
  const int t = lane & 15, g = lane >> 4;
  auto element = [](const uint4& w, int e) {
    const uint32_t x = e < 2 ? w.x : e < 4 ? w.y : e < 6 ? w.z : w.w;
    return (e & 1) ? hi16<bf16_t>(x) : lo16<bf16_t>(x);
  };
  // 1 / |row|, and eight channels of a row over its norm, rounded to bf16 (the reference's operand)
  auto inverse_norm = [](const uint4 (&w)[4]) {
    float a = 0.f, b = 0.f;
#pragma unroll
    for (int s = 0; s < 4; ++s) {
      a = dot2<bf16_t>(w[s].x, w[s].x, a);
      b = dot2<bf16_t>(w[s].y, w[s].y, b);
      a = dot2<bf16_t>(w[s].z, w[s].z, a);
      b = dot2<bf16_t>(w[s].w, w[s].w, b);
    }
    return fast_rsqrt(token_sum(a + b) + 1e-6f);
  };
  auto normalised = [&](const uint4& w, float inv, float (&x)[8]) {
#pragma unroll
    for (int e = 0; e < 8; e += 2) {
      const uint32_t w2 = pack2<bf16_t>(element(w, e) * inv, element(w, e + 1) * inv);
      x[e] = lo16<bf16_t>(w2);
      x[e + 1] = hi16<bf16_t>(w2);
    }
  };
  auto half_piece = [](const float (&x)[8]) {
    return make_uint4(pack2<f16_t>(x[0], x[1]), pack2<f16_t>(x[2], x[3]), pack2<f16_t>(x[4], x[5]), pack2<f16_t>(x[6], x[7]));
  };
  // rows past the sequence: no decay, beta = 0.  (The whole division and expf: v_exp_f32 of the scaled logit and v_rcp_f32 are 3e-7
  // from the sigmoid above -4 and 9e-7 at -12, and a token's write is proportional to it.)
  const float beta = valid ? 1.f / (1.f + expf(-to_float(bf16_t{rows.beta}))) : 0.f, ib = valid ? gate.inv_bound : 1e30f;
  const float k_inv = inverse_norm(rows.k);
  float q_inv = 0.f;
  if constexpr (OUT) q_inv = inverse_norm(rows.q);
  f32x4_t m = {0.f, 0.f, 0.f, 0.f}, pq = {0.f, 0.f, 0.f, 0.f};    // m[r] = M[t][4 g + r], pq[r] = P[t][4 g + r]
  float first[4][8];
#pragma unroll
  for (int s = 0; s < 4; ++s) {                   // eight channels at a time
    float (&ex)[8] = first[s];                    // e^{R} of the token before: e^{G_last} in the first token's lanes
    float kd[8], ku[8], up[8];                    // k e^{R}, k e^{-R}, e^{-R}
#pragma unroll
    for (int e = 0; e < 8; ++e) {
      const float w = __builtin_amdgcn_exp2f(fmaf(element(rows.g[s], e), gate.slope, gate.bias[32 * s + 8 * g + e]));
      ex[e] = row16_suffix(fast_rcp(fmaf(w, ib, ib)));
    }
    normalised(rows.k[s], k_inv, kd);
#pragma unroll
    for (int e = 0; e < 8; ++e) {
      up[e] = __builtin_amdgcn_exp2f(-row16_next(ex[e]));
      ex[e] = __builtin_amdgcn_exp2f(ex[e]);
      ku[e] = kd[e] * up[e];
    }
    times_next(kd, ex);
    // k e^{G} = e^{G_last} k e^{-R}
    float x[8];
#pragma unroll
    for (int e = 0; e < 8; ++e) x[e] = row16_lane<0>(ex[e]) * ku[e];
    *reinterpret_cast<uint4*>(slot + Slot::K + 1024 * s + 16 * lane) = half_piece(x);
    uint32_t hi[4], lo[4];
#pragma unroll
    for (int e = 0; e < 8; e += 2) pack2_pair_small(kd[e], kd[e + 1], hi[e / 2], lo[e / 2]);
    const int at = 1024 * s + turned_piece(lane);
    *reinterpret_cast<uint4*>(slot + Slot::TH + at) = make_uint4(hi[0], hi[1], hi[2], hi[3]);
    *reinterpret_cast<uint4*>(slot + Slot::TL + at) = make_uint4(lo[0], lo[1], lo[2], lo[3]);
    const bf16x8_t ku_hi = round_bf16(ku), kd_hi = round_bf16(kd);
    m = mfma16(kd_hi, rest_bf16(ku, ku_hi), m);
    const bf16x8_t kd_lo = rest_bf16(kd, kd_hi);
    m = mfma16(kd_lo, ku_hi, m);
    m = mfma16(kd_hi, ku_hi, m);
    if constexpr (OUT) {
      float qu[8];                                // q e^{-R}
      normalised(rows.q[s], q_inv, qu);
#pragma unroll
      for (int e = 0; e < 8; ++e) qu[e] *= up[e];
      const bf16x8_t qu_hi = round_bf16(qu);
      pq = mfma16(kd_lo, qu_hi, pq);
      pq = mfma16(kd_hi, qu_hi, pq);
      times_first(qu, ex);
      *reinterpret_cast<uint4*>(slot + Slot::Q + 1024 * s + 16 * lane) = half_piece(qu);
    }
  }
  store_row(m, beta, scratch, lane);
  own_lds_order();
  if (t == 0) {
#pragma unroll
    for (int s = 0; s < 4; ++s) {
      float* const f = reinterpret_cast<float*>(slot + Slot::F) + 32 * s + 8 * g;
      *reinterpret_cast<float4*>(f) = make_float4(first[s][0], first[s][1], first[s][2], first[s][3]);
      *reinterpret_cast<float4*>(f + 4) = make_float4(first[s][4], first[s][5], first[s][6], first[s][7]);
    }
  }
  loaded();
  if constexpr (OUT) {
#pragma unroll
    for (int r = 0; r < 4; ++r) pq[r] = 4 * g + r <= t ? pq[r] : 0.f;
    *reinterpret_cast<uint2*>(slot + Slot::P + 8 * lane) = make_uint2(pack2<f16_t>(pq[0], pq[1]), pack2<f16_t>(pq[2], pq[3]));
  }
  solve_and_store_w(beta, scratch, slot + Slot::W, lane);
}

// A producing wavefront: every PRODUCERS-th sub-chunk of the chain, from `pw`, into the ring.
template <bool OUT, int PRODUCERS>
__device__ __forceinline__ void kda_produce(const KdaPrefillParams& p, KdaLds<OUT>& lds, const Chain& chain, int lane, int pw,
                                            uint32_t readers) {
  const int subs = (chain.tokens + SUB - 1) / SUB;
  KdaRows<OUT> rows;
  if (pw < subs) {
    rows.seek(p, chain, pw, lane);
    rows.load();
  }
  const KdaGate gate(p, chain.head, lds.bias, lane);
  for (int i = pw; i < subs; i += PRODUCERS) {
    wait_count(&lds.flags.done[i % RING], readers * (uint32_t)(i / RING));
    char* const slot = lds.slots + (i % RING) * KDA_SLOT_BYTES<OUT>;
    kda_sub_chunk<OUT>(gate, rows, SUB * i + (lane & 15) < chain.tokens, slot, slot + KdaSlot::W, lane, [&]() {
      if (i + PRODUCERS < subs) {
        rows.advance(p, chain, i + PRODUCERS, PRODUCERS, lane);
        rows.load();
      }
    });
    slot_filled(&lds.flags, i, lane);
  }
}

// The same from prepared sub-chunks: every COPIERS-th slot of the workspace goes to the ring as it lies, asynchronously, two
// in flight per wavefront.
template <bool OUT, int COPIERS>
__device__ __forceinline__ void kda_copy(const KdaPrefillParams& p, KdaLds<OUT>& lds, const Chain& chain, int lane, int cw, uint32_t readers) {
  constexpr int PIECES = KDA_SLOT_BYTES<OUT> / 1024, REST = KDA_SLOT_BYTES<OUT> % 1024, COPIES = PIECES + (REST ? 1 : 0);
  const int subs = (chain.tokens + SUB - 1) / SUB;
  const char* const first = uniform_pointer(p.prepared + (chain.slot * p.H + chain.head) * KdaSlot::BYTES);
  const int64_t pitch = (int64_t)p.H * KdaSlot::BYTES;
  for (int i = cw; i < subs; i += COPIERS) {
    wait_count(&lds.flags.done[i % RING], readers * (uint32_t)(i / RING));
    const char* const from = first + i * pitch;
    const uint32_t to = lds_address(lds.slots) + (i % RING) * KDA_SLOT_BYTES<OUT>;
#pragma unroll
    for (int j = 0; j < PIECES; ++j) dma16(from, 1024u * j + 16u * lane, to + 1024u * j);
    if (REST && lane < REST / 16) dma16(from, 1024u * PIECES + 16u * lane, to + 1024u * PIECES);
    if (i >= COPIERS) {
      wait_vmcnt<COPIES>();
      slot_filled(&lds.flags, i - COPIERS, lane);
    }
  }
  if (cw < subs) {
    wait_vmcnt<0>();
    slot_filled(&lds.flags, (subs - 1 - cw) / COPIERS * COPIERS + cw, lane);
  }
}

// Prepares sub-chunks in the workspace: one wavefront per (sub-chunk, head), heads fastest.
constexpr int PREPARE_WAVES = 4;
__global__ __launch_bounds__(64 * PREPARE_WAVES) void kda_prepare_kernel(const KdaPrefillParams p) {
  __shared__ __align__(16) char scratch[PREPARE_WAVES][1024];
  __shared__ float bias[PREPARE_WAVES][128];
  const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int64_t index = (int64_t)blockIdx.x * PREPARE_WAVES + wave, number = index / p.H;
  Chain chain{};
  chain.head = (int)(index - number * p.H);
  int i = -1;
  for (int base = 0; base < p.N; base += 64) {
    const int n = base + lane;
    const int2 range = n < p.N ? sequence_tokens(p.cu_seqlens, n, p.T) : make_int2(0, 0);
    const int64_t at = number - first_slot(n, range.x);
    const unsigned long long owner = __ballot(at >= 0 && SUB * at < range.y);
    if (owner != 0) {
      const int l = __builtin_amdgcn_readfirstlane(__ffsll((long long)owner) - 1);
      chain.token = __builtin_amdgcn_readlane(range.x, l);
      chain.tokens = __builtin_amdgcn_readlane(range.y, l);
      i = __builtin_amdgcn_readlane((int)at, l);
    }
  }
  if (i < 0) return;
  KdaRows<true> rows;
  rows.seek(p, chain, i, lane);
  rows.load();
  const KdaGate gate(p, chain.head, bias[wave], lane);
  kda_sub_chunk<true>(gate, rows, SUB * i + (lane & 15) < chain.tokens, p.prepared + index * KdaSlot::BYTES, scratch[wave], lane, []() {});
}

// A computing wavefront: 16 NB columns of V from `col0`, the lane's NB adjacent ones at col0 + NB (lane % 16).  St[nb] is S^T
// in accumulator blocks (subchunk.h); OT[nb][r] the output of token 4 g + r.
template <int NB, bool OUT>
__device__ __forceinline__ void kda_compute(const KdaPrefillParams& p, KdaLds<OUT>& lds, const Chain& chain, int lane, int col0) {
  using Slot = KdaSlot;
  const int n = lane & 15, g = lane >> 4, vcol = col0 + NB * n;
  fp16_saturates();
  const int subs = (chain.tokens + SUB - 1) / SUB;
  f32x4_t St[NB][8];
#pragma unroll
  for (int nb = 0; nb < NB; ++nb)
#pragma unroll
    for (int b = 0; b < 8; ++b) {
      const int c = 32 * (b >> 1) + 8 * g + 4 * (b & 1);        // the block's first channel in this lane
      if (chain.identity) {
        St[nb][b] = f32x4_t{c == vcol + nb ? 1.f : 0.f, c + 1 == vcol + nb ? 1.f : 0.f, c + 2 == vcol + nb ? 1.f : 0.f,
                            c + 3 == vcol + nb ? 1.f : 0.f};
      } else if (chain.init != nullptr) {
        const float4 x = *reinterpret_cast<const float4*>(chain.init + (int64_t)(vcol + nb) * 128 + c);
        St[nb][b] = f32x4_t{x.x, x.y, x.z, x.w};
      } else {
        St[nb][b] = f32x4_t{0.f, 0.f, 0.f, 0.f};
      }
    }
  auto store_state = [&](float* tile) {
#pragma unroll
    for (int nb = 0; nb < NB; ++nb)
#pragma unroll
      for (int b = 0; b < 8; ++b)
        *reinterpret_cast<float4*>(tile + (int64_t)(vcol + nb) * 128 + 32 * (b >> 1) + 8 * g + 4 * (b & 1)) =
            make_float4(St[nb][b][0], St[nb][b][1], St[nb][b][2], St[nb][b][3]);
  };

  // V: NB adjacent values of rows 4 g + r of a sub-chunk, requested AHEAD sub-chunks ahead; o likewise.  Both through buffers that
  // end with the chain (rows beyond read as zero and are not written), so that a step has no branch for them.
  const uint32_t v_pitch = (uint32_t)(p.stride_v * 2), o_pitch = (uint32_t)p.H * 256u;
  const char* const v_rows = reinterpret_cast<const char*>(p.v) + (chain.token * p.stride_v + (int64_t)chain.head * 128) * 2;
  char* const o_rows = reinterpret_cast<char*>(p.o) + (chain.token * p.H + chain.head) * 256;
  uint32_t v_at = (uint32_t)(4 * g) * v_pitch + 2u * vcol, o_at = (uint32_t)(4 * g) * o_pitch + 2u * vcol;
  const int tokens_v = chain.identity ? 0 : chain.tokens;
  constexpr int AHEAD = 2;
  uint32_t vraw[AHEAD][4];
  auto load_v = [&](int first, uint32_t (&w)[4]) {             // the sub-chunk that starts at token `first` of the chain
    const auto rows = rows_resource(v_rows + (int64_t)first * v_pitch, tokens_v - first, v_pitch);
    asm volatile("" : "+v"(v_at));                 // (the four offsets are formed here, not kept in registers)
#pragma unroll
    for (int r = 0; r < 4; ++r) {
      if constexpr (NB == 2) w[r] = __builtin_amdgcn_raw_buffer_load_b32(rows, v_at + r * v_pitch, 0, 0);
      else w[r] = __builtin_amdgcn_raw_buffer_load_b16(rows, v_at + r * v_pitch, 0, 0);
    }
  };
  // the row operands of a sub-chunk, requested before the step before it ends
  bf16x8_t ka[4], qa[OUT ? 4 : 1];
  auto load_rows = [&](int i) {
    const char* const slot = lds.slots + (i % RING) * KDA_SLOT_BYTES<OUT> + 16 * lane;
#pragma unroll
    for (int s = 0; s < 4; ++s) {
      ka[s] = lds_granule(slot + Slot::K + 1024 * s);
      if (OUT && s < 2) qa[s] = lds_granule(slot + Slot::Q + 1024 * s);
    }
  };
  struct Turned { bf16x8_t t[2]; float4 f[2]; };               // blocks 2 s, 2 s + 1: [k e^{G_last - G} hi, lo] by channels, e^{G_last}
  const int turned = turned_offset(lane);
  auto load_turned = [&](const char* slot, int s) {
    Turned r;
#pragma unroll
    for (int h = 0; h < 2; ++h) {
      r.t[h] = pair_of(lds_turned(slot + Slot::TH + turned + 1024 * s + 8 * h), lds_turned(slot + Slot::TL + turned + 1024 * s + 8 * h));
      r.f[h] = *reinterpret_cast<const float4*>(slot + Slot::F + 32 * g + 128 * s + 16 * h);
    }
    return r;
  };
  const f32x4_t zero = {0.f, 0.f, 0.f, 0.f};
  // LDS requests stay on their side of a fence, arithmetic may cross it
  auto lds_fence = []() { __builtin_amdgcn_sched_barrier(0x000F); };
  auto step = [&](int i, uint32_t (&vraw)[4]) {
    const char* const slot = lds.slots + (i % RING) * KDA_SLOT_BYTES<OUT>;
    const int first = SUB * i;
    f32x4_t KS[NB], OT[NB];
    if constexpr (OUT) {                           // (all four of q ahead: 2-5 % slower)
#pragma unroll
      for (int s = 2; s < 4; ++s) qa[s] = lds_granule(slot + Slot::Q + 1024 * s + 16 * lane);
    }
    const bf16x8_t w = lds_granule(slot + Slot::W + 16 * lane);
    const uint32_t next_full = read_count(&lds.flags.full[(i + 1) % RING]);
    lds_fence();
#pragma unroll
    for (int nb = 0; nb < NB; ++nb) KS[nb] = OT[nb] = zero;
#pragma unroll
    for (int s = 0; s < 4; ++s)
#pragma unroll
      for (int nb = 0; nb < NB; ++nb) {
        const bf16x8_t sb = half8(St[nb][2 * s], St[nb][2 * s + 1]);        // (saturating: fp16_saturates)
        KS[nb] = mfma16h(ka[s], sb, KS[nb]);
        if constexpr (OUT) OT[nb] = mfma16h(qa[s], sb, OT[nb]);
      }
    Turned b0 = load_turned(slot, 0);
    Turned b1 = load_turned(slot, 1);
    lds_fence();
    bf16x8_t uh[NB], ul[NB];
    QuadPair u[NB];
#pragma unroll
    for (int nb = 0; nb < NB; ++nb) {
      f32x4_t x;
#pragma unroll
      for (int r = 0; r < 4; ++r) x[r] = (nb == 0 ? lo16<bf16_t>(vraw[r]) : hi16<bf16_t>(vraw[r])) - KS[nb][r];
      const QuadPair xp = quad_pair<true>(x);
      u[nb] = quad_pair<true>(mfma16h(w, pair_of(xp.hi, xp.hi), mfma16h(w, pair_of(xp.lo, xp.lo), zero)));
      uh[nb] = pair_of(u[nb].hi, u[nb].hi);
      ul[nb] = pair_of(u[nb].lo, u[nb].lo);
    }
    load_v(first + AHEAD * SUB, vraw);
    auto update = [&](const Turned& k, int s) {                // the small term first
#pragma unroll
      for (int h = 0; h < 2; ++h)
#pragma unroll
        for (int nb = 0; nb < NB; ++nb) {
          f32x4_t& st = St[nb][2 * s + h];
          st = f32x4_t{st[0] * k.f[h].x, st[1] * k.f[h].y, st[2] * k.f[h].z, st[3] * k.f[h].w};
          st = mfma16h(k.t[h], ul[nb], st);
        }
#pragma unroll
      for (int h = 0; h < 2; ++h)
#pragma unroll
        for (int nb = 0; nb < NB; ++nb) St[nb][2 * s + h] = mfma16h(k.t[h], uh[nb], St[nb][2 * s + h]);
    };
    if constexpr (OUT) {
      const uint2 pp = *reinterpret_cast<const uint2*>(slot + Slot::P + 8 * lane);
#pragma unroll
      for (int nb = 0; nb < NB; ++nb) OT[nb] = mfma16h(pair_of(pp, pp), pair_of(u[nb].hi, u[nb].lo), OT[nb]);
    }
    update(b0, 0);
    b0 = load_turned(slot, 2);
    lds_fence();
    update(b1, 1);
    b1 = load_turned(slot, 3);
    slot_done(&lds.flags, i, lane);                // (every read of the slot has been issued)
    lds_fence();
    update(b0, 2);
    if (i + 1 < subs) {
      if (!count_reached(next_full, (uint32_t)((i + 1) / RING) + 1u))
        wait_count(&lds.flags.full[(i + 1) % RING], (uint32_t)((i + 1) / RING) + 1u);
      asm volatile("" ::: "memory");
      load_rows(i + 1);
      lds_fence();
    }
    update(b1, 3);
    if constexpr (OUT) {
      const auto rows = rows_resource(o_rows + (int64_t)first * o_pitch, chain.tokens - first, o_pitch);
      asm volatile("" : "+v"(o_at));                 // (formed here as well)
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        if constexpr (NB == 2)
          __builtin_amdgcn_raw_buffer_store_b32(pack2<bf16_t>(p.scale * OT[0][r], p.scale * OT[1][r]), rows, o_at + r * o_pitch, 0, 0);
        else
          __builtin_amdgcn_raw_buffer_store_b16((short)from_float<bf16_t>(p.scale * OT[0][r]).bits, rows, o_at + r * o_pitch, 0, 0);
      }
    }
  };
#pragma unroll
  for (int a = 0; a < AHEAD; ++a) load_v(SUB * a, vraw[a]);
  if (subs > 0) {
    wait_count(&lds.flags.full[0], 1u);
    load_rows(0);
  }
  int i = 0;
  for (; i + AHEAD <= subs; i += AHEAD) {
#pragma unroll
    for (int a = 0; a < AHEAD; ++a) step(i + a, vraw[a]);
  }
#pragma unroll
  for (int a = 0; a < AHEAD - 1; ++a)
    if (i + a < subs) step(i + a, vraw[a]);
  if (chain.fin != nullptr) store_state(chain.fin);
}

__device__ __forceinline__ const float* kda_state_in(const KdaPrefillParams& p, int n, int head) {
  const int slot = p.h0 != nullptr ? (p.h0_indices ? p.h0_indices[n] : n) : -1;
  return slot >= 0 ? p.h0 + (int64_t)slot * p.h0_slot_stride + (int64_t)head * 16384 : nullptr;
}
__device__ __forceinline__ float* kda_state_out(const KdaPrefillParams& p, int n, int head) {
  const int slot = p.ht != nullptr ? (p.ht_indices ? p.ht_indices[n] : n) : -1;
  return slot >= 0 ? p.ht + (int64_t)slot * p.ht_slot_stride + (int64_t)head * 16384 : nullptr;
}

// The chain of logical index `index`: (sequence, head), or (segment, head) of those that the second sweep runs.
__device__ __forceinline__ Chain kda_chain(const KdaPrefillParams& p, int index, int lane) {
  Chain c{};
  const int item = index / p.H;
  c.head = index - item * p.H;
  if (p.pass == 0) {
    const int2 range = sequence_tokens(p.cu_seqlens, item, p.T);
    c.token = range.x;
    c.tokens = range.y;                              // 0: state untouched, no output
    c.slot = first_slot(item, range.x);
    c.init = kda_state_in(p, item, c.head);
    c.fin = kda_state_out(p, item, c.head);
    return c;
  }
  const Segment s = inline_segment(p.cu_seqlens, p.N, p.T, p.seg, p.split_from, true, item, lane);
  if (s.sequence < 0) return c;
  c.token = s.token;
  c.tokens = s.tokens;
  c.slot = s.slot;
  // the caller's state for a sequence of one segment, else what its predecessor ends in
  c.init = s.count == 1 ? kda_state_in(p, s.sequence, c.head) : p.seg.B + ((int64_t)(s.number - 1) * p.H + c.head) * 16384;
  if (s.index + 1 == s.count) c.fin = kda_state_out(p, s.sequence, c.head);
  return c;
}

// The final state of an empty sequence, which no chain reaches: the one it starts from (or zero), by the workgroups of
// (sequence, head) `index`, or of that segment and head.  (Copied ahead of the launch, for every sequence, it is a launch and up to 7 us: 18
// sequences of 12 heads, 28 MB.)  In the kernel of ragged sequences it stands BEHIND the sweep: ahead of it the two bodies came out
// slower (21 short sequences of 48 heads 108.7 us without it, 109.5 ahead, 106.5 behind; 18 of 12 heads 57.8 / 58.6 / 57.1); in the others
// ahead (364 + 124 tokens of 16 heads 30.0 / 30.4 / 30.7, 65 536 of 32 heads 1573 / 1574 / 1582).
template <int NB>
__device__ __forceinline__ void kda_empty_state(const KdaPrefillParams& p, int index, int half) {
  const int n = index / p.H, head = index - n * p.H;
  if (n >= p.N || sequence_tokens(p.cu_seqlens, n, p.T).y > 0) return;
  const float* const src = kda_state_in(p, n, head);
  float* const dst = kda_state_out(p, n, head);
  if (dst == nullptr) return;
  for (int i = 64 * 128 * half + 4 * threadIdx.x; i < 64 * 128 * (half + NB); i += 4 * blockDim.x)
    *reinterpret_cast<float4*>(dst + i) = src != nullptr ? *reinterpret_cast<const float4*>(src + i) : make_float4(0.f, 0.f, 0.f, 0.f);
}

constexpr int FEEDERS = 4;                         // producing or copying wavefronts of a workgroup
template <int NB, bool PREPARED, bool BEHIND>
__device__ __forceinline__ void kda_sweep(const KdaPrefillParams& p, KdaLds<true>& lds, int index, int half) {
  const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const Chain chain = kda_chain(p, index, lane);
  if (!BEHIND && p.empty_states && (p.pass == 2 || chain.tokens == 0)) kda_empty_state<NB>(p, index, half);
  if (chain.tokens > 0) {
    if (wave < 4) kda_compute<NB, true>(p, lds, chain, lane, 64 * half + 16 * NB * wave);
    else if (PREPARED) kda_copy<true, FEEDERS>(p, lds, chain, lane, wave - 4, 4);
    else kda_produce<true, FEEDERS>(p, lds, chain, lane, wave - 4, 4);
    if (!BEHIND || p.pass == 0) return;
  }
  if (BEHIND && p.empty_states) kda_empty_state<NB>(p, index, half);
}

// The rows of o beyond the last sequence, dealt to all workgroups of a launch.
__device__ __forceinline__ void kda_zero_tail(const KdaPrefillParams& p) {
  zero_tail(reinterpret_cast<uint16_t*>(p.o), p.cu_seqlens, p.N, p.T, p.H, blockIdx.x, gridDim.x);
}

// One workgroup per (sequence, head) or per (segment, head) in the second sweep over segments (NB = 2); NB = 1: two
// per chain, 64 V columns each, on one XCD: they read the same rows, which then come from memory once.
template <int NB, bool PREPARED>
__global__ __launch_bounds__(64 * (4 + FEEDERS), 1) void kda_sweep_kernel(const KdaPrefillParams p) {
  __shared__ KdaLds<true> lds;
  ring_reset(&lds.flags);
  kda_zero_tail(p);
  const int chains = (p.pass == 2 ? p.seg.max_segments : p.N) * p.H;
  const int wide = NB == 2 ? (int)blockIdx.x : xcd_grouped_index(blockIdx.x, 2, 2 * chains);
  if (wide < 0) return;
  kda_sweep<NB, PREPARED, false>(p, lds, NB == 2 ? wide : wide >> 1, NB == 2 ? 0 : wide & 1);
}

// Ragged whole sequences: the chains of the longest sequences as two halves (first in the grid: workgroups are
// dispatched in index order), those of the others whole, longest first (mixed_sweep_plan).
__global__ __launch_bounds__(64 * (4 + FEEDERS), 1) void kda_sweep_mixed_kernel(const KdaPrefillParams p) {
  __shared__ KdaLds<true> lds;
  ring_reset(&lds.flags);
  kda_zero_tail(p);
  if (blockIdx.x < p.split_grid) {
    const int wide = xcd_grouped_index(blockIdx.x, 2, 2 * p.n_long * p.H);
    if (wide < 0) return;
    const int chain = wide >> 1, k = chain / p.H;
    kda_sweep<1, false, true>(p, lds, p.seq_order[k] * p.H + chain - k * p.H, wide & 1);
  } else {
    const int chain = blockIdx.x - p.split_grid;
    if (chain >= (p.N - p.n_long) * p.H) return;
    const int k = chain / p.H;
    kda_sweep<2, false, true>(p, lds, p.seq_order[p.n_long + k] * p.H + chain - k * p.H, 0);
  }
}

// First sweep over segments.  A segment between the first and the last of its sequence is swept twice without
// output - from a zero state (its B summary) and from the identity with v = 0 (its transition matrix M) - and both sweeps
// multiply the same operands: wavefronts 0-3 carry the B columns (32 each), 4-7 the M columns, 8-11 form the operands.  A
// first segment is swept from its real start state and for good, with output: wavefronts 0-7 carry 16 columns each (with 32
// they need more registers than twelve wavefronts leave them), which takes about as long as the two roles of the others.  A
// sequence of one segment is left to the second sweep, which may run it as two halves (four of 400 to 600 tokens, 16 heads, that
// the kernels do not split: 51.9 us, swept here 62.5).
template <bool PREPARED>
__global__ __launch_bounds__(64 * (8 + FEEDERS), 1) void kda_first_sweep_kernel(const KdaPrefillParams p) {
  __shared__ union { KdaLds<true> out; KdaLds<false> lean; } lds;
  const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int item = blockIdx.x / p.H;
  const Segment s = inline_segment(p.cu_seqlens, p.N, p.T, p.seg, p.split_from, false, item, lane);
  if (s.sequence < 0) return;
  Chain chain{};
  chain.token = s.token;
  chain.tokens = s.tokens;
  chain.slot = s.slot;
  chain.head = blockIdx.x - item * p.H;
  const int64_t tile = ((int64_t)s.number * p.H + chain.head) * 16384;
  if (s.index == 0) {
    ring_reset(&lds.out.flags);
    chain.init = kda_state_in(p, s.sequence, chain.head);
    chain.fin = p.seg.B + tile;
    if (wave < 8) kda_compute<1, true>(p, lds.out, chain, lane, 16 * wave);
    else if (PREPARED) kda_copy<true, FEEDERS>(p, lds.out, chain, lane, wave - 8, 8);
    else kda_produce<true, FEEDERS>(p, lds.out, chain, lane, wave - 8, 8);
    return;
  }
  ring_reset(&lds.lean.flags);
  if (wave >= 8) {
    if (PREPARED) kda_copy<false, FEEDERS>(p, lds.lean, chain, lane, wave - 8, 8);
    else kda_produce<false, FEEDERS>(p, lds.lean, chain, lane, wave - 8, 8);
  } else {
    chain.identity = wave >= 4;
    chain.fin = (chain.identity ? p.seg.M : p.seg.B) + tile;
    kda_compute<2, false>(p, lds.lean, chain, lane, 32 * (wave & 3));
  }
}

// Segments of a split call (at most 64 chains).  A call is priced in us (of steps 4 % longer than they are now) from its longest sequence (L chunks) and its (segment, head)
// pairs: not split 13.5 + 2.84 L; split into segments of s chunks, 7.8 s for the two sweeps where the second one takes prepared
// sub-chunks as halves (pairs on half of the CUs at most; preparing them takes 0.2 per thousand tokens and heads), 12.7 s otherwise, and
// about 2 a segment for the combine step.  Segments are at least as long as gives every CU one pair of a sweep, which runs one
// segment less per split sequence than there are.  us per call, s = 3 / 4 / 8 / 16 / not split: one of 2048 tokens, 4 heads 63.4 / 64.4 /
// 83.2 / - / 94.6; 4096, 8 heads 94.5 / 83.8 / 94.9 / 141 / 168; 3000, 16 heads 88.3 / 88.3 / 94.7 / 142 / 132; 2048, 32 heads 125 / 84.6 / 97.0 / - /
// 101.  (The prices are from before first segments were swept once, for good; over fifty shapes their choice is 0-3 % from the best
// length, 5 % for one of 3000 tokens, 32 heads.)
// Splitting pays from sequences of about 15 + 0.13 chunks per chain on, 13 + 0.28 from 13 chains on (us split / not: 770 tokens, 1 head
// 48.5 / 42.9; 890 48.5 / 47.1; 960 49.4 / 49.6; 870, 4 heads 50.6 / 49.2; 960 51.3 / 52.3; 960, 8 heads 53.7 / 52.9; 1020 55.1 / 55.6; 870,
// 16 heads 56.7 / 53.2; 1150 62.8 / 65.3; 1150, 24 heads 66.9 / 65.3; 1250 67.3 / 69.0; 1300, 32 heads 72.1 / 73.4; 1400 75.7 / 77.4).
// The host knows the sum of several sequences only: where their mean is below that line the kernels decide by the longest one (count_segments), which costs
// 4 us where it turns out that nothing is split (six of 590 tokens, 4 heads 48.2 / 44.3, split 58.7; one of 3000 among
// short ones 76.9 / 143), and calls of less than 32 chunks are not split.
struct KdaSplit { int chunks, from; bool halves; };      // chunks of a segment (0: not split); KdaPrefillParams::split_from; see KdaWorkspaceLayout
static KdaSplit kda_split(int T, int N, int H, bool prepares) {
  const int chains = N * H, chunks = (T - 1) / CHUNK + 1, mean = (chunks + N - 1) / N, line = std::max(15 + chains / 8, 13 + 9 * chains / 32);
  KdaSplit split{0, 0, false};
  if (N == 1 ? chunks < line : T / CHUNK < 32) return split;
  const int per_head = std::max(1, CUS / H + (N == 1 ? 1 : 0)), least = std::max(3, ((N == 1 ? chunks : T / CHUNK) + per_head - 1) / per_head);
  double best = 0.;
  for (int s = least; s <= least + 16; ++s) {
    const double pairs = (N == 1 ? (chunks - 1) / s : (double)chunks / s - 0.5 * N) * H;
    const bool halves = prepares && pairs <= CUS / 2;
    const double price = halves ? 18.5 + 7.8 * s + 2.3 * mean / s + 2e-4 * T * H : 24. + 12.7 * s + 1.8 * mean / s;
    if (split.chunks == 0 || price < best) best = price, split = KdaSplit{s, 0, halves};
  }
  if (N > 1 && mean < line && (split.halves || 4 * mean < 3 * line))
    split = prepares ? KdaSplit{split.halves ? split.chunks : least, line, true} : KdaSplit{std::max(8, least), 0, false};
  return split;
}
// Calls of at most 128 chains leave half of the CUs without a sweep: kda_prepare_kernel forms their sub-chunks on all of them
// and the sweeps copy them (a step of 16 tokens then takes 0.7 us instead of 1.3), unless the sequences are so short that the
// second launch costs more than it saves (us per call, prepared / formed by the sweeps: 3 sequences of 47 tokens, 24 heads 19.0 /
// 15.5; of 157 28.1 / 25.4; of 507 47.5 / 52.7; three of 24, 71, 200, 12 heads 23.5 / 27.3) or the sub-chunks no longer stay
// in the last-level cache beside the inputs (MiB of them: 98, 3 of 1207 tokens, 24 heads 86.5 / 99.4; 131, 3 of 1207, 32 heads
// 115 / 100; 205, 3 of 2507, 24 heads 208 / 196).
constexpr int KDA_PREPARE_TOKENS = 96;
constexpr int64_t KDA_PREPARE_BYTES = (int64_t)112 << 20;
struct KdaWorkspaceLayout {
  size_t segM, segB, prepared, total;
  int seg_chunks, split_from, max_segments;
  int64_t slots;            // prepared sub-chunks (0: the sweeps form them)
  bool halves;              // two workgroups per chain
};
static KdaWorkspaceLayout kda_layout(int T, int N, int H) {
  KdaWorkspaceLayout L{};
  size_t off = 0;
  auto take = [&](size_t bytes) { const size_t at = off; off = align_up256(off + bytes); return at; };
  const int64_t chains = (int64_t)N * H, slots = T / SUB + N + 1;
  const bool prepares = slots * H * KdaSlot::BYTES <= KDA_PREPARE_BYTES;
  const KdaSplit split = chains <= 64 ? kda_split(T, N, H, prepares) : KdaSplit{0, 0, false};
  L.seg_chunks = split.chunks;
  L.split_from = split.from;
  L.max_segments = L.seg_chunks > 0 ? T / CHUNK / L.seg_chunks + N + 1 : 0;
  L.halves = L.seg_chunks > 0 ? split.halves : chains <= CUS / 2;
  L.slots = L.halves && prepares && (L.seg_chunks > 0 || T > KDA_PREPARE_TOKENS * (int64_t)N) ? slots : 0;
  const size_t states = (size_t)L.max_segments * H * 16384 * 4;
  L.segM = take(states); L.segB = take(states);
  L.prepared = take((size_t)L.slots * H * KdaSlot::BYTES);
  L.total = off > 0 ? off : 256;                 // (never empty: a null workspace is refused)
  return L;
}

}  // namespace pla

using namespace pla;

extern "C" int64_t pla_kda_prefill_workspace_bytes(int T, int N, int H) {
  if (T <= 0 || N <= 0 || H <= 0) return 0;
  return (int64_t)kda_layout(T, N, H).total;
}

// The share of a KDA chain's chunk time that one of its two half workgroups takes, and how much longer a chunk takes
// on a full chip than on an idle one (mixed_sweep_plan).  Measured, us per call without the plan / at (0.72, 0.05) / (0.8, 0.05)
// / (0.9, 0.05): 8000 + 7000 + 1000 + 2000 + 3000 tokens of 32 heads 728 / 597 / 599 / 645; eight ragged sequences of 32 810
// tokens 671 / 615 / 612 / 613; twelve of 700 to 6000 tokens 564 / 478 / 479 / 481; 18 of 121 to 999 tokens of 12 heads 111 / 102 /
// 102 / 102.
constexpr double KDA_HALF_COST = 0.8, KDA_FILL_COST = 0.05;

// Whether the output shares memory with an input that the sweeps read where no kernel prepares their sub-chunks (q, k, g, beta and
// the gate's parameters).  In place: every such input is the output's very rows, which a workgroup that sweeps all columns of a
// chain has read before it writes them; two workgroups of one chain would each overwrite rows that the other has yet to read.
enum class KdaOverlap { none, in_place, other };
static KdaOverlap kda_overlap(const KdaPrefillParams& p) {
  const uintptr_t o_begin = (uintptr_t)p.o, row = (uintptr_t)p.H * 256, o_end = o_begin + (uintptr_t)p.T * row;
  KdaOverlap found = KdaOverlap::none;
  auto look = [&](const void* base, int64_t pitch, uintptr_t bytes, bool rows_of_out) {
    const uintptr_t begin = (uintptr_t)base, end = begin + (uintptr_t)((p.T - 1) * pitch) + bytes;
    if (end <= o_begin || begin >= o_end) return;
    const bool same = rows_of_out && begin == o_begin && (p.T == 1 || pitch == (int64_t)row);
    if (!same) found = KdaOverlap::other;
    else if (found == KdaOverlap::none) found = KdaOverlap::in_place;
  };
  look(p.q, 2 * p.stride_q, row, true);
  look(p.k, 2 * p.stride_k, row, true);
  look(p.g, 2 * p.stride_g, row, true);
  look(p.beta, 2 * p.stride_beta, (uintptr_t)p.H * 2, false);
  look(p.A_log, 0, (uintptr_t)p.H * 4, false);
  look(p.dt_bias, 0, (uintptr_t)p.H * 512, false);
  return found;
}

static int kda_prefill_run(
    const void* q, const void* k, const void* v, const void* g, const void* beta,
    int64_t stride_q, int64_t stride_k, int64_t stride_v, int64_t stride_g, int64_t stride_beta,
    const float* A_log, const float* dt_bias, float lower_bound, float scale,
    const int32_t* cu_seqlens, int N, int T,
    const float* h0, const int32_t* h0_indices, int64_t h0_slot_stride,
    float* ht, const int32_t* ht_indices, int64_t ht_slot_stride,
    void* o, void* workspace, int64_t workspace_bytes,
    int H, int K, int V, int act_dtype, void* stream, const int32_t* raw_cu_seqlens, bool empty_states) {
  PLA_REQUIRE(K == 128 && V == 128, "KDA prefill requires head_dim K == V == 128, got K=%d, V=%d", K, V);
  PLA_REQUIRE(T > 0 && N > 0 && H > 0, "KDA prefill needs at least one token, sequence and head");
  PLA_REQUIRE(act_dtype == PLA_BF16, "KDA prefill takes bf16 activations");
  PLA_REQUIRE(q && k && v && g && beta && A_log && dt_bias && o && cu_seqlens && workspace, "null tensor pointer");
  PLA_REQUIRE(lower_bound <= 0.f && lower_bound >= -5.f, "lower_bound must lie in [-5, 0], got %g", (double)lower_bound);
  PLA_REQUIRE(((uintptr_t)q % 16 == 0) && ((uintptr_t)k % 16 == 0) && ((uintptr_t)g % 16 == 0) && stride_q % 8 == 0 &&
                  stride_k % 8 == 0 && stride_g % 8 == 0,
              "q/k/g rows require 16-byte alignment");
  PLA_REQUIRE(((uintptr_t)v % 16 == 0) && stride_v % 8 == 0, "v rows require 16-byte alignment");
  PLA_REQUIRE(((uintptr_t)o % 16 == 0), "out requires 16-byte alignment");
  const KdaWorkspaceLayout L = kda_layout(T, N, H);
  PLA_REQUIRE(workspace_bytes >= (int64_t)L.total, "workspace too small: need %zu bytes", L.total);
  PLA_REQUIRE((uintptr_t)workspace % 256 == 0, "workspace requires 256-byte alignment");
  if (h0) PLA_REQUIRE((uintptr_t)h0 % 16 == 0 && h0_slot_stride % 4 == 0, "state requires 16-byte alignment");
  if (ht) PLA_REQUIRE((uintptr_t)ht % 16 == 0 && ht_slot_stride % 4 == 0, "state requires 16-byte alignment");

  char* ws = reinterpret_cast<char*>(workspace);
  KdaPrefillParams p{};
  p.q = q; p.k = k; p.v = v; p.g = g; p.beta = beta;
  p.stride_q = stride_q; p.stride_k = stride_k; p.stride_v = stride_v; p.stride_g = stride_g; p.stride_beta = stride_beta;
  p.A_log = A_log; p.dt_bias = dt_bias; p.lower_bound = lower_bound; p.scale = scale;
  p.cu_seqlens = cu_seqlens; p.N = N; p.T = T;
  p.h0 = h0; p.h0_indices = h0_indices; p.h0_slot_stride = h0_slot_stride;
  p.ht = ht; p.ht_indices = ht_indices; p.ht_slot_stride = ht_slot_stride;
  p.o = o;
  p.H = H;
  p.empty_states = empty_states;

  hipStream_t s = reinterpret_cast<hipStream_t>(stream);
  const bool segmented = L.seg_chunks > 0, prepared = L.slots > 0;
  const KdaOverlap overlap = prepared ? KdaOverlap::none : kda_overlap(p);     // (prepared: all read ahead of the sweep)
  PLA_REQUIRE(overlap != KdaOverlap::other, "out shares memory with q, k, g, beta, A_log or dt_bias other than as the very rows of q, k or g");
  const bool whole_chains = overlap == KdaOverlap::in_place, halves = L.halves && !whole_chains;
  if (segmented) {
    // few, long sequences: sweep their segments concurrently (two sweeps and a combine step)
    p.seg.M = reinterpret_cast<float*>(ws + L.segM);
    p.seg.B = reinterpret_cast<float*>(ws + L.segB);
    p.seg.seg_chunks = L.seg_chunks;
    p.seg.max_segments = L.max_segments;
    p.split_from = L.split_from;
  }
  // Ragged whole sequences whose offsets the host holds: the chains of the longest sequences run as two halves where
  // that shortens the sweep (mixed_sweep_plan)
  bool mixed = false;
  if (!segmented && !L.halves && !whole_chains && raw_cu_seqlens != nullptr && N <= INLINE_TABLE_SEQUENCES) {
    int nc[INLINE_TABLE_SEQUENCES];
    for (int n = 0; n < N; ++n) nc[n] = (std::max(raw_cu_seqlens[n + 1] - raw_cu_seqlens[n], 0) + CHUNK - 1) / CHUNK;
    p.n_long = mixed_sweep_plan(nc, N, H, p.seq_order, KDA_HALF_COST, KDA_FILL_COST);
    // (more chains than CUs: the chains also start longest first - in the order of the sequences the last chain to
    // find a CU may be the longest one -, with or without halves)
    mixed = p.n_long > 0 || (int64_t)N * H > CUS;
    p.split_grid = xcd_grouped_grid(2 * (unsigned)p.n_long * H, 2);
  }
  const dim3 sweep_block(64 * (4 + FEEDERS)), first_block(64 * (8 + FEEDERS));
  const unsigned chains = (unsigned)N * H, segment_chains = (unsigned)L.max_segments * H;
  if (prepared) {
    p.prepared = ws + L.prepared;
    hipLaunchKernelGGL(kda_prepare_kernel, dim3((unsigned)((L.slots * H + PREPARE_WAVES - 1) / PREPARE_WAVES)), dim3(64 * PREPARE_WAVES), 0, s, p);
  }
  if (segmented) {
    p.pass = 1;
    hipLaunchKernelGGL(prepared ? kda_first_sweep_kernel<true> : kda_first_sweep_kernel<false>, dim3(segment_chains), first_block, 0, s, p);
    hipLaunchKernelGGL(segment_combine_kernel<false>, dim3(xcd_grouped_grid(chains * COMBINE_SPLIT, COMBINE_SPLIT)), dim3(256), 0, s, p.seg, cu_seqlens,
                       N, T, H, p.split_from);
    p.pass = 2;
  }
  const unsigned sweeps = segmented ? segment_chains : chains;
  if (mixed) hipLaunchKernelGGL(kda_sweep_mixed_kernel, dim3(p.split_grid + (unsigned)(N - p.n_long) * H), sweep_block, 0, s, p);
  else if (halves) hipLaunchKernelGGL((prepared ? kda_sweep_kernel<1, true> : kda_sweep_kernel<1, false>), dim3(xcd_grouped_grid(2 * sweeps, 2)), sweep_block, 0, s, p);
  else hipLaunchKernelGGL((kda_sweep_kernel<2, false>), dim3(sweeps), sweep_block, 0, s, p);
  return check_launch("kda prefill launch");
}

extern "C" int pla_kda_prefill_launch(
    const void* q, const void* k, const void* v, const void* g, const void* beta,
    int64_t stride_q, int64_t stride_k, int64_t stride_v, int64_t stride_g, int64_t stride_beta,
    const float* A_log, const float* dt_bias, float lower_bound, float scale,
    const int32_t* cu_seqlens, int N, int T,
    const float* h0, const int32_t* h0_indices, int64_t h0_slot_stride,
    float* ht, const int32_t* ht_indices, int64_t ht_slot_stride,
    void* o, void* workspace, int64_t workspace_bytes,
    int H, int K, int V, int act_dtype, void* stream) {
  return kda_prefill_run(q, k, v, g, beta, stride_q, stride_k, stride_v, stride_g, stride_beta, A_log, dt_bias, lower_bound, scale,
                         cu_seqlens, N, T, h0, h0_indices, h0_slot_stride, ht, ht_indices, ht_slot_stride, o, workspace,
                         workspace_bytes, H, K, V, act_dtype, stream, nullptr, false);
}

extern "C" int pla_kda_prefill_launch_raw(
    const void* q, const void* k, const void* v, const void* g, const void* beta,
    int64_t stride_q, int64_t stride_k, int64_t stride_v, int64_t stride_g, int64_t stride_beta,
    const float* A_log, const float* dt_bias, float lower_bound, float scale,
    const int32_t* cu_seqlens, int N, int T,
    const float* h0, const int32_t* h0_indices, int64_t h0_slot_stride,
    float* ht, const int32_t* ht_indices, int64_t ht_slot_stride,
    void* o, void* workspace, int64_t workspace_bytes,
    int H, int K, int V, int act_dtype, void* stream, const int32_t* raw_cu_seqlens) {
  return kda_prefill_run(q, k, v, g, beta, stride_q, stride_k, stride_v, stride_g, stride_beta, A_log, dt_bias, lower_bound, scale,
                         cu_seqlens, N, T, h0, h0_indices, h0_slot_stride, ht, ht_indices, ht_slot_stride, o, workspace,
                         workspace_bytes, H, K, V, act_dtype, stream, raw_cu_seqlens, false);
}

extern "C" int pla_kda_prefill_launch_states(
    const void* q, const void* k, const void* v, const void* g, const void* beta,
    int64_t stride_q, int64_t stride_k, int64_t stride_v, int64_t stride_g, int64_t stride_beta,
    const float* A_log, const float* dt_bias, float lower_bound, float scale,
    const int32_t* cu_seqlens, int N, int T,
    const float* h0, const int32_t* h0_indices, int64_t h0_slot_stride,
    float* ht, const int32_t* ht_indices, int64_t ht_slot_stride,
    void* o, void* workspace, int64_t workspace_bytes,
    int H, int K, int V, int act_dtype, void* stream, const int32_t* raw_cu_seqlens) {
  return kda_prefill_run(q, k, v, g, beta, stride_q, stride_k, stride_v, stride_g, stride_beta, A_log, dt_bias, lower_bound, scale,
                         cu_seqlens, N, T, h0, h0_indices, h0_slot_stride, ht, ht_indices, ht_slot_stride, o, workspace,
                         workspace_bytes, H, K, V, act_dtype, stream, raw_cu_seqlens, true);
}

extern "C" int pla_kda_prefill_halved_sequences(const int32_t* raw_cu_seqlens, int N, int T, int H) {
  if (raw_cu_seqlens == nullptr || N <= 0 || N > INLINE_TABLE_SEQUENCES || T <= 0 || H <= 0) return 0;
  const KdaWorkspaceLayout L = kda_layout(T, N, H);
  if (L.seg_chunks > 0 || (int64_t)N * H <= 128) return 0;
  int nc[INLINE_TABLE_SEQUENCES];
  unsigned char order[INLINE_TABLE_SEQUENCES];
  for (int n = 0; n < N; ++n) nc[n] = (std::max(raw_cu_seqlens[n + 1] - raw_cu_seqlens[n], 0) + CHUNK - 1) / CHUNK;
  return mixed_sweep_plan(nc, N, H, order, KDA_HALF_COST, KDA_FILL_COST);
}
