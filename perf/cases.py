"""What is timed of this framework: the operators as a serving program calls them, over the range it calls them in.

Seven operators, each through its public entry point:

  gdn_decode   one-token GDN decode from the packed QKV rows, state pool updated in place
  kda_decode   one-token KDA decode with the convolution, the gate and the gated norm in the same call
  gdn_verify   verify of a window of draft tokens, with a state snapshot after every token or without any
  kda_ring     KDA verify of every layer with replay records per slot, then one commit of the accepted prefixes
  kda_paged    the same over paged checkpoints, records per request row and the commit plan built on the device
  gdn_prefill  chunked prefill of packed variable-length sequences, pool updated in place
  kda_prefill  the same for KDA, from dense start states to dense final states

Head counts and draft windows are those of the decode and prefill caselists under tests/golden, batch sizes and
sequence lengths lie in the caselists' range.  Every input is drawn on the GPU from the seed.
"""
import math
from types import SimpleNamespace

import torch

from pla_amd.decode import (fused_sigmoid_gating_delta_rule_forward_k_last,
                            fused_sigmoid_gating_delta_rule_forward_k_last_packed)
from pla_amd.decode.kda import fused_kda_decode_mega_forward
from pla_amd.decode.kda_replayssm_sglang import commit_kda_replayssm_after_verify, fused_kda_decode_mtp_dspark
from pla_amd.decode.kda_replayssm_vllm import KDAReplayCommitContext, KDAReplayRecords, kda_replay_verify
from pla_amd.prefill.flashkdapro import flashkda_fwd
from pla_amd.prefill.flashqla import gdn_prefill_packed_qkv_fwd

D = 128
TILE = D * D                                  # elements of one (slot, value head) state tile
SCALE = D ** -0.5
# (q/k heads, value heads) of the GDN caselists; heads of the KDA caselists that the one-token step takes
GDN_HEADS = ((1, 8), (2, 6), (2, 16), (4, 8), (4, 12), (4, 32), (8, 16), (8, 24), (16, 32), (16, 48), (16, 64))
KDA_HEADS = (4, 6, 8, 12, 16, 24, 48, 64)
DTYPES = {"bf16": torch.bfloat16, "fp16": torch.float16, "fp32": torch.float32}


def listed():
    return [
        # a few concurrent chats: launch and latency count
        dict(name="gdn_decode_b8", op="gdn_decode", batch=8, H=16, HV=32, pad=0, act="bf16", state="fp32"),
        # the benchmark's decode step: a full batch, some entries of the captured batch padded
        dict(name="gdn_decode_b256", op="gdn_decode", batch=256, H=16, HV=32, pad=13, act="bf16", state="fp32"),
        # an odd batch on one of eight tensor-parallel ranks (12 heads), the whole step in one call
        dict(name="kda_decode_b69", op="kda_decode", batch=69, H=12, act="bf16", lower_bound=-5.0),
        # a small batch with four draft tokens, nothing but the outputs wanted: latency
        dict(name="gdn_verify_b6", op="gdn_verify", batch=6, tokens=4, H=16, HV=32, snapshots=False, act="bf16", state="fp32"),
        # speculative decoding that keeps the state after every draft token
        dict(name="gdn_verify_snapshots_b24", op="gdn_verify", batch=24, tokens=4, H=16, HV=32, snapshots=True, act="bf16",
             state="fp32"),
        # speculative decoding with replay records: four layers verified, then one commit for all of them
        dict(name="kda_ring_b64", op="kda_ring", batch=64, tokens=4, H=32, layers=4),
        # the same over paged checkpoints on one of eight ranks, the longest draft window of the caselists
        dict(name="kda_paged_b21", op="kda_paged", batch=21, tokens=8, H=12, layers=2, layout="SD"),
        # short prompts: a handful of chunks in all
        dict(name="gdn_prefill_short", op="gdn_prefill", lengths="24,200,71", H=16, HV=32, act="bf16", host_offsets=True),
        # the benchmark's prefill: eight prompts of very different lengths, 32 810 tokens
        dict(name="gdn_prefill_ragged", op="gdn_prefill", lengths="2646,6988,1342,6924,3410,2250,1978,7272", H=16, HV=32,
             act="bf16", host_offsets=True),
        # one long prompt: few chains, the sequence itself has to be split
        dict(name="gdn_prefill_long", op="gdn_prefill", lengths="16384", H=16, HV=32, act="bf16", host_offsets=True),
        # a batch of ordinary prompts on one of eight ranks
        dict(name="kda_prefill_ragged", op="kda_prefill",
             lengths="121,799,871,999,982,626,867,730,736,800,767,930,844,764,804,790,451,333", H=12, host_offsets=True),
        # the benchmark's KDA prefill: one prompt of 65 536 tokens
        dict(name="kda_prefill_long", op="kda_prefill", lengths="65536", H=32, host_offsets=False),
    ]


def _log_int(rng, lo, hi):
    return min(hi, max(lo, int(round(math.exp(rng.uniform(math.log(lo), math.log(hi + 0.5)))))))


def _lengths(rng, tokens):
    """1 to 24 sequences of very different lengths that sum to about `tokens`."""
    n = min(_log_int(rng, 1, 24), tokens)
    parts = [rng.uniform(0.2, 1.0) for _ in range(n)]
    return ",".join(str(max(1, int(tokens * p / sum(parts)))) for p in parts)


def draw(rng):
    op = rng.choice(("gdn_decode", "kda_decode", "gdn_verify", "kda_ring", "kda_paged", "gdn_prefill", "kda_prefill"))
    if op == "gdn_decode":
        H, HV = rng.choice(GDN_HEADS)
        batch = _log_int(rng, 4, 16384 // HV)
        return dict(op=op, batch=batch, H=H, HV=HV, pad=batch // 20 if rng.random() < 0.5 else 0,
                    act=rng.choice(("bf16", "bf16", "fp16")), state=rng.choice(("fp32", "fp32", "bf16")))
    if op == "kda_decode":
        H = rng.choice(KDA_HEADS)
        return dict(op=op, batch=_log_int(rng, 2, 12288 // H), H=H, act=rng.choice(("bf16", "bf16", "fp16")),
                    lower_bound=rng.choice((-5.0, None)))
    if op == "gdn_verify":
        H, HV = rng.choice(GDN_HEADS)
        snapshots = rng.random() < 0.5
        return dict(op=op, batch=_log_int(rng, 2, (4096 if snapshots else 12288) // HV), tokens=rng.randint(2, 8), H=H, HV=HV,
                    snapshots=snapshots, act="bf16", state=rng.choice(("fp32", "fp32", "bf16")))
    if op in ("kda_ring", "kda_paged"):
        H = rng.choice(KDA_HEADS + (32,))
        c = dict(op=op, batch=_log_int(rng, 2, 3072 // H), tokens=rng.randint(2, 8), H=H, layers=rng.randint(1, 4))
        return dict(c, layout=rng.choice(("SD", "DS"))) if op == "kda_paged" else c
    if op == "gdn_prefill":
        H, HV = rng.choice(GDN_HEADS)
        return dict(op=op, lengths=_lengths(rng, _log_int(rng, 64, 1048576 // HV)), H=H, HV=HV,
                    act=rng.choice(("bf16", "bf16", "fp16")), host_offsets=rng.random() < 0.7)
    H = rng.choice(KDA_HEADS + (32,))
    return dict(op=op, lengths=_lengths(rng, _log_int(rng, 64, 524288 // H)), H=H, host_offsets=rng.random() < 0.7)


class _Draw:
    """Seeded draws on the GPU."""

    def __init__(self, seed):
        self.device = torch.device("cuda", torch.cuda.current_device())
        self.g = torch.Generator(device=self.device).manual_seed(seed)

    def normal(self, *shape, dtype=torch.float32, scale=1.0):
        x = torch.empty(*shape, dtype=dtype, device=self.device)
        return x.normal_(0.0, scale, generator=self.g)

    def uniform(self, *shape, lo=0.0, hi=1.0):
        return torch.empty(*shape, device=self.device).uniform_(lo, hi, generator=self.g)

    def slots(self, slots, n, first=0):
        """n different slots of a pool, in no order."""
        return first + torch.randperm(slots - first, generator=self.g, device=self.device)[:n].to(torch.int32)

    def counts(self, n, hi):
        return torch.randint(1, hi + 1, (n,), generator=self.g, device=self.device, dtype=torch.int32)


def _even_offsets(batch, tokens, device):
    return torch.arange(0, batch * tokens + 1, tokens, dtype=torch.int32, device=device)


def _gdn_decode(c, r):
    B, H, HV, act = c["batch"], c["H"], c["HV"], DTYPES[c["act"]]
    slots = B + B // 2 + 3
    indices = r.slots(slots, B)
    indices[B - c["pad"]:] = -1
    args = dict(mixed_qkv=r.normal(B, (2 * H + HV) * D, dtype=act), a=r.normal(B, HV, dtype=act), b=r.normal(B, HV, dtype=act),
                A_log=r.uniform(HV, hi=math.log(16.0)), dt_bias=r.uniform(HV, lo=-1.0).to(act), softplus_beta=1.0,
                softplus_threshold=20.0, scale=SCALE,
                initial_state_source=r.normal(slots, HV, D, D, dtype=DTYPES[c["state"]], scale=0.1),
                initial_state_indices=indices, out=torch.empty(B, 1, HV, D, dtype=act, device=r.device),
                use_qk_l2norm_in_kernel=True, cu_seqlens=_even_offsets(B, 1, r.device), is_kda=False, is_sglang=True)

    def run():
        out = fused_sigmoid_gating_delta_rule_forward_k_last_packed(**args)
        return out, args["initial_state_source"]
    return run


def _kda_decode(c, r):
    B, H, act = c["batch"], c["H"], DTYPES[c["act"]]
    dim, slots = H * D, B + B // 2 + 3
    # one page per slot: three conv taps of every channel, then the FP32 state
    conv_elems = 9 * dim
    page = conv_elems * 2 + H * TILE * 4
    cache = torch.zeros(slots * page, dtype=torch.uint8, device=r.device)
    conv = torch.as_strided(cache.view(act), (slots, 3 * dim, 3), (page // 2, 1, 3 * dim))
    state = torch.as_strided(cache.view(torch.float32), (slots, H, D, D), (page // 4, TILE, D, 1), conv_elems // 2)
    conv.copy_(r.normal(slots, 3 * dim, 3, scale=0.3))
    state.copy_(r.normal(slots, H, D, D, scale=0.1))
    out = torch.empty(1, B, H, D, dtype=act, device=r.device)
    args = dict(x=r.normal(B, 3 * dim, dtype=act), weight=r.normal(3, 4, dim, scale=0.3), bias=None, conv_state=conv,
                raw_g=r.normal(1, B, H, D, dtype=act), raw_beta=r.normal(1, B, H, dtype=act), a_log=r.normal(H, scale=0.5),
                dt_bias=r.normal(dim, scale=0.1), state_indices=r.slots(slots, B), state=state, out=out,
                lower_bound=c["lower_bound"], output_gate=r.normal(B, H, D, dtype=act), norm_weight=r.uniform(D, lo=0.75, hi=1.25),
                norm_eps=1e-5)

    def run():
        fused_kda_decode_mega_forward(**args)
        return out, state, conv
    return run


def _gdn_verify(c, r):
    B, T, H, HV, act, sdt = c["batch"], c["tokens"], c["H"], c["HV"], DTYPES[c["act"]], DTYPES[c["state"]]
    slots = B + B // 2 + 3
    mixed = r.normal(B, T, (2 * H + HV) * D, dtype=act)
    q, k, v = (t.contiguous().view(B, T, -1, D) for t in mixed.split((H * D, H * D, HV * D), dim=2))
    snapshots = torch.zeros(B, T, HV, D, D, dtype=sdt, device=r.device) if c["snapshots"] else None
    args = dict(A_log=r.uniform(HV, hi=math.log(16.0)), a=r.normal(B, T, HV, dtype=act),
                dt_bias=r.uniform(HV, lo=-1.0).to(act), softplus_beta=1.0, softplus_threshold=20.0, q=q, k=k, v=v,
                b=r.normal(B, T, HV, dtype=act), initial_state_source=r.normal(slots, HV, D, D, dtype=sdt, scale=0.1),
                initial_state_indices=r.slots(slots, B), scale=SCALE, use_qk_l2norm_in_kernel=True, cu_seqlens=None,
                is_kda=False, disable_state_update=True, intermediate_states_buffer=snapshots,
                intermediate_state_indices=r.slots(B, B) if c["snapshots"] else None,
                cache_steps_or_num_accept=T if c["snapshots"] else None, retrieve_parent_token=None,
                out=torch.empty(B, T, HV, D, dtype=act, device=r.device))

    def run():
        return fused_sigmoid_gating_delta_rule_forward_k_last(**args), snapshots
    return run


def _kda_ring(c, r):
    B, T, H, L = c["batch"], c["tokens"], c["H"], c["layers"]
    dim, slots, bf16 = H * D, B + B // 2 + 3, torch.bfloat16
    ring = max(8, T)
    spec = SimpleNamespace(
        temporal=r.normal(L, slots, H, D, D, scale=0.1),
        replayssm_rawv=torch.zeros(L, slots, H, ring, D, dtype=bf16, device=r.device),
        replayssm_rawk=torch.zeros(L, slots, H, ring, D, dtype=bf16, device=r.device),
        replayssm_g=torch.zeros(L, slots, H, ring, D, device=r.device),
        replayssm_beta=torch.zeros(L, slots, H, ring, device=r.device),
        conv=[r.normal(L, slots, dim, 3, dtype=bf16, scale=0.3) for _ in range(3)],
        intermediate_conv_window=[torch.zeros(L, B, T, dim, 3, dtype=bf16, device=r.device) for _ in range(3)])
    indices = r.slots(slots, B)
    accepted = r.counts(B, T)
    shared = dict(intermediate_state_indices=torch.arange(B, dtype=torch.int32, device=r.device), ssm_state_indices=indices,
                  cu_seqlens=_even_offsets(B, T, r.device), lower_bound=-5.0, scale=SCALE, onorm_eps=1e-6)
    verify = []
    for l in range(L):
        rows = r.normal(1, B * T, 3 * dim, dtype=bf16, scale=0.5)
        x_q, x_k, x_v = (rows[:, :, i * dim:(i + 1) * dim].view(1, B * T, H, D) for i in range(3))
        w_q, w_k, w_v = (r.normal(dim, 4, scale=0.3) for _ in range(3))
        verify.append(dict(
            shared, x_q=x_q, x_k=x_k, x_v=x_v, w_q=w_q, w_k=w_k, w_v=w_v, cs_q=spec.conv[0][l], cs_k=spec.conv[1][l],
            cs_v=spec.conv[2][l], g=r.normal(1, B * T, H, D, dtype=bf16, scale=0.5), beta=r.normal(1, B * T, H, dtype=bf16),
            A_log=r.uniform(H, lo=0.5), dt_bias=r.normal(dim, scale=0.1), recurrent_state=spec.temporal[l],
            intermediate_conv_q=spec.intermediate_conv_window[0][l], intermediate_conv_k=spec.intermediate_conv_window[1][l],
            intermediate_conv_v=spec.intermediate_conv_window[2][l], replayssm_rawv=spec.replayssm_rawv[l],
            replayssm_rawk=spec.replayssm_rawk[l], replayssm_g=spec.replayssm_g[l], replayssm_beta=spec.replayssm_beta[l],
            onorm_gate=r.normal(1, B * T, H, D, dtype=bf16), onorm_weight=r.uniform(D, lo=0.75, hi=1.25),
            out=torch.empty(1, B * T, H, D, dtype=bf16, device=r.device)))
    last = accepted - 1

    def run():
        outs = [fused_kda_decode_mtp_dspark(**call) for call in verify]
        commit_kda_replayssm_after_verify(spec_state=spec, state_batch_indices=indices, accept_lens=accepted,
                                          last_correct_step_indices=last)
        return (outs, spec.temporal, spec.conv, spec.intermediate_conv_window, spec.replayssm_rawv, spec.replayssm_rawk,
                spec.replayssm_g, spec.replayssm_beta)
    return run


def _kda_paged(c, r):
    B, Q, H, L, layout = c["batch"], c["tokens"], c["H"], c["layers"], c["layout"]
    dim, slots, history = H * D, B + B // 2 + 3, Q + 2
    channels, T = 3 * dim, B * Q
    conv_shape, conv_stride = ((channels, history), (history, 1)) if layout == "DS" else ((history, channels), (channels, 1))
    state_at = -(-channels * history * 2 // 16) * 16
    page = -(-(state_at + H * TILE * 4) // 256) * 256
    indices = r.slots(slots, B, first=1)                       # slot 0 is the null block
    offsets = _even_offsets(B, Q, r.device)
    sampled = r.counts(B, Q)
    layers, verify = [], []
    for _ in range(L):
        raw = torch.zeros(slots * page, dtype=torch.uint8, device=r.device)
        conv = raw.view(torch.bfloat16).as_strided((slots, *conv_shape), (page // 2, *conv_stride))
        state = raw.view(torch.float32).as_strided((slots, H, D, D), (page // 4, TILE, D, 1), state_at // 4)
        conv.copy_(r.normal(slots, *conv_shape, scale=0.3))
        state.copy_(r.normal(slots, H, D, D, scale=0.1))
        records = KDAReplayRecords(*(torch.zeros_like(t) for t in vars(KDAReplayRecords.allocate(B, H, Q, r.device)).values()))
        rows = r.normal(T, 4 * dim + H, dtype=torch.bfloat16, scale=0.5)
        layers.append(SimpleNamespace(kv_cache=(conv, state), replay_records=records))
        verify.append(dict(mixed_qkv=rows[:, :3 * dim], raw_g=rows[:, 3 * dim:4 * dim], raw_beta=rows[:, 4 * dim:],
                           conv_weight=r.normal(channels, 4, scale=0.3), A_log=r.normal(H, scale=0.1),
                           dt_bias=r.normal(dim, scale=0.2), lower_bound=-5.0, conv_state=conv, checkpoint_state=state,
                           records=records, query_start_loc=offsets, state_indices=indices, conv_state_layout=layout,
                           null_block_id=0, out=torch.empty(T, dim, dtype=torch.bfloat16, device=r.device)))
    context = KDAReplayCommitContext.create(layers, Q, B, layout, 0)

    def run():
        outs = [kda_replay_verify(**call) for call in verify]
        context.commit(sampled, indices, offsets, token_capacity=T)
        return outs, [(*l.kv_cache, *vars(l.replay_records).values()) for l in layers]
    return run


def _split_lengths(c):
    lengths = [int(x) for x in c["lengths"].split(",")]
    offsets = [0]
    for n in lengths:
        offsets.append(offsets[-1] + n)
    return len(lengths), offsets[-1], offsets


def _gdn_prefill(c, r):
    H, HV, act = c["H"], c["HV"], DTYPES[c["act"]]
    N, T, offsets = _split_lengths(c)
    slots = max(8, N + N // 2)
    pool = r.normal(slots, HV, D, D, scale=0.1)
    args = (r.normal(T, (2 * H + HV) * D, dtype=act), r.normal(T, HV, dtype=act), r.normal(T, HV, dtype=act),
            r.uniform(HV, hi=math.log(16.0)), r.uniform(HV, lo=-1.0),
            torch.tensor(offsets, dtype=torch.int32).to(r.device))
    more = dict(num_qk_heads=H, num_v_heads=HV, scale=SCALE, initial_state=pool, initial_state_indices=r.slots(slots, N),
                raw_cu_seqlens=tuple(offsets) if c["host_offsets"] else None, output_final_state=False)

    def run():
        g_cum, _, o, _, _ = gdn_prefill_packed_qkv_fwd(*args, **more)
        return o, pool, g_cum
    return run


def _kda_prefill(c, r):
    H = c["H"]
    N, T, offsets = _split_lengths(c)
    # half of the heads forget within a few tokens, the others over thousands: the lower-bound gate is
    # g = -5 sigmoid(raw), so a mean of -1 gives g about -1.3 a token and a mean of -7 about -0.005
    gate = r.normal(T, H, D, scale=0.5)
    gate[:, :H // 2] -= 1.0
    gate[:, H // 2:] -= 7.0
    q, k, v = (r.normal(T, H, D, dtype=torch.bfloat16) for _ in range(3))
    out = torch.empty(T, H, D, dtype=torch.bfloat16, device=r.device)
    final = torch.empty(N, H, D, D, device=r.device)
    args = (q, k, v, gate.to(torch.bfloat16), r.normal(T, H, dtype=torch.bfloat16), torch.zeros(H, device=r.device),
            r.normal(H, D, scale=0.1), out)
    more = dict(scale=SCALE, lower_bound=-5.0, initial_state=r.normal(N, H, D, D, scale=0.1), final_state=final,
                cu_seqlens=torch.tensor(offsets, dtype=torch.int32).to(r.device),
                raw_cu_seqlens=tuple(offsets) if c["host_offsets"] else None)

    def run():
        flashkda_fwd(*args, **more)
        return out, final
    return run


_PREPARE = dict(gdn_decode=_gdn_decode, kda_decode=_kda_decode, gdn_verify=_gdn_verify, kda_ring=_kda_ring,
                kda_paged=_kda_paged, gdn_prefill=_gdn_prefill, kda_prefill=_kda_prefill)


def prepare(case, seed):
    return _PREPARE[case["op"]](case, _Draw(seed))


def run(state):
    return state()


def work(case):
    """Bytes: every input and state tile read once, every output, record and updated tile written once.  Operations: the
    recurrence per token and state element (decay, two products with a row, one rank-one update: 7), for the prefill
    the dense chunk-64 form (three K x V and two 64 x V products per value head, two 64 x K per q/k head)."""
    op, H = case["op"], case["H"]
    if op.endswith("prefill"):
        HV = case.get("HV", H)
        N, T, _ = _split_lengths(case)
        row = (2 * H + 2 * HV) * D * 2 + (HV * D * 2 + HV * 2 if op == "kda_prefill" else 2 * HV * 2 + HV * 4)
        return dict(bytes=T * row + N * HV * 2 * TILE * 4, flops=T * 2 * (HV * (3 * TILE + 2 * 64 * D) + H * 2 * 64 * D))
    B, T = case["batch"], case.get("tokens", 1)
    if op == "gdn_decode":
        HV, n = case["HV"], B - case["pad"]
        tile = TILE * (4 if case["state"] == "fp32" else 2)
        return dict(bytes=n * HV * (2 * tile + 4) + n * (2 * H + HV) * D * 2 + B * HV * D * 2, flops=n * HV * 7 * TILE)
    if op == "gdn_verify":
        HV = case["HV"]
        tile = TILE * (4 if case["state"] == "fp32" else 2)
        return dict(bytes=B * HV * tile * (1 + T * case["snapshots"]) + B * T * ((2 * H + 2 * HV) * D * 2 + HV * 4),
                    flops=B * T * HV * 7 * TILE)
    dim = H * D
    if op == "kda_decode":
        return dict(bytes=B * (H * 2 * TILE * 4 + 2 * 9 * dim * 2 + 6 * dim * 2 + 2 * H) + 12 * dim * 4, flops=B * H * 7 * TILE)
    # verify: the state read, per token q, k, v, gate (and the norm's gate) in, the output, the records (k, v, log-decay,
    # beta) and the conv window of every channel out; commit: the mean of (T + 1) / 2 recorded tokens back in, the tile
    # read and written, one conv window moved
    token = (6 if op == "kda_ring" else 5) * dim * 2 + 2 * H + (dim * 8 + H * 4) + 9 * dim * 2
    per_layer = B * (3 * H * TILE * 4 + T * token + (T + 1) / 2 * (dim * 8 + H * 4) + 3 * 9 * dim * 2) + 12 * dim * 4
    return dict(bytes=case["layers"] * per_layer, flops=case["layers"] * B * H * 7 * TILE * (T + (T + 1) / 2))


def tolerance(case):
    """Four times the distance of the outputs from the oracle in 64 bits, measured per operator, rounded up.  16-bit
    outputs of the decode and verify operators are one rounding of an FP32 result (2-norm 1.7e-3, largest 3.9e-3 in
    bf16, an eighth in fp16; FP32 states 1e-7, fp16 activations over a bf16 pool take the pool's figure).  The prefill
    products take rounded operands (o 2.8e-3, largest 2.1e-2 in bf16; 8.6e-4 and 6.1e-3 in fp16; FP32 states up to
    2.7e-4 and 2e-3)."""
    half = case.get("act") == "fp16" and case.get("state", "fp32") == "fp32"
    if case["op"].endswith("prefill"):
        return {"rel": 3.5e-3, "max": 2.5e-2} if half else {"rel": 1.1e-2, "max": 8.5e-2}
    return {"rel": 9e-4, "max": 2e-3} if half else {"rel": 7e-3, "max": 1.6e-2}
