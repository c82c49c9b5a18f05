"""The replay entry points offer each call to the compiled host layer first: ordinary calls are taken there, calls that
need a copy or fail a check are not, and both layers leave the same bits everywhere."""
import dataclasses
import types

import pytest
import torch

from oracle import conv_window_scatter_reference
from pla_amd.decode import _C, kda_replayssm_sglang as ring, kda_replayssm_vllm as paged
from pla_amd.workloads import kda_replay_verify
from test_replay_vllm_gpu import inputs, pages, records_filled, vector

pytestmark = pytest.mark.gpu
D = 128


class _Counting:
    """pla.decode._C with a record of what each offered call answered."""

    def __init__(self):
        self.answers = []

    def __getattr__(self, name):
        def offered(*args):
            self.answers.append(getattr(_C, name)(*args))
            return self.answers[-1]
        return offered


def _ring_step(index_dtype, onorm):
    w = kda_replay_verify(5, 6, 4, seed=33, onorm=onorm, strided=False, index_dtype=index_dtype, pad_rows=(3,))
    out = ring.fused_kda_decode_mtp_dspark(**w)
    spec = types.SimpleNamespace(
        temporal=w["recurrent_state"][None], conv=[w[k][None] for k in ("cs_q", "cs_k", "cs_v")],
        intermediate_conv_window=[w["intermediate_conv_" + k][None] for k in "qkv"],
        **{k: w[k][None] for k in ("replayssm_rawv", "replayssm_rawk", "replayssm_g", "replayssm_beta")})
    accepted = torch.tensor([4, 0, 2, 3, 1], dtype=torch.int32, device="cuda")
    ring.commit_kda_replayssm_after_verify(spec_state=spec, state_batch_indices=w["ssm_state_indices"].int(),
                                           accept_lens=accepted, last_correct_step_indices=accepted.long() - 1)
    return [out, *(w[k] for k in sorted(w) if torch.is_tensor(w[k]))]


def _strided_ring_verify(index_dtype, copied_weight):
    """Mixed rows, transposed conv pools and window segments as SGLang passes them."""
    w = kda_replay_verify(4, 3, 5, seed=35, onorm=True, strided=True, index_dtype=index_dtype, pad_rows=(1,))
    if copied_weight:
        w["w_k"] = w["w_k"].t().contiguous().t()
    return [ring.fused_kda_decode_mtp_dspark(**w), *(w[k] for k in sorted(w) if torch.is_tensor(w[k]))]


def _aligned_step(layout, table_dtype, mapped):
    """Two layers, verify and a commit in align mode: boundary snapshots, a conflict, request rows mapped onto sampler rows."""
    gen = torch.Generator().manual_seed(18)
    layers = [pages(14, 2, 3, layout, gen) for _ in range(2)]
    x = inputs(2, 12, gen)
    x.pop("storage")
    offsets, slots = vector([0, 3, 5, 6, 9]), vector([5, 9, 2, 11])
    outs = []
    for layer in layers:
        layer.kv_cache, layer.replay_records = (layer.conv, layer.state), records_filled(4, 2, 3)
        outs.append(paged.kda_replay_verify(**x, conv_state=layer.conv, checkpoint_state=layer.state, records=layer.replay_records,
                                            query_start_loc=offsets, state_indices=slots, conv_state_layout=layout)[:9])
    context = paged.KDAReplayCommitContext.create(layers, 3, 4, layout, 0)
    rows = [3, 2, 1, 0] if mapped else [0, 1, 2, 3]
    at = lambda values: [values[rows.index(i)] for i in range(4)]                        # sampler order
    table = torch.zeros(4, 6, dtype=table_dtype, device="cuda")[:, ::2]                  # rows and columns with a stride
    table.copy_(torch.tensor(at([[5, 6, 7], [8, 9, 1], [3, 3, 4], [10, 12, 13]])))
    plan = context.commit(vector(at([3, 2, 1, 2])), slots, offsets, vector(rows) if mapped else None, table,
                          vector(at([2, 4, 3, 1]), table_dtype), 4, token_capacity=12)
    assert [t.tolist() for t in vars(plan).values()] == [[3, 2, 1, 2], [6, 9, 3, 10], [5, 0, 3, 0], [2, 0, 1, 0]]
    return [*outs, *(t for layer in layers for t in (layer.raw, *vars(layer.replay_records).values())), *vars(plan).values()]


def _paged_step(layout, index_dtype, strided):
    gen = torch.Generator().manual_seed(8)
    layer = pages(6, 4, 5, layout, gen)
    x = inputs(4, 12, gen)
    x.pop("storage")
    rec = records_filled(3, 4, 5)
    layer.kv_cache, layer.replay_records = (layer.conv, layer.state), rec
    offsets, slots = vector([0, 5, 7, 12], index_dtype, strided), vector([4, 0, 2], index_dtype, strided)
    out = paged.kda_replay_verify(**x, conv_state=layer.conv, checkpoint_state=layer.state, records=rec,
                                  query_start_loc=offsets, state_indices=slots, conv_state_layout=layout)
    context = paged.KDAReplayCommitContext.create([layer], 5, 3, layout, 0)
    plan = context.commit(vector([3, 2, 5], index_dtype, strided), slots, offsets, token_capacity=12)
    return [out[:5], out[7:], layer.raw, *vars(rec).values(), *vars(plan).values()]


@pytest.mark.parametrize("step,args,taken", [
    (_ring_step, (torch.int32, False), [True, True]),
    (_ring_step, (torch.int64, True), [True, True]),
    (_paged_step, ("SD", torch.int32, False), [True, True]),
    (_paged_step, ("DS", torch.int64, False), [True, False]),          # the fold takes 32-bit source slots: a copy
    (_paged_step, ("DS", torch.int32, True), [False, False]),          # strided index vectors: copies
    (_strided_ring_verify, (torch.int64, False), [True]),
    (_strided_ring_verify, (torch.int32, True), [False]),              # a conv weight that needs a copy
    (_aligned_step, ("SD", torch.int32, False), [True, True, True]),
    (_aligned_step, ("DS", torch.int64, True), [True, True, True]),
])
def test_both_host_layers_leave_the_same_bits(monkeypatch, step, args, taken):
    native = _Counting()
    for module in (ring, paged):
        monkeypatch.setattr(module, "_compiled", lambda: native)
    got = step(*args)
    assert native.answers == taken
    for module in (ring, paged):
        monkeypatch.setattr(module, "_compiled", lambda: False)
    want = step(*args)
    torch.cuda.synchronize()
    for a, b in zip(got, want):
        assert torch.equal(a.cpu().view(torch.uint8) if a.is_contiguous() else a.cpu(), b.cpu().view(torch.uint8) if b.is_contiguous() else b.cpu())


def _ring_call():
    return ring.fused_kda_decode_mtp_dspark, dict(kda_replay_verify(3, 4, 3, seed=2, strided=False),
                                                  out=torch.zeros(1, 9, 4, D, dtype=torch.bfloat16, device="cuda"))


def _ring_commit_call():
    w = kda_replay_verify(3, 4, 3, seed=2, strided=False, onorm=False)
    return ring.commit_kda_replayssm_after_verify, dict(
        temporal=w["recurrent_state"][None], **{k: w[k][None] for k in ("replayssm_rawv", "replayssm_rawk", "replayssm_g", "replayssm_beta")},
        conv=[w[k][None] for k in ("cs_q", "cs_k", "cs_v")],
        intermediate_conv_window=[w["intermediate_conv_" + k][None] for k in "qkv"],
        state_batch_indices=w["ssm_state_indices"], accept_lens=vector([1, 3, 2]), last_correct_step_indices=vector([0, 2, 1]))


def _paged_call():
    gen = torch.Generator().manual_seed(3)
    layer, x = pages(6, 2, 3, "DS", gen), inputs(2, 12, gen)
    x.pop("storage")
    return paged.kda_replay_verify, dict(x, conv_state=layer.conv, checkpoint_state=layer.state, records=records_filled(4, 2, 3),
                                         query_start_loc=vector([0, 3, 5, 6]), state_indices=vector([4, 1, 2]), conv_state_layout="DS",
                                         out=torch.zeros(12, 256, dtype=torch.bfloat16, device="cuda"))


def _paged_commit_call():
    layer = pages(6, 2, 3, "DS", torch.Generator().manual_seed(3))
    layer.kv_cache, layer.replay_records = (layer.conv, layer.state), records_filled(4, 2, 3)
    context = paged.KDAReplayCommitContext.create([layer], 3, 4, "DS", 0)
    return context.commit, dict(num_sampled=vector([1, 3, 2]), state_indices=vector([4, 1, 2]), query_start_loc=vector([0, 3, 5, 6]),
                                token_capacity=12)


def _every_other(t):
    return torch.zeros(*t.shape[:-1], 2 * t.shape[-1], dtype=t.dtype, device="cuda")[..., ::2]


def _shifted(t):
    return torch.zeros(t.numel() + 1, dtype=t.dtype, device="cuda")[1:].view(t.shape)


def _records(**changes):
    return lambda a: dict(records=dataclasses.replace(a["records"], **{k: f(getattr(a["records"], k)) for k, f in changes.items()}))


def _with(**changes):
    return lambda a: {k: f(a[k]) if callable(f) else f for k, f in changes.items()}


_short, _narrow, _cpu, _float = (lambda t: t[:-1]), (lambda t: t[:, :-1]), (lambda t: t.cpu()), (lambda t: t.float())
_half, _double = (lambda t: t.half()), (lambda t: t.double())
REFUSED = [(call, change) for call, changes in [
    (_ring_call, [
        _with(recurrent_state=lambda t: t.bfloat16()), _with(recurrent_state=_shifted), _with(recurrent_state=_short),
        _with(replayssm_rawv=lambda t: t[:, :, :2]), _with(replayssm_rawk=_half), _with(replayssm_g=_half), _with(replayssm_g=_every_other),
        _with(replayssm_beta=lambda t: t[:, :, :-1]), _with(replayssm_beta=_every_other),
        _with(x_q=_half), _with(x_k=_narrow), _with(x_v=_every_other), _with(g=_every_other), _with(g=_float),
        _with(beta=_float), _with(beta=_every_other), _with(w_q=_short), _with(w_k=_double), _with(A_log=_short), _with(dt_bias=_double),
        _with(cs_q=_short), _with(cs_v=_float), _with(cs_k=lambda t: t[..., :1].expand(-1, -1, 3)),
        _with(intermediate_conv_q=_float), _with(intermediate_conv_k=lambda t: t[:, :2]), _with(intermediate_conv_v=lambda t: t[..., :2]),
        _with(intermediate_conv_q=lambda t: t[..., :1].expand(-1, -1, -1, 3)),
        _with(ssm_state_indices=_short), _with(ssm_state_indices=_float), _with(ssm_state_indices=_cpu),
        _with(intermediate_state_indices=lambda t: t[:2]), _with(intermediate_state_indices=_cpu),
        _with(cu_seqlens=lambda t: vector([0, 2, 4, 6, 9])), _with(cu_seqlens=_cpu), _with(cu_seqlens=_float),
        _with(out=_half), _with(out=_every_other),
        _with(onorm_gate=_narrow), _with(onorm_gate=_every_other), _with(onorm_weight=_half), _with(onorm_weight=_short),
        _with(onorm_eps=float("nan")), _with(onorm_eps=-1.0)]),
    (_ring_commit_call, [
        _with(temporal=lambda t: t.bfloat16()), _with(replayssm_rawv=lambda t: t[:, :, :1]), _with(replayssm_rawk=_float),
        _with(replayssm_g=_half), _with(replayssm_g=_every_other), _with(replayssm_beta=_every_other),
        _with(accept_lens=lambda t: t.long()), _with(accept_lens=_short), _with(state_batch_indices=lambda t: t.long()),
        # from here on the fold is valid: both layers run it and then refuse the conv rollback
        _with(last_correct_step_indices=None), _with(last_correct_step_indices=_short), _with(last_correct_step_indices=_float),
        _with(last_correct_step_indices=_cpu), _with(conv=lambda c: c[:2]),
        _with(conv=lambda c: [t.half() for t in c], intermediate_conv_window=lambda c: [t.half() for t in c]),
        _with(conv=lambda c: [t.float() for t in c]), _with(conv=lambda c: [_every_other(t) for t in c]),
        _with(conv=lambda c: [t[..., :2].contiguous() for t in c])]),
    (_paged_call, [
        _with(null_block_id=3), _with(conv_state_layout="XX"), _with(checkpoint_state=lambda t: t.bfloat16()),
        _with(checkpoint_state=_every_other), _with(conv_state=_short), _with(conv_state=_half), _with(conv_state=_narrow),
        _with(conv_state=lambda t: t[..., :2]), _with(conv_state=lambda t: t[:, :, :1].expand(-1, -1, 5)),
        _with(mixed_qkv=_narrow), _with(mixed_qkv=_float), _with(mixed_qkv=_every_other), _with(raw_g=_short), _with(raw_g=_every_other),
        _with(raw_beta=_float), _with(conv_weight=lambda t: t.t().contiguous().t()), _with(conv_weight=_double), _with(A_log=_double),
        _with(dt_bias=_short), _with(out=_half), _with(out=_every_other), _with(out=_short),
        _with(lower_bound=0.0), _with(lower_bound=float("nan")), _with(lower_bound=float("-inf")), _with(scale=float("inf")),
        _with(query_start_loc=_short), _with(query_start_loc=_cpu), _with(state_indices=_float), _with(state_indices=lambda t: t[None]),
        _with(query_start_loc=lambda t: vector([0, 1, 2, 3, 4, 5]), state_indices=lambda t: vector([4, 1, 2, 3, 5])),
        _records(g=_half), _records(beta=lambda t: t[:, :1]), _records(rawk=lambda t: t.transpose(1, 2).contiguous().transpose(1, 2)),
        _records(rawv=_shifted), _records(conv=_float), _records(conv=_short),
        lambda a: dict(out=a["records"].rawv.view(12, 256)), lambda a: dict(records=dataclasses.replace(a["records"], rawk=a["records"].rawv))]),
    (_paged_commit_call, [
        _with(token_capacity=-1), _with(token_capacity=2 ** 31), _with(num_sampled=_cpu), _with(num_sampled=_short), _with(num_sampled=_float),
        _with(query_start_loc=_short), _with(state_indices=_float), _with(state_indices=lambda t: vector([4, 1, 2, 3, 5]),
                                                                          query_start_loc=lambda t: vector([0, 1, 2, 3, 4, 5])),
        lambda a: dict(request_indices=vector([0, 1])), lambda a: dict(request_indices=vector([0, 1, 2]).float()),
        *(lambda a, table=table, computed=computed: dict(block_table=table(), num_computed_tokens=computed(), mamba_block_size=4)
          for table, computed in [(lambda: vector([1, 2, 3]), lambda: vector([0, 0, 0])),
                                  (lambda: torch.ones(3, 2, device="cuda"), lambda: vector([0, 0, 0])),
                                  (lambda: torch.ones(3, 2, dtype=torch.int32), lambda: vector([0, 0, 0])),
                                  (lambda: torch.ones(3, 2, dtype=torch.int32, device="cuda"), lambda: vector([0, 0]))])])] for change in changes]


@pytest.mark.parametrize("index", range(len(REFUSED)))
def test_both_host_layers_refuse_the_same_calls(monkeypatch, index):
    """One argument changed: the compiled layer leaves the call to the facade, which words the error, and what the call
    would have written is left alike."""
    make, change = REFUSED[index]
    seen = []
    for native in (_Counting(), False):
        for module in (ring, paged):
            monkeypatch.setattr(module, "_compiled", lambda: native)
        entry, args = make()
        args.update(change(args))
        if make is _ring_commit_call:
            names = ("temporal", "replayssm_rawv", "replayssm_rawk", "replayssm_g", "replayssm_beta", "conv", "intermediate_conv_window")
            spec = types.SimpleNamespace(**{k: args.pop(k) for k in names})
            args["spec_state"] = spec
        with pytest.raises((RuntimeError, ValueError, AssertionError)) as error:
            entry(**args)
        torch.cuda.synchronize()
        if native:
            assert native.answers in ([False], []), "the compiled layer took a call that the facade refuses"
        after = [args.get("out"), args.get("recurrent_state"), *vars(args.get("records", types.SimpleNamespace())).values()]
        if make is _ring_commit_call:
            after += [spec.temporal, *spec.conv]
        seen.append((error.type, str(error.value), [t.cpu() for t in after if t is not None]))
    assert seen[0][:2] == seen[1][:2]
    assert all(torch.equal(a, b) for a, b in zip(seen[0][2], seen[1][2]))


@pytest.mark.parametrize("layout", ["dense", "tap_major", "mixed", "interleaved", "shifted", "overlapping"])
@pytest.mark.parametrize("heads,dtype,index_dtype", [(1, torch.bfloat16, torch.int32), (4, torch.bfloat16, torch.int64),
                                                     (2, torch.float32, torch.int32)])
def test_conv_rollback_of_three_pools(layout, heads, dtype, index_dtype):
    """Pools that roll back in one launch of 16-byte pieces (dense, tap_major), in one launch by channel (mixed, shifted)
    and in a launch each (interleaved, overlapping): every pool is the oracle's, bit for bit."""
    layers, slots, rows, steps, dim = 2, 7, 5, 4, heads * D
    g = torch.Generator().manual_seed(heads)

    def filled(shape):
        return torch.randn(*shape, generator=g).to(dtype).cuda()

    if layout == "tap_major":
        conv = [filled((layers, slots, 3, dim)).transpose(-1, -2) for _ in range(3)]
    elif layout == "shifted":                            # bases off the 16-byte boundary
        conv = [filled((layers * slots * dim * 3 + 1,))[1:].view(layers, slots, dim, 3) for _ in range(3)]
    else:
        conv = [filled((layers, slots, dim, 3)) for _ in range(3)]
    if layout in ("tap_major", "mixed"):
        windows = [filled((layers, rows, steps, 3, dim)).transpose(-1, -2) for _ in range(3)]
    elif layout == "interleaved":                        # one tensor of all channels
        windows = list(filled((layers, rows, steps, 3 * dim, 3)).split(dim, dim=3))
    else:
        windows = [filled((layers, rows, steps, dim, 3)) for _ in range(3)]
    if layout == "overlapping":
        conv[2] = conv[0]                                # the last pool's windows win
    indices = torch.tensor([4, -1, 0, 6, 2], dtype=index_dtype)
    last = torch.tensor([3, 2, -1, 0, 1], dtype=index_dtype)
    want = [c.cpu().clone() for c in conv]
    for i in range(3):
        want[i] = conv_window_scatter_reference(want[i] if i < 2 or layout != "overlapping" else want[0], windows[i].cpu(), indices, last)
    if layout == "overlapping":
        want[0] = want[2]
    state = torch.zeros(layers, slots, heads, D, D, device="cuda")
    rec = torch.zeros(layers, slots, heads, 8, D, device="cuda")
    spec = types.SimpleNamespace(temporal=state, replayssm_rawv=rec.bfloat16(), replayssm_rawk=rec.bfloat16(), replayssm_g=rec,
                                 replayssm_beta=rec[..., 0].contiguous(), conv=conv, intermediate_conv_window=windows)
    ring.commit_kda_replayssm_after_verify(spec_state=spec, state_batch_indices=indices.int().cuda(), accept_lens=last.int().cuda() + 1,
                                           last_correct_step_indices=last.cuda())
    torch.cuda.synchronize()
    for c, expected in zip(conv, want):
        assert torch.equal(c.cpu(), expected)
