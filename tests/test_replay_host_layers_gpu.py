"""The replay entry points offer each call to the compiled host layer first: ordinary calls are taken there, calls that
need a copy or fail a check are not, and both layers leave the same bits everywhere."""
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
