"""The replay entry points offer each call to the compiled host layer first: ordinary calls are taken there, calls that
need a copy or fail a check are not, and both layers leave the same bits everywhere."""
import types

import pytest
import torch

from pla_amd.decode import _C, kda_replayssm_sglang as ring, kda_replayssm_vllm as paged
from pla_amd.workloads import kda_replay_verify
from test_replay_vllm_gpu import inputs, pages, records_filled, vector

pytestmark = pytest.mark.gpu


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
