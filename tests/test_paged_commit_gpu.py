"""The paged commit, in one launch or with its plan ahead, against plan, fold and conv windows in three, bit for bit (the arithmetic
of a tile is the same), on both sides of the line between them; and the plan of large batches, whose look-ups are spread over workgroups, against
the oracle."""
import pytest
import torch

from test_replay_vllm_gpu import inputs, pages, records_filled, vector

pytestmark = pytest.mark.gpu
BLOCK = 8


def _context(requests, heads, q, n_layers, layout, capacity, seed):
    from pla_amd.decode.kda_replayssm_vllm import KDAReplayCommitContext, kda_replay_verify
    gen = torch.Generator().manual_seed(seed)
    slots = requests + requests // 2 + 3
    layers = [pages(slots, heads, q, layout, gen) for _ in range(n_layers)]
    x = {k: v for k, v in inputs(heads, requests * q, gen).items() if k != "storage"}
    source = (1 + torch.randperm(slots - 1, generator=gen)[:requests]).tolist()
    offsets = list(range(0, requests * q + 1, q))
    for layer in layers:
        layer.replay_records = records_filled(capacity, heads, q)
        layer.kv_cache = (layer.conv, layer.state)
        kda_replay_verify(**x, conv_state=layer.conv, checkpoint_state=layer.state, records=layer.replay_records,
                          query_start_loc=vector(offsets), state_indices=vector(source), conv_state_layout=layout, null_block_id=0)
    return KDAReplayCommitContext.create(layers, q, capacity, layout, 0), layers, source, offsets, slots, gen


def _wide(t):
    return int(t is not None and t.dtype == torch.int64)


def _three_launches(ctx, sampled, source, offsets, mapping, table, computed, tokens):
    from pla_amd import _lib
    N, R, layers = source.numel(), ctx._capacity, ctx._table.shape[0]
    scratch, plan = torch.full((4, R), -9, dtype=torch.int32, device="cuda"), torch.full((4, R), -9, dtype=torch.int32, device="cuda")
    stream, ptr = torch.cuda.current_stream().cuda_stream, lambda t: None if t is None else t.data_ptr()
    rows, cols = (0, 0) if table is None else table.shape
    _lib.call("pla_kda_commit_plan_launch", sampled.data_ptr(), _wide(sampled), source.data_ptr(), 0, offsets.data_ptr(), _wide(offsets),
              ptr(mapping), _wide(mapping), ptr(computed), _wide(computed), ptr(table), _wide(table), N, R, sampled.numel(),
              rows, cols, ctx._slots, ctx._q, 0, tokens, cols,
              0 if table is None else 1, 0 if table is None else BLOCK, scratch.data_ptr(), plan.data_ptr(), stream)
    rows4 = [plan[c].data_ptr() for c in range(4)]
    _lib.call("pla_kda_fold_native_launch", ctx._table.data_ptr(), layers, source.data_ptr(), *rows4, N, ctx._heads, ctx._q,
              ctx._slots, 0, stream)
    _lib.call("pla_kda_conv_native_launch", ctx._table.data_ptr(), layers, *rows4, N, ctx._channels, ctx._q, ctx._rows,
              ctx._slots, stream)
    return plan


# one request; few tiles (8 rows per wavefront) and more (16 rows); more requests than threads of a workgroup; the largest
# number of tiles of one launch, and one request more than that; beyond it the conv windows stand behind the tiles of the fold, with 16
# and with 32 rows per wavefront, in both layouts, with whole workgroups of channels and with a remainder
@pytest.mark.parametrize("requests,heads,q,n_layers,layout,capacity", [
    (1, 1, 1, 1, "SD", 1), (5, 3, 4, 2, "DS", 9), (17, 6, 8, 2, "SD", 20), (260, 1, 2, 1, "DS", 300), (20, 8, 3, 2, "SD", 20),
    (21, 8, 3, 2, "SD", 21), (115, 3, 4, 1, "DS", 120), (64, 8, 3, 2, "SD", 64), (180, 3, 2, 1, "SD", 181), (70, 4, 8, 2, "DS", 70)])
@pytest.mark.parametrize("mode", ["plain", "mapping", "align", "mapping 64 bits", "align 64 bits"])
def test_commit_in_one_launch_equals_three(requests, heads, q, n_layers, layout, capacity, mode):
    from pla_amd import _lib
    assert _lib.load().pla_kda_commit_launches(requests, heads, n_layers) == (3 if requests * heads * n_layers > 320 else 1)
    mode, dtype = mode.split()[0], torch.int64 if "64" in mode else torch.int32
    ctx, layers, source, offsets, slots, gen = _context(requests, heads, q, n_layers, layout, capacity, 31 + requests)
    ri = lambda lo, hi, n: torch.randint(lo, hi, (n,), generator=gen)
    sampled = vector(ri(0, q + 2, requests + 2).tolist(), dtype)
    if requests > 16:                                            # no slot, a slot beyond the pool, two requests of one slot
        source[1], source[2], source[4] = 0, slots + 5, source[3]
    d_source, d_offsets = vector(source), vector(offsets, dtype)
    mapping = vector(ri(-1, requests + 3, requests).tolist(), dtype) if mode == "mapping" else None
    table = computed = None
    kw = {}
    if mode == "align":                                          # the blocks of a request: its source, then free or foreign slots
        free = [s for s in range(1, slots) if s not in source]
        cells = [[source[b] if 0 < source[b] < slots else 1, free[b % len(free)], (7 * b) % slots] for b in range(requests)]
        table = torch.tensor(cells + [[1, 2, 3]] * 2, dtype=dtype, device="cuda")
        computed = vector(ri(0, 2 * BLOCK, requests + 2).tolist(), dtype)
        kw = dict(block_table=table, num_computed_tokens=computed, mamba_block_size=BLOCK)
    before = [(layer.state.clone(), layer.conv.clone()) for layer in layers]
    want_plan = _three_launches(ctx, sampled, d_source, d_offsets, mapping, table, computed, offsets[-1])
    want = [(layer.state.clone(), layer.conv.clone()) for layer in layers]
    assert requests < 17 or (want_plan[0] > 0).any()

    def one_call():
        ptr = lambda t: None if t is None else t.data_ptr()
        grid, cols = (table.shape, table.shape[1]) if table is not None else ((0, 0), 0)
        _lib.call("pla_kda_commit_launch", ctx._table.data_ptr(), n_layers, heads, ctx._channels, ctx._rows, sampled.data_ptr(),
                  _wide(sampled), d_source.data_ptr(), d_offsets.data_ptr(), _wide(d_offsets), ptr(mapping), _wide(mapping),
                  ptr(computed), _wide(computed), ptr(table), _wide(table), requests, capacity, sampled.numel(), *grid, slots, q, 0,
                  offsets[-1], cols, 1 if cols else 0, BLOCK if cols else 0, ctx._candidate.data_ptr(), ctx._buffer.data_ptr(),
                  torch.cuda.current_stream().cuda_stream)
    for commit in (one_call, lambda: ctx.commit(sampled, d_source, d_offsets, request_indices=mapping, token_capacity=offsets[-1], **kw)):
        for layer, (state, conv) in zip(layers, before):
            layer.state.copy_(state)
            layer.conv.copy_(conv)
        ctx._buffer.fill_(-9)
        commit()
        torch.cuda.synchronize()
        assert torch.equal(ctx._buffer, want_plan)
        for layer, (state, conv) in zip(layers, want):
            assert torch.equal(layer.state, state) and torch.equal(layer.conv, conv)


def test_commit_takes_its_sources_from_its_own_plan():
    """The final slots of a commit as the sources of the next: the plan is overwritten while it is an input."""
    ctx, layers, source, offsets, slots, gen = _context(6, 2, 4, 1, "SD", 6, 77)
    args = dict(num_sampled=vector([2, 1, 4, 3, 1, 2]), query_start_loc=vector(offsets), token_capacity=offsets[-1])
    plan = ctx.commit(state_indices=vector(source), **args)
    before = layers[0].state.clone(), layers[0].conv.clone()
    ctx.commit(state_indices=plan.final_state_indices.clone(), **args)
    want = layers[0].state.clone(), layers[0].conv.clone(), ctx._buffer.clone()
    layers[0].state.copy_(before[0])
    layers[0].conv.copy_(before[1])
    ctx.commit(state_indices=plan.final_state_indices, **args)
    assert torch.equal(layers[0].state, want[0]) and torch.equal(layers[0].conv, want[1]) and torch.equal(ctx._buffer, want[2])
    assert plan.final_state_indices.tolist() == source


# every workgroup decides on four requests: batches of one share and of many, the largest whose claims LDS holds and the next
# one, a capacity far above the batch (whose workgroups only clear rows), 64-bit inputs
@pytest.mark.parametrize("batch,capacity,wide", [(1, 1, 0), (4, 5, 0), (5, 9, 1), (300, 5000, 0), (768, 768, 1), (3072, 3072, 0),
                                                 (3073, 3073, 0), (3100, 5003, 1), (4096, 4097, 0)])
@pytest.mark.parametrize("align", [False, True])
def test_commit_plan_of_many_requests_matches_the_oracle(batch, capacity, wide, align):
    from oracle import replay_commit_plan_reference
    from pla_amd import _lib
    gen = torch.Generator().manual_seed(batch + int(align))
    ri = lambda lo, hi, n: torch.randint(lo, hi, (n,), generator=gen)
    slots, q, rows, cols = 40 * batch + 2, 4, batch + 3, 5
    offsets = [0] + ri(1, q + 1, batch).cumsum(0).tolist()
    source = ri(1, slots, batch)
    some = ri(0, batch, batch // 50 + 1)
    source[some] = source[ri(0, batch, batch // 50 + 1)]              # clashes, and slots that do not exist
    source[ri(0, batch, batch // 100)] = slots + 3
    # (few requests commit in a large batch: the oracle compares each of them with every other one)
    sampled = ri(0, q + 2, rows) * (torch.rand(rows, generator=gen) < max(0.02, min(1.0, 100 / batch)))
    computed = ri(0, BLOCK * cols, rows)
    table = ri(1, slots, rows * cols).reshape(rows, cols)
    lists = [t.tolist() for t in (sampled, source, computed, table)]
    want = replay_commit_plan_reference(lists[0], lists[1], offsets, slots=slots, Q=q, token_capacity=offsets[-1], null_block_id=0,
                                        block_table=lists[3] if align else None, num_computed_tokens=lists[2] if align else None,
                                        block_size=BLOCK if align else None, capacity=capacity)
    dtype = torch.int64 if wide else torch.int32
    d_sampled, d_source, d_offsets, d_computed, d_table = (torch.as_tensor(x).to(dtype).cuda() for x in (sampled, source, offsets, computed, table))
    scratch, plan = (torch.full((4, capacity), -9, dtype=torch.int32, device="cuda") for _ in range(2))
    _lib.call("pla_kda_commit_plan_launch", d_sampled.data_ptr(), wide, d_source.data_ptr(), wide, d_offsets.data_ptr(), wide, None, 0,
              d_computed.data_ptr() if align else None, wide, d_table.data_ptr() if align else None, wide, batch, capacity, rows,
              rows if align else 0, cols if align else 0, slots, q, 0, offsets[-1], cols if align else 0, 1 if align else 0,
              BLOCK if align else 0, scratch.data_ptr(), plan.data_ptr(), torch.cuda.current_stream().cuda_stream)
    torch.cuda.synchronize()
    assert plan.cpu().tolist() == want
    assert batch < 50 or sum(n > 0 for n in want[0]) >= 20
