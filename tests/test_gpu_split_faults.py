"""Hand-off failures of the sequence split and of the training outputs fail
closed: NaN where a block's results, or the start state they are chained from,
are not trustworthy, and the caller's state untouched whichever block of its
sequence and head failed, so that the step can be run again.

The failures are forced from the host: a spin limit of zero polls (every
block's first wait gives up), or key waves of chosen blocks that never publish
their operators.  Every kernel still runs to its end."""

from __future__ import annotations

import numpy as np
import pytest
import torch

import test_gpu_statetune as st
from wkv7_testlib import (
    assert_output_close,
    assert_state_close,
    make_case,
    oracle_expect,
    require_gpu,
    to_np,
    tokens,
)

pytestmark = pytest.mark.gpu

from flashrwkv2_amd.tmix.wkv7 import (  # noqa: E402
    prepare_tmix_wkv7_recurrent_metadata,
    pretrain_tmix_wkv7_recurrent_bf16,
    statetune_tmix_wkv7_recurrent_fp32io16,
)

SPLIT = 3
LATER, SUMMARIES = 2, 3     # _set_handoff_stall: the blocks that stall


class _Forced:
    """The spin limit and the stalled blocks, restored at the end."""

    def __init__(self, polls, stall=0):
        self.polls, self.stall = polls, stall

    def __enter__(self):
        C = require_gpu()
        C.handoff_fault_count(reset=True)
        C._set_handoff_spin_limit(self.polls)
        C._set_handoff_stall(self.stall)

    def __exit__(self, *exc):
        C = require_gpu()
        torch.cuda.synchronize()
        C._set_handoff_stall(0)
        C._set_handoff_spin_limit(-1)


def _split(case, pool, pieces):
    """The split on an fp32 or bf16 pool; and the run again after the failure."""
    C = require_gpu()
    if pool.dtype == torch.bfloat16:
        C._chunk_split_pieces = pieces
        try:
            return C.infer_tmix_wkv7_chunk_bf16_forward_varlen(
                *tokens(case), state_pool=pool, cu_seqlens=case["cu_seqlens"],
                state_indices=case["state_indices"],
                max_seqlen=int(case["cu_seqlens"].diff().max()))[0]
        finally:
            C._chunk_split_pieces = None
    ticket = prepare_tmix_wkv7_recurrent_metadata(
        case["cu_seqlens"], case["state_indices"], total_tokens=case["r"].shape[0],
        state_pool_size=pool.shape[0])
    out = torch.empty_like(case["v"])
    C.tmix_wkv7_recurrent_fp32_kernel_forced(
        SPLIT, case["cu_seqlens"], case["state_indices"], pool, *tokens(case), out, 1.0, None,
        ticket, split_pieces=pieces)
    return out


def _bounds(lengths, plan):
    """Token rows (lo, hi) of every sequence's pieces."""
    _, plen, lead, _ = plan
    first, rows, at = lead or plen, [], 0
    for n in lengths:
        cuts = [0, *range(first, n, plen), n]
        rows.append([(at + lo, at + hi) for lo, hi in zip(cuts, cuts[1:])])
        at += n
    return rows


CASES = [
    ((700, 64, 1, 129, 1024), (4, 320), torch.float32),   # one to four pieces
    ((700, 64, 1, 129, 1024), 4, torch.bfloat16),
    ((200, 96), (2, 112), torch.float32),                 # no summary
]


@pytest.mark.parametrize("lengths,pieces,dtype", CASES)
def test_every_wait_gives_up(lengths, pieces, dtype):
    C = require_gpu()
    print(f"case split, spin limit 0, {lengths} {pieces} {dtype}", flush=True)
    H = 2
    case = make_case(lengths=lengths, num_heads=H, seed=5)
    pool = case["state_pool"].to(dtype)
    before = pool.clone()
    rows = _bounds(lengths, C.split_plan(len(lengths), H, 64, max(lengths), pieces))
    with _Forced(0):
        out = _split(case, pool, pieces)
    # first pieces and summaries count; the later pieces fail with them
    assert C.handoff_fault_count(reset=True) == H * sum(1 + max(0, len(r) - 2) for r in rows)
    assert torch.isnan(out.float()).all() and torch.equal(pool, before)
    y_ref, pool_ref = oracle_expect(case, state_pool=before)
    assert_output_close(_split(case, pool, pieces), y_ref)
    active = case["state_indices"].long()
    assert_state_close(pool[active], pool_ref[active.cpu().numpy()],
                       **({} if dtype == torch.float32 else {"rmse": 4e-3, "fro": 8e-3}))
    assert C.handoff_fault_count(reset=True) == 0


@pytest.mark.parametrize("lengths,pieces,dtype", CASES[:2])
def test_summaries_give_up(lengths, pieces, dtype):
    """The pieces chained over a failed summary are NaN and their sequence's state
    is untouched; the pieces before, and sequences without one, are right."""
    C = require_gpu()
    print(f"case split, summaries stalled, {lengths} {pieces} {dtype}", flush=True)
    H = 2
    case = make_case(lengths=lengths, num_heads=H, seed=6)
    pool = case["state_pool"].to(dtype)
    before = pool.clone()
    y_ref, pool_ref = oracle_expect(case, state_pool=before)
    rows = _bounds(lengths, C.split_plan(len(lengths), H, 64, max(lengths), pieces))
    with _Forced(20000, SUMMARIES):
        out = _split(case, pool, pieces)
    assert C.handoff_fault_count(reset=True) == H * sum(max(0, len(r) - 2) for r in rows)
    slots = case["state_indices"].tolist()
    for slot, pcs in zip(slots, rows):
        good = pcs[:2][-1][1]
        assert_output_close(out[pcs[0][0]:good], y_ref[pcs[0][0]:good])
        assert torch.isnan(out[good:pcs[-1][1]].float()).all()
        if len(pcs) > 2:
            assert torch.equal(pool[slot], before[slot])
        else:
            assert_state_close(pool[slot:slot + 1], pool_ref[slot:slot + 1],
                               **({} if dtype == torch.float32 else {"rmse": 4e-3, "fro": 8e-3}))
    idle = [i for i in range(pool.shape[0]) if i not in slots]
    assert torch.equal(pool[idle], before[idle])


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("polls", [500, 20000])
def test_a_middle_piece_gives_up_before_and_after_the_last_one_stored(polls, dtype):
    """Pieces 1 and 2 of four give up after about 50 us and 2 ms, the last one of
    4 096 tokens takes about 0.3 ms: the state is untouched either way."""
    C = require_gpu()
    print(f"case split, middle pieces stalled, {polls} polls {dtype}", flush=True)
    lengths, pieces, H = (16384, 600), (4, 4096), 1
    case = make_case(lengths=lengths, num_heads=H, seed=7)
    pool = case["state_pool"].to(dtype)
    before = pool.clone()
    y_ref, pool_ref = oracle_expect(case, state_pool=before)
    (pcs, short) = _bounds(lengths, C.split_plan(2, H, 64, max(lengths), pieces))
    assert len(pcs) == 4 and len(short) == 1
    with _Forced(polls, LATER):
        out = _split(case, pool, pieces)
    assert C.handoff_fault_count(reset=True) == 2
    assert torch.isnan(out[pcs[1][0]:pcs[2][1]].float()).all()
    assert torch.isfinite(out[:pcs[0][1]].float()).all()
    assert_output_close(out[pcs[3][0]:], y_ref[pcs[3][0]:])   # the last piece, the short one
    slots = case["state_indices"].tolist()
    assert torch.equal(pool[slots[0]], before[slots[0]])
    s = slots[1]
    assert_state_close(pool[s:s + 1], pool_ref[s:s + 1],
                       **({} if dtype == torch.float32 else {"rmse": 4e-3, "fro": 8e-3}))


@pytest.mark.parametrize("batch,tokens_,heads", [(1, 512, 1), (2, 1040, 3), (2, 64, 160)])
def test_training_passes_give_up(batch, tokens_, heads):
    """Split and whole: y and sa, then dv, are NaN, and so is the loss's gradient."""
    C = require_gpu()
    from flashrwkv2_amd import _native as N

    print(f"case training fault B={batch} T={tokens_} H={heads}", flush=True)
    floats = N.load().fr2_wkv7_pretrain_split_workspace_floats(batch, tokens_, heads, 64)
    assert (floats > 0) == (batch * heads < 128)
    g = torch.Generator().manual_seed(tokens_)
    shape = (batch, tokens_, heads * 64)
    vals = [(torch.randn(shape, generator=g) * 0.1).to(torch.bfloat16).cuda().requires_grad_()
            for _ in range(6)]
    heads_of = [t.detach().view(batch, tokens_, heads, 64) for t in vals]
    y = torch.zeros_like(heads_of[3])
    bnd = torch.empty((batch, heads, tokens_ // 16, 64, 64), device="cuda")
    sa = torch.zeros(y.shape, device="cuda")
    with _Forced(0):
        C.pretrain_tmix_wkv7_recurrent_forward(*heads_of, y, bnd, sa, 64)
    assert C.handoff_fault_count(reset=True) >= batch * heads
    assert torch.isnan(y.float()).all() and torch.isnan(sa).all()
    y = pretrain_tmix_wkv7_recurrent_bf16(*vals, head_size=64)
    torch.cuda.synchronize()
    assert C.handoff_fault_count(reset=True) == 0 and torch.isfinite(y.float()).all()
    with _Forced(0):
        y.backward(torch.ones_like(y))
    assert C.handoff_fault_count(reset=True) >= batch * heads
    assert torch.isnan(vals[3].grad.float()).all()


@pytest.mark.parametrize("heads", [2, 96])
def test_row_blocks_give_up(heads):
    """Chunks out of row order, short blocks, a sequence without tokens: NaN in the
    rows of the list and no others, the state as it was, and in the backward NaN
    for dv and the initial state's gradient."""
    C = require_gpu()
    print(f"case row blocks fault H={heads}", flush=True)
    offsets, lens = [0, 3, 3, 5], [700, 3, 601, 20, 1]
    starts, at = [0] * 5, 0
    for c in (3, 0, 4, 2, 1):
        starts[c] = at + 1
        at += 1 + lens[c]
    meta = st._meta(offsets, starts, [s + n for s, n in zip(starts, lens)])
    used = torch.zeros(at, dtype=torch.bool)
    for s, n in zip(starts, lens):
        used[s:s + n] = True
    used = used.cuda()
    g = torch.Generator().manual_seed(heads)
    vals = st._structured(at, heads, 64, torch.bfloat16, g)
    state0 = torch.randn((3, heads, 64, 64), generator=g).cuda()
    state, y = state0.clone(), torch.zeros_like(vals[3])
    sa = torch.zeros(y.shape, device="cuda")
    bnd = torch.empty((5, heads, 64, 64), device="cuda")
    with _Forced(0):
        C.statetune_tmix_wkv7_recurrent_fp32io16_forward(*meta, state, *vals, y, bnd, sa, 1.0)
    assert C.handoff_fault_count(reset=True) >= 2 * heads
    for x in (y.float(), sa):
        assert torch.isnan(x[used]).all() and (x[~used] == 0).all()
    assert torch.equal(state, state0)
    leaves = [t.requires_grad_() for t in vals]
    init = state0.clone().requires_grad_()
    y, final, _, _ = statetune_tmix_wkv7_recurrent_fp32io16(init, *meta, *leaves)
    torch.cuda.synchronize()
    assert C.handoff_fault_count(reset=True) == 0
    assert np.isfinite(to_np(y[used])).all()
    with _Forced(0):
        torch.autograd.backward([y, final], [torch.ones_like(y), torch.ones_like(final)])
    assert C.handoff_fault_count(reset=True) >= 2 * heads
    assert torch.isnan(vals[3].grad[used].float()).all()
    assert torch.isnan(init.grad[[0, 2]]).all()
    assert torch.equal(init.grad[1], torch.ones_like(final[1]))   # a sequence without tokens
