"""The fp32 chunked kernel of head sizes 128 and 256 (csrc/chunk_wide.hip)
against the fp64 oracle, around its 16-token chunks, its two sets of key waves
(odd and even chunk counts), ragged and one-token segments, decay bias and
scale, and with the training forward's outputs.  Final states meet 1e-6
relative (fp32 sums of at most a few hundred terms, 2^-24 each) and are no
further from fp64 than a token-by-token fp32 evaluation; y meets the gates of
the other kernels (its own 16-bit rounding dominates)."""

from __future__ import annotations

import numpy as np
import pytest
import torch

import oracle
from wkv7_testlib import (
    assert_output_close,
    make_case,
    oracle_expect,
    relative_rmse,
    require_gpu,
    to_np,
    tokens,
)

pytestmark = pytest.mark.gpu

from flashrwkv2_amd.tmix.wkv7 import (  # noqa: E402
    infer_tmix_wkv7_recurrent_fp32io16_forward_varlen as wkv7,
    prepare_tmix_wkv7_recurrent_metadata as prepare,
)

STATE_REL = 1.0e-6


@pytest.mark.parametrize("head_size", [128, 256])
@pytest.mark.parametrize("lengths,heads,dtype", [
    ((16,), 1, torch.bfloat16),              # one whole chunk
    ((17, 15, 31), 2, torch.float16),        # partial last chunks
    ((1, 300, 2, 48, 33), 3, torch.bfloat16),
    ((80, 96), 2, torch.float16),            # five and six chunks
])
def test_wide_heads_match_the_oracle(head_size, lengths, heads, dtype):
    C = require_gpu()
    print(f"case wide D={head_size} lengths={lengths} {dtype}", flush=True)
    assert C.dispatch_kernel_name(len(lengths), heads, head_size, sum(lengths),
                                  max(lengths), dtype).startswith("chunk_wide_kernel")
    case = make_case(dtype=dtype, head_size=head_size, lengths=lengths, num_heads=heads,
                     with_decay_bias=True, seed=head_size + heads)
    before = case["state_pool"].clone()
    y_ref, pool_ref = oracle_expect(case, scale=0.75)
    out = wkv7(*tokens(case), state_pool=case["state_pool"], cu_seqlens=case["cu_seqlens"],
               state_indices=case["state_indices"], decay_bias=case["decay_bias"], scale=0.75)
    torch.cuda.synchronize()
    assert_output_close(out, y_ref)
    active = case["state_indices"].long()
    got = to_np(case["state_pool"][active]).astype(np.float64)
    want = pool_ref[active.cpu().numpy()]
    assert np.linalg.norm(got - want) / np.linalg.norm(want) <= STATE_REL
    idle = [i for i in range(before.shape[0]) if i not in set(active.tolist())]
    assert torch.equal(case["state_pool"][idle], before[idle])


@pytest.mark.parametrize("batch,tokens_,heads,head_size", [(2, 112, 2, 128), (1, 80, 1, 256)])
def test_wide_training_forward_outputs(batch, tokens_, heads, head_size):
    """y, every token's sa and the state after every 16 tokens."""
    C = require_gpu()
    g = torch.Generator().manual_seed(head_size)
    shape = (batch, tokens_, heads, head_size)
    kk = torch.randn(shape, generator=g)
    kk = kk / kk.norm(dim=-1, keepdim=True)
    vals = [torch.randn(shape, generator=g) for _ in range(4)]
    vals += [-kk, kk * torch.sigmoid(torch.randn(shape, generator=g))]
    x = [t.to(torch.bfloat16).cuda() for t in vals]
    y = torch.empty_like(x[3])
    bnd = torch.empty((batch, heads, tokens_ // 16, head_size, head_size), device="cuda")
    sa = torch.empty(shape, device="cuda")
    C.pretrain_tmix_wkv7_recurrent_forward(*x, y, bnd, sa, head_size)
    torch.cuda.synchronize()
    flat = [to_np(t).reshape(batch * tokens_, heads, head_size) for t in x]
    cu = np.arange(0, batch * tokens_ + 1, tokens_, dtype=np.int32)
    y_ref, _, sa_ref, bnd_ref = oracle.wkv7_f64(*flat, cu_seqlens=cu, want_sa=True,
                                                boundary_len=16)
    assert_output_close(y.reshape(flat[0].shape), y_ref)
    assert relative_rmse(to_np(sa).reshape(sa_ref.shape), sa_ref) <= STATE_REL
    assert relative_rmse(to_np(bnd), bnd_ref) <= STATE_REL


@pytest.mark.parametrize("head_size", [128, 256])
def test_wide_rl_infctx_replay(head_size):
    """Chunks from their own start states, with decay bias and scale: y and sa, and
    the start states untouched."""
    C = require_gpu()
    lengths, heads = (33, 17, 64, 1), 2
    assert C.dispatch_kernel_name(len(lengths), heads, head_size, sum(lengths),
                                  0).startswith("chunk_wide_kernel")
    case = make_case(dtype=torch.bfloat16, head_size=head_size, lengths=lengths, num_heads=heads,
                     with_decay_bias=True, seed=head_size + 1)
    g = torch.Generator().manual_seed(head_size)
    starts = torch.randn((len(lengths), heads, head_size, head_size), generator=g).cuda()
    before, cu = starts.clone(), case["cu_seqlens"]
    out, sa = torch.empty_like(case["v"]), torch.empty(case["v"].shape, device="cuda")
    C.rl_infctx_tmix_wkv7_chunk_fp32io16_backward_replay(
        cu[:-1].contiguous(), cu[1:].contiguous(), starts, *tokens(case), out, sa, 0.75,
        case["decay_bias"])
    torch.cuda.synchronize()
    y_ref, _, sa_ref, _ = oracle.wkv7_f64(
        *(to_np(t) for t in tokens(case)), cu_seqlens=to_np(cu),
        state_indices=np.arange(len(lengths), dtype=np.int32), state_pool=to_np(starts),
        decay_bias=to_np(case["decay_bias"]), scale=0.75, want_sa=True)
    assert_output_close(out, y_ref)
    assert relative_rmse(to_np(sa), sa_ref) <= STATE_REL
    assert torch.equal(starts, before)


def _token_serial_f32(x):
    """Final states and sa of [B, T, H, D] inputs from a zero state, token by token
    in fp32 (sums over keys in pairs)."""
    r, logits, k, v, a, b = (t.float() for t in x)
    w = torch.exp(-float(np.exp(-0.5)) * torch.sigmoid(logits))
    B, T, H, D = r.shape
    state = torch.zeros((B, H, D, D), device=r.device)
    sa = torch.empty((B, T, H, D), device=r.device)
    for t in range(T):
        parts = a[:, t, :, :, None] * state
        while parts.shape[2] > 1:
            parts = parts[:, :, 0::2] + parts[:, :, 1::2]
        sa[:, t] = parts[:, :, 0]
        state = w[:, t, :, :, None] * state + (
            b[:, t, :, :, None] * sa[:, t, :, None, :] + k[:, t, :, :, None] * v[:, t, :, None, :])
    return state, sa


@pytest.mark.parametrize("decay", [(-6.0, -0.5), (-9.0, -4.0)])
@pytest.mark.parametrize("head_size", [128, 256])
def test_wide_training_forward_is_as_exact_as_token_by_token(head_size, decay):
    """Errors against fp64 of the state after every 16 tokens and of sa, next to those
    of a token-by-token fp32 evaluation of the same inputs.  Both are sums of
    thousands of roundings, so their size is steady: a quarter more is allowed."""
    C = require_gpu()
    batch, tokens_, heads = 2, 256, 2
    g = torch.Generator().manual_seed(head_size)
    shape = (batch, tokens_, heads, head_size)
    kk = torch.nn.functional.normalize(torch.randn(shape, generator=g), dim=-1)
    p = torch.exp(torch.rand(shape, generator=g) * (decay[1] - decay[0]) + decay[0] + 0.5)
    vals = [torch.randn(shape, generator=g), torch.logit(p.clamp(max=1 - 2.0 ** -23)),
            torch.randn(shape, generator=g), torch.randn(shape, generator=g),
            -kk, kk * torch.sigmoid(torch.randn(shape, generator=g))]
    x = [t.to(torch.bfloat16).cuda() for t in vals]
    y = torch.empty_like(x[3])
    bnd = torch.empty((batch, heads, tokens_ // 16, head_size, head_size), device="cuda")
    sa = torch.empty(shape, device="cuda")
    C.pretrain_tmix_wkv7_recurrent_forward(*x, y, bnd, sa, head_size)
    serial_state, serial_sa = _token_serial_f32(x)
    flat = [to_np(t).reshape(batch * tokens_, heads, head_size) for t in x]
    cu = np.arange(0, batch * tokens_ + 1, tokens_, dtype=np.int32)
    _, _, sa_ref, bnd_ref = oracle.wkv7_f64(*flat, cu_seqlens=cu, want_sa=True, boundary_len=16)
    for name, got, serial, want in (
            ("state", bnd[:, :, -1], serial_state, bnd_ref.reshape(bnd.shape)[:, :, -1]),
            ("sa", sa.reshape(sa_ref.shape), serial_sa.reshape(sa_ref.shape), sa_ref)):
        err, limit = relative_rmse(to_np(got), want), 1.25 * relative_rmse(to_np(serial), want)
        print(f"D={head_size} decay {decay} {name}: {err:.3e}, allowed {limit:.3e}", flush=True)
        assert err <= limit


@pytest.mark.parametrize("head_size", [128, 256])
@pytest.mark.parametrize("name,value", [("v", float("inf")), ("k", float("nan")),
                                        ("a", float("-inf")), ("b", float("inf")),
                                        ("decay_logits", float("nan")), ("r", float("nan"))])
def test_wide_non_finite_token_leaves_the_tokens_before_it(head_size, name, value):
    """A non-finite value in the middle of a 16-token chunk: what is finite token
    by token (the earlier tokens of its chunk, the other columns where only v is
    concerned, the other segments) is finite and right here too."""
    C = require_gpu()
    print(f"case wide non-finite D={head_size} {name}={value}", flush=True)
    case = make_case(dtype=torch.bfloat16, head_size=head_size, lengths=(40, 48), num_heads=2,
                     with_decay_bias=True, seed=head_size)
    case[name][27, 1, 70] = value
    C.handoff_fault_count(reset=True)
    y_ref, pool_ref = oracle_expect(case)
    out = wkv7(*tokens(case), state_pool=case["state_pool"], cu_seqlens=case["cu_seqlens"],
               state_indices=case["state_indices"], decay_bias=case["decay_bias"])
    torch.cuda.synchronize()
    assert C.handoff_fault_count(reset=True) == 0
    for got, want, rel in ((to_np(out), y_ref, 2.0e-3),
                           (to_np(case["state_pool"]), pool_ref, STATE_REL)):
        live = np.isfinite(want)
        assert live.any() and np.array_equal(np.isfinite(got), live)
        got, want = got[live].astype(np.float64), want[live]
        assert np.linalg.norm(got - want) / np.linalg.norm(want) <= rel


def test_wide_training_forward_non_finite_token():
    """sa and the state after every 16 tokens before and after a non-finite key."""
    C = require_gpu()
    case = make_case(dtype=torch.bfloat16, head_size=128, lengths=(48,), num_heads=1, seed=9)
    case["k"][21, 0, 3] = float("inf")
    x = [t.view(1, 48, 1, 128) for t in tokens(case)]
    y = torch.empty_like(x[3])
    bnd = torch.empty((1, 1, 3, 128, 128), device="cuda")
    sa = torch.empty((1, 48, 1, 128), device="cuda")
    C.pretrain_tmix_wkv7_recurrent_forward(*x, y, bnd, sa, 128)
    torch.cuda.synchronize()
    _, _, sa_ref, bnd_ref = oracle.wkv7_f64(*(to_np(t).reshape(48, 1, 128) for t in x),
                                            cu_seqlens=np.array([0, 48], dtype=np.int32),
                                            want_sa=True, boundary_len=16)
    for got, want in ((to_np(sa).reshape(sa_ref.shape), sa_ref),
                      (to_np(bnd).reshape(bnd_ref.shape), bnd_ref)):
        live = np.isfinite(want)
        assert live.any() and not live.all() and np.array_equal(np.isfinite(got), live)
        assert relative_rmse(got[live], want[live]) <= STATE_REL
    assert torch.isfinite(y[0, :21].float()).all()


@pytest.mark.parametrize("head_size", [128, 256])
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
def test_wide_hand_off_give_up_fails_closed(head_size, dtype):
    """With the bounded waits' limit at zero polls the state waves give up at
    once: NaN outputs, the state untouched, one fault per workgroup, and the
    same call is right again with the limit restored.  The token-serial kernel,
    forced, has no hand-off: no fault."""
    C = require_gpu()
    case = make_case(dtype=dtype, head_size=head_size, lengths=(64, 40), num_heads=2, seed=3)
    pool = case["state_pool"]
    before = pool.clone()
    ticket = prepare(case["cu_seqlens"], case["state_indices"], total_tokens=104,
                     state_pool_size=pool.shape[0])
    serial_pool, serial = pool.clone(), torch.empty_like(case["v"])
    C.handoff_fault_count(reset=True)
    C._set_handoff_spin_limit(0)
    try:
        C.tmix_wkv7_recurrent_fp32_kernel_forced(0, case["cu_seqlens"], case["state_indices"],
                                                 serial_pool, *tokens(case), serial, 1.0, None,
                                                 ticket)
        torch.cuda.synchronize()
        assert C.handoff_fault_count(reset=True) == 0
        out = wkv7(*tokens(case), state_pool=pool, cu_seqlens=case["cu_seqlens"],
                   state_indices=case["state_indices"])
        torch.cuda.synchronize()
    finally:
        C._set_handoff_spin_limit(-1)
    assert torch.isnan(out.float()).all() and torch.equal(pool, before)
    # sequences x heads x groups of 64 columns
    assert C.handoff_fault_count(reset=True) == 2 * 2 * (head_size // 64)
    y_ref, _ = oracle_expect(case)
    assert_output_close(serial, y_ref)
    out = wkv7(*tokens(case), state_pool=pool, cu_seqlens=case["cu_seqlens"],
               state_indices=case["state_indices"])
    torch.cuda.synchronize()
    assert_output_close(out, y_ref)
    assert C.handoff_fault_count(reset=True) == 0


@pytest.mark.parametrize("head_size", [128, 256])
def test_wide_training_forward_give_up_fails_closed(head_size):
    """The form with sa and the 16-token states: NaN in y and sa, counted."""
    C = require_gpu()
    x = [t.view(1, 64, 2, head_size) for t in tokens(make_case(head_size=head_size, lengths=(64,),
                                                               num_heads=2, seed=4))]
    y = torch.zeros_like(x[3])
    bnd = torch.empty((1, 2, 4, head_size, head_size), device="cuda")
    sa = torch.zeros((1, 64, 2, head_size), device="cuda")
    C.handoff_fault_count(reset=True)
    C._set_handoff_spin_limit(0)
    try:
        C.pretrain_tmix_wkv7_recurrent_forward(*x, y, bnd, sa, head_size)
        torch.cuda.synchronize()
    finally:
        C._set_handoff_spin_limit(-1)
    assert C.handoff_fault_count(reset=True) == 2 * (head_size // 64)
    assert torch.isnan(y.float()).all() and torch.isnan(sa).all()
