"""The training forward and backward on the sequence split (few (batch, head)
units: both passes cut each sequence into pieces) and on the kernels that take
over around its limits, against the fp64 oracle with the gates of the unsplit
tests: y, sa and every 16-token snapshot of the forward, and all six gradients.
The lengths cover the most pieces a unit gets, a last piece of one chunk and a
unit count just inside and outside the split."""

from __future__ import annotations

import pytest
import torch

import test_gpu_other_entries as entry_tests
import test_gpu_pretrain_backward as bwd_tests
from wkv7_testlib import require_gpu

pytestmark = pytest.mark.gpu

SHAPES = [
    # batch, tokens, heads, split into pieces
    (1, 512, 1, True),       # the most pieces: 7 of 80 tokens
    (2, 1040, 3, True),      # 10 pieces, the last of one chunk or a few
    (1, 4096, 2, True),
    (2, 1088, 64, True),     # 128 units: three pieces
    (1, 256, 2, False),      # too short to gain: the ring kernel, whole
    (1, 1088, 129, False),   # one unit too many for two pieces after the first
]


@pytest.mark.parametrize("batch,tokens,heads,split", SHAPES)
def test_training_passes_match_the_oracle(batch, tokens, heads, split):
    require_gpu()
    from flashrwkv2_amd import _native as N

    print(f"case train split B={batch} T={tokens} H={heads}", flush=True)
    floats = N.load().fr2_wkv7_pretrain_split_workspace_floats(batch, tokens, heads, 64)
    assert (floats > 0) == split
    entry_tests.test_pretrain_forward_matches_oracle(batch, tokens, heads, 64, True)
    vals, dy = bwd_tests._case(batch, tokens, heads, 64, seed=tokens + heads, rwkv=True,
                               logit_scale=1.5)
    got = bwd_tests._run(vals, dy, 64)
    bwd_tests._check(got, bwd_tests._expected(vals, dy, 64))


def test_split_entries_without_a_workspace_run_whole():
    """A null split workspace is the unsplit pass: the same results within the
    fp32 rounding that the split re-orders, and NaN never appears."""
    C = require_gpu()
    from flashrwkv2_amd import _native as N

    lib = N.load()
    B, T, H = 1, 1024, 2
    vals, _ = bwd_tests._case(B, T, H, 64, seed=3, rwkv=True)
    x = [t.detach().view(B, T, H, 64) for t in vals]
    outs = []
    for split in (True, False):
        y = torch.empty_like(x[3])
        bnd = torch.empty((B, H, T // 16, 64, 64), device="cuda")
        sa = torch.empty((B, T, H, 64), device="cuda")
        if split:
            C.pretrain_tmix_wkv7_recurrent_forward(*x, y, bnd, sa, 64)
        else:
            N.check(lib.fr2_wkv7_pretrain_forward(
                B, T, H, 64, *(t.data_ptr() for t in (*x, y, bnd, sa)),
                torch.cuda.current_stream().cuda_stream), "pretrain forward")
        torch.cuda.synchronize()
        outs.append((bnd, sa))
    for a, b in zip(*outs):
        assert torch.isfinite(a).all()
        assert ((a - b).norm() / b.norm()).item() <= 1e-4
