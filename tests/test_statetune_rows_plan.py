"""The row blocks of a StateTune chunk list (native host logic, CPU) against
the padded grid of the same list: the same tokens in the same 16-token blocks,
and a list neither takes is refused by both."""

from __future__ import annotations

import numpy as np
import pytest
import torch

from flashrwkv2_amd._statetune_plan import statetune_padded_plan, statetune_rows_plan


def _both(offsets, starts, ends, T, H=2):
    B, n = len(offsets) - 1, len(starts)
    t = lambda x: torch.tensor(x, dtype=torch.int32)   # noqa: E731
    grid = statetune_padded_plan(t(offsets), t(starts), t(ends), B, n, T, 64, torch.bfloat16)
    meta = np.array([*offsets, *starts, *ends], dtype=np.int32)
    return grid, statetune_rows_plan(meta, B, n, T, H), B, n


def _random_list(rng):
    B = int(rng.integers(1, 6))
    offsets, starts, ends, t = [0], [], [], 0
    for _ in range(B):
        for _ in range(int(rng.integers(0, 5))):
            t += int(rng.integers(0, 4))
            n = int(rng.choice([0, 1, 15, 16, 17, 40, 300]))
            starts.append(t)
            ends.append(t + n)
            t += n
        offsets.append(len(starts))
    if not starts:
        starts, ends, offsets[-1] = [0], [16], 1
        t = 16
    order = rng.permutation(len(starts))   # chunks in any order of their rows
    return offsets, [starts[i] for i in order], [ends[i] for i in order], t + int(rng.integers(0, 3))


@pytest.mark.parametrize("seed", range(40))
def test_rows_match_the_padded_grid(seed):
    rng = np.random.default_rng(seed)
    offsets, starts, ends, T = _random_list(rng)
    H = int(rng.choice([1, 4, 64]))
    grid, rows, B, n = _both(offsets, starts, ends, max(T, 1), H)
    assert (grid is None) == (rows is None)
    if grid is None:
        return
    Tp, row_source, chunk_seq, pstart, first = grid
    table, (blocks, spans, every, most) = rows
    row_blocks, rest = table[:2 * blocks].reshape(-1, 2), table[2 * blocks:]
    seq_blocks, seq_spans, rest = rest[:B + 1], rest[B + 1:2 * B + 2], rest[2 * B + 2:]
    span_list, rest = rest[:2 * spans].reshape(-1, 2), rest[2 * spans:]
    cseq, cblock, cfirst = rest[:n], rest[n:2 * n], rest[2 * n:]
    assert cseq.tolist() == chunk_seq.tolist() and cfirst.tolist() == first.tolist()
    assert most == np.diff(seq_blocks).max() and blocks == seq_blocks[-1]
    for b in range(B):
        blk = row_blocks[seq_blocks[b]:seq_blocks[b + 1]]
        want = row_source[b * Tp:(b + 1) * Tp].reshape(-1, 16)
        for j, (row0, cnt) in enumerate(blk):
            assert want[j].tolist() == [*range(row0, row0 + cnt), *[-1] * (16 - cnt)]
        assert (want[len(blk):] == -1).all()
        assert seq_spans[b + 1] - seq_spans[b] == -(-len(blk) // every)
    assert [(cblock[c] - seq_blocks[cseq[c]]) * 16 for c in range(n)] == pstart.tolist()
    assert sorted(map(tuple, span_list)) == [
        (b, i) for b in range(B) for i in range(seq_spans[b + 1] - seq_spans[b])]


@pytest.mark.parametrize("B,H", [(65535, 1), (65536, 1), (40000, 60000)])
def test_more_sequences_or_chunks_than_a_grid_holds(B, H):
    """Such a list is left to the token-serial kernels, which take it."""
    ends = np.arange(1, B + 1, dtype=np.int32) * 16
    ends[-1] += 1   # (not uniform)
    meta = np.concatenate([np.arange(B + 1), ends[:1] * 0, ends[:-1], ends]).astype(np.int32)
    rows = statetune_rows_plan(meta, B, B, int(ends[-1]), H)
    assert (rows is not None) == (B == 65535)


@pytest.mark.parametrize("offsets,starts,ends,T", [
    ([0, 1, 2], [0, 48], [64, 112], 112),          # rows in two chunks
    ([0, 1, 2], [0, 64], [64, 129], 128),          # past the end
    ([0, 1, 2], [-1, 64], [64, 128], 128),
    ([0, 1, 2], [0, 64], [64, 60], 128),           # negative length
    ([0, 2, 1], [0, 64], [64, 128], 128),          # offsets not increasing
    ([1, 1, 2], [0, 64], [64, 128], 128),
    ([0, 9], list(range(9)), list(range(1, 10)), 9),   # nine one-token chunks: 16x blocks
    ([0, 1], [0], [0], 16),                        # no tokens
    # one long sequence among short ones: filled up to it, more than four times the
    # tokens, which the fp32 token-serial kernels keep
    ([0, 2, 3, 4, 5, 6, 7], [0, 128, 256, 257, 258, 259, 260],
     [128, 256, 257, 258, 259, 260, 261], 261),
])
def test_lists_that_are_refused(offsets, starts, ends, T):
    grid, rows, _, _ = _both(offsets, starts, ends, T)
    assert grid is None and rows is None
