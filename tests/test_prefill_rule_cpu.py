"""Which kernels a prefill of 32-token chunks runs (csrc/prefill_rule.h), on the CPU."""

from __future__ import annotations

import pytest

from tests.prefill_rule import plan, reads_qkv, side

LIMIT = (0x7fffffff // 2 - 128) // 32   # largest gate row stride of the whole-head kernels


@pytest.mark.parametrize("lengths", [[32], [100] * 8, [300] * 8, [290, 1, 0, 70, 33] + [0] * 254])
def test_gate_rows_beyond_32_bit_offsets_take_the_norm_pass(lengths):
    """A chunk's gate rows and the one after them fit 31 bits up to LIMIT; beyond (and for rows that go
    backwards) no whole-head kernel runs."""
    assert 2 * (32 * LIMIT + 128) <= 0x7fffffff < 2 * (32 * (LIMIT + 1) + 128)
    assert plan(lengths, 32, LIMIT) == plan(lengths, 32)
    assert plan(lengths, 32, LIMIT)[1]
    for row in (LIMIT + 1, 70_000_000, 1 << 40, -4096):
        assert plan(lengths, 32, row)[1:] == (False, True)
        assert side(lengths, 32, row) == "rows"


@pytest.mark.parametrize("lengths", [[32], [200], [100] * 8, [300] * 8])
def test_qkv_rows_that_overlap_or_lie_far_apart(lengths):
    """Overlapping rows (one expanded over the tokens, say) are read by the whole-head kernels
    alone; rows beyond 31-bit offsets in a chunk, and backward ones, by neither side."""
    width, rows = 8192, plan(lengths, 32)[2]
    limit = (0x7fffffff // 2 - width) // 32
    assert reads_qkv(lengths, 32, width, width) and reads_qkv(lengths, 32, limit, width)
    for row in (0, 64, width - 1):
        assert reads_qkv(lengths, 32, row, width) == (not rows)
    for row in (limit + 1, 1 << 40, -width):
        assert not reads_qkv(lengths, 32, row, width)


def test_more_pairs_than_the_row_block_grid_holds():
    """roundup(pairs, 8) x 4 row blocks x 512 threads stays under 2^32; beyond, whole heads alone."""
    lengths = [40] * 65_534 + [3000]
    assert (len(lengths) * 32 + 7) // 8 * 8 * 4 * 512 < 1 << 32
    assert plan(lengths, 32)[1:] == (True, True)
    assert plan(lengths + [40], 32)[1:] == (True, False)


@pytest.mark.parametrize("lengths,heads,faster", [
    ([6000] + [40] * 300, 32, "rows"), ([3000] + [33] * 90, 48, "rows"),
    ([512] + [40] * 28, 32, "rows"), ([1024] + [64] * 50, 32, "rows"),
    ([8192] + [20] * 511, 32, "rows"), ([4096] + [16] * 15, 32, "rows"),
    ([2048] + [32] * 260, 32, "own"), ([512] + [40] * 48, 32, "own"), ([32] * 512, 32, "own"),
    ([64] * 16, 32, "own"), ([100] * 28 + [2000] * 4, 32, "records"), ([1024] * 32, 32, "records"),
    ([3000] * 3, 48, "records"), ([1000] * 4, 32, "rows")])
def test_the_faster_side_is_taken(lengths, heads, faster):
    """Batches whose two sides were measured 5% or more apart (equal ones of 128 pairs apart)."""
    assert side(lengths, heads) == faster
