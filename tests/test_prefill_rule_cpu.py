"""Which kernels a prefill of 32-token chunks runs (csrc/prefill_rule.h), on the CPU."""

from __future__ import annotations

import pytest

from tests.prefill_rule import plan, side

LIMIT = (0x7fffffff // 2 - 128) // 31   # largest gate row stride of the whole-head kernels


@pytest.mark.parametrize("lengths", [[32], [100] * 8, [300] * 8, [290, 1, 0, 70, 33] + [0] * 254])
def test_gate_rows_beyond_32_bit_offsets_take_the_norm_pass(lengths):
    """The last byte of a chunk's gate rows fits 31 bits up to LIMIT; beyond (and for rows that go
    backwards) no whole-head kernel runs."""
    assert 2 * (31 * LIMIT + 128) <= 0x7fffffff < 2 * (31 * (LIMIT + 1) + 128)
    assert plan(lengths, 32, LIMIT) == plan(lengths, 32)
    assert plan(lengths, 32, LIMIT)[1]
    for row in (LIMIT + 1, 70_000_000, 1 << 40, -4096):
        assert plan(lengths, 32, row)[1:] == (False, True)
        assert side(lengths, 32, row) == "rows"
