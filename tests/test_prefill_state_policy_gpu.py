"""The token-serial prefill on both sides of the number of state tiles from which it streams
them, against the oracle (the parity helpers' tolerances)."""

from __future__ import annotations

import pytest
import torch

from lightdelta_amd import ops
from tests.test_prefill_gpu import announce, prefill_case
from tests.test_prefill_heads_gpu import check

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("sequences", [128, 129])
def test_streamed_state_tiles(gpu, sequences):
    """4096 and 4128 tiles of 32 v-heads: one to five tokens, empty sequences, zero and given
    initial states, a padding slot."""
    announce(test="prefill_state_policy", sequences=sequences)
    saved = ops.prefill_algorithm()
    ops.set_prefill_algorithm("token_serial")
    try:
        case = prefill_case(gpu, [(1, 2, 0, 5, 4)[i % 5] for i in range(sequences)], seed=sequences,
                            w_dtype=torch.bfloat16)
        case["has_initial"][1::3] = False
        case["slots"][8] = -1
        check(case)
    finally:
        ops.set_prefill_algorithm(saved)
