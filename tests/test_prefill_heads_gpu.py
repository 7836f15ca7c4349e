"""The 32-token chunked prefill with a whole head per workgroup (csrc/prefill_heads.hip): prompt
lengths at the edges of its chunks, every head grouping, both sides of the rule that picks it,
and rows of gate and qkv that start at no 16-byte boundary, against the oracle (the parity
helpers' tolerances)."""

from __future__ import annotations

import pytest
import torch

from lightdelta_amd import ops
from oracle.decode import expected_prefill
from tests.parity import assert_bf16_outputs, assert_states
from tests.prefill_rule import plan, reads_qkv, side
from tests.test_prefill_gpu import PREFILL, announce, prefill_case, run

pytestmark = pytest.mark.gpu


@pytest.fixture(autouse=True)
def chunked_32():
    saved = ops.prefill_algorithm()
    ops.set_prefill_algorithm("chunked_32")
    yield
    ops.set_prefill_algorithm(saved)


def check(case):
    exp_out, exp_pool, pre = expected_prefill(*[case[k] for k in PREFILL], 1e-6, return_pre=True)
    before = case["pool"].clone()
    run(case)
    torch.cuda.synchronize()
    assert_bf16_outputs(case["out"], exp_out, pre)
    assert_states(case["pool"], exp_pool)
    assert torch.equal(case["pool"][0], before[0])


@pytest.mark.parametrize("heads,times", [((1, 1), 12), ((2, 6), 2), ((16, 16), 1), ((4, 32), 1),
                                         ((16, 48), 1)])
def test_chunk_edges(gpu, heads, times):
    """Lengths one below, at and above one, two and three chunks, one token, none (repeated until
    there are sequences enough for whole heads); zero and given initial states; a padding slot."""
    lengths = [1, 31, 32, 33, 0, 63, 64, 65, 96, 97, 2] * times
    assert side(lengths, heads[1]) == "own"
    announce(test="heads_chunk_edges", heads=heads, lengths=lengths)
    case = prefill_case(gpu, lengths, heads=heads, seed=heads[1], dt_dtype=torch.bfloat16,
                        w_dtype=torch.bfloat16)
    case["has_initial"][1::2] = False
    case["slots"][6] = -1
    check(case)


@pytest.mark.parametrize("heads,times", [((1, 1), 24), ((2, 6), 4), ((16, 16), 2), ((4, 32), 1),
                                         ((16, 48), 1)])
def test_record_chunk_edges(gpu, heads, times):
    """The same where the chunks' records come from a launch ahead."""
    lengths = [257, 288, 289, 319, 321, 290, 0, 577] * times
    assert side(lengths, heads[1]) == "records"
    announce(test="heads_record_chunk_edges", heads=heads, lengths=lengths)
    case = prefill_case(gpu, lengths, heads=heads, seed=heads[1], w_dtype=torch.bfloat16)
    case["has_initial"][1::2] = False
    case["slots"][3] = -1
    check(case)


@pytest.mark.parametrize("lengths,taken", [
    ([128], "own"), ([129], "rows"), ([64, 64], "own"), ([128, 128], "rows"), ([129, 128], "rows"),
    ([86, 85, 85], "own"), ([86, 85, 86], "rows"), ([64] * 4, "own"), ([65, 64, 64, 64], "rows"),
    ([256] * 4, "rows"), ([257, 256, 256, 256], "rows"), ([80, 33, 70, 81, 90], "own"),
    ([330, 40, 10, 1, 70], "rows"), ([300, 256, 280, 270, 256], "records")])
def test_both_sides_of_the_rule(gpu, lengths, taken):
    """Batches of up to 128 (sequence, head) pairs at the limits of the short chains, and 160 pairs,
    decided on the device: short prompts, a long one among short ones, equal longer ones."""
    assert side(lengths, 32) == taken
    announce(test="heads_rule", lengths=lengths, taken=taken)
    check(prefill_case(gpu, lengths, seed=len(lengths)))


@pytest.mark.parametrize("heads,lengths,taken", [
    ((16, 48), [290, 353, 261], "records"), ((16, 48), [256] * 3, "own"),
    ((16, 32), [270] + [250] * 5, "own"), ((16, 32), [270, 253, 253, 253, 252], "records")])
def test_both_sides_of_the_record_rule(gpu, heads, lengths, taken):
    """A mean of up to 256 tokens, where a workgroup prepares its chunks itself (nine of them
    here: three rounds of four), and above, where a launch ahead writes their records."""
    assert side(lengths, heads[1]) == taken
    announce(test="heads_records", heads=heads, lengths=lengths)
    check(prefill_case(gpu, lengths, heads=heads, seed=sum(lengths), dt_dtype=torch.bfloat16))


@pytest.mark.parametrize("lengths", [[290, 1, 0, 70, 33] + [0] * 254 + [40], [3, 0, 1, 34] * 65,
                                     [33] + [0] * 255 + [300, 7, 0]])
def test_many_sequences(gpu, lengths):
    """Over 8,192 (sequence, head) pairs: batches for the row-block scan (one long prompt, its
    workgroups' first or last item) and one for the whole-head kernels, decided on the device,
    each replayed from a graph too."""
    assert all(plan(lengths, 32)[1:])
    assert side(lengths, 32) == ("rows" if max(lengths) > 256 else "own")
    announce(test="heads_many", sequences=len(lengths))
    case = prefill_case(gpu, lengths, seed=7)
    pool0 = case["pool"].clone()
    check(case)
    out, pool = case["out"].clone(), case["pool"].clone()
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        run(case)
    for _ in range(3):
        case["pool"].copy_(pool0)
        graph.replay()
        torch.cuda.synchronize()
        assert torch.equal(case["out"], out)
        assert torch.equal(case["pool"], pool)


@pytest.mark.parametrize("lengths", [[70, 33, 1, 0, 64, 90], [300, 270, 0, 290, 280, 500]])
@pytest.mark.parametrize("what", ["qkv", "gate", "out"])
def test_unaligned_rows_give_the_aligned_bits(gpu, what, lengths):
    assert side(lengths, 32) == ("own" if 33 in lengths else "records")
    announce(test="heads_unaligned", what=what, lengths=lengths)
    case = prefill_case(gpu, lengths, seed=3)
    pool0 = case["pool"].clone()
    run(case)
    torch.cuda.synchronize()
    ref_out, ref_pool = case["out"].clone(), case["pool"].clone()
    n = case["qkv"].shape[0]
    if what == "out":
        flat = torch.zeros(n * 32 * 128 + 1, dtype=torch.bfloat16, device=gpu)
        case["out"] = flat[1:].view(n, 32, 128)
    else:
        rows = case[what].reshape(n, -1)
        moved = torch.empty(n, rows.shape[1] + 3, dtype=torch.bfloat16, device=gpu)[:, 1:-2]
        moved.copy_(rows)
        case[what] = moved if what == "qkv" else moved.unflatten(1, (32, 128))
    case["pool"].copy_(pool0)
    run(case)
    torch.cuda.synchronize()
    assert torch.equal(case["out"], ref_out)
    assert torch.equal(case["pool"], ref_pool)


def test_rows_of_one_shared_token(gpu):
    """qkv and gate as one row expanded over the tokens (row stride 0)."""
    assert side([40] * 6, 32, 0) == "own"
    announce(test="heads_expanded_rows")
    case = prefill_case(gpu, [40] * 6, seed=4)
    n = case["qkv"].shape[0]
    case["qkv"] = case["qkv"][:1].expand(n, -1)
    case["gate"] = case["gate"][:1].expand(n, -1, -1)
    check(case)


@pytest.mark.parametrize("row", [33_554_427, 33_554_428, 69_273_700])
def test_far_apart_gate_rows(gpu, row):
    """Gate rows at the largest stride whose offsets within a chunk fit 31 bits (whole heads), one
    element farther apart, and so far that 32 bits would wrap (row blocks and the norm pass)."""
    lengths = [33]
    assert side(lengths, 32, row) == ("own" if row == 33_554_427 else "rows")
    announce(test="heads_far_gate_rows", row=row)
    case = prefill_case(gpu, lengths, seed=5)
    far = torch.empty(32 * row + 4096, dtype=torch.bfloat16, device=gpu)
    far = far.as_strided((33, 32, 128), (row, 128, 1))
    far.copy_(case["gate"])
    case["gate"] = far
    check(case)


@pytest.mark.parametrize("lengths", [[130], [300, 40, 1], [330, 40, 10, 1, 70], [40] * 6])
@pytest.mark.parametrize("row", [0, 64, 4096])
def test_overlapping_qkv_rows(gpu, row, lengths):
    """qkv rows closer together than they are long, for batches of either side."""
    announce(test="heads_overlapping_rows", row=row, lengths=lengths)
    case = prefill_case(gpu, lengths, seed=6)
    n, width = case["qkv"].shape
    assert reads_qkv(lengths, 32, row, width) == (lengths == [40] * 6)
    flat = case["qkv"].reshape(-1)[:(n - 1) * row + width].clone()
    case["qkv"] = flat.as_strided((n, width), (row, 1))
    check(case)


@pytest.mark.parametrize("lengths", [[33], [130]])
@pytest.mark.parametrize("row", [33_554_175, 33_554_176, 69_273_700])
def test_far_apart_qkv_rows(gpu, row, lengths):
    """As for the gate's rows, on either side."""
    announce(test="heads_far_qkv_rows", row=row, lengths=lengths)
    case = prefill_case(gpu, lengths, seed=7)
    n, width = case["qkv"].shape
    assert reads_qkv(lengths, 32, row, width) == (row == 33_554_175)
    far = torch.empty((n - 1) * row + width, dtype=torch.bfloat16, device=gpu)
    far = far.as_strided((n, width), (row, 1))
    far.copy_(case["qkv"])
    case["qkv"] = far
    check(case)


@pytest.mark.parametrize("lengths", [[5, 33, 64, 1], [270, 290, 300, 280, 265]])
@pytest.mark.parametrize("value", [3.3e38, float("inf")])
@pytest.mark.parametrize("where", ["last", "middle"])
def test_decays_to_zero(gpu, where, value, lengths):
    """Log decays near -3e38 (finite, but not in units of log 2) and infinite: the state before
    them is gone, what follows is as from a zero state."""
    assert side(lengths, 32) == ("own" if len(lengths) == 4 else "records")
    announce(test="heads_decay_to_zero", where=where, value=value, lengths=lengths)
    case = prefill_case(gpu, lengths, seed=8)
    case["a_log"].fill_(-0.1)
    case["a"] = case["a"].clone()
    ends = case["cu_seqlens"][1:].long() - 1
    case["a"][ends if where == "last" else ends - torch.tensor(lengths, device=gpu) // 2] = value
    check(case)
