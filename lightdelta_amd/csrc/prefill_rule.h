// Which kernels a chunked prefill of 32-token chunks runs: host arithmetic on sizes and strides
// alone, and the part that the chunk index kernel decides from the lengths (constexpr functions
// are host and device ones).
#pragma once

#include <cstdint>

namespace ld {

// The whole-head kernels (prefill_heads.hip: a workgroup per (sequence, v-head)) or
// chunk_prep32_kernel and chunk_scan32_kernel (a head's rows over four workgroups).  A chunk
// takes a lone workgroup of the first 3.2 us and of the second 2.3 us, but with the chip full a
// (chunk, v-head) takes the first 17 ns and the second 30 ns; so it is decided by how many
// heads' chains the batch keeps going beside its longest: heads x chunks / longest chain, the
// number of (sequence, head) pairs if the prompts are equally long.  Over short chains the
// launches and records that the first saves decide.
struct HeadsRule {
  int num_v_heads;
  int short_chunks;   // whole heads up to this many chunks in the longest chain
  int chains;         // or from this many chains
  constexpr bool whole_heads(int64_t chunks, int64_t longest) const {
    return longest <= short_chunks || chunks * num_v_heads > chains * longest;
  }
};

// Prompts up to this mean length have their records prepared by the scan's own workgroups, which
// saves the record launch and the records (us, with records / own: 1 x 64 26.5 / 19.7, 16 x 64
// 41.9 / 31.9, 8 x 128 39.5 / 28.4, 8 x 256 53.2 / 49.4, 32 x 256 169 / 155, 1024 x 32 1266 /
// 1196) but lengthens a chunk's step in its chain by 1 us (13 prompts up to 3000 tokens 265 / 338,
// 8 x 1024 161 / 177).
constexpr int64_t kOwnTokens = 256;

// Whether a chunk's 32 rows (`used` elements of 2 bytes, `row` elements apart), and the row
// after them, begin within the 31 bits that offsets from its first row and sizes of resources
// over them have.
constexpr bool chunk_rows_fit(int64_t row, int64_t used) {
  return row >= 0 && row <= (0x7fffffff / 2 - used) / 32;
}

struct Plan32 {
  bool own;     // the whole-head kernels prepare their chunks themselves
  bool heads;   // launch the whole-head kernels
  bool rows;    // launch the others; with both, HeadsRule decides on the device
  HeadsRule rule;
};

// The row-block scan's grid of 4 x 512 threads a (sequence, head) pair, in multiples of 8, has to
// hold less than 2^32.
constexpr int64_t kRowPairs = (1 << 21) - 8;

// Where the host's numbers leave no choice only one side is launched; else both are, and the
// other side's workgroups return at once: 4 to 10 us of launches, 20 to 40 where whole heads run
// over 8,192 pairs and more (65,536 row-block workgroups take 18 us to return; us, one side / both:
// 512 x 32 620 / 640, 1024 x 32 1216 / 1257).  A grid that fits the chip and takes its workgroups'
// pairs from a queue returns in 2 us but is slower where its batch comes: one of 8192 and 511 of
// 20 tokens 1,203 us against 1,028 (1,020 by the row blocks alone), with the 8192 last 1,619
// against 1,404; at six waves a SIMD and without spills still 1,113 and 1,770.  us, row blocks /
// whole heads / decided: 32 x 1024 985 / 586 / 590, 512 prompts of 8 to 56 994 / 631 / 680, 16 x 64
// 52 / 32 / 40, one of 4096 and 15 of 16 277 / 430 / 284, one of 1000 and 30 of 40 108 / 162 / 112,
// 5 of 1 to 6000 179 / 272 / 184, 32 of 1 to 1000 206 / 179 / 191.
constexpr Plan32 plan_chunks32(int64_t num_tokens, int64_t num_sequences, int num_v_heads,
                               int64_t gate_row) {
  const int64_t pairs = num_sequences * num_v_heads;
  Plan32 plan{};
  plan.own = num_tokens <= kOwnTokens * num_sequences;
  plan.rule.num_v_heads = num_v_heads;
  plan.rule.short_chunks = !plan.own ? 0 : pairs > 64 ? 8 : 4;
  plan.rule.chains = plan.own ? 128 : 96;
  // (the whole-head kernels' gate offsets are of 32 bits, the norm pass's of 64)
  if (!chunk_rows_fit(gate_row, 128)) {
    plan.rows = true;
    return plan;
  }
  plan.rows = (num_tokens + 31) / 32 > plan.rule.short_chunks && num_v_heads <= plan.rule.chains;
  // (up to 128 pairs the launches in vain would take what the decision gains: 3 x 100 34 / 34 us,
  // 4 x 128 36 / 34, 4 x 1024 131 / 131)
  plan.heads = !plan.rows || pairs > 128;
  if (pairs > kRowPairs) plan.rows = false;
  return plan;
}

// Whether these kernels read qkv with such rows rightly; if not, the 64-token form does, whose
// preparation alone reads qkv, by 64-bit addresses.  The row-block scan's reads of v end at
// `rows` row strides from the chunk's start: short of the last rows where rows overlap (a row
// expanded over the tokens).
constexpr bool reads_qkv32(const Plan32& plan, int64_t qkv_row, int64_t qkv_width) {
  return chunk_rows_fit(qkv_row, qkv_width) && (!plan.rows || qkv_row >= qkv_width);
}

}  // namespace ld
