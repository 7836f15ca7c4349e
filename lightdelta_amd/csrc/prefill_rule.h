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
//   Where workgroups prepare their own chunks (4.6 us a chunk) the line is 150 such chains.  us,
// row blocks / whole heads, 32 v-heads: one of 6000 and 300 of 40 tokens (134 chains) 897 / 1020,
// and 340 (148) 975 / 1040, 20 of 1 to 600 (142) 84 / 96, 22 (149) 97 / 128, one of 512 and 28 of
// 40 (144) 82 / 100, one of 1024 and 50 of 64 (132) 174 / 189; the other way one of 2048 and 230 of
// 32 (147) 457 / 430, 24 of 1 to 1500 (130) 226 / 223; beyond, 24 of 1 to 600 (160) 120 / 119, one
// of 2048 and 250 of 32 (157) 497 / 441, one of 512 and 36 of 40 (176) 98 / 106, 32 of 1 to 1500
// (171) 303 / 288.  With records (3.3 us) it is 96, about which the order of the prompts decides:
// 16 of 1 to 3000 (85) 277 / 276, 18 (93) 349 / 293, 11 at 48 v-heads (97) 283 / 257, 5 of 500 to
// 1500 (115) 187 / 176; 22 of 1 to 8000 (97) 886 / 959, one of 4000 and 8 of 1000 (98) 417 / 466.
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
// 8 x 1024 161 / 177).  With the chip full the other workgroup of a CU covers that, and the rule,
// which looks at the mean alone, gives up 1 to 3% beyond it: 32 x 1024 610 / 591, 64 x 512 607 / 589,
// 32 x 2048 1141 / 1118, 64 x 300 405 / 395, 16 x 1024 306 / 298, 13 x 1000 268 / 271.
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
// other side's workgroups return at once: 4 to 10 us of launches, 20 over 8,192 pairs (us, row blocks
// / whole heads / so
// decided: 32 x 1024 985 / 586 / 590, 512 prompts of 8 to 56 994 / 631 / 658, 16 x 64 52 / 32 / 40,
// one of 4096 and 15 of 16 277 / 430 / 284, one of 1000 and 30 of 40 108 / 162 / 112, 5 of 1 to 6000
// 179 / 272 / 184, 32 of 1 to 1000 206 / 179 / 191).
constexpr Plan32 plan_chunks32(int64_t num_tokens, int64_t num_sequences, int num_v_heads,
                               int64_t gate_row) {
  const int64_t pairs = num_sequences * num_v_heads;
  Plan32 plan{};
  plan.own = num_tokens <= kOwnTokens * num_sequences;
  plan.rule.num_v_heads = num_v_heads;
  plan.rule.short_chunks = !plan.own ? 0 : pairs > 64 ? 8 : 4;
  plan.rule.chains = plan.own ? 150 : 96;
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
