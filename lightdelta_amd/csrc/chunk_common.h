// Device helpers shared by the chunked-prefill kernels (prefill_chunked.hip,
// prefill_heads.hip): the exact three-way bf16 split of fp32 values, buffer-resource loads and
// the chunk search.
#pragma once

#include "gdn_common.h"

namespace ld {
namespace {

typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
// x = s1 + s2 + s3 exactly, in bf16 (each part the round-to-nearest-even of what the
// earlier ones leave, and every remainder exact in fp32: 8 + 8 + 8 bits of x's 24), so a
// product of an exact bf16 operand with x runs on the bf16 matrix cores as three products
// with exact terms and fp32 sums.  p[i] holds part i + 1 of four values.
struct Split4 {
  uint2 p[3];
};

typedef float f32x2 __attribute__((ext_vector_type(2)));
typedef __bf16 bf16x2 __attribute__((ext_vector_type(2)));

// two values to a packed bf16 pair (round to nearest even, one v_cvt_pk_bf16_f32)
__device__ __forceinline__ uint32_t bf16_pair(f32x2 v) {
  return __builtin_bit_cast(uint32_t, __builtin_convertvector(v, bf16x2));
}

// Each remainder r - s in one instruction: a dot product of the rounded pair with (-1, 0)
// or (0, -1) added to r (v_dot2c_f32_bf16; exact products, and the sum is r - s, which
// fp32 holds exactly).  (-1, 0) is set in an SGPR: as an operand the compiler encodes it
// as the inline constant -1.0, which this instruction reads as the fp32 word 0xbf800000,
// i.e. (0, -1).  Being an intrinsic, the first remainder also keeps a product passed as x
// rounded to fp32 (x - s1 written out would be contracted into an fma of its factors).
__device__ __forceinline__ Split4 split4(f32x4 x) {
  Split4 sp;
  uint32_t minus_lo_bits;
  asm("s_mov_b32 %0, 0xbf80" : "=s"(minus_lo_bits));
  const bf16x2 minus_lo = __builtin_bit_cast(bf16x2, minus_lo_bits);
  const bf16x2 minus_hi = __builtin_bit_cast(bf16x2, 0xbf800000u);
#pragma unroll
  for (int j = 0; j < 2; ++j) {
    f32x2 r = {x[2 * j], x[2 * j + 1]};
#pragma unroll
    for (int i = 0; i < 3; ++i) {
      const uint32_t w = bf16_pair(r);
      (j == 0 ? sp.p[i].x : sp.p[i].y) = w;
      if (i < 2) {
        const bf16x2 s = __builtin_bit_cast(bf16x2, w);
        r = f32x2{__builtin_amdgcn_fdot2_f32_bf16(s, minus_lo, r.x, false),
                  __builtin_amdgcn_fdot2_f32_bf16(s, minus_hi, r.y, false)};
      }
    }
  }
  return sp;
}

// Buffer resource over one chunk record (raw, byte-addressed; word 3 = 0x00020000, the
// gfx9 raw-buffer format) and a 16-byte load at lane offset + uniform offset: the address
// stays a scalar resource plus one offset register, whatever the compiler's register
// pressure.
__device__ __forceinline__ __amdgpu_buffer_rsrc_t record_resource(const float* r, int bytes) {
  return __builtin_amdgcn_make_buffer_rsrc(const_cast<float*>(r), 0, bytes, 0x00020000);
}

// The state tile of (slot, head) as a buffer resource: over its 64 KiB when the sequence
// starts from it, else over 0 bytes, whose loads return zeros without touching memory.  Its
// loads then need no branch and go out together (a branch per load, as `from_slot ? load :
// 0` compiles, waited for each load before the next was issued).  Callers pass the whole
// offset per lane, so the range check sees all of it.
__device__ __forceinline__ __amdgpu_buffer_rsrc_t state_resource(const DecodeParams& p, int slot,
                                                                 int head, bool from_slot) {
  // (uniform: readfirstlane keeps the resource in scalar registers, where a vector-held one
  // would put each load in a loop over its distinct values)
  return record_resource(
      p.state + static_cast<int64_t>(slot) * p.state_slot + static_cast<int64_t>(head) * kDim * kDim,
      __builtin_amdgcn_readfirstlane(from_slot ? kDim * kDim * 4 : 0));
}

// bf16 by the hardware's round-to-nearest-even conversion (v_cvt_pk_bf16_f32): the same
// value as f32_to_bf16 for every finite input
__device__ __forceinline__ uint16_t to_bf16(float f) {
  return __builtin_bit_cast(uint16_t, static_cast<__bf16>(f));
}

__device__ __forceinline__ f32x4 load16(__amdgpu_buffer_rsrc_t rsrc, uint32_t lane16,
                                        int byte_offset) {
  return __builtin_bit_cast(
      f32x4, __builtin_amdgcn_raw_buffer_load_b128(rsrc, static_cast<int>(lane16), byte_offset, 0));
}

__device__ __forceinline__ u32x4 load16u(__amdgpu_buffer_rsrc_t rsrc, uint32_t lane16,
                                         int byte_offset) {
  return __builtin_bit_cast(
      u32x4, __builtin_amdgcn_raw_buffer_load_b128(rsrc, static_cast<int>(lane16), byte_offset, 0));
}

__device__ __forceinline__ float load4(__amdgpu_buffer_rsrc_t rsrc, int byte_offset) {
  return __builtin_bit_cast(float, __builtin_amdgcn_raw_buffer_load_b32(rsrc, 0, byte_offset, 0));
}

// Global chunk g -> (sequence, first row, tokens): the last n with chunk_start[n] <= g
// (empty sequences come before it), by a 64-way search with one wave-wide load per level
// (one level up to 64 sequences, two up to 4096; a binary search took one dependent load per
// halving); false past the last chunk.  Called by every lane of a wave; the results are
// uniform.  C: tokens per chunk.
template <int C>
__device__ bool find_chunk(const int32_t* cu, const int32_t* chunk_start, int num_sequences,
                           int g, int& seq, int& t0, int& len) {
  if (g >= chunk_start[num_sequences]) return false;
  const int lane = threadIdx.x & 63;
  int lo = 0;              // chunk_start[lo] <= g throughout
  int count = num_sequences;
  for (;;) {
    const int step = (count + 63) >> 6;   // entries per lane at this level
    const bool in = lane * step < count;
    const int idx = lo + (in ? lane * step : 0);
    const int start = chunk_start[idx];
    int row0 = 0, row1 = 0;
    if (step == 1) {   // the last level: the rows of every candidate in the same round trip
      row0 = cu[idx];
      row1 = cu[idx + 1];
    }
    const int k = 63 - __clzll(static_cast<long long>(__ballot(in && start <= g)));
    if (step == 1) {
      seq = lo + k;
      t0 = __builtin_amdgcn_readlane(row0, k) + (g - __builtin_amdgcn_readlane(start, k)) * C;
      len = min(C, __builtin_amdgcn_readlane(row1, k) - t0);
      return true;
    }
    lo += k * step;
    count = min(step, count - k * step);
  }
}

}  // namespace
}  // namespace ld
