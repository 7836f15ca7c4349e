// Chunked prefill for gfx950, 32-token chunks, one workgroup per (sequence, v-head): the scan
// of prefill_chunked.hip's 32-token form with the whole head's state in registers and the
// gated RMSNorm fused in.
//
// Four waves; wave w owns state rows v = 32 w .. 32 w + 31 as S^T in the accumulator layout of
// v_mfma_f32_32x32x16_bf16 (fp32, 64 registers).  For lane l, lj = l % 32 and hi = l / 32; a
// 32 x 32 accumulator holds rows i(r) = 8 (r / 4) + 4 hi + r % 4, r < 16, of column lj, and an
// operand A[i = lj][k = 8 hi + e] or B[k = 8 hi + e][j = lj], e < 8.  The summation index may
// be assigned to (step, hi, e) freely as long as both operands agree, so an accumulator's
// registers 8 u .. 8 u + 7 are directly the B operand of step u once split into bf16 planes:
// nothing of the chain S -> Y -> X -> V_new -> S' moves between lanes or waves.
//   state tile T < 4:  row i of the accumulator is k = 32 T + key_of(i), chosen so that step u
//                      takes k = 32 T + 16 u + 8 hi + e: 16 consecutive bytes of a q or k row
//   tokens:            row i of an accumulator over the chunk is token i, so step u of a
//                      product over tokens takes token 16 u + 8 (e / 4) + 4 hi + e % 4
// Per chunk and wave (rows past the sequence's end are zeros):
//   Y = K S^T, O = Q S^T    (q, k as stored against S's exact three-way split: 24 products each)
//   X = V - diag(ws) Y
//   V_new = T X             (T = (I + A)^-1 diag(beta); six of the nine products of planes)
//   O = diag(sq) O + P X    (P = P0 T: P0 V_new without waiting for V_new; the same)
//   S' = exp(G_n-1) S + K^T (ck V_new)   (24 products)
// and the chunk's raw outputs go through LDS (bf16, the reference's rounding point) to the
// gated RMSNorm of whole rows.  q, k and v come from qkv through LDS, the transposed operands
// by ds_read_b64_tr_b16; T, P (as planes) and the per-token scales are prepared by the
// workgroup itself (short prompts) or come as records from a launch ahead.
//
// Of the planes' products of T X and P X, those of planes (1, 2), (2, 1) and (2, 2) are left out.
// A plane 1 is up to 2^-8 and a plane 2 up to 2^-17 of its value, so a term t x lacks up to 2^-24
// of |t x| (two products of up to 2^-25): the size of an fp32 rounding, one of which each term of
// the fp32 products that the row-block scan forms here has.  The states' relative error against
// 64 bits is 0.9e-7 to 1.0e-7, the row blocks' 1.9e-7 to 7.3e-7 (for the decays' sums, below).
//
// What bounds it: vector issue, and matrix instructions beside it.  A wave's chunk is 96 matrix
// instructions (3,072 cycles of a matrix core) and, with the norm and its share of the rest, 900
// vector ones (4,100 cycles of issue with the matrix ones').  With two workgroups a CU a chunk
// takes 10,800 cycles, of which a SIMD's vector issue is busy 8,300 and its matrix core 6,100
// (counters at 32 x 1024 tokens and 32 v-heads, 433 us at 1.89 GHz; 2.33 GHz where fewer
// workgroups run, so the power limit has a part).  That is 0.95 PFLOP/s of bf16 products (a large
// bf16 GEMM reaches 1.17), where chunk_scan32_kernel and the norm pass took 820 us: with a head's
// rows over four workgroups every wave re-read S's planes from LDS and the raw outputs crossed
// HBM twice more.  The whole prefill, with the prep below, went from 992 to 576 us there, 257 to
// 169 us at 8 x 1024, 1,710 to 1,213 us at 1024 x 32.  Products and vector work are laid out by
// hand, slot by slot: as the compiler scheduled the same code, 32 x 1024 took 685 us.  Spilled
// registers: none with records ahead, 15 where the workgroups prepare their chunks (17 and 47
// where rows are not at 16-byte boundaries).
#include "chunk_common.h"

namespace ld {
namespace {

typedef float f32x16 __attribute__((ext_vector_type(16)));
typedef __bf16 bf16x4 __attribute__((ext_vector_type(4)));
typedef short s16x4 __attribute__((ext_vector_type(4)));

constexpr int kTok = 32;                       // tokens per chunk
constexpr int kTileRow = kDim * 2;             // bytes of a q, k, v or raw-output row in LDS
constexpr int kTileSize = kTok * kTileRow;

// 16-byte pieces of row r are stored at piece ^ swizzle(r): a column of pieces over 16 rows
// (operand A of the products with S) and 4 x 4 element blocks of 4 rows (transposed reads)
// each cover every bank once.
__device__ __forceinline__ constexpr int swizzle(int row) {
  return ((row & 3) << 2) | ((row >> 2) & 3);
}

__device__ __forceinline__ f32x16 mfma32(bf16x8 a, bf16x8 b, f32x16 c) {
  return __builtin_amdgcn_mfma_f32_32x32x16_bf16(a, b, c, 0, 0, 0);
}

// Fixes the order of pure operations: a value is defined ahead of this point and not used
// before it, and the points keep their order in the program.  (Left to itself the compiler
// lines the splits up ahead of the matrix instructions that should run beside them; it
// emits nothing for a pin.)
template <typename T>
__device__ __forceinline__ void pin(T& x) {
  asm volatile("" : "+v"(x));
}

// The exact split of eight values (a lane's registers 8 u .. 8 u + 7 of an accumulator) into
// planes that are B operands, in five stages: 0, 2, 4 round (4 instructions), 1, 3 take the
// remainders (16: each value less its plane's, exact).  split4's remainder is one v_dot2c, but
// that does not run beside a matrix instruction: with 8 of them behind each, a matrix
// instruction of 32 cycles took 81 (78 with two waves a SIMD); with 8 of these, 46 (42).
struct Split8 {
  float r[8];
  u32x4 w[3];
  __device__ __forceinline__ void set(f32x4 lo, f32x4 hi) {
#pragma unroll
    for (int e = 0; e < 4; ++e) {
      r[e] = lo[e];
      r[4 + e] = hi[e];
    }
  }
  __device__ __forceinline__ void stage(int i) {  // 0 .. 4
    if (i & 1) {
#pragma unroll
      for (int j = 0; j < 4; ++j) {
        const uint32_t pair = w[i >> 1][j];
        r[2 * j] -= __builtin_bit_cast(float, pair << 16);
        r[2 * j + 1] -= __builtin_bit_cast(float, pair & 0xffff0000u);
      }
      asm volatile("" : "+v"(r[0]), "+v"(r[1]), "+v"(r[2]), "+v"(r[3]), "+v"(r[4]), "+v"(r[5]),
                   "+v"(r[6]), "+v"(r[7]));
    } else {
#pragma unroll
      for (int j = 0; j < 4; ++j) w[i >> 1][j] = bf16_pair(f32x2{r[2 * j], r[2 * j + 1]});
      pin(w[i >> 1]);
    }
  }
  __device__ __forceinline__ void all() {
#pragma unroll
    for (int i = 0; i < 5; ++i) stage(i);
  }
  __device__ __forceinline__ bf16x8 plane(int i) const {
    return __builtin_bit_cast(bf16x8, w[i]);
  }
};
__device__ __forceinline__ f32x4 quad(const f32x16& x, int q) {
  return f32x4{x[4 * q], x[4 * q + 1], x[4 * q + 2], x[4 * q + 3]};
}

// A matrix instruction in its place of the schedule (First: of a sum that starts at zero).
template <bool First = false>
__device__ __forceinline__ void product(bf16x8 a, bf16x8 b, f32x16& c) {
  if constexpr (First) {
    pin(a);
    c = mfma32(a, b, f32x16{});
  } else {
    pin(c);
    c = mfma32(a, b, c);
  }
  pin(c);
}

// 4 x 16 block of bf16 transposed on the way from LDS: within 16 lanes, lane m gives the
// address of row m / 4, elements 4 (m % 4) .. + 3, and receives rows 0 .. 3 of column m.
__device__ __forceinline__ bf16x4 read_tr(const uint8_t* at) {
  const auto p = (__attribute__((address_space(3))) s16x4*)(at);
  return __builtin_bit_cast(bf16x4, __builtin_amdgcn_ds_read_tr16_b64_v4i16(p));
}

__device__ __forceinline__ void lds_barrier() {
  asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory");
}

// Keeps LDS accesses of a wave in program order past the compiler (the hardware runs them in
// order).
__device__ __forceinline__ void lds_order() { asm volatile("" ::: "memory"); }

// Sixteen bytes of a row at a lane's byte offset + a uniform one: one load, or (rows not at
// 16-byte boundaries) eight of one element.
template <bool Wide>
__device__ __forceinline__ u32x4 load_piece(__amdgpu_buffer_rsrc_t rs, uint32_t offset,
                                            int uniform) {
  if constexpr (Wide) return load16u(rs, offset, uniform);
  u32x4 out;
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    const uint32_t lo = __builtin_amdgcn_raw_buffer_load_b16(rs, static_cast<int>(offset + 4 * i), uniform, 0);
    const uint32_t hi = __builtin_amdgcn_raw_buffer_load_b16(rs, static_cast<int>(offset + 4 * i + 2), uniform, 0);
    out[i] = (lo & 0xffffu) | (hi << 16);
  }
  return out;
}

// The gated RMSNorm of a chunk's rows, a thread's 16 columns of one token, in slices that fit
// beside matrix instructions and hold eight independent operations where the arithmetic
// allows: 0: the raw outputs' reads, 1-4: squares, 5: the row's sum over its 8 threads, 6:
// rstd, 7-14: columns 0 .. 7, 15-22: columns 8 .. 15.  Arithmetic as prefill_norm_kernel's.
struct Norm {
  u32x4 raw[2], gate[2], y[2];
  float ss[2], rstd, g[8], t[8];
  __device__ __forceinline__ static float low(uint32_t pair) { return __builtin_bit_cast(float, pair << 16); }
  __device__ __forceinline__ static float high(uint32_t pair) {
    return __builtin_bit_cast(float, pair & 0xffff0000u);
  }
  __device__ __forceinline__ void pin8(float (&x)[8]) {
    asm volatile("" : "+v"(x[0]), "+v"(x[1]), "+v"(x[2]), "+v"(x[3]), "+v"(x[4]), "+v"(x[5]),
                 "+v"(x[6]), "+v"(x[7]));
  }
  __device__ __forceinline__ void slice(int i, const uint8_t* raw0, const uint8_t* raw1,
                                        const float* weight, float eps) {
    if (i == 0) {
      raw[0] = *reinterpret_cast<const u32x4*>(raw0);
      raw[1] = *reinterpret_cast<const u32x4*>(raw1);
      ss[0] = ss[1] = 0.0f;
    } else if (i < 5) {
#pragma unroll
      for (int h = 0; h < 2; ++h) {
        const uint32_t bits = raw[h][i - 1];
        ss[h] = fmaf(low(bits), low(bits), ss[h]);
        ss[h] = fmaf(high(bits), high(bits), ss[h]);
      }
      pin(ss[0]);
      pin(ss[1]);
    } else if (i == 5) {
      ss[0] += ss[1];
      ss[0] += dpp<kDppQuadXor1>(ss[0]);
      ss[0] += dpp<kDppQuadXor2>(ss[0]);
      ss[0] += dpp<kDppRowHalfMirror>(ss[0]);
      pin(ss[0]);
    } else if (i == 6) {
      rstd = fast_rsqrt(ss[0] / static_cast<float>(kDim) + eps);
      pin(rstd);
    } else {
      const int h = (i - 7) >> 3;
      switch ((i - 7) & 7) {
        case 0:
#pragma unroll
          for (int e = 0; e < 8; ++e) {
            const uint32_t pair = gate[h][e >> 1];
            g[e] = e & 1 ? high(pair) : low(pair);
          }
          pin8(g);
          break;
        case 1:
#pragma unroll
          for (int e = 0; e < 8; ++e) t[e] = __expf(-g[e]);
          pin8(t);
          break;
        case 2:
#pragma unroll
          for (int e = 0; e < 8; ++e) t[e] += 1.0f;
          pin8(t);
          break;
        case 3:
#pragma unroll
          for (int e = 0; e < 8; ++e) t[e] = fast_rcp(t[e]);
          pin8(t);
          break;
        case 4:
#pragma unroll
          for (int e = 0; e < 8; ++e) t[e] *= g[e];   // silu
          pin8(t);
          break;
        case 5:
#pragma unroll
          for (int e = 0; e < 8; ++e) {
            const uint32_t pair = raw[h][e >> 1];
            g[e] = (e & 1 ? high(pair) : low(pair)) * rstd;
          }
          pin8(g);
          break;
        case 6: {
          const f32x4 w0 = *reinterpret_cast<const f32x4*>(weight + 8 * h);
          const f32x4 w1 = *reinterpret_cast<const f32x4*>(weight + 8 * h + 4);
#pragma unroll
          for (int e = 0; e < 8; ++e) g[e] *= e < 4 ? w0[e & 3] : w1[e & 3];
          pin8(g);
          break;
        }
        default:
#pragma unroll
          for (int d = 0; d < 4; ++d)
            y[h][d] = bf16_pair(f32x2{g[2 * d] * t[2 * d], g[2 * d + 1] * t[2 * d + 1]});
          pin(y[h]);
      }
    }
  }
};

// ---- a chunk's T, P and scales, by one wave ------------------------------------------------
// Every fourth chunk each wave does one of the next four alone, so nothing waits on another
// wave: q and k come as operands of v_mfma_f32_16x16x32_bf16 (for lane l, li = l % 16 and
// lg = l / 16: row 16 a + li, 16 bytes at k = 32 s + 8 lg), which give the raw products K K^T
// and K Q^T below the diagonal and, from the diagonals of K K^T and Q Q^T, the squared norms;
// then the gates, -A to LDS, the inverses of I + A's two diagonal blocks (a column per lane),
// T10 = -T1 A10 T0 and P = P0 T as 16 x 16 x 4 fp32 products with summation index k = 4 lg +
// step, for which P0's tiles, T10 and the first product are operands as they are.

// What the chunks' products read of it, in LDS, offsets in bytes: T = (I + A)^-1 diag(beta) and
// P = P0 T (32 x 32 fp32, lower triangular) as their exact bf16 planes in operand order.  Of a
// step u, a lane (hi, lj) of the product holds row lj, tokens 16 u + 8 (e / 4) + 4 hi + e % 4,
// e < 8, as 16 bytes; plane i of step 0 is at 1024 i + (32 hi + lj) * 16, of step 1 (whose rows
// below 16 are zeros and not stored) at 3072 + 512 i + (16 hi + lj - 16) * 16.  Then the
// per-token scales in fp32 (offsets of kSq, .. in 16-byte pieces from kScales) sq = rq scale
// exp(G), ck = rk exp(G_n-1 - G), ws = rk exp(G), and exp(G_n-1).
struct Record {
  static constexpr int kT = 0;
  static constexpr int kP = 4608;
  static constexpr int kScales = 9216;
  static constexpr int kSq = 0;
  static constexpr int kCk = 8;
  static constexpr int kWs = 16;
  static constexpr int kGamma = kScales + 384;
  static constexpr int kBytes = static_cast<int>(kHeadRecordBytes);
};

// The wave's working memory, in the place of the planes it writes at the end.
struct PrepScratch {
  static constexpr int kARow = kTok + 4;   // padded rows (floats)
  static constexpr int kTRow = 20;
  float a[kTok][kARow];                    // -A
  float t[3][16][kTRow];                   // T0, T1, T10
  float g[kTok], glo[kTok];                // G / ln 2 as a sum of two floats
  float beta[kTok], rq[kTok], rk[kTok];
};
static_assert(sizeof(PrepScratch) <= Record::kScales, "the scratch fits the planes' place");

__device__ __forceinline__ f32x4 mfma16(bf16x8 a, bf16x8 b, f32x4 c) {
  return __builtin_amdgcn_mfma_f32_16x16x32_bf16(a, b, c, 0, 0, 0);
}

// c[4 lg + r][li] + sum over k of a[li][k] b[k][li], the lane's a[li][4 lg + st] and
// b[4 lg + st][li]
__device__ __forceinline__ f32x4 mfma_f32(f32x4 a, f32x4 b, f32x4 c) {
#pragma unroll
  for (int st = 0; st < 4; ++st) c = __builtin_amdgcn_mfma_f32_16x16x4f32(a[st], b[st], c, 0, 0, 0);
  return c;
}

// Inclusive sums over the 32 lanes of each half wave (lane 32 + i as lane i), in 64 bits: decays
// between two tokens are differences of these sums, and rounded to 32 bits the sums' error (half
// an ulp of up to about 70) was most of the states': against 64 bits 1.9e-7 to 7.3e-7 over six
// workloads, 0.9e-7 to 1.0e-7 this way.
template <int Ctrl>
__device__ __forceinline__ double dpp64(double x) {
  const uint64_t u = __builtin_bit_cast(uint64_t, x);
  const uint32_t lo = __builtin_amdgcn_update_dpp(0, static_cast<int>(u), Ctrl, 0xF, 0xF, false);
  const uint32_t hi = __builtin_amdgcn_update_dpp(0, static_cast<int>(u >> 32), Ctrl, 0xF, 0xF, false);
  return __builtin_bit_cast(double, (static_cast<uint64_t>(hi) << 32) | lo);
}
__device__ __forceinline__ double prefix_sum32(double x, int lane) {
  x += dpp64<0x111>(x);   // row_shr:1, 2, 4, 8: zeros from below the row
  x += dpp64<0x112>(x);
  x += dpp64<0x114>(x);
  x += dpp64<0x118>(x);
  const uint64_t u = __builtin_bit_cast(uint64_t, x);
  const uint32_t lo = __builtin_amdgcn_readlane(static_cast<int>(u), 15);
  const uint32_t hi = __builtin_amdgcn_readlane(static_cast<int>(u >> 32), 15);
  const double row0 = __builtin_bit_cast(double, (static_cast<uint64_t>(hi) << 32) | lo);
  return x + ((lane & 16) != 0 ? row0 : 0.0);
}

// q and k of one chunk as loaded (zeros past its end), and the gates of one v-head, of token
// lane % 32.
struct PrepInputs {
  u32x4 q[2][4], k[2][4];
};
struct PrepGates {
  uint16_t a, b;
  float a_log, dt_bias;
};

template <bool Wide>
__device__ __forceinline__ void prep_fetch(PrepInputs& x, const DecodeParams& p, int t0, int len,
                                           int key_head, int lane) {
  const int li = lane & 15;
  const int lg = lane >> 4;
  const uint32_t row_bytes = static_cast<uint32_t>(p.qkv_row) * 2;
  const __amdgpu_buffer_rsrc_t rows = __builtin_amdgcn_make_buffer_rsrc(
      const_cast<uint16_t*>(p.qkv + static_cast<int64_t>(t0) * p.qkv_row), 0,
      (len - 1) * static_cast<int>(row_bytes) + (2 * p.num_k_heads + p.num_v_heads) * kTileRow,
      0x00020000);
#pragma unroll
  for (int a = 0; a < 2; ++a) {
    const uint32_t at = 16 * a + li < len ? (16 * a + li) * row_bytes + lg * 16 : 0xfffff000u;
#pragma unroll
    for (int s = 0; s < 4; ++s) {
      x.k[a][s] = load_piece<Wide>(rows, at, (p.num_k_heads + key_head) * kTileRow + s * 64);
      x.q[a][s] = load_piece<Wide>(rows, at, key_head * kTileRow + s * 64);
    }
  }
}

template <bool DtBf16>
__device__ __forceinline__ void prep_gates(PrepGates& x, const DecodeParams& p, int t0, int len,
                                           int head, int lane) {
  const int64_t tok = t0 + min(lane & 31, len - 1);
  x.a = p.a[tok * p.a_row + head];
  x.b = p.b[tok * p.b_row + head];
  x.a_log = p.a_log[head];
  x.dt_bias = load_param(p.dt_bias, head, DtBf16);
}

// kk: raw tiles of K K^T (0,0), (1,0), (1,1), rows 4 lg + r, column li; kq: K Q^T of P's tiles
// (0,0), (1,0), (1,1): row li of P0, columns 4 lg + r (exact products, fp32 sums).
struct PrepTiles {
  f32x4 kk[3], kq[3];
};

// The part that depends on q and k alone: the raw tiles, and the inverse norms to the scratch.
__device__ __forceinline__ void prep_tiles(PrepTiles& x, const PrepInputs& in, float scale, int len,
                                           PrepScratch& sc, int lane) {
  const int li = lane & 15;
  const int lg = lane >> 4;
  {
    f32x4 qq[2];
#pragma unroll
    for (int i = 0; i < 3; ++i) x.kk[i] = x.kq[i] = f32x4{0.0f, 0.0f, 0.0f, 0.0f};
    qq[0] = qq[1] = x.kk[0];
#pragma unroll
    for (int s = 0; s < 4; ++s) {
      const bf16x8 k0 = __builtin_bit_cast(bf16x8, in.k[0][s]);
      const bf16x8 k1 = __builtin_bit_cast(bf16x8, in.k[1][s]);
      const bf16x8 q0 = __builtin_bit_cast(bf16x8, in.q[0][s]);
      const bf16x8 q1 = __builtin_bit_cast(bf16x8, in.q[1][s]);
      x.kk[0] = mfma16(k0, k0, x.kk[0]);
      x.kk[1] = mfma16(k1, k0, x.kk[1]);
      x.kk[2] = mfma16(k1, k1, x.kk[2]);
      x.kq[0] = mfma16(k0, q0, x.kq[0]);
      x.kq[1] = mfma16(k0, q1, x.kq[1]);
      x.kq[2] = mfma16(k1, q1, x.kq[2]);
      qq[0] = mfma16(q0, q0, qq[0]);
      qq[1] = mfma16(q1, q1, qq[1]);
    }
    // the inverse norms, from the lanes that hold a diagonal entry (register li % 4 of the lanes
    // with li / 4 = lg); rows past the end: q's are zeros, k's too
    if ((li >> 2) == lg) {
#pragma unroll
      for (int a = 0; a < 2; ++a) {
        const f32x4 dq = qq[a];
        const f32x4 dk = x.kk[2 * a];
        const int r = li & 3;
        const float q2 = r < 2 ? (r == 0 ? dq[0] : dq[1]) : (r == 2 ? dq[2] : dq[3]);
        const float k2 = r < 2 ? (r == 0 ? dk[0] : dk[1]) : (r == 2 ? dk[2] : dk[3]);
        const bool live = 16 * a + li < len;
        sc.rq[16 * a + li] = live ? fast_rsqrt(q2 + 1e-6f) * scale : 0.0f;
        sc.rk[16 * a + li] = live ? fast_rsqrt(k2 + 1e-6f) : 0.0f;
      }
    }
  }
}

// One v-head's T, P and scales to `rec` (in LDS, where the scratch may be in the planes' place,
// or in memory).
__device__ __forceinline__ void prep_head(const PrepTiles& x, const PrepGates& in, int len,
                                          PrepScratch& sc, uint8_t* rec, int lane) {
  const int li = lane & 15;
  const int lg = lane >> 4;
  const int token = lane & 31;
  const auto at4 = [](const float* x) __attribute__((always_inline)) {
    return *reinterpret_cast<const f32x4*>(x);
  };
  {
    // gates and the in-chunk cumulative log decay: the token-serial form's arithmetic
    {
      const bool live = token < len;
      const float xa = bf16_to_f32(in.a) + in.dt_bias;
      // (a log decay below -1e6, whose decay is 0 in any form, as -1e6: sums in log2 units stay
      // finite and keep the bits of the decays after it; NaN stays)
      const float decay = -__expf(in.a_log) * softplus(xa);
      const float gl = live ? (decay < -1e6f ? -1e6f : decay) : 0.0f;
      const float beta = live ? sigmoid(bf16_to_f32(in.b)) : 0.0f;
      const double sum = prefix_sum32(gl, lane) * 1.4426950408889634;   // exp2 from here on
      const float G = static_cast<float>(sum);
      const float glo = static_cast<float>(sum - static_cast<double>(G));
      const float last = __int_as_float(__builtin_amdgcn_readlane(__float_as_int(G), 31));
      const float last_lo = __int_as_float(__builtin_amdgcn_readlane(__float_as_int(glo), 31));
      const float eg = __builtin_amdgcn_exp2f(G);
      const float rk = sc.rk[token];
      float* const scales = reinterpret_cast<float*>(rec + Record::kScales);
      if (lane < kTok) {
        sc.g[token] = G;
        sc.glo[token] = glo;
        sc.beta[token] = beta;
        scales[4 * Record::kSq + token] = sc.rq[token] * eg;
        scales[4 * Record::kWs + token] = eg * rk;
      } else {
        scales[4 * Record::kCk + token] = rk * __builtin_amdgcn_exp2f((last - G) + (last_lo - glo));
        if (token == 0) *reinterpret_cast<float*>(rec + Record::kGamma) = __builtin_amdgcn_exp2f(last);
      }
    }
    lds_order();

    // -A to LDS (tile i, rows 4 lg + r, column li), zeros from the diagonal on
#pragma unroll
    for (int i = 0; i < 3; ++i) {
      const int mt = i > 0 ? 1 : 0, nt = i > 1 ? 1 : 0;
      const int mcol = 16 * nt + li;
      const float gm = sc.g[mcol];
      const float glm = sc.glo[mcol];
      const float rkm = sc.rk[mcol];
      const f32x4 gi = at4(&sc.g[16 * mt + 4 * lg]);
      const f32x4 gli = at4(&sc.glo[16 * mt + 4 * lg]);
      const f32x4 bi = at4(&sc.beta[16 * mt + 4 * lg]);
      const f32x4 rki = at4(&sc.rk[16 * mt + 4 * lg]);
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        const float na = -(bi[r] * __builtin_amdgcn_exp2f((gi[r] - gm) + (gli[r] - glm)) * ((rki[r] * rkm) * x.kk[i][r]));
        sc.a[16 * mt + 4 * lg + r][mcol] = i == 1 || li < 4 * lg + r ? na : 0.0f;
      }
    }
    // P0's tiles: row li, columns 4 lg + r
    f32x4 p0[3];
#pragma unroll
    for (int i = 0; i < 3; ++i) {
      const int mt = i > 0 ? 1 : 0, nt = i > 1 ? 1 : 0;
      const float gi = sc.g[16 * mt + li];
      const float gli = sc.glo[16 * mt + li];
      const float rqi = sc.rq[16 * mt + li];
      const f32x4 gm = at4(&sc.g[16 * nt + 4 * lg]);
      const f32x4 glm = at4(&sc.glo[16 * nt + 4 * lg]);
      const f32x4 rkm = at4(&sc.rk[16 * nt + 4 * lg]);
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        const float pv = __builtin_amdgcn_exp2f((gi - gm[r]) + (gli - glm[r])) * ((rqi * rkm[r]) * x.kq[i][r]);
        p0[i][r] = (i == 1 || 4 * lg + r <= li) && 16 * mt + li < len ? pv : 0.0f;
      }
    }
    lds_order();
    // T0 and T1: column li of block lane / 16 (lanes 32 .. 63 repeat), row by row: col[i] =
    // delta(i, li) + sum over m < i of (-A)[i][m] col[m], the terms in order of m
    {
      const int block = (lane >> 4) & 1;
      const float* const ab = &sc.a[16 * block][16 * block];
      float col[16];
#pragma unroll
      for (int i = 0; i < 16; ++i) col[i] = i == li ? 1.0f : 0.0f;
#pragma unroll
      for (int mc = 0; mc < 15; ++mc)
#pragma unroll
        for (int i = mc + 1; i < 16; ++i) col[i] = fmaf(ab[i * PrepScratch::kARow + mc], col[mc], col[i]);
      if (lane < 32) {
#pragma unroll
        for (int i = 0; i < 16; ++i) sc.t[block][i][li] = col[i];
      }
    }
    lds_order();
    f32x4 t0k, t1k;   // T0, T1 [4 lg + r][li]
#pragma unroll
    for (int r = 0; r < 4; ++r) {
      t0k[r] = sc.t[0][4 * lg + r][li];
      t1k[r] = sc.t[1][4 * lg + r][li];
    }
    const f32x4 t0r = at4(&sc.t[0][li][4 * lg]);   // T0, T1 [li][4 lg + r]
    const f32x4 t1r = at4(&sc.t[1][li][4 * lg]);
    const f32x4 a10 = at4(&sc.a[16 + li][4 * lg]);
    const f32x4 zero = {0.0f, 0.0f, 0.0f, 0.0f};
    const f32x4 z = mfma_f32(a10, t0k, zero);      // -A10 T0
    const f32x4 t10k = mfma_f32(t1r, z, zero);     // T10 [4 lg + r][li]
#pragma unroll
    for (int r = 0; r < 4; ++r) sc.t[2][4 * lg + r][li] = t10k[r];
    // P = P0 T, transposed (T^T P0^T): row li, columns 4 lg + r
    f32x4 pt[3];
    pt[0] = mfma_f32(t0k, p0[0], zero);
    pt[1] = mfma_f32(t10k, p0[2], mfma_f32(t0k, p0[1], zero));
    pt[2] = mfma_f32(t1k, p0[2], zero);
    lds_order();
    const f32x4 t10r = at4(&sc.t[2][li][4 * lg]);
    const f32x4 b0 = at4(&sc.beta[4 * lg]);
    const f32x4 b1 = at4(&sc.beta[16 + 4 * lg]);
    lds_order();   // the planes may take the scratch's place: its last reads are above
    // to the planes: tile (mt, nt), row li, columns 4 lg ..
    auto put = [&](int base, int mt, int nt, f32x4 x) __attribute__((always_inline)) {
      const Split4 sp = split4(x);
      uint8_t* const at = rec + base + (lg >> 1) * 8 + li * 16 +
                          (nt == 0 ? (lg & 1) * 512 + mt * 256 : 3072 + (lg & 1) * 256);
#pragma unroll
      for (int pl = 0; pl < 3; ++pl)
        *reinterpret_cast<uint2*>(at + pl * (nt == 0 ? 1024 : 512)) = sp.p[pl];
    };
    put(Record::kT, 0, 0, t0r * b0);
    put(Record::kT, 1, 0, t10r * b0);
    put(Record::kT, 1, 1, t1r * b1);
    put(Record::kP, 0, 0, pt[0] * b0);
    put(Record::kP, 1, 0, pt[1] * b0);
    put(Record::kP, 1, 1, pt[2] * b1);
  }
}

// The records of every chunk in a launch of their own, one wave per (chunk, k-head) running the
// group's v-heads in turn: for longer prompts, where a head's workgroup would do its chunks'
// preparation in its own chain.  Bound by memory and by the latency of a unit's chain: at
// 32 x 1024 tokens, 32 v-heads, 114 us for 0.59 GB (134 us at four waves a SIMD, which spills),
// where a workgroup of four waves with a barrier per phase took 169 us (0.69 GB, with the
// planes' zero rows and the decay's sums in 32 bits).
template <bool DtBf16, bool Wide>
__global__ __launch_bounds__(kThreads) __attribute__((amdgpu_waves_per_eu(3, 3)))
void chunk_prep_heads_kernel(const DecodeParams p, int num_sequences, float* ws,
                             const int32_t* chunk_start, const int32_t* form, int records) {
  if (form != nullptr && *form == 0) return;
  __shared__ __attribute__((aligned(16))) PrepScratch scratch[kWaves];
  const int lane = threadIdx.x & 63;
  const int wave = __builtin_amdgcn_readfirstlane(static_cast<int>(threadIdx.x) >> 6);
  const int64_t unit = static_cast<int64_t>(blockIdx.x) * kWaves + wave;   // chunk * H + k-head
  const int g = static_cast<int>(unit / p.num_k_heads);
  if (g >= records) return;
  const int key_head = static_cast<int>(unit - static_cast<int64_t>(g) * p.num_k_heads);
  int seq = 0, t0 = 0, len = 0;
  if (!find_chunk<kTok>(p.cu, chunk_start, num_sequences, g, seq, t0, len)) return;
  PrepScratch& sc = scratch[wave];
  PrepGates gates, next;
  prep_gates<DtBf16>(next, p, t0, len, key_head * p.group, lane);
  PrepTiles tiles;
  {
    PrepInputs in;
    prep_fetch<Wide>(in, p, t0, len, key_head, lane);
    prep_tiles(tiles, in, p.scale, len, sc, lane);
  }
  for (int member = 0; member < p.group; ++member) {
    const int head = key_head * p.group + member;
    gates = next;
    if (member + 1 < p.group) prep_gates<DtBf16>(next, p, t0, len, head + 1, lane);
    lds_order();
    prep_head(tiles, gates, len, sc,
              reinterpret_cast<uint8_t*>(ws) +
                  (static_cast<int64_t>(g) * p.num_v_heads + head) * Record::kBytes, lane);
    lds_order();   // (the next v-head rewrites the scratch)
  }
}

// Own: the workgroup prepares its chunks itself (no workspace), a wave per chunk, four at a
// time; else their records are in `ws`.
template <bool Own, bool DtBf16, bool WBf16, bool Wide>
__global__ __launch_bounds__(kThreads) __attribute__((amdgpu_waves_per_eu(2, 2)))
void chunk_heads_kernel(const DecodeParams p, int num_sequences, const float* ws,
                        const int32_t* chunk_start, const int32_t* form, int records) {
  if (form != nullptr && *form == 0) return;   // (another form's batch)
  using R = Record;
  // Workgroups go to the 8 XCDs round-robin by id; the v-heads of one (sequence, k-head) read
  // the same q and k, so they are given ids on one XCD.
  const int xcd = blockIdx.x & 7;
  const int rank = blockIdx.x >> 3;
  const int unit = (rank / p.group) * 8 + xcd;
  if (unit >= num_sequences * p.num_k_heads) return;
  const int seq = unit / p.num_k_heads;
  const int key_head = unit - seq * p.num_k_heads;
  const int head = key_head * p.group + rank % p.group;
  const int tid = threadIdx.x;
  const int lane = tid & 63;
  const int w = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int lj = lane & 31;
  const int hi = lane >> 5;
  const int bos = p.cu[seq];
  const int eos = p.cu[seq + 1];
  const int slot = p.indices[seq];
  const bool from_slot = slot > 0 && p.has_initial[seq] != 0;
  const int gbase = Own ? 0 : chunk_start[seq];
  // (bounded by the records the workspace holds, whatever cu_seqlens says)
  const int chunks = min((eos - bos + kTok - 1) / kTok, Own ? 0x7fffffff : max(records - gbase, 0));

  constexpr int kRing = Own ? kWaves : 1;
  // In LDS a record is as it was prepared (Own), its step 1 zeroed as it is read, or, where the
  // room is there, with the zero rows: T's and P's plane i of step u at 3072 u + 1024 i (7 us of
  // 583 at 32 x 1024).
  constexpr int kLdsP = Own ? R::kP : 6144;
  constexpr int kLdsScales = Own ? R::kScales : 12288;
  constexpr int kLdsRecord = kLdsScales + R::kBytes - R::kScales;
  __shared__ __attribute__((aligned(16))) uint8_t sK[kTileSize];
  __shared__ __attribute__((aligned(16))) uint8_t sQ[kTileSize];
  // v of the chunk, then in its place the raw outputs (a wave reads and writes its own 32
  // columns of both); two, as the norm reads one while the next chunk's v arrives
  __shared__ __attribute__((aligned(16))) uint8_t sV[2][kTileSize];
  __shared__ __attribute__((aligned(16))) uint8_t sRec[kRing][kLdsRecord];   // chunk c's in c % kRing
  __shared__ __attribute__((aligned(16))) float sW[kDim];

  if (tid < kDim) sW[tid] = load_param(p.norm_weight, tid, WBf16);

  // ---- operands of one chunk, in registers on their way to LDS ----
  const uint32_t row_bytes = static_cast<uint32_t>(p.qkv_row) * 2;
  const int srow = tid >> 4;         // row (+ 16 for the second piece) and piece of this thread
  const int spiece = tid & 15;
  const uint32_t src = srow * row_bytes + spiece * 16;
  const int q_col = key_head * kTileRow;
  const int k_col = (p.num_k_heads + key_head) * kTileRow;
  const int v_col = (2 * p.num_k_heads + head) * kTileRow;
  const int qkv_bytes = (2 * p.num_k_heads + p.num_v_heads) * kTileRow;
  const uint32_t dst = srow * kTileRow + ((spiece ^ swizzle(srow)) << 4);
  auto lds_at = [](int byte) __attribute__((always_inline)) {   // of a record's byte (not Own)
    const int base = byte < R::kP ? 0 : kLdsP;
    const int at = byte < R::kP ? byte : byte - R::kP;
    const int step1 = at - 3072;
    return base + (at < 3072 ? at
                             : 3072 + (step1 >> 9) * 1024 + ((step1 >> 8) & 1) * 512 + 256 + (step1 & 255));
  };
  const int rec_at[2] = {lds_at(tid * 16), lds_at(4096 + tid * 16)};
  const int rest_at = lds_at(8192 + tid * 4);
  if constexpr (!Own) {
    for (int i = tid; i < 2 * 3 * 2 * 16; i += kThreads)   // matrix, plane, hi, 16-byte piece
      *reinterpret_cast<u32x4*>(sRec[0] + (i / 96) * kLdsP + 3072 + ((i / 32) % 3) * 1024 +
                                ((i >> 4) & 1) * 512 + (i & 15) * 16) = u32x4{0u, 0u, 0u, 0u};
  }
  struct Staged {
    u32x4 q[2], k[2], v[2], rec[2];
    uint32_t rest[2];   // the record's last 1.5 KiB
  };
  // Where chunk c's operands are (past the last chunk: resources over 0 bytes, whose loads
  // return zeros), and its load i of 6 (Own) or 10.
  struct Source {
    __amdgpu_buffer_rsrc_t rows, rec;
    uint32_t at[2];
  };
  auto source = [&](int c) __attribute__((always_inline)) {
    Source x;
    const int t0 = bos + min(c, max(chunks - 1, 0)) * kTok;
    const int live = c < chunks ? min(kTok, eos - t0) : 0;   // rows of the chunk
    x.rows = __builtin_amdgcn_make_buffer_rsrc(
        const_cast<uint16_t*>(p.qkv + static_cast<int64_t>(t0) * p.qkv_row), 0,
        live > 0 ? (live - 1) * static_cast<int>(row_bytes) + qkv_bytes : 0, 0x00020000);
    if constexpr (!Own)
      x.rec = record_resource(
          ws + (static_cast<int64_t>(gbase + min(c, max(chunks - 1, 0))) * p.num_v_heads + head) *
                   (R::kBytes / 4),
          c < chunks ? R::kBytes : 0);
    // rows past the chunk's end: an offset past the resource, so zeros
#pragma unroll
    for (int i = 0; i < 2; ++i) x.at[i] = srow + 16 * i < live ? src + i * 16 * row_bytes : 0xfffff000u;
    return x;
  };
  auto fetch = [&](Staged& x, const Source& from, int i) __attribute__((always_inline)) {
    if (i < 2)
      x.k[i] = load_piece<Wide>(from.rows, from.at[i], k_col);
    else if (i < 4)
      x.q[i - 2] = load_piece<Wide>(from.rows, from.at[i - 2], q_col);
    else if (i < 6)
      x.v[i - 4] = load_piece<Wide>(from.rows, from.at[i - 4], v_col);
    else if (Own)
      return;
    else if (i < 8)
      x.rec[i - 6] = load16u(from.rec, tid * 16 + (i - 6) * 4096, 0);
    else   // (past the record's end: zeros)
      x.rest[i - 8] = __builtin_amdgcn_raw_buffer_load_b32(from.rec, tid * 4 + 8192 + (i - 8) * 1024, 0, 0);
  };
  auto put = [&](const Staged& x, int buf) __attribute__((always_inline)) {
#pragma unroll
    for (int i = 0; i < 2; ++i) {
      *reinterpret_cast<u32x4*>(sK + dst + i * 16 * kTileRow) = x.k[i];
      *reinterpret_cast<u32x4*>(sQ + dst + i * 16 * kTileRow) = x.q[i];
      *reinterpret_cast<u32x4*>(sV[buf] + dst + i * 16 * kTileRow) = x.v[i];
    }
    if constexpr (!Own) {
#pragma unroll
      for (int i = 0; i < 2; ++i) *reinterpret_cast<u32x4*>(sRec[0] + rec_at[i]) = x.rec[i];
      *reinterpret_cast<uint32_t*>(sRec[0] + rest_at) = x.rest[0];
      if (tid < (R::kBytes - R::kScales) / 4)
        *reinterpret_cast<uint32_t*>(sRec[0] + kLdsScales + tid * 4) = x.rest[1];
    }
  };
  static_assert(R::kScales == 8192 + 1024 && R::kBytes - R::kScales <= 1024, "the record's loads");

  // The chunk that this wave prepares first: its loads go out ahead of the state's and return
  // first.
  PrepInputs first;
  PrepGates first_gates;
  auto prep_rows = [&](int c) __attribute__((always_inline)) { return min(kTok, eos - bos - c * kTok); };
  auto prepare_fetch = [&](PrepInputs& in, PrepGates& gates, int c) __attribute__((always_inline)) {
    prep_fetch<Wide>(in, p, bos + c * kTok, prep_rows(c), key_head, lane);
    prep_gates<DtBf16>(gates, p, bos + c * kTok, prep_rows(c), head, lane);
  };
  auto prepare = [&](const PrepInputs& in, const PrepGates& gates, int c) __attribute__((always_inline)) {
    PrepScratch& sc = *reinterpret_cast<PrepScratch*>(sRec[w & (kRing - 1)]);
    PrepTiles tiles;
    prep_tiles(tiles, in, p.scale, prep_rows(c), sc, lane);
    lds_order();
    prep_head(tiles, gates, prep_rows(c), sc, sRec[w & (kRing - 1)], lane);
  };
  if (Own && w < chunks) prepare_fetch(first, first_gates, w);
  asm volatile("" ::: "memory");
  Staged staged;
  if (chunks > 0) {
    const Source from = source(0);
#pragma unroll
    for (int i = 0; i < 10; ++i) fetch(staged, from, i);
  }
  asm volatile("" ::: "memory");

  // st[T][8 u + 4 h + r] = S[32 w + lj][32 T + 16 u + 8 hi + 4 h + r]
  f32x16 st[4];
  {
    const __amdgpu_buffer_rsrc_t srs = state_resource(p, slot, head, from_slot);
    const uint32_t at = static_cast<uint32_t>(((32 * w + lj) * kDim + 8 * hi) * 4);
#pragma unroll
    for (int T = 0; T < 4; ++T)
#pragma unroll
      for (int q = 0; q < 4; ++q) {
        const f32x4 x = load16(srs, at + (32 * T + 16 * (q >> 1) + 4 * (q & 1)) * 4, 0);
#pragma unroll
        for (int r = 0; r < 4; ++r) st[T][4 * q + r] = x[r];
      }
  }

  // lane addresses of the operands (the swizzle's parts that depend on the step are XORed in)
  const uint32_t a_at = lj * kTileRow + ((hi ^ swizzle(lj)) << 4);       // ^ ((4 T + 2 u) << 4)
  const int m = lane & 15;
  const int c16 = (lane >> 4) & 1;
  const uint32_t tr_row = (4 * hi + (m >> 2)) * kTileRow;
  // transposed k: rows 16 u + 8 h + .., columns key_of(16 c16 + ..)   ^ (T << 6) ^ (h << 5)
  const uint32_t kt_at =
      tr_row + (((2 * c16 + (m & 1)) ^ ((m >> 2) << 2) ^ hi) << 4) + ((m >> 1) & 1) * 8;
  // transposed v: rows 8 q + .., the wave's columns   ^ ((q & 1) << 5)
  const uint32_t vt_at =
      tr_row + (((4 * w + 2 * c16 + ((m & 3) >> 1)) ^ ((m >> 2) << 2) ^ hi) << 4) + (m & 1) * 8;
  // raw outputs: row 8 q + 4 hi + e, column 32 w + lj   ^ (e << 6) ^ ((q & 1) << 5)
  const uint32_t raw_at =
      4 * hi * kTileRow + (((4 * w + (lj >> 3)) ^ hi) << 4) + (lj & 7) * 2;

  // The norm of chunk c - 1 runs beside chunk c's products; thread = (token, 16 columns).
  // Resources over the chunk's rows of gate and out (before the first chunk: over 0 bytes,
  // whose loads return zeros and whose stores are dropped).
  const int ntok = tid >> 3;
  const int ncol = (tid & 7) * 16;
  const uint32_t gate_bytes = static_cast<uint32_t>(p.gate_row) * 2;
  const uint32_t out_bytes = static_cast<uint32_t>(p.num_v_heads) * kTileRow;
  const uint32_t raw0_at = ntok * kTileRow + (((ncol >> 3) ^ swizzle(ntok)) << 4);
  const uint32_t raw1_at = ntok * kTileRow + ((((ncol >> 3) + 1) ^ swizzle(ntok)) << 4);
  auto chunk_rows = [&](const uint16_t* base, int64_t row, int c) __attribute__((always_inline)) {
    const int t0 = bos + max(c, 0) * kTok;
    return __builtin_amdgcn_make_buffer_rsrc(
        const_cast<uint16_t*>(base + static_cast<int64_t>(t0) * row + static_cast<int64_t>(head) * kDim),
        0, c >= 0 ? (min(kTok, eos - t0) - 1) * static_cast<int>(row * 2) + kTileRow : 0, 0x00020000);
  };
  auto load_gate = [&](u32x4 (&to)[2], int c) __attribute__((always_inline)) {
    const __amdgpu_buffer_rsrc_t rows = chunk_rows(p.gate, p.gate_row, c);
#pragma unroll
    for (int i = 0; i < 2; ++i)
      to[i] = load_piece<Wide>(rows, ntok * gate_bytes + ncol * 2 + 16 * i, 0);
  };
  auto store_norm = [&](const Norm& norm, int c) __attribute__((always_inline)) {
    const __amdgpu_buffer_rsrc_t rows = chunk_rows(p.out, static_cast<int64_t>(p.num_v_heads) * kDim, c);
#pragma unroll
    for (int i = 0; i < 2; ++i) {
      const int at = static_cast<int>(ntok * out_bytes) + ncol * 2 + 16 * i;
      if constexpr (Wide) {
        __builtin_amdgcn_raw_buffer_store_b128(norm.y[i], rows, at, 0, 0);
      } else {
#pragma unroll
        for (int d = 0; d < 4; ++d) {
          __builtin_amdgcn_raw_buffer_store_b16(static_cast<uint16_t>(norm.y[i][d]), rows, at + 4 * d, 0, 0);
          __builtin_amdgcn_raw_buffer_store_b16(static_cast<uint16_t>(norm.y[i][d] >> 16), rows, at + 4 * d + 2, 0, 0);
        }
      }
    }
  };

  if (Own && w < chunks) prepare(first, first_gates, w);
  // (the state's loads are waited for here: inside the loop the waits would be counted
  // against later chunks' loads)
#pragma unroll
  for (int T = 0; T < 4; ++T) pin(st[T]);
  Norm norm;
  u32x4 gate[2] = {};   // of the chunk whose raw outputs are next to be normalised
  for (int c = 0; c < chunks; ++c) {
    const int buf = c & 1;
    if (Own && c > 0 && (c & (kWaves - 1)) == 0 && c + w < chunks) {
      PrepInputs in;
      PrepGates gates;
      prepare_fetch(in, gates, c + w);
      prepare(in, gates, c + w);
    }
    const uint8_t* const rec = sRec[c & (kRing - 1)];
    const f32x4* const scales = reinterpret_cast<const f32x4*>(rec + kLdsScales) + hi;
    put(staged, buf);
    lds_barrier();   // the chunk's operands and the previous chunk's raw outputs are in LDS

    // The next chunk's loads go out between the products below (a burst of them holds the wave
    // until the last is accepted, and in registers before they are due).
    const Source from = source(c + 1);
    auto prefetch = [&](int i) __attribute__((always_inline)) {
      asm volatile("" ::: "memory");
      fetch(staged, from, i);
      asm volatile("" ::: "memory");
    };
    const uint8_t* const last_raw = sV[buf ^ 1];
    auto normalise = [&](int i) __attribute__((always_inline)) {
      norm.slice(i, last_raw + raw0_at, last_raw + raw1_at, sW + ncol, p.eps);
    };

    // Y = K S^T and O = Q S^T: step n = 2 T + u takes k = 32 T + 16 u + ..; beside its products
    // the next step's operands are read and its S split, and S is scaled once split.  The last
    // two steps' O products come after Y's, beside X = V - diag(ws) Y (ws and v are zero past
    // the sequence's end) and its split.
    f32x16 y, o;
    auto operand = [&](const uint8_t* tile, int n) __attribute__((always_inline)) {
      return *reinterpret_cast<const bf16x8*>(tile + (a_at ^ (n << 5)));
    };
    const float gamma = *reinterpret_cast<const float*>(rec + kLdsScales + R::kGamma - R::kScales);
    Split8 now, next, held;
    bf16x8 ka = operand(sK, 0), qa = operand(sQ, 0), q6;
    now.set(quad(st[0], 0), quad(st[0], 1));
    now.all();
    bf16x4 vt[4];
    f32x4 wsc[4], xs[4];
    auto scale_state = [&](int T, int u) __attribute__((always_inline)) {
#pragma unroll
      for (int e = 8 * u; e < 8 * u + 8; ++e) st[T][e] *= gamma;
      pin(st[T]);
    };
#pragma unroll
    for (int n = 0; n < 8; ++n) {
      const bf16x8 kc = ka, qc = qa;
      if (n == 1 || n == 3 || n == 5) prefetch(n >> 1);
      if (n < 7) {
        ka = operand(sK, n + 1);
        qa = operand(sQ, n + 1);
        next.set(quad(st[(n + 1) >> 1], 2 * ((n + 1) & 1)), quad(st[(n + 1) >> 1], 2 * ((n + 1) & 1) + 1));
      }
      if (n < 6) {
        if (n == 0) product<true>(kc, now.plane(2), y); else product(kc, now.plane(2), y);
        next.stage(0);
        if (n == 0) product<true>(qc, now.plane(2), o); else product(qc, now.plane(2), o);
        next.stage(1);
        product(kc, now.plane(1), y);
        next.stage(2);
        product(qc, now.plane(1), o);
        next.stage(3);
        product(kc, now.plane(0), y);
        next.stage(4);
        product(qc, now.plane(0), o);
        if (n > 0) scale_state((n - 1) >> 1, (n - 1) & 1);
        now = next;
      } else if (n == 6) {
        product(kc, now.plane(2), y);
        next.stage(0);
        next.stage(1);
        product(kc, now.plane(1), y);
        next.stage(2);
        next.stage(3);
        product(kc, now.plane(0), y);
        next.stage(4);
        held = now;
        q6 = qc;
        now = next;
      } else {
#pragma unroll
        for (int q = 0; q < 4; ++q)
          vt[q] = read_tr(sV[buf] + (vt_at ^ ((q & 1) << 5)) + 8 * q * kTileRow);
#pragma unroll
        for (int q = 0; q < 4; ++q) wsc[q] = scales[R::kWs + 2 * q];
        product(kc, now.plane(2), y);
        scale_state(2, 1);
        product(kc, now.plane(1), y);
        scale_state(3, 0);
        product(kc, now.plane(0), y);
        scale_state(3, 1);
        product(q6, held.plane(2), o);
#pragma unroll
        for (int q = 0; q < 4; ++q) {
#pragma unroll
          for (int r = 0; r < 4; ++r) xs[q][r] = static_cast<float>(vt[q][r]);
          pin(xs[q]);
        }
        product(q6, held.plane(1), o);
        product(q6, held.plane(0), o);
#pragma unroll
        for (int q = 0; q < 4; ++q) {
#pragma unroll
          for (int r = 0; r < 4; ++r) xs[q][r] = fmaf(-wsc[q][r], y[4 * q + r], xs[q][r]);
          pin(xs[q]);
        }
        held.set(xs[0], xs[1]);
        next.set(xs[2], xs[3]);
        held.stage(0);
        held.stage(1);
        product(qc, now.plane(2), o);
        held.stage(2);
        product(qc, now.plane(1), o);
        held.stage(3);
        product(qc, now.plane(0), o);
        held.stage(4);
      }
    }
    // V_new = T X and O = diag(sq) O + P X, T and P as planes (held, next: X's), the smallest
    // products of a step first
    auto weight = [&](int base, int u, int i) __attribute__((always_inline)) {
      if (u == 0 || !Own)
        return *reinterpret_cast<const bf16x8*>(rec + base + u * 3072 + i * 1024 + lane * 16);
      u32x4 x = *reinterpret_cast<const u32x4*>(rec + base + 3072 + i * 512 + (16 * hi + (lj & 15)) * 16);
#pragma unroll
      for (int d = 0; d < 4; ++d) x[d] = lj < 16 ? 0u : x[d];   // rows above the triangle
      return __builtin_bit_cast(bf16x8, x);
    };
    // the six products of a step; NEXT, UN: the matrix and step whose planes replace the
    // current ones as they fall free
#define LD_PRODUCTS(FIRST, ACC, X, SLOT, NEXT, UN)                                            \
  product<FIRST>(wt[2], X.plane(0), ACC); wt[2] = weight(NEXT, UN, 2); SLOT(0);               \
  product(wt[1], X.plane(1), ACC); SLOT(1);                                                   \
  product(wt[0], X.plane(2), ACC); SLOT(2);                                                   \
  product(wt[1], X.plane(0), ACC); wt[1] = weight(NEXT, UN, 1); SLOT(3);                      \
  product(wt[0], X.plane(1), ACC); SLOT(4);                                                   \
  product(wt[0], X.plane(0), ACC); wt[0] = weight(NEXT, UN, 0); SLOT(5);
    f32x16 vn;
    bf16x8 wt[3];
#pragma unroll
    for (int i = 0; i < 3; ++i) wt[i] = weight(R::kT, 0, i);
    f32x4 sq[4], ck[4];
#pragma unroll
    for (int q = 0; q < 4; ++q) sq[q] = scales[R::kSq + 2 * q];
    auto slot_t0 = [&](int i) __attribute__((always_inline)) {
      if (i < 5) next.stage(i);
      if (i % 2 == 0) prefetch(3 + i / 2);
    };
    LD_PRODUCTS(true, vn, held, slot_t0, R::kT, 1)
    auto slot_t1 = [&](int i) __attribute__((always_inline)) {
      if (i < 2) {
#pragma unroll
        for (int q = 2 * i; q < 2 * i + 2; ++q)
#pragma unroll
          for (int r = 0; r < 4; ++r) o[4 * q + r] *= sq[q][r];
        pin(o);
      } else {
        normalise(i - 2);
      }
    };
    LD_PRODUCTS(false, vn, next, slot_t1, kLdsP, 0)
#pragma unroll
    for (int q = 0; q < 2; ++q) ck[q] = scales[R::kCk + 2 * q];
    // beside P X: the split of ck V_new (now: step 0, last: step 1)
    Split8 last;
    auto scaled_vn = [&](int q, Split8& to) __attribute__((always_inline)) {
      f32x4 lo = quad(vn, q) * ck[q];
      f32x4 hi = quad(vn, q + 1) * ck[q + 1];
      pin(lo);   // rounded: the first remainder is of the product's fp32 value
      pin(hi);
      to.set(lo, hi);
    };
    auto slot_p0 = [&](int i) __attribute__((always_inline)) {
      if (!Own && i % 3 == 0) prefetch(6 + i / 3);
      if (i == 0) {
        normalise(4);
      } else if (i == 1) {
        scaled_vn(0, now);
        now.stage(0);
      } else {
        now.stage(i - 1);
      }
      if (i >= 4) ck[i - 2] = scales[R::kCk + 2 * (i - 2)];
    };
    LD_PRODUCTS(false, o, held, slot_p0, kLdsP, 1)
    auto slot_p1 = [&](int i) __attribute__((always_inline)) {
      if (!Own && i % 3 == 0) prefetch(8 + i / 3);
      if (i == 0)
        scaled_vn(2, last);
      else
        last.stage(i - 1);
    };
    LD_PRODUCTS(false, o, next, slot_p1, kLdsP, 1)
#undef LD_PRODUCTS
    // S' = exp(G_n-1) S + K^T (ck V_new); beside it the raw outputs to LDS, rounded to bf16, and
    // the previous chunk's norm
    auto key_t = [&](int i) __attribute__((always_inline)) {   // tile i % 4, step i / 4
      const int T = i & 3, u = i >> 2;
      const bf16x4 k0 = read_tr(sK + (kt_at ^ (T << 6)) + 16 * u * kTileRow);
      const bf16x4 k1 = read_tr(sK + (kt_at ^ (T << 6) ^ (1 << 5)) + (16 * u + 8) * kTileRow);
      return __builtin_shufflevector(k0, k1, 0, 1, 2, 3, 4, 5, 6, 7);
    };
    norm.gate[0] = gate[0];
    norm.gate[1] = gate[1];
    asm volatile("" ::: "memory");
    load_gate(gate, c);
    asm volatile("" ::: "memory");
    bf16x8 kt = key_t(0);
#pragma unroll
    for (int i = 0; i < 8; ++i) {
      const bf16x8 kc = kt;
      if (i < 7) kt = key_t(i + 1);
#pragma unroll
      for (int pl = 2; pl >= 0; --pl) {
        product(kc, i < 4 ? now.plane(pl) : last.plane(pl), st[i & 3]);
        const int n = 3 * i + 2 - pl;   // 0 .. 23
        if (n < 2) normalise(5 + n);
        else if (n >= 4 && n < 20) normalise(n + 3);
        if (n >= 2 && n % 3 == 2) {   // two tokens in each of eight slots
#pragma unroll
          for (int e = 0; e < 2; ++e) {
            const int tok = 2 * ((n - 2) / 3) + e, q = tok >> 2;
            *reinterpret_cast<uint16_t*>(sV[buf] + (raw_at ^ ((tok & 3) << 6) ^ ((q & 1) << 5)) +
                                         (8 * q + (tok & 3)) * kTileRow) = to_bf16(o[tok]);
          }
        }
      }
    }
    store_norm(norm, c - 1);
    lds_barrier();   // every read of the operands is done
  }
  if (slot > 0) {
    float* tile = p.state + static_cast<int64_t>(slot) * p.state_slot +
                  static_cast<int64_t>(head) * kDim * kDim + (32 * w + lj) * kDim + 8 * hi;
#pragma unroll
    for (int T = 0; T < 4; ++T)
#pragma unroll
      for (int q = 0; q < 4; ++q)
        *reinterpret_cast<f32x4*>(tile + 32 * T + 16 * (q >> 1) + 4 * (q & 1)) = quad(st[T], q);
  }
  if (chunks > 0) {   // the last chunk's norm (its raw outputs are complete past the barrier)
    norm.gate[0] = gate[0];
    norm.gate[1] = gate[1];
    const uint8_t* const last_raw = sV[(chunks - 1) & 1];
#pragma unroll
    for (int i = 0; i < 23; ++i)
      norm.slice(i, last_raw + raw0_at, last_raw + raw1_at, sW + ncol, p.eps);
    store_norm(norm, chunks - 1);
  }
}

}  // namespace

int launch_chunk_heads(const DecodeParams& p, int num_sequences, bool own, float* ws,
                       const int32_t* chunk_start, const int32_t* form, int records,
                       bool dt_bf16, bool w_bf16, hipStream_t stream) {
  const int64_t units = static_cast<int64_t>(num_sequences) * p.num_k_heads;
  const int64_t groups = (units + 7) / 8 * 8 * p.group;
  const int64_t prep_groups = (static_cast<int64_t>(records) * p.num_k_heads + kWaves - 1) / kWaves;
  if (groups > 0x7fffffff || prep_groups > 0x7fffffff)
    return fail(LD_ERR_INVALID_ARGUMENT, "prefill too large");
  const auto at16 = [](const void* base, int64_t row) {
    return (reinterpret_cast<uintptr_t>(base) & 15) == 0 && (row & 7) == 0;
  };
  const bool wide_qkv = at16(p.qkv, p.qkv_row);
  const bool wide = wide_qkv && at16(p.gate, p.gate_row) && at16(p.out, 0);
#define LD_HEADS(O, D, W) (wide ? chunk_heads_kernel<O, D, W, true> : chunk_heads_kernel<O, D, W, false>)
  const auto kernel = !own      ? (w_bf16 ? LD_HEADS(false, false, true) : LD_HEADS(false, false, false))
                      : dt_bf16 ? (w_bf16 ? LD_HEADS(true, true, true) : LD_HEADS(true, true, false))
                                : (w_bf16 ? LD_HEADS(true, false, true) : LD_HEADS(true, false, false));
#undef LD_HEADS
  if (!own) {
    const auto prep = dt_bf16 ? (wide_qkv ? chunk_prep_heads_kernel<true, true> : chunk_prep_heads_kernel<true, false>)
                              : (wide_qkv ? chunk_prep_heads_kernel<false, true> : chunk_prep_heads_kernel<false, false>);
    hipLaunchKernelGGL(prep, dim3(static_cast<uint32_t>(prep_groups)), dim3(kThreads), 0, stream, p,
                       num_sequences, ws, chunk_start, form, records);
  }
  hipLaunchKernelGGL(kernel, dim3(static_cast<uint32_t>(groups)), dim3(kThreads), 0, stream, p,
                     num_sequences, ws, chunk_start, form, records);
  return check_launch("ld_gdn_prefill (chunked)");
}

}  // namespace ld
