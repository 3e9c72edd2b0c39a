// gemm_skinny_impl.hpp -- y = x W^T for a few tokens (batch_m 2 .. 64), the packed
// weights decoded straight into MFMA operands: one launch, no workspace.
//
// Reference behaviour: CodebookMatrix::gemv_cpu (codebook.rs:350-417), the
// Q8_0 / Q4_0 block dots (llm_prefill.rs:45-54, q4_0.rs:99-147) and, for
// larger batches, PackedTensor::gemm_cpu (llm_prefill.rs:156-255); with the
// gated epilogue, the runner's [gate; up] step (llm_cpu.rs:448-464).
//
// A call of this size should cost the stream of its packed weights.  With one
// FMA per weight per token on the VALU it costs the arithmetic instead, so
// the products go to v_mfma_f32_16x16x32_bf16: 16 tokens (A, rows past the
// batch repeat the last one and are never stored) by 16 weight rows (B).
//
// Exact operands.  bf16 has f32's range, so no operand needs a scale; a second
// term of an f32 value is kept times 2^8 and a third times 2^16, as bf16 ends at
// 2^-133 and f32 at 2^-149 (unscaled, activations of 2^-126 came out 4.5e-3 off):
//   * g64: an f16 table entry is two bf16 terms (8 + 3 significant bits);
//   * cb4: an f32 centroid is three (8 + 8 + 8 bits); a 128-column group's
//     products are summed in fresh accumulators and scaled once, as the
//     reference's GEMV does; the CSR residuals are added on the VALU;
//   * Q8_0 / Q4_0: the int8 value / q - 8 is one term; a 32-column block's
//     products are summed in a fresh accumulator and scaled once;
//   * bf16 activations are one term, f32 ones three.
// Every product of two terms is exact in fp32.  Of an f32 activation's terms
// the product of the two last (2^-32 of the whole) is left out where a weight
// has three.  The product of the leading terms has accumulators of its own:
// an infinite activation makes it infinite with the right sign while the
// other products may be NaN (0 * Inf), so an infinite leading sum is the
// tile's.  An output that is not finite after all is computed anew from its
// definition (plain_dot).
//
// Mapping.  A workgroup is eight waves: RG row groups of 16 weight rows by KW
// = 8 / RG K-ways.  K is walked in phases of PH columns: the phase's
// activations are staged in LDS once for all waves (rows padded by 16 bytes:
// the 16 rows of a fragment read fall in distinct banks), the next phase's
// activations and weights are requested before a phase is multiplied, and
// wave kw takes the phase's chunks kw, kw + KW, ...  The K-ways are added
// through LDS in a fixed tree, so results do not depend on timing, and a
// chunk's sum is formed apart before it is added: short chains of roundings
// (relative error of 2048-column products 0.7 .. 0.9e-7, the kernels before 0.7
// .. 1.05e-7).
//
// Weights.  Lane l (row l % 16, group g = l / 16) loads 16 bytes (cb4, Q4_0:
// 32 columns) or 32 (Q8_0; g64: 64 columns and the whole table of its
// 64-column group), 64 or 128 contiguous bytes of a row per instruction.
//   * cb4, g64: the lane's 8 columns of MFMA step j are 8 j .. 8 j + 7 of its
//     own contiguous range; the MFMA sums k in any order, so the activations
//     are read from LDS at the same columns.
//   * Q4_0, Q8_0: the k slots of one MFMA must share a block, so the four
//     lane groups exchange dwords (v_permlane32_swap / v_permlane16_swap, a
//     4 x 4 transpose in four instructions): afterwards each group holds its
//     quarter of every block.  Q4_0's quarter is bytes 4 g .. 4 g + 3, i.e.
//     columns 4 g + b and 16 + 4 g + b; the activations are staged in that
//     order (column c of a block at 2 (c % 16) + c / 16).
// What bounds it.  Up to a few thousand rows a call is one round of workgroups
// and their latency: a load, a barrier, one to eight chunks, the sum (lab
// copies without the MFMAs or the cb4 table reads ran level at 2048 x 12288; the
// cb4 residuals cost 2 of its 11 us: a dependent load and the gathers).  So the
// tiles are made small where rows are few: half tiles (Tile's HALF) put 256
// workgroups on a 2048-row matrix instead of 128 (M = 4, 6144 -> 2048: cb4
// 12.3 -> 8.2 us, g64 12.3 -> 7.5, Q4_0 9.0 -> 6.9; 2048 -> 2048 5.7 -> 4.2, -, 4.2
// -> 3.3), and three workgroups per CU are asked for up to 8 tokens (cb4 2048
// -> 12288, M = 4: 12.0 -> 11.2 us).  From 32768 rows the streaming form
// (skinny_stream_kernel) drops the per-tile latency (151936 x 2048, M = 4: cb4
// 178 -> 75 us, g64 133 -> 67 for 311 MB, Q4_0 67 -> 61).
//
// Decode through LDS: cb4 reads its table entry's three terms in one 8-byte
// read (16 entries on distinct banks); g64 builds its lane's table (two
// terms in a word, entry e of lane l at word 64 e + l: no conflicts); Q4_0
// reads both nibbles of a byte as a pair from a 256-word table.
#pragma once
#include <algorithm>
#include <type_traits>

#include "act.hpp"
#include "common.hpp"

#pragma clang fp contract(off)

namespace vxt {

namespace sk {

typedef float f32x4_t __attribute__((ext_vector_type(4)));
typedef __bf16 bf16x8_t __attribute__((ext_vector_type(8)));
typedef uint32_t u32x2 __attribute__((ext_vector_type(2)));
// The tables and planes in LDS are written and read through may_alias types
// of different widths.
typedef uint32_t __attribute__((may_alias)) u32_alias_t;
typedef u32x2 __attribute__((may_alias)) u32x2_alias_t;
typedef u32x4 __attribute__((may_alias)) u32x4_alias_t;
typedef uint16_t __attribute__((may_alias)) u16_alias_t;
typedef float __attribute__((may_alias)) f32_alias_t;
#define LDS_AS __attribute__((address_space(3)))
typedef LDS_AS u32_alias_t lds_u32;
typedef LDS_AS u32x2_alias_t lds_u32x2;
typedef LDS_AS u32x4_alias_t lds_u32x4;
typedef LDS_AS u16_alias_t lds_u16;
typedef LDS_AS f32_alias_t lds_f32;

constexpr int kWaves = 8;
constexpr int kThreads = 64 * kWaves;
constexpr uint32_t kStreamRows = 32768;
constexpr uint32_t kHalfRows = 4096;
constexpr uint32_t kHalfRowsF32 = 2048;   // one workgroup per CU: one round

// f32 as three bf16 terms, each the high half of a word (what the low halves
// hold is not read): v = h + m 2^-8 + l 2^-16 exactly, subnormals too.  Inf and
// NaN are h alone; canonicalising sets a NaN's quiet bit, so the cut keeps it one.
constexpr float kTerm1 = 1.0f / 256.0f, kTerm2 = 1.0f / 65536.0f;
__device__ __forceinline__ void split3(float v, uint32_t& h, uint32_t& m, uint32_t& l) {
  auto cut = [](float f) { return __uint_as_float(__float_as_uint(f) & 0xffff0000u); };
  const float r = __builtin_isfinite(v) ? (v - cut(v)) * 256.0f : 0.0f;
  h = __float_as_uint(__builtin_canonicalizef(v));
  m = __float_as_uint(r);
  l = __float_as_uint((r - cut(r)) * 256.0f);
}

__device__ __forceinline__ uint32_t lo_pair(uint32_t a, uint32_t b) { return __builtin_amdgcn_perm(b, a, 0x05040100u); }
__device__ __forceinline__ uint32_t hi_pair(uint32_t a, uint32_t b) { return __builtin_amdgcn_perm(b, a, 0x07060302u); }

__device__ __forceinline__ void swap32(uint32_t& a, uint32_t& b) {
  const auto r = __builtin_amdgcn_permlane32_swap(a, b, false, false);
  a = r[0];
  b = r[1];
}
__device__ __forceinline__ void swap16(uint32_t& a, uint32_t& b) {
  const auto r = __builtin_amdgcn_permlane16_swap(a, b, false, false);
  a = r[0];
  b = r[1];
}
// w[i] of lane group g becomes w[g] of lane group i: a 4 x 4 transpose over
// (lane group, register).
__device__ __forceinline__ void transpose4(uint32_t (&w)[4]) {
  swap32(w[0], w[2]);
  swap32(w[1], w[3]);
  swap16(w[0], w[1]);
  swap16(w[2], w[3]);
}

template <uint32_t KIND>
struct W;
template <>
struct W<KIND_CB4> {
  uint4 q;
  uint32_t sc;
};
template <>
struct W<KIND_G64> {
  uint4 q0, q1, l0, l1;
};
template <>
struct W<KIND_Q40> {
  uint4 q;
  uint32_t sc;
};
template <>
struct W<KIND_Q8> {
  uint4 a, b;
  uint32_t sc;
};

// Columns of one chunk (four lane groups), weight terms.
template <uint32_t KIND>
constexpr int kChunk = KIND == KIND_G64 ? 256 : 128;
template <uint32_t KIND>
constexpr int kTerms = KIND == KIND_CB4 ? 3 : KIND == KIND_G64 ? 2 : 1;

// Decode tables in LDS, ahead of the activations.
template <uint32_t KIND>
constexpr uint32_t kTabBytes = KIND == KIND_CB4 ? 384u : KIND == KIND_G64 ? kWaves * 4096u : KIND == KIND_Q40 ? 1024u : 0u;

using Args = SkinnyArgs;

// What a wave needs to multiply chunks of its 16 weight rows.
// HALF: 8 weight rows, up to 8 tokens; rows and tokens 8 .. 15 of an operand
// are rows and tokens 0 .. 7 again over the other half of a 2 x CH column
// chunk, so the diagonal quarters of the result hold the two halves' sums.
template <uint32_t KIND, int XT, int TT, bool HALF = false>
struct Tile {
  uint32_t base;        // decode tables in LDS
  uint32_t wave;
  uint32_t r, g, lane;
  uint32_t cols;
  uint32_t ctab;        // cb4: the row's centroid table
  bool skip_zero;       // cb4: a zero scale skips its group, whatever the activations
  uint32_t plane;       // bytes of one staged activation plane
  uint32_t arow[TT];    // the lane's token row of each token tile
  f32x4_t acc[TT], accl[TT], accr[TT];   // leading products; the others; cb4 residuals

  __device__ __forceinline__ void clear() {
#pragma unroll
    for (int i = 0; i < TT; ++i) acc[i] = accl[i] = accr[i] = f32x4_t{0.0f, 0.0f, 0.0f, 0.0f};
  }

  // One MFMA step: the B terms against the activations at column position c.
  // The lesser products go to an accumulator for each power of 2^-8 that the
  // terms' products carry (g64's two terms carry none), 2^-24 in lo[0]: shorter
  // chains of dependent MFMAs too.
  template <int WT>
  __device__ __forceinline__ void step(const bf16x8_t (&b)[WT], uint32_t c, f32x4_t (&hi)[TT], f32x4_t (&lo)[3][TT]) {
#pragma unroll
    for (int i = 0; i < TT; ++i) {
#pragma unroll
      for (int xt = 0; xt < XT; ++xt) {
        const bf16x8_t av = __builtin_bit_cast(bf16x8_t, *(lds_u32x4*)(size_t)(arow[i] + xt * plane + c * 2u));
#pragma unroll
        for (int wt = 0; wt < WT; ++wt) {
          if (wt + xt > 3) continue;
          if (wt + xt == 0) {
            hi[i] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(av, b[wt], hi[i], 0, 0, 0);
          } else {
            f32x4_t& l = lo[((KIND == KIND_CB4 ? wt : 0) + xt) % 3][i];
            l = __builtin_amdgcn_mfma_f32_16x16x32_bf16(av, b[wt], l, 0, 0, 0);
          }
        }
      }
    }
  }

  // The lesser products' sum of a chunk; sums that were never formed stay out.
  __device__ __forceinline__ float lesser(const f32x4_t (&lo)[3][TT], int i, int k) const {
    float v = KIND == KIND_G64 ? lo[0][i][k] : KIND == KIND_CB4 && XT > 1 ? lo[0][i][k] * (kTerm1 * kTerm2) : 0.0f;
    if constexpr (KIND == KIND_CB4 || XT > 1) v = __builtin_fmaf(lo[1][i][k], kTerm1, __builtin_fmaf(lo[2][i][k], kTerm2, v));
    return v;
  }

  // Weights of columns past the row's end, zeroed: an Inf or NaN there must
  // not meet the zero activations.  Dword d holds columns c + 2 d, c + 2 d + 1.
  __device__ __forceinline__ void mask_tail(uint32_t c, uint32_t (&d)[4]) const {
#pragma unroll
    for (uint32_t j = 0; j < 4; ++j) {
      const uint32_t k = c + 2u * j;
      d[j] &= k + 1u < cols ? ~0u : k < cols ? 0xffffu : 0u;
    }
  }

  // Chunk c of the rows, its activations at column position `at`.
  template <bool TAIL>
  __device__ __forceinline__ void chunk(const W<KIND>& w, uint32_t c, uint32_t at) {
    constexpr uint32_t CH = kChunk<KIND>;
    const f32x4_t z = {0.0f, 0.0f, 0.0f, 0.0f};
    if constexpr (KIND == KIND_CB4) {
      f32x4_t fh[TT], fl[3][TT];
#pragma unroll
      for (int i = 0; i < TT; ++i) fh[i] = fl[0][i] = fl[1][i] = fl[2][i] = z;
      const uint32_t wd[4] = {w.q.x, w.q.y, w.q.z, w.q.w};
#pragma unroll
      for (uint32_t j = 0; j < 4; ++j) {
        u32x2 e[8];
#pragma unroll
        for (int k = 0; k < 8; ++k) e[k] = *(lds_u32x2*)(size_t)((((wd[j] >> (4 * k)) & 15u) << 3) + ctab);
        uint32_t d[3][4];
#pragma unroll
        for (int k = 0; k < 4; ++k) {
          d[0][k] = lo_pair(e[2 * k].x, e[2 * k + 1].x);
          d[1][k] = hi_pair(e[2 * k].x, e[2 * k + 1].x);
          d[2][k] = lo_pair(e[2 * k].y, e[2 * k + 1].y);
        }
        bf16x8_t b[3];
#pragma unroll
        for (int k = 0; k < 3; ++k) {
          if constexpr (TAIL) mask_tail(c * CH + 32u * g + 8u * j, d[k]);
          const u32x4 v = {d[k][0], d[k][1], d[k][2], d[k][3]};
          b[k] = __builtin_bit_cast(bf16x8_t, v);
        }
        step(b, at + 32u * g + 8u * j, fh, fl);
      }
      const float s = c * CH < cols ? f16_to_f32(w.sc) : 0.0f;
      const bool skip = skip_zero && s == 0.0f;
#pragma unroll
      for (int i = 0; i < TT; ++i)
#pragma unroll
        for (int k = 0; k < 4; ++k) {
          acc[i][k] = skip ? acc[i][k] : __builtin_fmaf(s, fh[i][k], acc[i][k]);
          accl[i][k] = skip ? accl[i][k] : __builtin_fmaf(s, lesser(fl, i, k), accl[i][k]);
        }
    } else if constexpr (KIND == KIND_G64) {
      // the lane's table: two terms of each f16 entry in one word
      const uint32_t tab = base + wave * 4096u;
      const uint32_t le[8] = {w.l0.x, w.l0.y, w.l0.z, w.l0.w, w.l1.x, w.l1.y, w.l1.z, w.l1.w};
#pragma unroll
      for (int e = 0; e < 16; ++e) {
        const float v = f16_to_f32((le[e >> 1] >> (16 * (e & 1))) & 0xffffu);
        // An infinite entry's second term is NaN: its sum is dropped for the
        // infinite (or NaN) leading one.  The widening quiets a NaN, so the
        // cut keeps it one.
        const float lo = v - __uint_as_float(__float_as_uint(v) & 0xffff0000u);
        *(lds_u32*)(size_t)(tab + 256u * e + 4u * lane) = hi_pair(__float_as_uint(v), __float_as_uint(lo));
      }
      // a table word's address: byte 0 the lane's column, byte 1 the block and the nibble
      const uint32_t lbyte = lane * 4u, rep = ((tab >> 8) & 0xffu) * 0x01010101u;
      const uint32_t wd[8] = {w.q0.x, w.q0.y, w.q0.z, w.q0.w, w.q1.x, w.q1.y, w.q1.z, w.q1.w};
      f32x4_t fh[2][TT], fl[3][TT];   // two chains of leading products: half the roundings in a row
#pragma unroll
      for (int i = 0; i < TT; ++i) fh[0][i] = fh[1][i] = fl[0][i] = fl[1][i] = fl[2][i] = z;
#pragma unroll
      for (uint32_t j = 0; j < 8; ++j) {
        const uint32_t we = (wd[j] & 0x0F0F0F0Fu) | rep, wo = ((wd[j] >> 4) & 0x0F0F0F0Fu) | rep;
        uint32_t d[2][4];
#pragma unroll
        for (uint32_t k = 0; k < 4; ++k) {
          const uint32_t sel = 0x0c0c0000u | ((4u + k) << 8);
          const uint32_t e0 = *(lds_u32*)(size_t)__builtin_amdgcn_perm(we, lbyte, sel);
          const uint32_t e1 = *(lds_u32*)(size_t)__builtin_amdgcn_perm(wo, lbyte, sel);
          d[0][k] = lo_pair(e0, e1);
          d[1][k] = hi_pair(e0, e1);
        }
        bf16x8_t b[2];
#pragma unroll
        for (int k = 0; k < 2; ++k) {
          if constexpr (TAIL) mask_tail(c * CH + 64u * g + 8u * j, d[k]);
          const u32x4 v = {d[k][0], d[k][1], d[k][2], d[k][3]};
          b[k] = __builtin_bit_cast(bf16x8_t, v);
        }
        step(b, at + 64u * g + 8u * j, fh[j & 1], fl);
      }
#pragma unroll
      for (int i = 0; i < TT; ++i)
#pragma unroll
        for (int k = 0; k < 4; ++k) {
          acc[i][k] += fh[0][i][k] + fh[1][i][k];
          accl[i][k] += lesser(fl, i, k);
        }
    } else {
      // Blocks past the row hold a repeated block: scale 0 (its products are
      // zero, the staged activations there being zero).
      uint32_t s4[4];
      {
        const uint32_t v = c * 4u + g < (cols + 31u) / 32u ? w.sc : 0u;
        uint32_t e = v, o = v;
        swap16(e, o);   // e: groups 0, 0, 2, 2; o: 1, 1, 3, 3
        s4[0] = s4[2] = e;
        swap32(s4[0], s4[2]);
        s4[1] = s4[3] = o;
        swap32(s4[1], s4[3]);
      }
      uint32_t q[2][4] = {};
      if constexpr (KIND == KIND_Q40) {
        q[0][0] = w.q.x; q[0][1] = w.q.y; q[0][2] = w.q.z; q[0][3] = w.q.w;
        transpose4(q[0]);
      } else {
        q[0][0] = w.a.x; q[0][1] = w.a.z; q[0][2] = w.b.x; q[0][3] = w.b.z;   // even dwords
        q[1][0] = w.a.y; q[1][1] = w.a.w; q[1][2] = w.b.y; q[1][3] = w.b.w;
        transpose4(q[0]);
        transpose4(q[1]);
      }
      f32x4_t ch[TT], cl[TT];   // the chunk's sums: a short chain of roundings at a small magnitude
#pragma unroll
      for (int i = 0; i < TT; ++i) ch[i] = cl[i] = z;
#pragma unroll
      for (uint32_t j = 0; j < 4; ++j) {
        uint32_t d[4];
        if constexpr (KIND == KIND_Q40) {
#pragma unroll
          for (int k = 0; k < 4; ++k) d[k] = *(lds_u32*)(size_t)(base + (((q[0][j] >> (8 * k)) & 0xffu) << 2));
        } else {
#pragma unroll
          for (int k = 0; k < 4; ++k) {
            const uint32_t v = q[k >> 1][j] >> (16 * (k & 1));
            const float f0 = (float)(int8_t)(v & 0xffu), f1 = (float)(int8_t)((v >> 8) & 0xffu);
            d[k] = hi_pair(__float_as_uint(f0), __float_as_uint(f1));
          }
        }
        const u32x4 v = {d[0], d[1], d[2], d[3]};
        const bf16x8_t b[1] = {__builtin_bit_cast(bf16x8_t, v)};
        f32x4_t fh[TT], fl[3][TT];
#pragma unroll
        for (int i = 0; i < TT; ++i) fh[i] = fl[0][i] = fl[1][i] = fl[2][i] = z;
        step(b, at + 32u * j + 8u * g, fh, fl);
        const float s = f16_to_f32(s4[j]);
#pragma unroll
        for (int i = 0; i < TT; ++i)
#pragma unroll
          for (int k = 0; k < 4; ++k) {
            ch[i][k] = __builtin_fmaf(s, fh[i][k], ch[i][k]);
            if constexpr (XT > 1) cl[i][k] = __builtin_fmaf(s, lesser(fl, i, k), cl[i][k]);
          }
      }
#pragma unroll
      for (int i = 0; i < TT; ++i)
#pragma unroll
        for (int k = 0; k < 4; ++k) {
          acc[i][k] += ch[i][k];
          if constexpr (XT > 1) accl[i][k] += cl[i][k];
        }
    }
  }

  // cb4 residuals of the lane's row, entries [os, oe): this wave (HALF: each
  // half of it) takes entries os + kw + KW * n.  Lane group g holds entry n = 4 k + g of round
  // k; the groups pass their entries on (three swaps) and each adds the
  // products of its own four tokens, gathered from the staged activations.
  // Entries outside columns [c0, c0 + span) belong to another phase.
  template <int KW, int KP>
  __device__ __forceinline__ void residuals(const uint32_t* __restrict__ outl, const uint32_t (&pre)[KP], uint32_t os,
                                            uint32_t oe, uint32_t kw, uint32_t M, uint32_t xoff, uint32_t xs,
                                            uint32_t c0, uint32_t span) {
    auto round = [&](uint32_t k, uint32_t mine) {
      uint32_t e = mine, o = mine, q[4];
      swap16(e, o);
      q[0] = q[2] = e;
      swap32(q[0], q[2]);
      q[1] = q[3] = o;
      swap32(q[1], q[3]);
      float v[4];
      uint32_t at[4];
      bool on[4];
#pragma unroll
      for (uint32_t j = 0; j < 4; ++j) {   // entries past the row's or of another phase: weight 0 of a staged column
        const uint32_t col = (q[j] & 0xffffu) - c0;
        on[j] = os + kw + KW * (4u * k + j) < oe && col < span;
        v[j] = f16_to_f32(q[j] >> 16);
        at[j] = xoff + (on[j] ? col * 2u : 0u);
      }
#pragma unroll
      for (int tt = 0; tt < TT; ++tt)
#pragma unroll
        for (int i = 0; i < 4; ++i) {
          const uint32_t m = std::min(16u * tt + 4u * (HALF ? g & 1u : g) + i, M - 1u);
          float xv[4];
#pragma unroll
          for (int j = 0; j < 4; ++j) {
            xv[j] = 0.0f;
#pragma unroll
            for (int xt = XT - 1; xt >= 0; --xt)   // the terms' sum is exact, smallest first
              xv[j] = __builtin_fmaf(bf16_to_f32(*(lds_u16*)(size_t)(at[j] + xt * plane + m * xs)),
                                     xt == 2 ? kTerm2 : xt == 1 ? kTerm1 : 1.0f, xv[j]);
          }
#pragma unroll
          for (int j = 0; j < 4; ++j) accr[tt][i] = on[j] ? __builtin_fmaf(v[j], xv[j], accr[tt][i]) : accr[tt][i];
        }
    };
#pragma unroll
    for (int k = 0; k < KP; ++k) {
      if (!__any(os + kw + KW * 4u * k < oe)) return;
      round(k, pre[k]);
    }
    for (uint32_t k = KP; __any(os + kw + KW * 4u * k < oe); ++k) {
      const uint32_t i = os + kw + KW * (4u * k + g);
      round(k, i < oe ? outl[i] : 0u);
    }
  }

  // The tile's sum for token 16 i + 4 g + k, row r.
  __device__ __forceinline__ float sum(int i, int k) const {
    const float v = __builtin_isinf(acc[i][k]) ? acc[i][k] : acc[i][k] + accl[i][k];
    return v + accr[i][k];
  }
};

// The lane's packed bytes of its row, and the loads of one chunk (clamped
// into the row).
template <uint32_t KIND>
struct Row {
  const char* wp;
  const uint16_t* sp;
  __device__ __forceinline__ void set(const DevTensor& t, uint32_t row) {
    wp = static_cast<const char*>(t.p0) + (size_t)row * (KIND == KIND_Q8 ? t.kp : t.kp / 2);
    sp = t.p1 + (size_t)row * (KIND == KIND_CB4 ? t.kp / 128 : KIND == KIND_G64 ? t.kp / 64 * 16 : t.kp / 32);
  }
  __device__ __forceinline__ void load(uint32_t cols, uint32_t c, uint32_t g, W<KIND>& w) const {
    if constexpr (KIND == KIND_CB4) {
      const uint32_t cc = std::min(c, (cols + 127u) / 128u - 1u);
      w.q = load_nt16(wp + cc * 64u + g * 16u);
      w.sc = sp[cc];
    } else if constexpr (KIND == KIND_G64) {
      const uint32_t gg = std::min(c * 4u + g, (cols + 63u) / 64u - 1u);
      w.q0 = load_nt16(wp + gg * 32u);
      w.q1 = load_nt16(wp + gg * 32u + 16u);
      w.l0 = load_nt16(sp + gg * 16u);
      w.l1 = load_nt16(sp + gg * 16u + 8u);
    } else {
      const uint32_t b = std::min(c * 4u + g, (cols + 31u) / 32u - 1u);
      if constexpr (KIND == KIND_Q40) {
        w.q = load_nt16(wp + b * 16u);
      } else {
        w.a = load_nt16(wp + b * 32u);
        w.b = load_nt16(wp + b * 32u + 16u);
      }
      w.sc = sp[b];
    }
  }
};

// Activations: phase columns [c0, c0 + PH) of every token (zero from column
// `cols` on; rows of ld columns), global ->
// registers -> LDS rows of PH * 2 + 16 bytes per plane.
template <uint32_t KIND, int XT, int CAP, int PH>
struct Stage {
  static constexpr uint32_t XS = PH * 2 + 16;
  static constexpr int NP = (CAP * PH / 8 + kThreads - 1) / kThreads;   // pieces of 8 columns per thread
  uint4 v[NP][XT == 3 ? 2 : 1];

  __device__ __forceinline__ void load(const Args& a, uint32_t ld, uint32_t cols, uint32_t c0) {
#pragma unroll
    for (int i = 0; i < NP; ++i) {
      const uint32_t u = threadIdx.x + (uint32_t)i * kThreads;
      const uint32_t m = std::min(u / (PH / 8), a.M - 1u);
      const uint32_t c = c0 + (u % (PH / 8)) * 8u;
      if (a.x_vec) {   // rows of whole 16-byte pieces
        const size_t o = (size_t)m * ld + std::min(c, ld - 8u);
        if constexpr (XT == 3) {
          const u32x4* q = reinterpret_cast<const u32x4*>(static_cast<const float*>(a.x) + o);
          const u32x4 v0 = q[0], v1 = q[1];
          v[i][0] = make_uint4(v0.x, v0.y, v0.z, v0.w);
          v[i][1] = make_uint4(v1.x, v1.y, v1.z, v1.w);
        } else {
          const u32x4 v0 = *reinterpret_cast<const u32x4*>(static_cast<const uint16_t*>(a.x) + o);
          v[i][0] = make_uint4(v0.x, v0.y, v0.z, v0.w);
        }
      } else {
        uint32_t e[8];
#pragma unroll
        for (uint32_t j = 0; j < 8; ++j) {
          const size_t o = (size_t)m * ld + std::min(c + j, ld - 1u);
          e[j] = XT == 3 ? static_cast<const uint32_t*>(a.x)[o] : (uint32_t)static_cast<const uint16_t*>(a.x)[o];
          if (c + j >= cols) e[j] = 0;
        }
        if constexpr (XT == 3) {
          v[i][0] = make_uint4(e[0], e[1], e[2], e[3]);
          v[i][1] = make_uint4(e[4], e[5], e[6], e[7]);
        } else {
          v[i][0] = make_uint4(e[0] | e[1] << 16, e[2] | e[3] << 16, e[4] | e[5] << 16, e[6] | e[7] << 16);
        }
      }
    }
  }

  // One piece's 8 bf16 at column c8 of the phase.
  __device__ __forceinline__ static void put(uint32_t row_at, uint32_t c8, const uint32_t (&d)[4]) {
    if constexpr (KIND == KIND_Q40) {
      // columns c8 .. c8 + 7 lie in one half of a block: column c at 2 (c % 16) + half
      const uint32_t at = row_at + (c8 & ~31u) * 2u + ((c8 & 15u) * 2u + ((c8 >> 4) & 1u)) * 2u;
#pragma unroll
      for (int j = 0; j < 4; ++j) {
        *(lds_u16*)(size_t)(at + 8u * j) = (uint16_t)d[j];
        *(lds_u16*)(size_t)(at + 8u * j + 4u) = (uint16_t)(d[j] >> 16);
      }
    } else {
      const u32x4 w = {d[0], d[1], d[2], d[3]};
      *(lds_u32x4*)(size_t)(row_at + c8 * 2u) = w;
    }
  }

  __device__ __forceinline__ void write(uint32_t xoff, uint32_t M, uint32_t cols, uint32_t c0) const {
    const uint32_t plane = M * XS;
#pragma unroll
    for (int i = 0; i < NP; ++i) {
      const uint32_t u = threadIdx.x + (uint32_t)i * kThreads;
      const uint32_t m = u / (PH / 8), c8 = (u % (PH / 8)) * 8u;
      if (m >= M) continue;
      const bool live = c0 + c8 < cols;   // past the row: zero (a piece is whole with x_vec, else zeroed as loaded)
      const uint32_t at = xoff + m * XS;
      if constexpr (XT == 3) {
        const uint32_t e[8] = {v[i][0].x, v[i][0].y, v[i][0].z, v[i][0].w, v[i][1].x, v[i][1].y, v[i][1].z, v[i][1].w};
        uint32_t h[8], mm[8], l[8];
#pragma unroll
        for (int j = 0; j < 8; ++j) split3(live ? __uint_as_float(e[j]) : 0.0f, h[j], mm[j], l[j]);
        const uint32_t dh[4] = {hi_pair(h[0], h[1]), hi_pair(h[2], h[3]), hi_pair(h[4], h[5]), hi_pair(h[6], h[7])};
        const uint32_t dm[4] = {hi_pair(mm[0], mm[1]), hi_pair(mm[2], mm[3]), hi_pair(mm[4], mm[5]),
                                hi_pair(mm[6], mm[7])};
        const uint32_t dl[4] = {hi_pair(l[0], l[1]), hi_pair(l[2], l[3]), hi_pair(l[4], l[5]), hi_pair(l[6], l[7])};
        put(at, c8, dh);
        put(at + plane, c8, dm);
        put(at + 2u * plane, c8, dl);
      } else {
        const uint32_t d[4] = {live ? v[i][0].x : 0u, live ? v[i][0].y : 0u, live ? v[i][0].z : 0u,
                               live ? v[i][0].w : 0u};
        put(at, c8, d);
      }
    }
  }
};

// One output by its definition, in f64, columns [k0, k1): for a sum that came
// out infinite or NaN.  The kernels sum a group's or a block's products before
// its scale, so values near f32's end overflow where the result does not (cb4,
// N(0, 1) * 2^124: 80 % of the outputs at 16 tokens), and they add cb4's
// residuals apart, so an infinite activation at a residual's column meets two
// weights where gemm_cpu has their sum (llm_prefill.rs:156-255).  Run by the
// lane that stores the output, one column at a time: only for such outputs.
// gemv: gemv_cpu's form, residuals apart and zero scales skipped
// (codebook.rs:376-417).
template <uint32_t KIND, int XT>
__device__ __forceinline__ float plain_dot(const DevTensor& t, uint32_t row, const void* x, uint32_t k0, uint32_t k1,
                                           bool gemv) {
  auto xat = [&](uint32_t c) {
    return XT == 3 ? static_cast<const float*>(x)[c] : bf16_to_f32(static_cast<const uint16_t*>(x)[c]);
  };
  const uint8_t* w = static_cast<const uint8_t*>(t.p0) + (size_t)row * (KIND == KIND_Q8 ? t.kp : t.kp / 2);
  const uint16_t* sp = t.p1 + (size_t)row * (KIND == KIND_CB4 ? t.kp / 128 : KIND == KIND_G64 ? t.kp / 64 * 16 : t.kp / 32);
  const float* cent = t.cent + (KIND == KIND_CB4 ? cent_table(t, row) * 16u : 0u);
  const uint32_t os = KIND == KIND_CB4 ? t.row_ptr[row] : 0u, oe = KIND == KIND_CB4 ? t.row_ptr[row + 1] : 0u;
  double s = 0.0;
  for (uint32_t c = k0; c < k1 && !__builtin_isnan(s); ++c) {
    const float xv = xat(c);
    float v;
    if constexpr (KIND == KIND_CB4) {
      const float sc = f16_to_f32(sp[c / 128u]);
      if (gemv && sc == 0.0f) continue;
      v = sc * cent[(w[c / 2u] >> (4u * (c & 1u))) & 15u];
      if (!gemv && !__builtin_isfinite(xv))
        for (uint32_t i = os; i < oe; ++i)
          if ((t.outliers[i] & 0xffffu) == c) v += f16_to_f32(t.outliers[i] >> 16);
    } else if constexpr (KIND == KIND_G64) {
      v = f16_to_f32(sp[(c / 64u) * 16u + ((w[c / 2u] >> (4u * (c & 1u))) & 15u)]);
    } else if constexpr (KIND == KIND_Q40) {
      v = (float)((int)((w[c / 32u * 16u + (c & 15u)] >> ((c & 16u) >> 2)) & 15u) - 8) * f16_to_f32(sp[c / 32u]);
    } else {
      v = (float)(int8_t)w[c] * f16_to_f32(sp[c / 32u]);
    }
    s += (double)v * (double)xv;
  }
  for (uint32_t i = os; i < oe; ++i) {
    const uint32_t c = t.outliers[i] & 0xffffu;
    const float xv = c >= k0 && c < k1 ? xat(c) : 0.0f;
    if (c >= k0 && c < k1 && (gemv || __builtin_isfinite(xv)))
      s += (double)f16_to_f32(t.outliers[i] >> 16) * (double)xv;
  }
  return (float)s;
}

// Whether an output that is not finite is computed anew.  Q8_0 and Q4_0 in
// the GEMV's range keep the reference's block dots, which overflow as the sums
// here do (llm_prefill.rs:45-54, q4_0.rs:109-145).
template <uint32_t KIND>
__device__ __forceinline__ bool redone(float v, const Args& a) {
  return !__builtin_isfinite(v) && !((KIND == KIND_Q8 || KIND == KIND_Q40) && a.skip_zero);
}

// Decode tables shared by the workgroup (before a barrier).
template <uint32_t KIND>
__device__ __forceinline__ void write_tables(const DevTensor& t, uint32_t base) {
  const uint32_t tid = threadIdx.x;
  if constexpr (KIND == KIND_CB4) {
    if (tid < 48u) {
      uint32_t h, m, l;
      split3(t.cent[tid], h, m, l);
      const u32x2 v = {hi_pair(h, m), l >> 16};
      *(lds_u32x2*)(size_t)(base + (tid >> 4) * 128u + (tid & 15u) * 8u) = v;
    }
  } else if constexpr (KIND == KIND_Q40) {
    if (tid < 256u) {
      const float f0 = (float)(int)(tid & 15u) - 8.0f, f1 = (float)(int)(tid >> 4) - 8.0f;
      *(lds_u32*)(size_t)(base + tid * 4u) = hi_pair(__float_as_uint(f0), __float_as_uint(f1));
    }
  }
}

// Waves per SIMD asked of the compiler: a workgroup is mostly latency (a
// load, a barrier, a few chunks, a sum), so three workgroups per CU beat two.
template <uint32_t KIND, int XT, int CAP, int NC>
constexpr int Occ = XT == 1 && CAP <= 8 && NC * kChunk<KIND> <= 256 ? 6 : 4;

// TT tiles of 16 tokens; CAP: the most tokens of this instantiation; RG row
// groups; NC chunks per wave and phase.  MULTI: several phases (K > PH).
template <uint32_t KIND, int XT, int TT, int CAP, int RG, int NC, bool MULTI, bool GLU, bool HALF>
__global__ __launch_bounds__(kThreads, (MULTI ? 2 : Occ<KIND, XT, CAP, NC>)) void skinny_kernel(DevTensor t, Args a) {
  // CH: columns of a chunk per lane group set; WC: columns a wave takes at once
  constexpr int KW = kWaves / RG, CH = kChunk<KIND>, WC = HALF ? 2 * CH : CH, PH = NC * KW * WC;
  constexpr uint32_t RT = HALF ? 8 : 16;   // weight rows of a tile
  constexpr uint32_t GH = RT / 2;          // gated form: gate rows of a tile, their up rows following
  static_assert(!HALF || (TT == 1 && CAP <= 8), "half tiles: up to 8 tokens");
  using St = Stage<KIND, XT, CAP, PH>;
  constexpr uint32_t XS = St::XS;
  extern __shared__ __attribute__((aligned(4096))) uint32_t smem[];
  const uint32_t base = (uint32_t)(size_t)((const LDS_AS uint32_t*)smem);
  const uint32_t xoff = base + kTabBytes<KIND>;

  const uint32_t tid = threadIdx.x, lane = tid & 63u, wave = tid >> 6;
  const uint32_t r = lane & 15u, g = lane >> 4;
  const uint32_t kw = wave % KW, rg = wave / KW;
  // K range of this block (grid.z): columns [k0, k1); its fp32 sums go to
  // slice blockIdx.z of a partial buffer where there are several.
  const uint32_t k0 = blockIdx.z * a.kslice, cols = std::min(t.cols, k0 + a.kslice);
  const uint32_t c_first = k0 / WC, nch = (cols + WC - 1) / WC;
  const uint32_t h = HALF ? r >> 3 : 0u;
  auto lane_chunk = [&](uint32_t c) { return HALF ? 2u * c + h : c; };
  // Tokens past CAP run as further blocks of the grid.
  a.x = static_cast<const char*>(a.x) + (size_t)blockIdx.y * CAP * t.cols * (XT == 3 ? 4u : 2u);
  a.y = static_cast<char*>(a.y) +
        ((size_t)blockIdx.z * a.M + (size_t)blockIdx.y * CAP) * (GLU ? a.y_stride : t.rows) * (a.y_bf16 ? 2u : 4u);
  a.M = std::min(a.M - blockIdx.y * CAP, (uint32_t)CAP);
  const uint32_t M = a.M;
  uint32_t row;
  if constexpr (GLU) {
    const uint32_t o = blockIdx.x * (GH * RG) + GH * rg + r % GH;
    row = (r % RT < GH ? 0u : a.n_ff) + std::min(o, a.n_ff - 1u);
  } else {
    row = std::min(blockIdx.x * (RT * RG) + RT * rg + r % RT, t.rows - 1u);
  }
  // The CSR bounds first: the entries' loads wait for them.
  uint32_t os = 0, oe = 0;
  if constexpr (KIND == KIND_CB4) {
    os = t.row_ptr[row];
    oe = t.row_ptr[row + 1];
  }
  St st;
  st.load(a, t.cols, cols, k0);
  Row<KIND> rw;
  rw.set(t, row);
  W<KIND> wr[MULTI ? 2 : 1][NC];
#pragma unroll
  for (int i = 0; i < NC; ++i)
    if (MULTI || i == 0 || c_first + kw + KW * i < nch) rw.load(cols, lane_chunk(c_first + kw + KW * i), g, wr[0][i]);
  write_tables<KIND>(t, base);
  constexpr int KP = KIND == KIND_CB4 ? (MULTI || PH > 2048 ? 2 : 1) : 1;
  constexpr int kWays = HALF ? 2 * KW : KW;           // shares of a row's residuals
  const uint32_t way = HALF ? 2u * kw + h : kw;
  uint32_t pre[KP] = {};
  if constexpr (KIND == KIND_CB4) {
#pragma unroll
    for (int k = 0; k < KP; ++k) {
      const uint32_t i = os + way + kWays * (4u * k + g);
      pre[k] = i < oe ? t.outliers[i] : 0u;
    }
  }
  Tile<KIND, XT, TT, HALF> tile;
  tile.base = base;
  tile.wave = wave;
  tile.r = r;
  tile.g = g;
  tile.lane = lane;
  tile.cols = cols;
  tile.ctab = KIND == KIND_CB4 ? base + cent_table(t, row) * 128u : 0u;
  tile.skip_zero = a.skip_zero != 0;
  tile.plane = M * XS;
#pragma unroll
  for (int i = 0; i < TT; ++i) tile.arow[i] = xoff + std::min(HALF ? r & 7u : 16u * i + r, M - 1u) * XS;
  tile.clear();

  auto phase = [&](uint32_t p, const W<KIND> (&w)[NC]) {
#pragma unroll
    for (int i = 0; i < NC; ++i) {
      const uint32_t cl = kw + KW * i, c = c_first + p * (PH / WC) + cl;
      if (c >= nch) break;
      if ((c + 1u) * WC > cols)
        tile.template chunk<true>(w[i], lane_chunk(c), lane_chunk(cl) * CH);
      else
        tile.template chunk<false>(w[i], lane_chunk(c), lane_chunk(cl) * CH);
    }
    if constexpr (KIND == KIND_CB4)
      tile.template residuals<kWays, KP>(t.outliers, pre, os, oe, way, M, xoff, XS, k0 + p * PH, std::min((uint32_t)PH, cols - k0 - p * PH));
  };
  if constexpr (!MULTI) {
    st.write(xoff, M, cols, k0);
    lds_barrier();
    phase(0, wr[0]);
    lds_barrier();
  } else {
    const uint32_t nph = (cols - k0 + PH - 1) / PH;
    auto request = [&](uint32_t p, W<KIND> (&w)[NC]) {
      st.load(a, t.cols, cols, k0 + p * PH);
#pragma unroll
      for (int i = 0; i < NC; ++i) rw.load(cols, lane_chunk(c_first + p * (PH / WC) + kw + KW * i), g, w[i]);
    };
    for (uint32_t p = 0; p < nph; p += 2) {
      st.write(xoff, M, cols, k0 + p * PH);
      lds_barrier();
      if (p + 1 < nph) request(p + 1, wr[1]);
      phase(p, wr[0]);
      lds_barrier();
      if (p + 1 < nph) {
        st.write(xoff, M, cols, k0 + (p + 1) * PH);
        lds_barrier();
        if (p + 2 < nph) request(p + 2, wr[0]);
        phase(p + 1, wr[1]);
        lds_barrier();
      }
    }
  }

  // ---- K-ways added in order, epilogue -------------------------------------------
#pragma unroll
  for (int i = 0; i < TT; ++i)
#pragma unroll
    for (int k = 0; k < 4; ++k)
      *(lds_f32*)(size_t)(xoff + (((wave * TT + i) * 4u + k) * 64u + lane) * 4u) = tile.sum(i, k);
  lds_barrier();
  // the K-ways pairwise: fewer roundings than one after the other
  auto total = [&](uint32_t gr, uint32_t tt, uint32_t k, uint32_t ln) {
    float v[KW];
#pragma unroll
    for (uint32_t w = 0; w < (uint32_t)KW; ++w) {
      auto part = [&](uint32_t l) {
        return *(lds_f32*)(size_t)(xoff + ((((gr * KW + w) * TT + tt) * 4u + k) * 64u + l) * 4u);
      };
      v[w] = part(ln);
      if constexpr (HALF) v[w] += part(ln + 40u);   // group + 2, row + 8: the other half of the columns
    }
#pragma unroll
    for (int d = 1; d < KW; d *= 2)
#pragma unroll
      for (int w = 0; w + d < KW; w += 2 * d) v[w] += v[w + d];
    return v[0];
  };
  // outputs of a tile: lanes (g, r) with g < GQ, r < WD, four tokens each
  constexpr uint32_t WD = GLU ? GH : RT, GQ = HALF ? 2 : 4, kPer = 4 * GQ * WD;
  constexpr uint32_t kOut = RG * TT * kPer;
  // Output u; false if it has to be redone.  The redoing pass is one of its
  // own: it holds nothing live here.
  auto output = [&](uint32_t u, auto redo_) {
    constexpr bool REDO = decltype(redo_)::value;
    const uint32_t e = u % kPer, tt = u / kPer % TT, grp = u / kPer / TT;
    const uint32_t k = e / (GQ * WD), ln = e / WD % GQ * 16u + e % WD;
    const uint32_t m = tt * 16u + 4u * (ln >> 4) + k;
    const uint32_t o = blockIdx.x * ((GLU ? GH : RT) * RG) + (GLU ? GH : RT) * grp + (ln & 15u);
    const uint32_t lim = GLU ? a.y_stride : t.rows;
    if (m >= M || o >= lim) return true;
    const void* xm = static_cast<const char*>(a.x) + (size_t)m * t.cols * (XT == 3 ? 4u : 2u);
    float v = total(grp, tt, k, ln);
    bool ok = !redone<KIND>(v, a);
    if (REDO && !ok) v = plain_dot<KIND, XT>(t, o, xm, k0, cols, a.skip_zero != 0);
    if constexpr (GLU) {
      float up = total(grp, tt, k, ln + GH);
      const bool up_ok = !redone<KIND>(up, a);
      if (o >= a.n_ff) {
        v = 0.0f;   // zero padding up to the row stride
        ok = true;
      } else {
        if (REDO && !up_ok) up = plain_dot<KIND, XT>(t, a.n_ff + o, xm, k0, cols, a.skip_zero != 0);
        ok = ok && up_ok;
        v = gated_act(v, up, a.gelu != 0);
      }
    }
    const size_t at = (size_t)m * lim + o;
    if (a.y_bf16)
      static_cast<uint16_t*>(a.y)[at] = f32_to_bf16(v);
    else
      static_cast<float*>(a.y)[at] = v;
    return ok;
  };
  bool ok = true;
  for (uint32_t u = tid; u < kOut; u += kThreads) ok = output(u, std::false_type{}) && ok;
  if (__builtin_expect(!ok, 0))
    for (uint32_t u = tid; u < kOut; u += kThreads) output(u, std::true_type{});
}

// Many rows (an LM head): each wave streams whole 16-row tiles, wv, wv +
// waves, ..., over all of K, D chunks requested ahead across tile
// boundaries; the activations are staged once per workgroup and no sum
// crosses waves.
template <uint32_t KIND, int CAP, int PH, int D>
__global__ __launch_bounds__(kThreads, 4) void skinny_stream_kernel(DevTensor t, Args a) {
  constexpr uint32_t CH = kChunk<KIND>;
  using St = Stage<KIND, 1, CAP, PH>;
  constexpr uint32_t XS = St::XS;
  extern __shared__ __attribute__((aligned(4096))) uint32_t smem[];
  const uint32_t base = (uint32_t)(size_t)((const LDS_AS uint32_t*)smem);
  const uint32_t xoff = base + kTabBytes<KIND>;
  const uint32_t tid = threadIdx.x, lane = tid & 63u, wave = tid >> 6;
  const uint32_t r = lane & 15u, g = lane >> 4;
  const uint32_t M = a.M, cols = t.cols, rows = t.rows;
  const uint32_t nch = (cols + CH - 1) / CH, nchp = (nch + D - 1) / D * D;
  const uint32_t tiles = (rows + 15u) / 16u, nwv = gridDim.x * kWaves;
  uint32_t ti = blockIdx.x * kWaves + wave;
  {
    St st;
    st.load(a, cols, cols, 0);
    write_tables<KIND>(t, base);
    st.write(xoff, M, cols, 0);
  }
  // prefetch position: chunk pc of tile pt
  uint32_t pt = ti, pc = 0;
  Row<KIND> rw;
  auto at_tile = [&](uint32_t tl) { rw.set(t, std::min(tl * 16u + r, rows - 1u)); };
  at_tile(pt);
  W<KIND> w[D];
  auto fetch = [&](W<KIND>& d) {
    rw.load(cols, pc, g, d);
    if (++pc == nchp) {
      pc = 0;
      pt += nwv;
      at_tile(std::min(pt, tiles - 1u));
    }
  };
#pragma unroll
  for (int i = 0; i < D; ++i) fetch(w[i]);
  lds_barrier();
  Tile<KIND, 1, 1> tile;
  tile.base = base;
  tile.wave = wave;
  tile.r = r;
  tile.g = g;
  tile.lane = lane;
  tile.cols = cols;
  tile.skip_zero = a.skip_zero != 0;
  tile.plane = M * XS;
  tile.arow[0] = xoff + std::min(r, M - 1u) * XS;
  for (; ti < tiles; ti += nwv) {
    const uint32_t row = std::min(ti * 16u + r, rows - 1u);
    tile.ctab = KIND == KIND_CB4 ? base + cent_table(t, row) * 128u : 0u;
    tile.clear();
    f32x4_t th = {0.0f, 0.0f, 0.0f, 0.0f}, tl = th;   // sums of earlier rounds of D chunks: shorter chains of roundings
    constexpr int KP = KIND == KIND_CB4 ? 6 : 1;
    uint32_t os = 0, oe = 0, pre[KP] = {};
    if constexpr (KIND == KIND_CB4) {
      os = t.row_ptr[row];
      oe = t.row_ptr[row + 1];
#pragma unroll
      for (int k = 0; k < KP; ++k) {
        const uint32_t i = os + 4u * k + g;
        pre[k] = i < oe ? t.outliers[i] : 0u;
      }
    }
    for (uint32_t c0 = 0; c0 < nchp; c0 += D) {
#pragma unroll
      for (uint32_t i = 0; i < (uint32_t)D; ++i) {
        const uint32_t c = c0 + i;
        if ((c + 1u) * CH <= cols)
          tile.template chunk<false>(w[i], c, c * CH);
        else if (c < nch)
          tile.template chunk<true>(w[i], c, c * CH);
        fetch(w[i]);
      }
#pragma unroll
      for (int k = 0; k < 4; ++k) {
        th[k] += tile.acc[0][k];
        tl[k] += tile.accl[0][k];
        tile.acc[0][k] = tile.accl[0][k] = 0.0f;
      }
    }
    tile.acc[0] = th;
    tile.accl[0] = tl;
    if constexpr (KIND == KIND_CB4)
      tile.template residuals<1, KP>(t.outliers, pre, os, oe, 0, M, xoff, XS, 0, PH);
    const uint32_t o = ti * 16u + r;
    auto store = [&](uint32_t m, float v) {
      const size_t at = (size_t)m * rows + o;
      if (a.y_bf16)
        static_cast<uint16_t*>(a.y)[at] = f32_to_bf16(v);
      else
        static_cast<float*>(a.y)[at] = v;
    };
    uint32_t redo = 0;
#pragma unroll
    for (uint32_t k = 0; k < 4; ++k) {
      const float v = tile.sum(0, k);
      if (4u * g + k < M && o < rows) {
        store(4u * g + k, v);
        redo |= redone<KIND>(v, a) ? 1u << k : 0u;
      }
    }
    for (; __builtin_expect(redo != 0, 0); redo &= redo - 1u) {
      const uint32_t m = 4u * g + (uint32_t)__builtin_ctz(redo);
      store(m, plain_dot<KIND, 1>(t, o, static_cast<const uint16_t*>(a.x) + (size_t)m * cols, 0, cols, a.skip_zero != 0));
    }
  }
}

template <uint32_t KIND, int XT, int TT, int CAP, int RG, int NC, bool MULTI, bool GLU, bool HALF = false>
hipError_t launch(const DevTensor& t, const Args& a, uint32_t outs, hipStream_t s) {
  constexpr uint32_t xs = NC * (kWaves / RG) * kChunk<KIND> * (HALF ? 2 : 1) * 2 + 16;
  const uint32_t rows = std::min<uint32_t>(a.M, CAP);
  const size_t lds = kTabBytes<KIND> + std::max<size_t>((size_t)XT * rows * xs, (size_t)kWaves * TT * 1024);
  constexpr size_t most = kTabBytes<KIND> + std::max<size_t>((size_t)XT * CAP * xs, (size_t)kWaves * TT * 1024);
  static_assert(most <= 160 * 1024, "LDS budget");
  static const hipError_t attr = hipFuncSetAttribute(
      reinterpret_cast<const void*>(&skinny_kernel<KIND, XT, TT, CAP, RG, NC, MULTI, GLU, HALF>),
      hipFuncAttributeMaxDynamicSharedMemorySize, (int)most);
  if (attr != hipSuccess) return attr;
  constexpr uint32_t per = (HALF ? 8 : 16) / (GLU ? 2 : 1) * RG;
  hipLaunchKernelGGL((skinny_kernel<KIND, XT, TT, CAP, RG, NC, MULTI, GLU, HALF>),
                     dim3((outs + per - 1) / per, (a.M + CAP - 1) / CAP, (t.cols + a.kslice - 1) / a.kslice), dim3(kThreads), lds, s, t, a);
  return hipGetLastError();
}

template <uint32_t KIND, int CAP, int PH, int D>
hipError_t launch_stream(const DevTensor& t, const Args& a, hipStream_t s) {
  const size_t lds = kTabBytes<KIND> + (size_t)a.M * (PH * 2 + 16);
  constexpr size_t most = kTabBytes<KIND> + (size_t)CAP * (PH * 2 + 16);
  static_assert(most <= 160 * 1024, "LDS budget");
  static const hipError_t attr = hipFuncSetAttribute(reinterpret_cast<const void*>(&skinny_stream_kernel<KIND, CAP, PH, D>),
                                                     hipFuncAttributeMaxDynamicSharedMemorySize, (int)most);
  if (attr != hipSuccess) return attr;
  const uint32_t wgs = ((t.rows + 15) / 16 + kWaves - 1) / kWaves;
  hipLaunchKernelGGL((skinny_stream_kernel<KIND, CAP, PH, D>), dim3(std::min<uint32_t>(wgs, 512u)), dim3(kThreads),
                     lds, s, t, a);
  return hipGetLastError();
}

// Phase length: all of K where its activations fit about 64 KB of LDS (two
// workgroups per CU), else several phases.
template <uint32_t KIND>
hipError_t launch_plain(const DevTensor& t, const Args& a, bool x_bf16, hipStream_t s) {
  constexpr int N1 = 256 / kChunk<KIND>;   // chunks per wave of 2048 columns
  constexpr bool G = KIND == KIND_G64;
  const uint32_t K = t.cols, M = a.M, n = t.rows;
  if (!x_bf16) {
    // Half tiles: one round of 256 workgroups at most, and a K whose phases they
    // halve (4 tokens, us: cb4 4096 -> 1024 13.3 -> 9.0, 8192 -> 1024 27.6 -> 18.1, g64
    // 4096 -> 1024 9.0 -> 6.5; 8 tokens Q8_0 4096 -> 1024 12.1 -> 8.0; from 2049 rows on,
    // two rounds, 4 tokens of cb4 3072 -> 4096 12.4 against 16.1).
    const bool half = n <= kHalfRowsF32 && K > (G ? 2048u : M <= 4 ? 512u : 1024u);
    if constexpr (!G) {
      if (M <= 4 && half && K <= 2048) return launch<KIND, 3, 1, 4, 1, 1, false, false, true>(t, a, n, s);
      if (M > 4 && M <= 8 && half) return launch<KIND, 3, 1, 8, 1, 1, true, false, true>(t, a, n, s);
    }
    if (M <= 4) {
      if (half) return launch<KIND, 3, 1, 4, 1, 1, true, false, true>(t, a, n, s);
      return K <= 2048 ? launch<KIND, 3, 1, 4, 1, N1, false, false>(t, a, n, s)
                       : launch<KIND, 3, 1, 4, 1, N1, true, false>(t, a, n, s);
    }
    return launch<KIND, 3, 1, 16, G ? 2 : 1, 1, true, false>(t, a, n, s);   // 1024 columns: four g64 chunks
  }
  if (n >= kStreamRows && K <= 2048 && M <= 16) {
    if (M <= 4) return launch_stream<KIND, 4, 2048, G ? 2 : 4>(t, a, s);
    return launch_stream<KIND, 16, 2048, G ? 2 : 4>(t, a, s);
  }
  // Half tiles where 16-row ones leave CUs without a workgroup.
  if (M <= 8 && n <= kHalfRows && (!G || K > 2048)) {
    if (M <= 4) {
      if constexpr (!G)
        if (K <= 2048) return launch<KIND, 1, 1, 4, 1, 1, false, false, true>(t, a, n, s);
      if (K <= 4096) return launch<KIND, 1, 1, 4, 1, N1, false, false, true>(t, a, n, s);
      if (K <= 8192) return launch<KIND, 1, 1, 4, 1, 2 * N1, false, false, true>(t, a, n, s);
      return launch<KIND, 1, 1, 4, 1, N1, true, false, true>(t, a, n, s);
    }
    if constexpr (!G)
      if (K <= 2048) return launch<KIND, 1, 1, 8, 1, 1, false, false, true>(t, a, n, s);
    if (K <= 4096) return launch<KIND, 1, 1, 8, 1, N1, false, false, true>(t, a, n, s);
    return launch<KIND, 1, 1, 8, 1, N1, true, false, true>(t, a, n, s);
  }
  if (M <= 4) {
    if (K <= 2048) return launch<KIND, 1, 1, 4, 1, N1, false, false>(t, a, n, s);
    if (K <= 4096) return launch<KIND, 1, 1, 4, 1, 2 * N1, false, false>(t, a, n, s);
    if (K <= 8192) return launch<KIND, 1, 1, 4, 1, 4 * N1, false, false>(t, a, n, s);
    return launch<KIND, 1, 1, 4, 1, 2 * N1, true, false>(t, a, n, s);
  }
  if (M <= 8) {
    if (K <= 2048) return launch<KIND, 1, 1, 8, 1, N1, false, false>(t, a, n, s);
    if (K <= 4096) return launch<KIND, 1, 1, 8, 1, 2 * N1, false, false>(t, a, n, s);
    return launch<KIND, 1, 1, 8, 1, 2 * N1, true, false>(t, a, n, s);
  }
  // More tokens: K ranges of at most 2048 columns (gemm_skinny.hip sums them), or one of several phases
  if (M <= 16)
    return std::min(K, a.kslice) <= 2048 ? launch<KIND, 1, 1, 16, 1, N1, false, false>(t, a, n, s)
                                         : launch<KIND, 1, 1, 16, 1, N1, true, false>(t, a, n, s);
  return launch<KIND, 1, 2, 32, 2, N1, true, false>(t, a, n, s);
}

template <uint32_t KIND>
hipError_t launch_glu(const DevTensor& t, const Args& a, bool x_bf16, hipStream_t s) {
  constexpr int N1 = 256 / kChunk<KIND>;
  constexpr bool G = KIND == KIND_G64;
  const uint32_t K = t.cols, M = a.M, n = a.y_stride;
  if (!x_bf16) {
    const bool half = t.rows <= kHalfRowsF32 && K > (G ? 2048u : M <= 4 ? 512u : 1024u);   // as the plain form
    if (M <= 4 && half) return launch<KIND, 3, 1, 4, 1, 1, true, true, true>(t, a, n, s);
    if constexpr (!G)
      if (M <= 8 && half) return launch<KIND, 3, 1, 8, 1, 1, true, true, true>(t, a, n, s);
    return M <= 4 ? launch<KIND, 3, 1, 4, 1, N1, true, true>(t, a, n, s)
                  : launch<KIND, 3, 1, 16, G ? 2 : 1, 1, true, true>(t, a, n, s);
  }
  // Half tiles for the sizes where the plain form takes them: up to 8 tokens the
  // sums are those of the plain form's skinny_kernel, bit for bit (not those of
  // its streaming form from kStreamRows, nor of the kernels that launch_gemv
  // keeps for two tokens of g64 and of Q8_0).
  if (M <= 8 && t.rows <= kHalfRows && (!G || K > 2048)) {
    if constexpr (!G)
      if (K <= 2048)
        return M <= 4 ? launch<KIND, 1, 1, 4, 1, 1, false, true, true>(t, a, n, s)
                      : launch<KIND, 1, 1, 8, 1, 1, false, true, true>(t, a, n, s);
    return launch<KIND, 1, 1, 8, 1, N1, true, true, true>(t, a, n, s);
  }
  if (M <= 4)
    return K <= 2048 ? launch<KIND, 1, 1, 4, 1, N1, false, true>(t, a, n, s)
                     : launch<KIND, 1, 1, 4, 1, N1, true, true>(t, a, n, s);
  if (M <= 8 && K <= 2048) return launch<KIND, 1, 1, 8, 1, N1, false, true>(t, a, n, s);
  if (M <= 16)
    return K <= 2048 ? launch<KIND, 1, 1, 16, 1, N1, false, true>(t, a, n, s)
                     : launch<KIND, 1, 1, 16, 1, N1, true, true>(t, a, n, s);
  return launch<KIND, 1, 2, 32, 2, N1, true, true>(t, a, n, s);
}

}  // namespace sk

}  // namespace vxt
