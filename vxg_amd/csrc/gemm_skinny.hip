// gemm_skinny.hip -- entry to the few-token MFMA kernels (gemm_skinny_impl.hpp),
// instantiated by weight kind in gemm_skinny_{cb4,g64,q40,q8}.hip.
#include <algorithm>

#include "common.hpp"

namespace vxt {

hipError_t launch_skinny_cb4(const DevTensor&, const SkinnyArgs&, bool, hipStream_t);
hipError_t launch_skinny_g64(const DevTensor&, const SkinnyArgs&, bool, hipStream_t);
hipError_t launch_skinny_q40(const DevTensor&, const SkinnyArgs&, bool, hipStream_t);
hipError_t launch_skinny_q8(const DevTensor&, const SkinnyArgs&, bool, hipStream_t);

hipError_t launch_gemm_reduce(const float* partial, uint32_t splits, const float* inv, const int32_t* xe, uint32_t m,
                              uint32_t n, void* y, bool y_bf16, hipStream_t s);

static hipError_t launch_any(const DevTensor& t, const SkinnyArgs& a, bool x_bf16, hipStream_t s) {
  switch (t.kind) {
    case KIND_CB4: return launch_skinny_cb4(t, a, x_bf16, s);
    case KIND_G64: return launch_skinny_g64(t, a, x_bf16, s);
    case KIND_Q40: return launch_skinny_q40(t, a, x_bf16, s);
    case KIND_Q8: return launch_skinny_q8(t, a, x_bf16, s);
    default: return hipErrorInvalidValue;
  }
}

static SkinnyArgs args(const DevTensor& t, const void* x, bool x_bf16, uint32_t m, void* y, bool y_bf16) {
  SkinnyArgs a{};
  a.x = x;
  a.y = y;
  a.M = m;
  const size_t esz = x_bf16 ? 2 : 4;
  a.x_vec = reinterpret_cast<uintptr_t>(x) % 16 == 0 && t.cols % 8 == 0 && ((size_t)t.cols * esz) % 16 == 0;
  a.y_bf16 = y_bf16;
  a.skip_zero = m <= 8;   // batch_m 1..8 is the GEMV, above the GEMM
  a.kslice = (t.cols + 1023u) / 1024u * 1024u;   // one range
  return a;
}

// K ranges of a call, each a set of workgroups of its own, summed by the
// split-K reduction; their columns (a multiple of 1024) in `cols`.  bf16
// activations above 8 tokens: 2048 columns, but all of K for g64 from 11 tokens and
// 8192 rows (16 tokens 2304 -> 12288 the sliced form takes 1.14 times as long, the
// fused kernel 0.95 times; cb4, Q8_0, Q4_0 in one range 1.1 .. 1.6 times as long).
// f32 ones past 2048 columns: a workgroup fills a CU and takes some 3 us per 1024
// columns, so the fewest ranges that cut rounds over the 256 CUs x columns by a
// sixth or more (16 tokens, us, one range and the two-phase path against this: cb4 8192 -> 2048 52 / 43 against
// 28.6, Q4_0 8192 -> 1024 42 / 32 against 14.6, g64 6144 -> 2048 35 / 26 against 14.6,
// Q8_0 12288 -> 512 42 / 31 against 10.8).
static uint32_t k_slices(const DevTensor& t, uint32_t m, bool x_bf16, uint32_t* cols = nullptr) {
  const uint32_t kt = (t.cols + 1023u) / 1024u;
  uint32_t per = kt;
  if (m > 8 && x_bf16) {
    if (!(t.kind == KIND_G64 && m > 10 && m <= 16 && t.rows >= 8192u)) per = 2;
  } else if (m > 8 && kt > 2) {
    const uint32_t tr = t.kind == KIND_G64 ? 32u : 16u, tiles = (t.rows + tr - 1u) / tr;   // rows of a workgroup
    auto cost = [&](uint32_t p) { return (tiles * ((kt + p - 1u) / p) + 255u) / 256u * p; };
    for (uint32_t p = kt - 1u; p > 0; --p)
      if (cost(p) * 6u <= cost(per) * 5u) per = p;
  }
  if (cols) *cols = per * 1024u;
  return (kt + per - 1u) / per;
}

// The most tokens of one call.
uint32_t skinny_max_m(bool x_bf16) { return x_bf16 ? 64u : 16u; }

size_t skinny_workspace_bytes(const DevTensor& t, uint32_t m, bool x_bf16) {
  const uint32_t sl = k_slices(t, m, x_bf16);
  return sl > 1 ? (size_t)sl * m * t.rows * 4 : 0;
}

hipError_t launch_skinny(const DevTensor& t, const void* x, bool x_bf16, uint32_t m, void* y, bool y_bf16, void* ws,
                         hipStream_t s) {
  uint32_t per;
  const uint32_t sl = k_slices(t, m, x_bf16, &per);
  SkinnyArgs a = args(t, x, x_bf16, m, sl > 1 ? ws : y, sl > 1 ? false : y_bf16);
  if (sl > 1) a.kslice = per;
  const hipError_t e = launch_any(t, a, x_bf16, s);
  if (e != hipSuccess || sl == 1) return e;
  return launch_gemm_reduce(static_cast<const float*>(ws), sl, nullptr, nullptr, m, t.rows, y, y_bf16, s);
}

// Whether a gated call takes the fused form: up to 8 tokens always (but Q8_0
// with 3 .. 8 aligned bf16 tokens, whose plain GEMV has kernels of its own: the
// staged form keeps its sums), above (in AUTO) up to 16, and up to 64 bf16 tokens
// while K fits one phase range and the decode, repeated for every 32 tokens, stays
// below the staged form's GEMM, f32 gate and up rows and element-wise pass (32 / 64
// tokens, K = 2048, n_ff = 6144, us against the staged form: cb4 27 / 40 against 58
// / 59, g64 20 / 29 against 25 / 34, Q4_0 22 / 32 against 41 / 40, Q8_0 18 / 26
// against 23 / 30).  f32 activations: where the plain form needs no K ranges.  g64
// leaves with many rows where its staged GEMM is the fused kernel and ahead
// (fused form over staged: 16 tokens n_ff = 11008, K = 512 1.50, 3072 1.13, 8192 1.16;
// 33 tokens 512 1.37; 17 tokens n_ff = 14336, 512 1.23), Q8_0 so above 32 tokens (33
// tokens 512, n_ff = 11008 1.56) and with few rows of a long K (16 tokens 8192,
// n_ff = 64 .. 1024 1.25; 1536 0.75).
bool skinny_glu_takes(const DevTensor& t, const void* x, uint32_t m, bool x_bf16, int mode) {
  if (m <= 8) return t.kind != KIND_Q8 || m == 2 || !args(t, x, x_bf16, m, nullptr, false).x_vec || !x_bf16;
  if (mode != kGemmAuto && mode != kGemmAutoOwn) return false;
  const uint32_t n_ff = t.rows / 2;
  if (x_bf16 && t.kind == KIND_G64 && m > 10) {
    if (t.cols < 1024 && n_ff > (m > 16 && m <= 32 ? 12288u : 8192u)) return false;
    if (t.cols > 2048 && n_ff >= 8192) return false;
  }
  if (x_bf16 && t.kind == KIND_Q8 && (m > 32 ? t.cols < 1024 && n_ff > 8192 : t.cols > 6144 && n_ff < 1536)) return false;
  if (m <= 16) return x_bf16 || k_slices(t, m, x_bf16) == 1;
  const size_t w = (size_t)t.cols * t.rows, M1 = 1000 * 1000;
  return m <= skinny_max_m(x_bf16) && t.cols <= 2048 && w <= (m <= 32 ? 34 : 26) * M1;
}

// Gated [gate; up] form: act[m][i] = f(gate_i) * up_i for i < rows / 2, zero
// up to act_stride.
hipError_t launch_skinny_glu(const DevTensor& t, const void* x, bool x_bf16, uint32_t m, void* act, bool act_bf16,
                             uint32_t act_stride, bool gelu, hipStream_t s) {
  SkinnyArgs a = args(t, x, x_bf16, m, act, act_bf16);
  a.glu = 1;
  a.n_ff = t.rows / 2;
  a.y_stride = act_stride;
  a.gelu = gelu;
  return launch_any(t, a, x_bf16, s);
}

}  // namespace vxt
