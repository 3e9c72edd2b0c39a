// gemv.hip -- dispatch of the decode GEMV (batch_m 1..8) by weight kind.
// The kernels live in gemv_impl.hpp and are instantiated in gemv_{q8,q40,cb4,g64}.hip.
#include "common.hpp"

namespace vxt {

hipError_t launch_gemv_q8(const DevTensor&, const void*, bool, uint32_t, void*, bool, hipStream_t);
hipError_t launch_gemv_q40(const DevTensor&, const void*, bool, uint32_t, void*, bool, hipStream_t);
hipError_t launch_gemv_cb4(const DevTensor&, const void*, bool, uint32_t, void*, bool, hipStream_t);
hipError_t launch_gemv_g64(const DevTensor&, const void*, bool, uint32_t, void*, bool, hipStream_t);
hipError_t launch_norm_q8(const DevTensor&, const NormIn&, int, void*, bool, uint32_t, hipStream_t);
hipError_t launch_norm_q40(const DevTensor&, const NormIn&, int, void*, bool, uint32_t, hipStream_t);
hipError_t launch_norm_cb4(const DevTensor&, const NormIn&, int, void*, bool, uint32_t, hipStream_t);
hipError_t launch_norm_g64(const DevTensor&, const NormIn&, int, void*, bool, uint32_t, hipStream_t);
hipError_t launch_glu_q8(const DevTensor&, const void*, bool, uint32_t, uint32_t, void*, bool, uint32_t, bool,
                         hipStream_t);
hipError_t launch_glu_q40(const DevTensor&, const void*, bool, uint32_t, uint32_t, void*, bool, uint32_t, bool,
                          hipStream_t);
hipError_t launch_glu_cb4(const DevTensor&, const void*, bool, uint32_t, uint32_t, void*, bool, uint32_t, bool,
                          hipStream_t);
hipError_t launch_glu_g64(const DevTensor&, const void*, bool, uint32_t, uint32_t, void*, bool, uint32_t, bool,
                          hipStream_t);

hipError_t launch_skinny(const DevTensor&, const void*, bool, uint32_t, void*, bool, void*, hipStream_t);

// Two tokens of a small g64 matrix (bf16 activations): the generic kernel has
// a wave for each row and no barrier between its waves.  Whole call, few-token
// kernel over this one: K = 2048 with 512 / 1024 / 2048 rows 1.31 / 1.31 / 1.13
// times as long (3.3 / 3.3 / 4.0 us here), K = 1024 1.12 / 1.13 / 0.97; at K =
// 2048 and 3072 rows 0.93, at K = 3072 and 512 rows 0.89.  Either kernel multiplies
// every bit of the table's entries.  cb4 and Q4_0 keep the few-token kernel
// there, which is the more exact one for them.
static bool two_token_gemv(const DevTensor& t, uint32_t m, bool x_bf16) {
  return t.kind == KIND_G64 && m == 2 && x_bf16 && t.cols <= 2048 && t.rows <= (t.cols <= 1024 ? 1024u : 2048u);
}

// Two tokens and more run on the few-token MFMA kernels, except Q8_0 with
// aligned bf16 activations (x_vec), whose own kernels stream int8 as fast or
// faster (2048 x 2048 / 2048 x 6144 / 151936 x 2048 at M = 4: 3.7 / 5.6 / 63
// us).  M = 4, K x N = 2048 x 6144 / 6144 x 2048 / 2048 x 151936 against the
// one-FMA-per-weight-per-token kernel before: cb4 22.3 / 19.1 / 543 -> 8.3 /
// 8.2 / 75 us, g64 20.3 / 18.7 / 459 -> 6.6 / 7.4 / 67, Q4_0 12.4 / 11.4 /
// 265 -> 6.0 / 7.0 / 61.
hipError_t launch_gemv(const DevTensor& t, const void* x, bool x_bf16, bool x_vec, uint32_t m, void* y,
                       bool y_bf16, hipStream_t s) {
  if (m >= 2 && (t.kind != KIND_Q8 || !x_bf16 || !x_vec) && !two_token_gemv(t, m, x_bf16))
    return launch_skinny(t, x, x_bf16, m, y, y_bf16, nullptr, s);
  switch (t.kind) {
    case KIND_Q8: return launch_gemv_q8(t, x, x_bf16, m, y, y_bf16, s);
    case KIND_Q40: return launch_gemv_q40(t, x, x_bf16, m, y, y_bf16, s);
    case KIND_CB4: return launch_gemv_cb4(t, x, x_bf16, m, y, y_bf16, s);
    case KIND_G64: return launch_gemv_g64(t, x, x_bf16, m, y, y_bf16, s);
    default: return hipErrorInvalidValue;
  }
}

// Two tokens of a gated call with bf16 in and out on the generic kernel: where
// the few-token kernel's workgroups (16 rows of gate and 16 of up) leave CUs
// idle.  Measured by kind, K and n_ff, few-token kernel over this one (whole
// calls):
//   K = 1536, 2048: g64 1.17 .. 1.23 up to n_ff = 1024, 0.97 .. 1.01 above; the
//   others 0.99 .. 1.14 up to 2048; at 3072 cb4 and Q8_0 1.12 and 1.06 with K =
//   2048, 0.91 and 0.90 with K = 1536; 0.65 .. 0.98 from 4096; K = 1024 0.5 .. 1.01;
//   K = 6144: cb4 1.04 .. 1.11, Q4_0 1.11 .. 1.18, g64 1.00 .. 1.06 up to n_ff =
//   2048, Q8_0 1.05 .. 1.09 up to 1024, 0.59 .. 0.96 above;
//   K = 3072, 4096, 8192: 0.80 .. 0.99 up to n_ff = 1024 (half tiles), then g64
//   1.01 .. 1.20 throughout, cb4 and Q4_0 1.10 .. 1.34 at 1536 and 2048 (cb4 at K =
//   8192 also 1.16 at 3072), 0.71 .. 1.02 above; Q8_0 0.79 .. 0.97.
// An f32 result keeps the few-token kernel, whose sums are the more exact.
bool two_token_glu(const DevTensor& t, uint32_t m, bool x_bf16, bool act_bf16) {
  if (m != 2 || !x_bf16 || !act_bf16 || t.cols <= 1024) return false;
  const uint32_t n_ff = t.rows / 2;
  if (t.cols <= 2048)
    return n_ff <= (t.kind == KIND_G64 ? 1024u : t.cols <= 1536 || t.kind == KIND_Q40 ? 2048u : 3072u);
  if (t.cols > 4096 && t.cols <= 6144) return n_ff <= (t.kind == KIND_Q8 ? 1024u : 2048u);
  if (t.kind == KIND_Q8 || n_ff <= 1024) return false;
  return t.kind == KIND_G64 || n_ff <= (t.kind == KIND_CB4 && t.cols > 6144 ? 3072u : 2048u);
}

// Gated gate/up GEMV (one token, or two that two_token_glu takes): t is [gate; up] with t.rows = 2 * n_ff.
hipError_t launch_gemv_glu(const DevTensor& t, const void* x, bool x_bf16, uint32_t m, void* act, bool act_bf16,
                           uint32_t act_stride, bool gelu, hipStream_t s) {
  const uint32_t n_ff = t.rows / 2;
  switch (t.kind) {
    case KIND_Q8: return launch_glu_q8(t, x, x_bf16, m, n_ff, act, act_bf16, act_stride, gelu, s);
    case KIND_Q40: return launch_glu_q40(t, x, x_bf16, m, n_ff, act, act_bf16, act_stride, gelu, s);
    case KIND_CB4: return launch_glu_cb4(t, x, x_bf16, m, n_ff, act, act_bf16, act_stride, gelu, s);
    case KIND_G64: return launch_glu_g64(t, x, x_bf16, m, n_ff, act, act_bf16, act_stride, gelu, s);
    default: return hipErrorInvalidValue;
  }
}

// Batch-1 GEMV whose x is bf16(rms_norm(cur [+ delta]) * w), built in each
// workgroup.  epi 0: y = W x; 1 / 2: gated SiLU / GELU-tanh over [gate; up].
hipError_t launch_gemv_norm(const DevTensor& t, const NormIn& nin, int epi, void* y, bool y_bf16, uint32_t y_stride,
                            hipStream_t s) {
  switch (t.kind) {
    case KIND_Q8: return launch_norm_q8(t, nin, epi, y, y_bf16, y_stride, s);
    case KIND_Q40: return launch_norm_q40(t, nin, epi, y, y_bf16, y_stride, s);
    case KIND_CB4: return launch_norm_cb4(t, nin, epi, y, y_bf16, y_stride, s);
    case KIND_G64: return launch_norm_g64(t, nin, epi, y, y_bf16, y_stride, s);
    default: return hipErrorInvalidValue;
  }
}

}  // namespace vxt
