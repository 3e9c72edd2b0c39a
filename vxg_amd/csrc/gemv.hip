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

// Two tokens and more run on the few-token MFMA kernels, except Q8_0 with
// aligned bf16 activations (x_vec), whose own kernels stream int8 as fast or
// faster (2048 x 2048 / 2048 x 6144 / 151936 x 2048 at M = 4: 3.7 / 5.6 / 63
// us).  M = 4, K x N = 2048 x 6144 / 6144 x 2048 / 2048 x 151936 against the
// one-FMA-per-weight-per-token kernel before: cb4 22.3 / 19.1 / 543 -> 8.3 /
// 8.2 / 75 us, g64 20.3 / 18.7 / 459 -> 6.6 / 7.4 / 67, Q4_0 12.4 / 11.4 /
// 265 -> 6.0 / 7.0 / 61.
hipError_t launch_gemv(const DevTensor& t, const void* x, bool x_bf16, bool x_vec, uint32_t m, void* y,
                       bool y_bf16, hipStream_t s) {
  if (m >= 2 && (t.kind != KIND_Q8 || !x_bf16 || !x_vec)) return launch_skinny(t, x, x_bf16, m, y, y_bf16, nullptr, s);
  switch (t.kind) {
    case KIND_Q8: return launch_gemv_q8(t, x, x_bf16, m, y, y_bf16, s);
    case KIND_Q40: return launch_gemv_q40(t, x, x_bf16, m, y, y_bf16, s);
    case KIND_CB4: return launch_gemv_cb4(t, x, x_bf16, m, y, y_bf16, s);
    case KIND_G64: return launch_gemv_g64(t, x, x_bf16, m, y, y_bf16, s);
    default: return hipErrorInvalidValue;
  }
}

// Gated gate/up GEMV (one token): t is [gate; up] with t.rows = 2 * n_ff.
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
