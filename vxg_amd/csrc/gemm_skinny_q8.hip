// gemm_skinny_q8.hip -- the few-token MFMA kernels (gemm_skinny_impl.hpp) for KIND_Q8.
#include "gemm_skinny_impl.hpp"

namespace vxt {

hipError_t launch_skinny_q8(const DevTensor& t, const SkinnyArgs& a, bool x_bf16, hipStream_t s) {
  return a.glu ? sk::launch_glu<KIND_Q8>(t, a, x_bf16, s) : sk::launch_plain<KIND_Q8>(t, a, x_bf16, s);
}

}  // namespace vxt
