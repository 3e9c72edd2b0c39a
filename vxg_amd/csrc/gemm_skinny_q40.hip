// gemm_skinny_q40.hip -- the few-token MFMA kernels (gemm_skinny_impl.hpp) for KIND_Q40.
#include "gemm_skinny_impl.hpp"

namespace vxt {

hipError_t launch_skinny_q40(const DevTensor& t, const SkinnyArgs& a, bool x_bf16, hipStream_t s) {
  return a.glu ? sk::launch_glu<KIND_Q40>(t, a, x_bf16, s) : sk::launch_plain<KIND_Q40>(t, a, x_bf16, s);
}

}  // namespace vxt
