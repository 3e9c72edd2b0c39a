// gemm_skinny_g64.hip -- the few-token MFMA kernels (gemm_skinny_impl.hpp) for KIND_G64.
#include "gemm_skinny_impl.hpp"

namespace vxt {

hipError_t launch_skinny_g64(const DevTensor& t, const SkinnyArgs& a, bool x_bf16, hipStream_t s) {
  return a.glu ? sk::launch_glu<KIND_G64>(t, a, x_bf16, s) : sk::launch_plain<KIND_G64>(t, a, x_bf16, s);
}

}  // namespace vxt
