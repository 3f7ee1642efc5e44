// The block-sparse attention (fp_attn_kernel.h) at head dim 256, compiled with
// the MFMAs in their vector-register form (see Ring there for why).
#include "fp_attn_kernel.h"

namespace fp {

hipError_t launch_merge_d256(const AttnArgs& a, int dtype, int block, hipStream_t s) {
  return dtype == FP_DTYPE_BF16 ? launch_merge_t<BF16, 256>(a, block, s)
                                : launch_merge_t<F16, 256>(a, block, s);
}

hipError_t launch_attn_d256(const AttnArgs& a, int dtype, int block, int64_t grid, bool persist,
                            hipStream_t s) {
  return dtype == FP_DTYPE_BF16 ? launch_attn_t<BF16, 256>(a, block, grid, persist, s)
                                : launch_attn_t<F16, 256>(a, block, grid, persist, s);
}

}  // namespace fp
