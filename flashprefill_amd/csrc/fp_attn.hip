// Launchers of the block-sparse attention (fp_attn_kernel.h) for 16-bit inputs;
// head dims 64 and 128 are compiled here.
#include "fp_attn_kernel.h"

namespace fp {

hipError_t launch_merge(const AttnArgs& a, int dtype, int head_dim, int block, hipStream_t s) {
  if (a.unit_slots <= 0 || dtype == FP_DTYPE_F32) return hipSuccess;
  if (head_dim == 256) return launch_merge_d256(a, dtype, block, s);
  if (head_dim == 128)
    return dtype == FP_DTYPE_BF16 ? launch_merge_t<BF16, 128>(a, block, s)
                                  : launch_merge_t<F16, 128>(a, block, s);
  return dtype == FP_DTYPE_BF16 ? launch_merge_t<BF16, 64>(a, block, s)
                                : launch_merge_t<F16, 64>(a, block, s);
}

hipError_t launch_attn(const AttnArgs& a, int dtype, int head_dim, int block, int64_t grid,
                       bool persist, hipStream_t s) {
  if (grid <= 0) return hipSuccess;
  if (head_dim == 256) return launch_attn_d256(a, dtype, block, grid, persist, s);
  if (head_dim == 128)
    return dtype == FP_DTYPE_BF16 ? launch_attn_t<BF16, 128>(a, block, grid, persist, s)
                                  : launch_attn_t<F16, 128>(a, block, grid, persist, s);
  return dtype == FP_DTYPE_BF16 ? launch_attn_t<BF16, 64>(a, block, grid, persist, s)
                                : launch_attn_t<F16, 64>(a, block, grid, persist, s);
}

}  // namespace fp
