// gemm_f16_mb4s.hip -- the fp16 / bf16 prefill GEMM (gemm_f16_tile.hpp) with 128-row tiles, K split over workgroups.
#include "gemm_f16_tile.hpp"

namespace cbk {

GemmKernel gemm_f16_mb4s(int dt, int bits, bool tail, bool gs128, int mode) {
    return kernel_of<4, true>(dt, bits, tail, gs128, mode);
}

}  // namespace cbk
