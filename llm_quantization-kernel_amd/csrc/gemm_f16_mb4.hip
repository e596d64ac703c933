// gemm_f16_mb4.hip -- the fp16 / bf16 prefill GEMM (gemm_f16_tile.hpp) with 128-row tiles, one workgroup per tile.
#include "gemm_f16_tile.hpp"

namespace cbk {

GemmKernel gemm_f16_mb4(int dt, int bits, bool tail, bool gs128, int mode) {
    return kernel_of<4, false>(dt, bits, tail, gs128, mode);
}

}  // namespace cbk
