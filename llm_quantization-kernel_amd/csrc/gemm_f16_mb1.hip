// gemm_f16_mb1.hip -- the fp16 / bf16 prefill GEMM (gemm_f16_tile.hpp) with 32-row tiles (K split or not).
#include "gemm_f16_tile.hpp"

namespace cbk {

GemmKernel gemm_f16_mb1(int dt, int bits, bool tail, bool gs128, int mode) {
    return kernel_of<1, true>(dt, bits, tail, gs128, mode);
}

}  // namespace cbk
