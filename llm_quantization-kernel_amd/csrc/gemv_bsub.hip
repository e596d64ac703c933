// gemv_bsub.hip -- the batched streaming decode of gemv_stream.hpp for groups finer than a 128-code
// unit: SUB = 2 (multiples of 64) or 4 (multiples of 32) sub-units a unit.
#include "gemv_stream.hpp"

namespace cbk {

const void* gemv_bstream_sub_kernel_for(int mode, int bits, bool mixed, int dt, int sub) {
    if (dt == DT_BF16)
        return sub == 2 ? bstream_kernel<4, DT_BF16, 2>(mode, bits, mixed)
                        : bstream_kernel<4, DT_BF16, 4>(mode, bits, mixed);
    if (dt == DT_F32)
        return sub == 2 ? bstream_kernel<4, DT_F32, 2>(mode, bits, mixed)
                        : bstream_kernel<4, DT_F32, 4>(mode, bits, mixed);
    return sub == 2 ? bstream_kernel<4, DT_F16, 2>(mode, bits, mixed) : bstream_kernel<4, DT_F16, 4>(mode, bits, mixed);
}

}  // namespace cbk
