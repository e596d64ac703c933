// gemv_stream.hip -- the streaming decode kernels of gemv_stream.hpp, groups of whole 128-code units
// for the batched one.
#include "gemv_stream.hpp"

namespace cbk {
namespace {

template <int MB, int RPW, int DT>
const void* stream_kernel(int mode, int bits, bool mixed) {
    if (mixed) return reinterpret_cast<const void*>(&gemv_stream_kernel<MODE_QKV, 0, MB, RPW, DT>);
#define CBK_STREAM_K(M)                                                                            \
    (bits == 2 ? reinterpret_cast<const void*>(&gemv_stream_kernel<M, 2, MB, RPW, DT>)             \
               : (bits == 3 ? reinterpret_cast<const void*>(&gemv_stream_kernel<M, 3, MB, RPW, DT>)\
                            : reinterpret_cast<const void*>(&gemv_stream_kernel<M, 4, MB, RPW, DT>)))
    if (mode == MODE_QKV) return CBK_STREAM_K(MODE_QKV);
    if (mode == MODE_GATEUP) return CBK_STREAM_K(MODE_GATEUP);
    return CBK_STREAM_K(MODE_GEMV);
#undef CBK_STREAM_K
}

}  // namespace

template <int DT>
const void* stream_kernel_dt(int mode, int bits, bool mixed, int mb, int rpw) {
    if constexpr (DT != DT_F32)                        // fp32 streams at batch 1 only
        if (mb > 1) return stream_kernel<2, STREAM_RPW, DT>(mode, bits, mixed);
    if (rpw == STREAM_RPW_WIDE && mode == MODE_GEMV && !mixed) {     // the host plans 8 rows for plain GEMVs only
        constexpr int W = STREAM_RPW_WIDE;
        return bits == 2 ? reinterpret_cast<const void*>(&gemv_stream_kernel<MODE_GEMV, 2, 1, W, DT>)
                         : (bits == 3 ? reinterpret_cast<const void*>(&gemv_stream_kernel<MODE_GEMV, 3, 1, W, DT>)
                                      : reinterpret_cast<const void*>(&gemv_stream_kernel<MODE_GEMV, 4, 1, W, DT>));
    }
    return stream_kernel<1, STREAM_RPW, DT>(mode, bits, mixed);
}

const void* gemv_stream_kernel_for(int mode, int bits, bool mixed, int mb, int rpw, int dt) {
    return dt == DT_BF16 ? stream_kernel_dt<DT_BF16>(mode, bits, mixed, mb, rpw)
                         : (dt == DT_F32 ? stream_kernel_dt<DT_F32>(mode, bits, mixed, mb, rpw)
                                         : stream_kernel_dt<DT_F16>(mode, bits, mixed, mb, rpw));
}

const void* gemv_bstream_kernel_for(int mode, int bits, bool mixed, int bsu, int dt, int sub) {
    if (sub > 1) return gemv_bstream_sub_kernel_for(mode, bits, mixed, dt, sub);
    if (dt == DT_BF16)
        return bsu == 8 ? bstream_kernel<8, DT_BF16, 1>(mode, bits, mixed)
                        : bstream_kernel<4, DT_BF16, 1>(mode, bits, mixed);
    if (dt == DT_F32)
        return bsu == 8 ? bstream_kernel<8, DT_F32, 1>(mode, bits, mixed)
                        : bstream_kernel<4, DT_F32, 1>(mode, bits, mixed);
    return bsu == 8 ? bstream_kernel<8, DT_F16, 1>(mode, bits, mixed) : bstream_kernel<4, DT_F16, 1>(mode, bits, mixed);
}

}  // namespace cbk
