// cbk_kernels.hpp -- launchers exported by the kernel translation units to abi.cpp.
#pragma once

#include <hip/hip_runtime.h>
#include "cbk_device.hpp"

namespace cbk {

// abi.cpp: every kernel launch goes through here.  While the measurement timer is
// armed (cbk_timer_start) the launch records start/stop events inside the dispatch
// (hipExtLaunchKernel), so cbk_timer_stop reports pure kernel durations.
hipError_t launch(const void* f, dim3 grid, dim3 block, void** args, size_t lds, hipStream_t stream);

// abi.cpp: raises kernel f's dynamic-LDS limit (on the current device) to cover `bytes`,
// once per kernel and device; the limit is only ever raised.
hipError_t lds_limit_raise(const void* f, int bytes);

// gemv_stream.hip: batch 1 or 2 (mb staged activation rows), fp16 or bf16, group size % 32 == 0.  A job is rpw * st_rw
// virtual rows x one K split; its workgroup has st_ks * st_rw waves, each over rpw rows
// (STREAM_RPW, or STREAM_RPW_WIDE at batch 1) and one K slice of 64 * STREAM_CPL chunks.
#ifndef CBK_STREAM_CPL
#define CBK_STREAM_CPL 1
#endif
constexpr int STREAM_CPL = CBK_STREAM_CPL;
constexpr int STREAM_RPW = 4;
constexpr int STREAM_RPW_WIDE = 8;
const void* gemv_stream_kernel_for(int mode, int bits, bool mixed, int mb, int rpw, int dt);
// gemv_stream.hip: batch 3..16, fp16 or bf16 (fp32: 2..8), group size % 128 == 0 (sub 1).  A job is 16 * st_rw virtual
// rows x one K split (over 128-code units); its workgroup has st_ks * st_rw waves, each
// over 16 rows and one K slice of bsu (4 or 8) units.
const void* gemv_bstream_kernel_for(int mode, int bits, bool mixed, int bsu, int dt, int sub);
// gemv_bsub.hip: the same with groups finer than a unit, sub 2 (multiples of 64) or 4 (of 32), bsu 4.
const void* gemv_bstream_sub_kernel_for(int mode, int bits, bool mixed, int dt, int sub);

// gemv_any.hip: any dtype / group size / alignment, on the fp32 matrix cores.  A job is
// 16 virtual rows x 16 batch rows x one K split, one workgroup of 64 to ANY_MAX_THREADS
// threads (whole waves) that share the split's chunks.
constexpr int ANY_MAX_THREADS = 1024;
const void* gemv_any_kernel_for(int dt, int mode);

// gemv_any.hip: the combine launch of split-K partials (P > 1 without arrival counters).
hipError_t launch_gemv_combine(const GemvArgs& A, int dt, int mode, hipStream_t stream);

struct GemmArgs {
    const void* x;          // [M, K]
    const uint32_t* w;      // packed [N, wpr]
    const void* s;          // scales [N, G]
    const void* z;          // zeros [N, G]
    const void* b;          // bias [N] or nullptr
    void* out;              // [M, N]
    int M, N, K, C, G, gs, wpr, bits, act;
    int xvec;               // x is 16-byte aligned and K % 8 == 0 (vector activation loads)
    FastDiv divG;           // by the group size
    // 16-bit matrix-core GEMM: K splits per tile, their partial tiles, an arrival counter per tile
    int S;
    float* partial;
    uint32_t* split_cnt;
    const uint32_t* w2;     // gate-up GEMM: the up projection's packed [N, wpr], scales, zeros
    const void* s2;
    const void* z2;
    // fused QKV: Q and K stored pair-interleaved per head of perm_hd rows (0: in order), the
    // RoPE tables [M, perm_hd] (nullptr: none) in fp32 or the activations' dtype
    const void* rope_cos;
    const void* rope_sin;
    int perm_hd, rope_f32;
    FastDiv divHD;          // by perm_hd
};

// The fused-QKV GEMM: a's fields common to the three projections, and each one's own.
struct GemmQkvArgs {
    GemmArgs a;
    const uint32_t* w[3];
    const void* s[3];
    const void* z[3];
    const void* b[3];
    void* out[3];
    int n[3], bits[3];
    int first[3];           // each projection's first tile
};
enum { GEMM_PLAIN = 0, GEMM_GATEUP = 1, GEMM_QKV = 2 };

// gemm.hip: fp16 / bf16 on the 16-bit matrix cores, any alignment.
hipError_t launch_gemm_mfma(const GemmArgs& A, int dt, hipStream_t stream);

// gemm_f32.hip: any dtype, fp32 operands on the fp32 matrix cores, W-hat unrounded.
hipError_t launch_gemm_f32(const GemmArgs& A, int dt, hipStream_t stream);

// gemm_f16.cpp: fp16 or bf16 (dt), K % 8 == 0, 16-byte aligned x.  gate_up: out =
// silu(x . W-hat^T) * (x . W2-hat^T), each factor rounded to the dtype first (no bias).
// A call's plan: tiles of 32 mb rows (mb 1, 2 or 4) x 128 columns, S K splits each.
struct GemmPlan {
    int mb = 4, S = 1;
    int64_t tiles = 0, partial_floats = 0;       // tiles, and the fp32 partial tiles of S > 1
};
// ntiles: 128-column tiles over all projections (64 output pairs a tile for gate-up); split: K
// splits allowed.
GemmPlan gemm_f16_plan(int64_t M, int64_t ntiles, int64_t K, bool split);
inline int64_t gemm_f16_ntiles(int64_t N, bool gate_up) { return gate_up ? (N + 63) / 64 : (N + 127) / 128; }
bool gemm_f16_supported(const GemmArgs& A);
// A.S, A.partial and A.split_cnt set when the plan has splits (S = 1 otherwise); without counters
// a combine launch follows.  mode: GEMM_PLAIN or GEMM_GATEUP.
hipError_t launch_gemm_f16(const GemmArgs& A, int dt, const GemmPlan& plan, hipStream_t stream, int mode);
hipError_t launch_gemm_f16_qkv(GemmQkvArgs& Q, int dt, const GemmPlan& plan, hipStream_t stream);

// The kernels of a tile height, one translation unit each (gemm_f16_mb*.hip).
struct GemmKernel {
    const void* f = nullptr;
    const void* combine = nullptr;
    int lds = 0, combine_lds = 0;
};
GemmKernel gemm_f16_mb1(int dt, int bits, bool tail, bool gs128, int mode);
GemmKernel gemm_f16_mb2(int dt, int bits, bool tail, bool gs128, int mode);
GemmKernel gemm_f16_mb4(int dt, int bits, bool tail, bool gs128, int mode);
GemmKernel gemm_f16_mb4s(int dt, int bits, bool tail, bool gs128, int mode);   // with K splits

// quant.hip: group-affine quantizer + bit packer (the format's producer).
struct QuantArgs {
    const void* w;          // [N, K] weights (fp16 / bf16 / fp32)
    uint32_t* packed;       // [N, wpr]
    void* scales;           // [N, G] in the metadata dtype
    void* zeros;            // [N, G]
    int N, K, G, gs, bits, wpr;
    int scheme;             // 0: reference.py quantize_affine, 1: crispybits_quant affine
};
hipError_t launch_quant_pack(const QuantArgs& A, int dt, int mdt, int cus, hipStream_t stream);

// unpack.hip
hipError_t launch_unpack(const uint32_t* packed, int N, int K, int bits, int32_t* codes, hipStream_t stream);

// probe.hip: one read-only streaming launch over `bytes` (the measurement floor).
hipError_t launch_stream_probe(const void* src, uint32_t bytes, int unroll, int block, bool store, uint32_t* sink,
                               hipStream_t stream);

}  // namespace cbk
