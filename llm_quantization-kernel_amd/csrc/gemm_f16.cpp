// gemm_f16.cpp -- the plan and the launch of the fp16 / bf16 prefill GEMM (gemm_f16_tile.hpp).
#include <algorithm>

#include "cbk_kernels.hpp"

namespace cbk {

namespace {
constexpr int BN = 128, BK = 128;
constexpr int CUS = 256;                     // of every gfx950 part: the plan needs no device
}  // namespace

bool gemm_f16_supported(const GemmArgs& A) {
    // 16-byte activation pieces, whole octets before K, 16-byte aligned packed /
    // scale / zero bases (the loads' aligned pieces and the zero scan), windows of
    // 8 groups spanning whole weight blocks (group size a multiple of 32), tensors
    // within the 32-bit range of a buffer descriptor
    const auto al16 = [](const void* p) { return (reinterpret_cast<uintptr_t>(p) & 15) == 0; };
    const long lim = 0x7FFFFFFF;                 // buffer offsets and ranges are 32-bit
    const bool up_ok = !A.w2 || (al16(A.w2) && al16(A.s2) && al16(A.z2));
    return A.K % 8 == 0 && A.K >= 8 && A.gs % 32 == 0 && al16(A.x) && al16(A.w) && al16(A.s) && al16(A.z) && up_ok &&
           (long)A.M * A.K * 2 < lim && (long)A.N * A.wpr * 4 < lim && (long)A.N * A.G * 2 < lim;
}

// The tile height and K splits of a call: the least of an estimated time over tiles of 32, 64 and
// 128 rows and every split that keeps two weight blocks (512 codes) per part.  A tile costs a
// fixed part (launch, first loads, epilogue) and a part per 128-code stage -- little less for
// 32 rows than for 128, the stage being bound by its instructions -- and tiles past one per CU
// cost another round; a split adds the round trip of its partial tiles.  The constants (us) are
// fitted to 2272 measured (shape, batch, tile, split) points: N 1024 .. 13824, K 512 .. 13824,
// batch 17 .. 1024, W4 / W3, fp16 / bf16, plain and gate-up, on 256 CUs.  Its pick is 0.6 % off
// the fastest point in the geometric mean, at worst 9 %, and 1.25x faster than the same kernel's
// 128-row tiles unsplit, at none of those points slower (W4, us: 11008 -> 4096 batch 32 68.0 -> 17.5, batch 256 68.9 -> 41.0;
// 4096^2 batch 128 29.9 -> 18.1).
GemmPlan gemm_f16_plan(int64_t M, int64_t ntiles, int64_t K, bool split) {
    struct Cost {
        int mb;
        double fixed, stage, split0, split1;
    };
    static constexpr Cost costs[] = {{4, 6.9, 0.70, 3.22, 2.70}, {2, 7.37, 0.57, 2.34, 0.99}, {1, 4.59, 0.65, 4.51, 0.34}};
    constexpr double round_per_mb = 4.7;
    constexpr int64_t max_split = 32;
    const int64_t nblk = (K + 2 * BK - 1) / (2 * BK);
    GemmPlan best;
    double best_t = 0;
    for (const Cost& c : costs) {
        const int64_t tiles = ((M + 32 * c.mb - 1) / (32 * c.mb)) * ntiles;
        for (int64_t S = 1; S == 1 || (split && S <= std::min(nblk / 2, max_split)); ++S) {
            const double stages = 2.0 * (double)((nblk + S - 1) / S), rounds = (double)((tiles * S + CUS - 1) / CUS);
            const double t = c.fixed + rounds * stages * c.stage + (rounds - 1) * round_per_mb * c.mb +
                             (S > 1 ? c.split0 + c.split1 * (double)S : 0.0);
            if (best.tiles && t >= best_t) continue;
            best_t = t;
            best.mb = c.mb;
            best.S = (int)S;
            best.tiles = tiles;
            best.partial_floats = S > 1 ? tiles * S * (32 * c.mb) * BN : 0;
        }
    }
    return best;
}

namespace {

GemmKernel kernel_for(const GemmArgs& A, int dt, int bits, const GemmPlan& p, int mode) {
    const bool tail = A.K % BK != 0, gs128 = A.gs == 128;
    return p.mb == 1   ? gemm_f16_mb1(dt, bits, tail, gs128, mode)
           : p.mb == 2 ? gemm_f16_mb2(dt, bits, tail, gs128, mode)
           : A.S > 1   ? gemm_f16_mb4s(dt, bits, tail, gs128, mode)
                       : gemm_f16_mb4(dt, bits, tail, gs128, mode);
}

hipError_t run(const GemmKernel& k, const GemmArgs& A, const GemmPlan& p, void** args, hipStream_t stream) {
    hipError_t e = lds_limit_raise(k.f, k.lds);
    if (e == hipSuccess) e = launch(k.f, dim3((uint32_t)(p.tiles * A.S)), dim3(512), args, (size_t)k.lds, stream);
    if (e != hipSuccess || A.S == 1 || A.split_cnt) return e;
    e = lds_limit_raise(k.combine, k.combine_lds);
    if (e == hipSuccess) e = launch(k.combine, dim3((uint32_t)p.tiles), dim3(512), args, (size_t)k.combine_lds, stream);
    return e;
}

}  // namespace

hipError_t launch_gemm_f16(const GemmArgs& A, int dt, const GemmPlan& p, hipStream_t stream, int mode) {
    void* args[] = {const_cast<GemmArgs*>(&A)};
    return run(kernel_for(A, dt, A.bits, p, mode), A, p, args, stream);
}

hipError_t launch_gemm_f16_qkv(GemmQkvArgs& Q, int dt, const GemmPlan& p, hipStream_t stream) {
    const int mtiles = (Q.a.M + 32 * p.mb - 1) / (32 * p.mb);
    Q.first[0] = 0;
    for (int i = 1; i < 3; ++i) Q.first[i] = Q.first[i - 1] + mtiles * (int)gemm_f16_ntiles(Q.n[i - 1], false);
    void* args[] = {&Q};
    return run(kernel_for(Q.a, dt, 4, p, GEMM_QKV), Q.a, p, args, stream);
}

}  // namespace cbk
