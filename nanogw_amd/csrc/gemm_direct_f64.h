// FP64 MFMA GEMM without LDS (v_mfma_f64_16x16x4f64): one wave owns a
// (16 FM) x (16 FN) tile of C = A B and reads its operand fragments straight
// from global memory into a ring of D register sets, D - 1 blocks of 16 k
// ahead of the block being multiplied.
//
// For products whose LDS tiles would leave most of the 1024 SIMDs idle: a
// 16 x 16 tile per wave gives four times as many waves as 64 x 64 tiles on four
// waves, eight times as many as 128 x 64, and the ring covers the memory
// latency that a lone wave per SIMD cannot hide behind others.  The k order of every sum is that of gemm_core_f64.h (blocks of 16,
// sub-step s of lane group g takes k = 4 g + s), so both cores give the same
// bits.
//
// The loader functors are those of operator_loaders.h.  Rows past an operand
// re-read its last row (their results are never stored); k past the end is
// zero in both operands.
#pragma once

#include "gemm_core_f64.h"

namespace ngw {

template <int FM, int FN>
struct AccDirect {
    f64x4 v[FM][FN];
};

template <int FM, int FN, int D, class AL, class BL>
__device__ __forceinline__ void gemm_f64_direct(const AL& al, const BL& bl, int m0, int n0, int K,
                                                AccDirect<FM, FN>& acc)
{
    const int lane = threadIdx.x & 63, r16 = lane & 15, k4 = 4 * (lane >> 4);
#pragma unroll
    for (int i = 0; i < FM; ++i)
#pragma unroll
        for (int j = 0; j < FN; ++j) acc.v[i][j] = f64x4{0.0, 0.0, 0.0, 0.0};
    typename AL::Handle ha[FM];
    typename BL::Handle hb[FN];
#pragma unroll
    for (int i = 0; i < FM; ++i) ha[i] = al.shift(al.row(min(m0 + 16 * i + r16, al.MN - 1)), k4);
#pragma unroll
    for (int j = 0; j < FN; ++j) hb[j] = bl.shift(bl.row(min(n0 + 16 * j + r16, bl.MN - 1)), k4);
    double ra[D][FM][4][AL::NRAW], rb[D][FN][4][BL::NRAW];
    const int nfull = K / 16, nblk = (K + 15) / 16;
    auto fetch = [&](int blk, auto uc) {
        constexpr int u = decltype(uc)::value;
        const int kb = 16 * blk;  // the handles hold this lane's k4
#pragma unroll
        for (int i = 0; i < FM; ++i)
#pragma unroll
            for (int s = 0; s < 4; ++s) al.fetch(ha[i], kb + s, ra[u][i][s]);
#pragma unroll
        for (int j = 0; j < FN; ++j)
#pragma unroll
            for (int s = 0; s < 4; ++s) bl.fetch(hb[j], kb + s, rb[u][j][s]);
    };
    auto multiply = [&](auto uc) {
        constexpr int u = decltype(uc)::value;
#pragma unroll
        for (int s = 0; s < 4; ++s) {
            double a[FM], b[FN];
#pragma unroll
            for (int i = 0; i < FM; ++i) a[i] = al.combine(ra[u][i][s]);
#pragma unroll
            for (int j = 0; j < FN; ++j) b[j] = bl.combine(rb[u][j][s]);
#pragma unroll
            for (int i = 0; i < FM; ++i)
#pragma unroll
                for (int j = 0; j < FN; ++j)
                    acc.v[i][j] = __builtin_amdgcn_mfma_f64_16x16x4f64(a[i], b[j], acc.v[i][j], 0, 0, 0);
        }
    };
    if (nfull > 0) {
        static_for<D - 1>([&](auto uc) { fetch(min(decltype(uc)::value, nfull - 1), uc); });
        // (the last turn skips what is past the end: a separate tail would be
        // more code to fetch for kernels that run a few microseconds)
        for (int t = 0; t < nfull; t += D)
            static_for<D>([&](auto uc) {
                constexpr int u = decltype(uc)::value;
                if (t + u >= nfull) return;
                fetch(min(t + u + D - 1, nfull - 1), std::integral_constant<int, (u + D - 1) % D>{});
                multiply(uc);
            });
    }
    if (nblk > nfull) {  // the last K mod 16
        double a[FM][4], b[FN][4];
#pragma unroll
        for (int s = 0; s < 4; ++s) {
            const int k = 16 * nfull + k4 + s, kc = min(k, K - 1) - k4;
#pragma unroll
            for (int i = 0; i < FM; ++i) {
                double r[AL::NRAW];
                al.fetch(ha[i], kc, r);
                a[i][s] = k < K ? al.combine(r) : 0.0;
            }
#pragma unroll
            for (int j = 0; j < FN; ++j) {
                double r[BL::NRAW];
                bl.fetch(hb[j], kc, r);
                b[j][s] = k < K ? bl.combine(r) : 0.0;
            }
        }
#pragma unroll
        for (int s = 0; s < 4; ++s)
#pragma unroll
            for (int i = 0; i < FM; ++i)
#pragma unroll
                for (int j = 0; j < FN; ++j)
                    acc.v[i][j] = __builtin_amdgcn_mfma_f64_16x16x4f64(a[i][s], b[j][s], acc.v[i][j], 0, 0, 0);
    }
}

// f(row, col, value) for every accumulator value of this lane, relative to
// the wave's tile.
template <int FM, int FN, class F>
__device__ __forceinline__ void for_acc_direct(const AccDirect<FM, FN>& acc, F&& f)
{
    const int lane = threadIdx.x & 63;
#pragma unroll
    for (int i = 0; i < FM; ++i)
#pragma unroll
        for (int j = 0; j < FN; ++j)
#pragma unroll
            for (int r = 0; r < 4; ++r) f(16 * i + (lane >> 4) + 4 * r, 16 * j + (lane & 15), acc.v[i][j][r]);
}

}  // namespace ngw
