// FP64 MFMA GEMM core for gfx950 (v_mfma_f64_16x16x4f64).
//
// C tile (BM x BN) of C = A B, K reduced in slabs of BK = 16:
//  * 256 threads = 4 waves in a 2 x 2 layout, each wave owns (BM/2) x (BN/2);
//  * LDS holds A and B slabs k-contiguous ([mn][BK + 2]) so that each lane
//    reads its 4 consecutive k of a fragment with two 16-byte loads; the k
//    order inside a slab is permuted (lane group g of MFMA sub-step s uses
//    k = 4 g + s), which leaves the sum unchanged;
//  * double-buffered LDS, two slabs ahead in registers, fragments one half
//    slab ahead; one barrier per slab;
//  * operands come through loader functors: a thread keeps a per-row handle
//    (pointer arithmetic done once per tile) and reads element k on demand.
//
// MFMA f64 16x16x4 lane layout (measured on gfx950):
//   A/B operand: lane l supplies row/col l%16 at k = l/16;
//   result     : lane l, component r holds row l/16 + 4r, col l%16.
#pragma once

#include "ngw_kernels.h"

#include <type_traits>

namespace ngw {

typedef double f64x4 __attribute__((ext_vector_type(4)));

constexpr int GK = 16;     // K slab
constexpr int GPAD = 2;    // LDS row padding (doubles); keeps rows 16-byte aligned
constexpr int GNT = 256;   // threads per workgroup

// Compile-time loop: f(std::integral_constant<int, 0>) ... f(<N - 1>).
template <int I, int N, class F>
__device__ __forceinline__ void static_for_impl(F&& f)
{
    if constexpr (I < N) {
        f(std::integral_constant<int, I>{});
        static_for_impl<I + 1, N>(f);
    }
}
template <int N, class F>
__device__ __forceinline__ void static_for(F&& f)
{
    static_for_impl<0, N>(f);
}

// Workgroup -> tile with each XCD owning a contiguous range of tiles (WGs are
// dispatched round-robin over the 8 XCDs); inside a range the M index runs
// fastest so neighbouring tiles share their B slab in that XCD's L2.
__device__ __forceinline__ int xcd_tile(int bid, int ntiles)
{
    const int x = bid & 7, local = bid >> 3;
    const int q = ntiles >> 3, r = ntiles & 7;
    const int start = x * q + (x < r ? x : r);
    return start + local;
}

template <int BM, int BN>
struct SmemF64 {
    double a[2][BM][GK + GPAD];
    double b[2][BN][GK + GPAD];
};

// Per-thread slab loader for one operand tile of MN rows.
// kContig operands: thread t reads k = t % 16 for rows t/16 + 16 i.
// otherwise       : thread t reads row t % MN for k = t/MN + (256/MN) i.
// Loader functors split an element into NRAW raw values (fetch) and a
// combine() applied when the slab is written to LDS, so that the prefetch of
// a later slab never has to complete before the current slab's MFMAs.  Rows
// past the operand read its row 0: they only reach results that no epilogue
// stores.
template <class L, int MN>
struct SlabLoader {
    static constexpr int PER = MN * GK / GNT;  // elements per thread
    static constexpr int NH = L::kContig ? PER : 1;
    typename L::Handle h[NH];
    int kk0;

    __device__ __forceinline__ void init(const L& ld, int mn0)
    {
        const int t = threadIdx.x;
        if (L::kContig) {
            kk0 = t % GK;
#pragma unroll
            for (int i = 0; i < PER; ++i) {
                const int mn = mn0 + t / GK + (GNT / GK) * i;
                h[i] = ld.shift(ld.row(mn < ld.MN ? mn : 0), kk0);
            }
        } else {
            kk0 = t / MN;
            const int mn = mn0 + t % MN;
            h[0] = ld.shift(ld.row(mn < ld.MN ? mn : 0), kk0);
        }
    }

    // k of element i relative to the handle (the handle holds kk0)
    __device__ static constexpr int kof(int k0, int i) { return L::kContig ? k0 : k0 + (GNT / MN) * i; }

    __device__ __forceinline__ void fetch(const L& ld, int k0, double (&raw)[PER][L::NRAW]) const
    {
#pragma unroll
        for (int i = 0; i < PER; ++i) ld.fetch(h[L::kContig ? i : 0], kof(k0, i), raw[i]);
    }
    __device__ __forceinline__ void put(double (*dst)[GK + GPAD], int i, double v) const
    {
        const int t = threadIdx.x;
        if (L::kContig)
            dst[t / GK + (GNT / GK) * i][kk0] = v;
        else
            dst[t % MN][kk0 + (GNT / MN) * i] = v;
    }
    __device__ __forceinline__ void store(const L& ld, double (*dst)[GK + GPAD],
                                          const double (&raw)[PER][L::NRAW]) const
    {
#pragma unroll
        for (int i = 0; i < PER; ++i) put(dst, i, ld.combine(raw[i]));
    }
    // the last K mod 16: k past the end is zero
    __device__ __forceinline__ void load_tail(const L& ld, int k0, int K, double (*dst)[GK + GPAD]) const
    {
#pragma unroll
        for (int i = 0; i < PER; ++i) {
            const int k = kof(k0, i) + kk0;
            double r[L::NRAW];
            ld.fetch(h[L::kContig ? i : 0], min(k, K - 1) - kk0, r);
            put(dst, i, k < K ? ld.combine(r) : 0.0);
        }
    }
};

template <int BM, int BN>
struct AccF64 {
    static constexpr int FM = BM / 32, FN = BN / 32;
    f64x4 v[FM][FN];
};

// A wave's operand fragments of one slab.
template <int FM, int FN>
struct FragF64 {
    double a[FM][4], b[FN][4];
};

template <int BM, int BN>
__device__ __forceinline__ void frag_read(const SmemF64<BM, BN>& sm, int cur, FragF64<BM / 32, BN / 32>& f)
{
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    const int wm = (wave & 1) * (BM / 2), wn = (wave >> 1) * (BN / 2);
    const int r16 = lane & 15, k4 = lane >> 4;
#pragma unroll
    for (int i = 0; i < BM / 32; ++i) {
        const double2* p = reinterpret_cast<const double2*>(&sm.a[cur][wm + 16 * i + r16][4 * k4]);
        const double2 x0 = p[0], x1 = p[1];
        f.a[i][0] = x0.x; f.a[i][1] = x0.y; f.a[i][2] = x1.x; f.a[i][3] = x1.y;
    }
#pragma unroll
    for (int j = 0; j < BN / 32; ++j) {
        const double2* p = reinterpret_cast<const double2*>(&sm.b[cur][wn + 16 * j + r16][4 * k4]);
        const double2 x0 = p[0], x1 = p[1];
        f.b[j][0] = x0.x; f.b[j][1] = x0.y; f.b[j][2] = x1.x; f.b[j][3] = x1.y;
    }
}

template <int S0, int S1, int BM, int BN>
__device__ __forceinline__ void frag_mfma(const FragF64<BM / 32, BN / 32>& f, AccF64<BM, BN>& acc)
{
#pragma unroll
    for (int s = S0; s < S1; ++s)
#pragma unroll
        for (int i = 0; i < BM / 32; ++i)
#pragma unroll
            for (int j = 0; j < BN / 32; ++j)
                acc.v[i][j] = __builtin_amdgcn_mfma_f64_16x16x4f64(f.a[i][s], f.b[j][s], acc.v[i][j], 0, 0, 0);
}

// C tile over K.  An FP64 MFMA occupies the matrix pipe for 64 cycles and
// everything else can issue under it, if it stands between the MFMAs of the
// same wave: in the first half of slab t the next slab goes from registers to
// LDS and the one after it is requested, in the second half the next slab's
// fragments are read, each spread over the half's MFMAs
// (sched_group_barrier).
template <int BM, int BN, class AL, class BL>
__device__ __forceinline__ void gemm_f64_tile(const AL& al, const BL& bl, int m0, int n0, int K,
                                              AccF64<BM, BN>& acc, SmemF64<BM, BN>& sm)
{
    constexpr int FM = BM / 32, FN = BN / 32;
    typedef SlabLoader<AL, BM> LA;
    typedef SlabLoader<BL, BN> LB;
#pragma unroll
    for (int i = 0; i < FM; ++i)
#pragma unroll
        for (int j = 0; j < FN; ++j) acc.v[i][j] = f64x4{0.0, 0.0, 0.0, 0.0};
    LA la;
    LB lb;
    la.init(al, m0);
    lb.init(bl, n0);
    double ra[LA::PER][AL::NRAW], rb[LB::PER][BL::NRAW];
    const int nfull = K / GK;
    FragF64<FM, FN> fr[2];
    if (nfull > 0) {
        la.fetch(al, 0, ra);
        lb.fetch(bl, 0, rb);
        la.store(al, sm.a[0], ra);
        lb.store(bl, sm.b[0], rb);
        const int k1 = min(1, nfull - 1) * GK;
        la.fetch(al, k1, ra);
        lb.fetch(bl, k1, rb);
        __syncthreads();
        frag_read<BM, BN>(sm, 0, fr[0]);
        // one slab: fragments in fr[u], the next slab's raw values in ra, rb;
        // requests past the last slab re-read it
        auto slab = [&](int t, auto uc) {
            constexpr int u = decltype(uc)::value;
            constexpr int NM = 2 * FM * FN, NW = LA::PER + LB::PER, NL = LA::PER * AL::NRAW + LB::PER * BL::NRAW;
            la.store(al, sm.a[u ^ 1], ra);
            lb.store(bl, sm.b[u ^ 1], rb);
            const int k = min(t + 2, nfull - 1) * GK;
            la.fetch(al, k, ra);
            lb.fetch(bl, k, rb);
            frag_mfma<0, 2, BM, BN>(fr[u], acc);
            static_for<NM>([&](auto) {
                __builtin_amdgcn_sched_group_barrier(0x008, 1, 0);                       // MFMA
                __builtin_amdgcn_sched_group_barrier(0x200, (NW + NM - 1) / NM, 0);      // DS write
                __builtin_amdgcn_sched_group_barrier(0x020, (NL + NM - 1) / NM, 0);      // VMEM read
            });
            __syncthreads();
            frag_read<BM, BN>(sm, u ^ 1, fr[u ^ 1]);
            frag_mfma<2, 4, BM, BN>(fr[u], acc);
            static_for<NM>([&](auto) {
                __builtin_amdgcn_sched_group_barrier(0x008, 1, 0);
                __builtin_amdgcn_sched_group_barrier(0x100, (2 * (FM + FN) + NM - 1) / NM, 0);  // DS read
            });
        };
        int t = 0;
        for (; t + 2 <= nfull; t += 2) {
            slab(t, std::integral_constant<int, 0>{});
            slab(t + 1, std::integral_constant<int, 1>{});
        }
        if (t < nfull) slab(t, std::integral_constant<int, 0>{});
    }
    if (K > nfull * GK) {
        __syncthreads();
        la.load_tail(al, nfull * GK, K, sm.a[0]);
        lb.load_tail(bl, nfull * GK, K, sm.b[0]);
        __syncthreads();
        frag_read<BM, BN>(sm, 0, fr[0]);
        frag_mfma<0, 4, BM, BN>(fr[0], acc);
    }
    __syncthreads();  // the caller may reuse the LDS
}

// Calls f(row, col, value) for every accumulator value of this thread
// (row, col relative to the tile origin).
template <int BM, int BN, class F>
__device__ __forceinline__ void for_acc_f64(const AccF64<BM, BN>& acc, F&& f)
{
    constexpr int FM = BM / 32, FN = BN / 32;
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    const int wm = (wave & 1) * (BM / 2), wn = (wave >> 1) * (BN / 2);
#pragma unroll
    for (int i = 0; i < FM; ++i)
#pragma unroll
        for (int j = 0; j < FN; ++j)
#pragma unroll
            for (int r = 0; r < 4; ++r)
                f(wm + 16 * i + (lane >> 4) + 4 * r, wn + 16 * j + (lane & 15), acc.v[i][j][r]);
}

}  // namespace ngw
