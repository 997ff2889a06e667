// FP64 ISDF-factored Casida operator kernels (gfx950 MFMA).
//
// The operator of NanoGW's Lanczos path (shared/apply_matvec_BLOCK.F90:25-208)
//   y = d o x' + beta s o C^T M C x',  x' = s o x (full) or x (TDA)
// with C(mu, (v,c)) = Psi_v(mu) Psi_c(mu) is applied WITHOUT forming C:
//   K1  T(mu, (v,b)) = sum_c PsiC(mu,c) x'_b(v,c)        GEMM Nmu x (nv B) x nc
//       t(mu, b)     = sum_v PsiV(mu,v) T(mu,(v,b))      (epilogue, LDS reduce)
//   K2  u(mu, b)     = sum_nu M(mu,nu) t(nu, b)          GEMM Nmu x B x Nmu
//   K3  Y(c, (v,b))  = sum_mu PsiC(mu,c) PsiV(mu,v) u(mu,b)  GEMM nc x (nv B) x Nmu
//       y = alpha (d o x' + beta s o Y) + gamma v0 [+ acc]   (epilogue)
// The epilogue also carries one Horner stage of p(H)
// (apply_matvec_BLOCK.F90:250-265) and the Lanczos "w = w + p(H) q" update
// (lanczos_spectra_BLOCK.F90:91-95).
//
// K1's reduction over v writes per-tile partial sums to a slot buffer instead
// of using atomics; a small kernel sums the slots in a fixed order.  A column's
// bits depend on its place in the call (where its slots are cut), not on how
// many columns follow, for calls of two and more; one column alone takes
// operator_f64_one, which splits the sums.

#include "gemm_direct_f64.h"
#include "operator_loaders.h"

namespace ngw {

static long tiles(long m, int bm, long n, int bn) { return (m + bm - 1) / bm * ((n + bn - 1) / bn); }

// ---------------------------------------------------------------- plain GEMMs
template <int BM, int BN, class AL, class BL>
__global__ __launch_bounds__(GNT) void gemm_plain_kernel(AL al, BL bl, int m, int n, int k, double alpha,
                                                         double* c, long ldc, int mtiles, int ntiles)
{
    __shared__ SmemF64<BM, BN> sm;
    const int tile = xcd_tile(blockIdx.x, ntiles);
    const int m0 = (tile % mtiles) * BM, n0 = (tile / mtiles) * BN;
    AccF64<BM, BN> acc;
    gemm_f64_tile<BM, BN>(al, bl, m0, n0, k, acc, sm);
    for_acc_f64<BM, BN>(acc, [&](int row, int col, double val) {
        int gm = m0 + row, gn = n0 + col;
        if (gm < m && gn < n) c[gm + (long)gn * ldc] = alpha * val;
    });
}

// Tiles of 64 x 128 (two waves per SIMD; TF/s, in brackets 128 x 128 with one:
// 67.2 (64.1) at 31461 x 2000 x 2000, 70.9 (69.1) at 4096^3, 55.8 (54.2) at
// 32768 x 480 x 480; 128 x 64 64.0, 66.9, 53.4), of 64 x 64 where the wide ones
// are fewer than the CUs (500 x 480 x 480: 30 us, 44 on 64 x 128, 74 on 128 x
// 128).  All tiles add a sum in the same order: the same bits.
template <class AL, class BL>
static int gemm_plain(hipStream_t s, const AL& al, const BL& bl, int m, int n, int k, double alpha, double* c, long ldc)
{
    auto go = [&](auto kernel, int bn) {
        const int mt = (m + 63) / 64, nt = (n + bn - 1) / bn;
        hipLaunchKernelGGL(kernel, dim3(mt * nt), dim3(GNT), 0, s, al, bl, m, n, k, alpha, c, ldc, mt, mt * nt);
    };
    if (m <= 0 || n <= 0) return NGW_OK;
    if (tiles(m, 64, n, 128) < NCU) go(gemm_plain_kernel<64, 64, AL, BL>, 64);
    else go(gemm_plain_kernel<64, 128, AL, BL>, 128);
    NGW_HIP(hipGetLastError());
    return NGW_OK;
}

int gemm_f64(hipStream_t s, int m, int n, int k, const double* a, long lda, const double* b,
             long ldb, double* c, long ldc)
{
    return gemm_plain(s, ColMajorA{a, lda, m}, ColMajorB{b, ldb, n}, m, n, k, 1.0, c, ldc);
}

// C = (A(:, :k1) B(:k1, :)) o (A B): the two products of a tile one after the
// other in registers, so that the result is written once (two products and an
// element-wise kernel move five times its size: the B blocks of a 97,000 x
// 2000 fit, k1 = 40, k = 440, 5.8 -> 3.7 ms).  128 x 64 tiles hold both
// accumulators at two waves per SIMD; 128 x 128, at one, take 0.9 ms more.
template <int BM, int BN>
__global__ __launch_bounds__(GNT) void gemm_pair_kernel(ColMajorA al, ColMajorB bl, int m, int n, int k1, int k,
                                                        double* c, long ldc, int mtiles, int ntiles)
{
    __shared__ SmemF64<BM, BN> sm;
    const int tile = xcd_tile(blockIdx.x, ntiles);
    const int m0 = (tile % mtiles) * BM, n0 = (tile / mtiles) * BN;
    AccF64<BM, BN> p, q;
    gemm_f64_tile<BM, BN>(al, bl, m0, n0, k1, p, sm);
    gemm_f64_tile<BM, BN>(al, bl, m0, n0, k, q, sm);
#pragma unroll
    for (int i = 0; i < BM / 32; ++i)
#pragma unroll
        for (int j = 0; j < BN / 32; ++j) q.v[i][j] *= p.v[i][j];
    for_acc_f64<BM, BN>(q, [&](int row, int col, double val) {
        const int gm = m0 + row, gn = n0 + col;
        if (gm < m && gn < n) c[gm + (long)gn * ldc] = val;
    });
}

int gemm_f64_pair(hipStream_t s, int m, int n, int k1, int k, const double* a, long lda, const double* b, long ldb,
                  double* c, long ldc)
{
    if (m <= 0 || n <= 0) return NGW_OK;
    constexpr int BM = 128, BN = 64;
    const int mt = (m + BM - 1) / BM, nt = (n + BN - 1) / BN;
    hipLaunchKernelGGL((gemm_pair_kernel<BM, BN>), dim3(mt * nt), dim3(GNT), 0, s, ColMajorA{a, lda, m},
                       ColMajorB{b, ldb, n}, m, n, k1, k, c, ldc, mt, mt * nt);
    NGW_HIP(hipGetLastError());
    return NGW_OK;
}

int gemm_f64_tn(hipStream_t s, int m, int n, int k, double alpha, const double* a, long lda,
                const double* b, long ldb, double* c, long ldc)
{
    return gemm_plain(s, ColMajorAT{a, lda, m}, ColMajorB{b, ldb, n}, m, n, k, alpha, c, ldc);
}

// C = alpha A^T B (n x n) where the product is symmetric: the 64 x 64 tiles on
// and above the diagonal, the k sum in S ranges.  2000 columns have 528 such
// tiles, two or three per CU, and k is the grid: without the ranges the CUs
// with three set the time (10.5 ms for k = 97,000, now 8.3; the full product on 128 x
// 128 tiles 11.4).  Range partials lie tile after tile; sym_sum_kernel adds
// them in order and writes each element and its mirror.  With one range (4033
// columns and more, or k below 4096) the tile is written as it is: partials
// would take half of C's size again.
constexpr int SYM = 64;
template <bool SPLIT>
__global__ __launch_bounds__(GNT) void gemm_sym_kernel(ColMajorAT al, ColMajorB bl, int k, int kc, int ntiles,
                                                       double* part, int n, double alpha, double* c, long ldc)
{
    __shared__ SmemF64<SYM, SYM> sm;
    const int id = xcd_tile(blockIdx.x, gridDim.x), split = id / ntiles, tile = id - split * ntiles;
    // tile = tn (tn + 1) / 2 + tm, tm <= tn
    int tn = (int)((sqrt(8.0 * tile + 1.0) - 1.0) * 0.5);
    if ((tn + 1) * (tn + 2) / 2 <= tile) ++tn;
    if (tn * (tn + 1) / 2 > tile) --tn;
    const long k0 = (long)split * kc;
    al.a += k0;
    bl.b += k0;
    AccF64<SYM, SYM> acc;
    const int m0 = (tile - tn * (tn + 1) / 2) * SYM, n0 = tn * SYM;
    gemm_f64_tile<SYM, SYM>(al, bl, m0, n0, min(kc, k - (int)k0), acc, sm);
    if constexpr (SPLIT) {
        double* o = part + (long)id * SYM * SYM;
        for_acc_f64<SYM, SYM>(acc, [&](int row, int col, double val) { o[row + col * SYM] = val; });
    } else {
        for_acc_f64<SYM, SYM>(acc, [&](int row, int col, double val) {
            const int gm = m0 + row, gn = n0 + col;
            if (gm >= n || gn >= n) return;
            c[gm + (long)gn * ldc] = alpha * val;
            if (m0 != n0) c[gn + (long)gm * ldc] = alpha * val;
        });
    }
}

__global__ __launch_bounds__(256) void sym_sum_kernel(const double* part, int S, int ntiles, int n, double alpha,
                                                      double* c, long ldc)
{
    const int tile = blockIdx.x;
    int tn = (int)((sqrt(8.0 * tile + 1.0) - 1.0) * 0.5);
    if ((tn + 1) * (tn + 2) / 2 <= tile) ++tn;
    if (tn * (tn + 1) / 2 > tile) --tn;
    const int m0 = (tile - tn * (tn + 1) / 2) * SYM, n0 = tn * SYM;
    for (int e = threadIdx.x; e < SYM * SYM; e += 256) {
        double s = 0.0;
        for (int p = 0; p < S; ++p) s += part[((long)p * ntiles + tile) * SYM * SYM + e];
        const int gm = m0 + e % SYM, gn = n0 + e / SYM;
        if (gm >= n || gn >= n) continue;
        const double v = alpha * s;
        c[gm + (long)gn * ldc] = v;
        if (m0 != n0) c[gn + (long)gm * ldc] = v;
    }
}

int gemm_f64_tn_sym(hipStream_t s, int n, int k, double alpha, const double* a, long lda, const double* b, long ldb,
                    double* c, long ldc, DevBuf& part)
{
    if (n <= 0) return NGW_OK;
    const int nt = (n + SYM - 1) / SYM, ntiles = nt * (nt + 1) / 2;
    // about eight workgroups per CU, ranges of at least 2048
    int S = std::max(1, std::min((8 * NCU + ntiles - 1) / ntiles, k / 2048));
    const int kc = (k + S - 1) / S;
    S = (k + kc - 1) / kc;
    const ColMajorAT al{a, lda, n};
    const ColMajorB bl{b, ldb, n};
    if (S == 1) {
        hipLaunchKernelGGL(gemm_sym_kernel<false>, dim3(ntiles), dim3(GNT), 0, s, al, bl, k, kc, ntiles, nullptr, n,
                           alpha, c, ldc);
        NGW_HIP(hipGetLastError());
        return NGW_OK;
    }
    NGW_TRY(part.ensure(sizeof(double) * (size_t)S * ntiles * SYM * SYM));
    hipLaunchKernelGGL(gemm_sym_kernel<true>, dim3(ntiles * S), dim3(GNT), 0, s, al, bl, k, kc, ntiles,
                       part.as<double>(), n, alpha, c, ldc);
    hipLaunchKernelGGL(sym_sum_kernel, dim3(ntiles), dim3(256), 0, s, part.as<const double>(), S, ntiles, n, alpha, c,
                       ldc);
    NGW_HIP(hipGetLastError());
    return NGW_OK;
}

// C = A B (column-major A m x k, B k x n) with the k sum split into ranges
// when the tiles alone are too few for the GPU (n of a few vectors): grid
// tiles x S, range partials added in range order by split_sum_kernel.
constexpr int GSM = 128, GSN = 64;
__global__ __launch_bounds__(GNT) void gemm_split_kernel(const double* a, long lda, const double* b, long ldb, int m,
                                                         int n, int k, int kc, int mtiles, int ntiles, double* part)
{
    __shared__ SmemF64<GSM, GSN> sm;
    const int split = blockIdx.y;
    const int tile = xcd_tile(blockIdx.x, mtiles * ntiles);
    const int m0 = (tile % mtiles) * GSM, n0 = (tile / mtiles) * GSN;
    const int k0 = split * kc, K = min(kc, k - k0);
    AccF64<GSM, GSN> acc;
    gemm_f64_tile<GSM, GSN>(ColMajorA{a + (long)k0 * lda, lda, m}, ColMajorB{b + k0, ldb, n}, m0, n0, K, acc, sm);
    const long mn = (long)m * n;
    for_acc_f64<GSM, GSN>(acc, [&](int row, int col, double val) {
        const int gm = m0 + row, gn = n0 + col;
        if (gm < m && gn < n) part[(long)split * mn + gm + (long)gn * m] = val;
    });
}

__global__ void split_sum_kernel(const double* part, int S, int m, int n, double* c, long ldc)
{
    const long mn = (long)m * n;
    for (long t = blockIdx.x * (long)blockDim.x + threadIdx.x; t < mn; t += (long)gridDim.x * blockDim.x) {
        double s = 0.0;
        for (int p = 0; p < S; ++p) s += part[(long)p * mn + t];
        const long gn = t / m, gm = t - gn * m;
        c[gm + gn * ldc] = s;
    }
}

// Splits of a sum of length k over `tiles` tiles: about 1024 workgroups in
// all, each range at least 64 long (four 16-deep slabs).
static int sum_splits(int tiles, int k)
{
    const int want = std::max(1, 1024 / std::max(tiles, 1));
    return std::max(1, std::min(want, (k + 63) / 64));
}

int gemm_f64_split(hipStream_t s, int m, int n, int k, const double* a, long lda, const double* b, long ldb,
                   double* c, long ldc, DevBuf& part)
{
    if (m <= 0 || n <= 0) return NGW_OK;
    const int mt = (m + GSM - 1) / GSM, nt = (n + GSN - 1) / GSN;
    int S = sum_splits(mt * nt, k);
    const int kc = (k + S - 1) / S;
    S = (k + kc - 1) / kc;
    NGW_TRY(part.ensure(sizeof(double) * (size_t)S * m * n));
    hipLaunchKernelGGL(gemm_split_kernel, dim3(mt * nt, S), dim3(GNT), 0, s, a, lda, b, ldb, m, n, k, kc, mt, nt,
                       part.as<double>());
    const long mn = (long)m * n;
    hipLaunchKernelGGL(split_sum_kernel, dim3((unsigned)std::min<long>((mn + 255) / 256, 4096)), dim3(256), 0, s,
                       part.as<const double>(), S, m, n, c, ldc);
    NGW_HIP(hipGetLastError());
    return NGW_OK;
}

// ---------------------------------------------------------------- K1
constexpr int K1N = 64;  // columns of a K1 tile: sizes the slots

template <int BM>
__global__ __launch_bounds__(GNT) void k1_f64_kernel(ColMajorA al, XprimeB bl, const double* psiv, long ldp,
                                                     int nmu, int nc, int nv, int nvec, double* tpart,
                                                     long ldt, int mtiles, int ntiles)
{
    __shared__ union {
        SmemF64<BM, K1N> ab;
        double red[BM][K1N + 2];
    } sm;
    const int tile = xcd_tile(blockIdx.x, ntiles);
    const int tm = tile % mtiles, tn = tile / mtiles;
    const int m0 = tm * BM, n0 = tn * K1N;
    const int N = nv * nvec;
    AccF64<BM, K1N> acc;
    gemm_f64_tile<BM, K1N>(al, bl, m0, n0, nc, acc, sm.ab);
    // T(mu, j) PsiV(mu, v(j)) into LDS, then per-(mu, b) sums over the tile's v range
    // (entries past nmu or N are never summed or stored: their loads are
    // clamped, not skipped, so that no branch stands between the loads)
    for_acc_f64<BM, K1N>(acc, [&](int row, int col, double val) {
        const int gm = min(m0 + row, nmu - 1), gn = n0 + col;
        sm.red[row][col] = val * psiv[gm + (long)(gn % nv) * ldp];
    });
    __syncthreads();
    const int nend = min(n0 + K1N, N);
    const int b_lo = n0 / nv, b_hi = (nend - 1) / nv;
    const int nbt = b_hi - b_lo + 1;
    for (int e = threadIdx.x; e < BM * nbt; e += GNT) {
        int row = e % BM, b = b_lo + e / BM;
        int c0 = max(n0, b * nv) - n0, c1 = min(nend, (b + 1) * nv) - n0;
        double s = 0.0;
        for (int cc = c0; cc < c1; ++cc) s += sm.red[row][cc];
        int gm = m0 + row;
        int slot = tn - (b * nv) / K1N;
        if (gm < nmu) tpart[((long)slot * nvec + b) * ldt + gm] = s;
    }
}

// K1 without LDS slabs for small products: four waves of 16 (16 FM) x 16
// tiles side by side make a (16 FM) x K1N tile, so the slot partial sums are
// those of k1_f64_kernel, bit for bit.  With at most two slots per vector
// (nv <= K1N) the second slot of a vector that has only one is set to zero,
// and K2 adds the two while it loads them (SlotPairB).
template <int FM, int D>
__global__ __launch_bounds__(GNT) void k1_direct_kernel(ColMajorA al, XprimeB bl, const double* psiv, long ldp,
                                                        int nmu, int nc, int nv, int nvec, double* tpart, long ldt,
                                                        int mtiles, int ntiles)
{
    __shared__ double red[16 * FM][K1N + 2];
    const int tile = xcd_tile(blockIdx.x, ntiles);
    const int tm = tile % mtiles, tn = tile / mtiles;
    const int m0 = tm * 16 * FM, n0 = tn * K1N;
    const int N = nv * nvec, wn = 16 * (threadIdx.x >> 6);
    AccDirect<FM, 1> acc;
    gemm_f64_direct<FM, 1, D>(al, bl, m0, n0 + wn, nc, acc);
    const int gn = n0 + wn + (threadIdx.x & 15);
    const double* pv = psiv + (long)(gn % nv) * ldp;
    for_acc_direct<FM, 1>(acc, [&](int row, int col, double val) {
        red[row][wn + col] = val * pv[min(m0 + row, nmu - 1)];
    });
    __syncthreads();
    const int nend = min(n0 + K1N, N);
    const int b_lo = n0 / nv, b_hi = (nend - 1) / nv;
    const int nbt = b_hi - b_lo + 1;
    for (int e = threadIdx.x; e < 16 * FM * nbt; e += GNT) {
        const int row = e % (16 * FM), b = b_lo + e / (16 * FM);
        const int first = (b * nv) / K1N, last = ((b + 1) * nv - 1) / K1N;
        const int c0 = max(n0, b * nv) - n0, c1 = min(nend, (b + 1) * nv) - n0;
        double s = 0.0;
        for (int cc = c0; cc < c1; ++cc) s += red[row][cc];
        const int gm = m0 + row, slot = tn - first;
        if (gm < nmu) {
            tpart[((long)slot * nvec + b) * ldt + gm] = s;
            if (first == last) tpart[((long)nvec + b) * ldt + gm] = 0.0;
        }
    }
}

int k1_slots(int nv) { return (nv - 1) / K1N + 2; }

// t(nu, b) = sum over the K1 tiles that covered vector b, in tile order.
__global__ void k1_reduce_kernel(const double* tpart, long ldt, int nmu, int nvec, int nv, double* t)
{
    const long i = blockIdx.x * (long)blockDim.x + threadIdx.x;
    if (i >= (long)nmu * nvec) return;
    const int b = (int)(i / nmu), nu = (int)(i - (long)b * nmu);
    const int first = (b * nv) / K1N, last = ((b + 1) * nv - 1) / K1N;
    double s = 0.0;
    for (int sl = 0; sl <= last - first; ++sl) s += tpart[((long)sl * nvec + b) * ldt + nu];
    t[nu + (long)b * nmu] = s;
}

int k1_reduce(hipStream_t s, const double* tpart, long ldt, int nmu, int nvec, int nv, double* t)
{
    long total = (long)nmu * nvec;
    hipLaunchKernelGGL(k1_reduce_kernel, dim3((unsigned)((total + 255) / 256)), dim3(256), 0, s, tpart, ldt, nmu,
                       nvec, nv, t);
    NGW_HIP(hipGetLastError());
    return NGW_OK;
}

// ---------------------------------------------------------------- K2
template <int BM, int BN, class BL>
__global__ __launch_bounds__(GNT) void k2_f64_kernel(ColMajorA al, BL bl, int nmu, int nvec, double* u,
                                                     long ldu, int mtiles, int ntiles)
{
    __shared__ SmemF64<BM, BN> sm;
    const int tile = xcd_tile(blockIdx.x, ntiles);
    const int m0 = (tile % mtiles) * BM, n0 = (tile / mtiles) * BN;
    AccF64<BM, BN> acc;
    gemm_f64_tile<BM, BN>(al, bl, m0, n0, nmu, acc, sm);
    for_acc_f64<BM, BN>(acc, [&](int row, int col, double val) {
        int gm = m0 + row, gn = n0 + col;
        if (gm < nmu && gn < nvec) u[gm + (long)gn * ldu] = val;
    });
}

template <int FM, int FN, int D, class BL>
__global__ __launch_bounds__(64) void k2_direct_kernel(ColMajorA al, BL bl, int nmu, int nvec, double* u,
                                                                 long ldu, int mtiles, int ntiles)
{
    const int tile = xcd_tile(blockIdx.x, ntiles);
    const int m0 = (tile % mtiles) * 16 * FM, n0 = (tile / mtiles) * 16 * FN;
    AccDirect<FM, FN> acc;
    gemm_f64_direct<FM, FN, D>(al, bl, m0, n0, nmu, acc);
    for_acc_direct<FM, FN>(acc, [&](int row, int col, double val) {
        const int gm = m0 + row, gn = n0 + col;
        if (gm < nmu && gn < nvec) u[gm + (long)gn * ldu] = val;
    });
}

// ---------------------------------------------------------------- K3
// Epilogue of NI x NJ fragments of four rows each (acc.v[i][j][r]: tile row
// 16 i + 4 r + lane / 16, tile column 16 j + lane % 16): the terms of one or
// two fragments are loaded before any of their results is stored.
template <int NI, int NJ, class V>
__device__ __forceinline__ void k3_epilogue(const OperatorEpilogue& ep, const V& v, int c0, int j0, int nc, int nv,
                                            int N)
{
    const int lane = threadIdx.x & 63;
#pragma unroll
    for (int j = 0; j < NJ; ++j) {
        const int col = j0 + 16 * j + (lane & 15);
        if (col >= N) continue;
        const int b = col / nv;
        const long base = col - b * nv;
        constexpr int CH = NI % 2 == 0 ? 2 : 1;  // fragment rows whose terms are in flight together
#pragma unroll
        for (int i0 = 0; i0 < NI; i0 += CH) {
            const int c = c0 + 16 * i0 + (lane >> 4);
            OperatorEpilogue::Terms t[4 * CH];
#pragma unroll
            for (int r = 0; r < 4 * CH; ++r) t[r] = ep.load(base + (long)min(c + 4 * r, nc - 1) * nv, b);
#pragma unroll
            for (int r = 0; r < 4 * CH; ++r)
                if (c + 4 * r < nc) ep.store(base + (long)(c + 4 * r) * nv, b, ep.value(t[r], v[i0 + r / 4][j][r % 4]));
        }
    }
}

template <int FM, int FN, int D>
__global__ __launch_bounds__(64) void k3_direct_kernel(ColMajorAT al, WeightedPsiVB bl, int nmu, int nc,
                                                                 int nv, int nvec, OperatorEpilogue ep, int mtiles,
                                                                 int ntiles)
{
    const int tile = xcd_tile(blockIdx.x, ntiles);
    const int m0 = (tile % mtiles) * 16 * FM, n0 = (tile / mtiles) * 16 * FN;
    const int N = nv * nvec;
    AccDirect<FM, FN> acc;
    gemm_f64_direct<FM, FN, D>(al, bl, m0, n0, nmu, acc);
    k3_epilogue<FM, FN>(ep, acc.v, m0, n0, nc, nv, N);
}

template <int BM, int BN>
__global__ __launch_bounds__(GNT) void k3_f64_kernel(ColMajorAT al, WeightedPsiVB bl, int nmu, int nc, int nv,
                                                     int nvec, OperatorEpilogue ep, int mtiles, int ntiles)
{
    __shared__ SmemF64<BM, BN> sm;
    const int tile = xcd_tile(blockIdx.x, ntiles);
    const int m0 = (tile % mtiles) * BM, n0 = (tile / mtiles) * BN;
    const int N = nv * nvec;
    AccF64<BM, BN> acc;
    gemm_f64_tile<BM, BN>(al, bl, m0, n0, nmu, acc, sm);
    const int wave = threadIdx.x >> 6;
    k3_epilogue<BM / 32, BN / 32>(ep, acc.v, m0 + (wave & 1) * (BM / 2), n0 + (wave >> 1) * (BN / 2), nc, nv, N);
}

// ---------------------------------------------------------------- one vector
// The operator on one vector (NanoGW's single-vector routines,
// apply_matvec_UltraLowMem.F90:25-222).  K1 and K3 have only nv columns, so a
// workgroup takes 32 rows and up to 64 v without LDS slabs
// (gemm_direct_f64.h), its four waves split the sum, and the sum is split
// further into S ranges over the grid where the row tiles are fewer than the
// CUs and the ranges stay long.  Partials are added in wave and range order:
// no atomics, and the result does not depend on scheduling.  A small operator
// is three launches of 7 us or less: 31 us a call at 480 x 8 x 56, against 45
// for seven launches on 128 x 64 LDS tiles; 66 against 115 at 3000 x 64 x
// 700, 160 against 203 at 5000 x 100 x 1500 (M alone is 38 us of reading).
constexpr int OVM = 32, OVW = 4;  // rows of a tile, waves that split its sum
constexpr double OV_BIG = 2.5e8;  // nmu nv nc from which K1 is bound by its operand reads

// This wave's part [k0, k0 + K) of a range of n, in blocks of 16.
__device__ __forceinline__ void ov_wave_range(int n, int& k0, int& K)
{
    const int kw = (n + 16 * OVW - 1) / (16 * OVW) * 16;
    k0 = min((int)(threadIdx.x >> 6) * kw, n);
    K = min(kw, n - k0);
}
template <int FN>
constexpr int ov_depth() { return FN >= 4 ? 2 : FN >= 2 ? 3 : 4; }

// part[(split nchunk + chunk) nmu + mu] = sum_{v in chunk} PsiV(mu, v) sum_{c in range} PsiC(mu, c) s x(v, c)
template <int FN>
__global__ __launch_bounds__(64 * OVW) void ov_k1_kernel(const double* psi, long ldp, const double* x,
                                                         const double* sx, int nmu, int nc, int nv, int kc,
                                                         double* part)
{
    __shared__ double red[OVW][OVM];
    const int m0 = blockIdx.x * OVM, chunk = blockIdx.y, split = blockIdx.z;
    const int v0 = chunk * 16 * FN, lane = threadIdx.x & 63;
    int k0, K;
    ov_wave_range(min(kc, nc - split * kc), k0, K);
    const long c0 = (long)split * kc + k0;
    AccDirect<OVM / 16, FN> acc;
    gemm_f64_direct<OVM / 16, FN, ov_depth<FN>()>(
        ColMajorA{psi + (nv + c0) * ldp, ldp, nmu},
        XprimeB{x + c0 * nv, sx ? sx + c0 * nv : nullptr, 0, nv, nv}, m0, v0, K, acc);
#pragma unroll
    for (int i = 0; i < OVM / 16; ++i) {
        double t[4] = {0.0, 0.0, 0.0, 0.0};
#pragma unroll
        for (int j = 0; j < FN; ++j) {
            // past the ends the load is clamped and counts as zero: a branch
            // would make every load wait for the one before it
            const int v = v0 + 16 * j + (lane & 15);
            const double* pv = psi + (long)min(v, nv - 1) * ldp;
#pragma unroll
            for (int r = 0; r < 4; ++r) {
                const double p = pv[min(m0 + 16 * i + (lane >> 4) + 4 * r, nmu - 1)];
                t[r] += v < nv ? acc.v[i][j][r] * p : 0.0;
            }
        }
#pragma unroll
        for (int r = 0; r < 4; ++r) {
#pragma unroll
            for (int off = 8; off > 0; off >>= 1) t[r] += __shfl_xor(t[r], off, 64);
            if ((lane & 15) == 0) red[threadIdx.x >> 6][16 * i + (lane >> 4) + 4 * r] = t[r];
        }
    }
    __syncthreads();
    const int gm = m0 + threadIdx.x;
    if (threadIdx.x < OVM && gm < nmu) {
        double s = 0.0;
#pragma unroll
        for (int w = 0; w < OVW; ++w) s += red[w][threadIdx.x];
        part[((long)split * gridDim.y + chunk) * nmu + gm] = s;
    }
}

// ov_k1_kernel for nv > 16: both operands run along memory by rows and
// columns, not along k, so a lane takes pairs of neighbouring rows (fragments
// 2 p and 2 p + 1) and of neighbouring columns (2 q, 2 q + 1) in 16-byte
// loads, half the loads of the fragment-by-fragment form.  No two waves share
// an operand line, so what a wave reads per MFMA is what bounds the large
// molecules (L2): 64 rows (FM = 4) on an x scaled beforehand instead of 32 on
// x and sqrtR take K1 of 5000 x 100 x 1500 from 65 to 57 us.
template <int FM, int FN>
__global__ __launch_bounds__(64 * OVW) void ov_k1_pair_kernel(const double* psi, long ldp, const double* x,
                                                              const double* sx, int nmu, int nc, int nv, int kc,
                                                              double* part)
{
    constexpr int P = FM / 2, Q = FN / 2, BM = 16 * FM;
    typedef double f64x2 __attribute__((ext_vector_type(2), aligned(8)));
    __shared__ double red[OVW][BM];
    const int m0 = blockIdx.x * BM, chunk = blockIdx.y, split = blockIdx.z;
    const int v0 = chunk * 16 * FN, lane = threadIdx.x & 63, r16 = lane & 15, k4 = lane >> 4;
    int k0, K;
    ov_wave_range(min(kc, nc - split * kc), k0, K);
    const long c0 = (long)split * kc + k0;
    // pairs that would leave the array start one element earlier: their first
    // element is then the pair's second
    int rbase[P], cbase[Q];
#pragma unroll
    for (int p = 0; p < P; ++p) rbase[p] = min(m0 + 32 * p + 2 * r16, nmu - 2);
#pragma unroll
    for (int q = 0; q < Q; ++q) cbase[q] = min(v0 + 32 * q + 2 * r16, nv - 2);
    const double* pa = psi + (nv + c0 + k4) * ldp;
    const double* px = x + (c0 + k4) * nv;
    const double* ps = sx ? sx + (c0 + k4) * nv : nullptr;
    f64x4 acc[FM][FN];
#pragma unroll
    for (int i = 0; i < FM; ++i)
#pragma unroll
        for (int j = 0; j < FN; ++j) acc[i][j] = f64x4{0.0, 0.0, 0.0, 0.0};
    // one step: four k (this lane's is 4 t + k4)
    struct Raw {
        f64x2 a[P], x[Q], s[Q];
    };
    const int steps = (K + 3) / 4;
    auto fetch = [&](int t, Raw& r) {
        const long k = min(4 * t + k4, K - 1) - k4;  // k past the end re-reads the last
#pragma unroll
        for (int p = 0; p < P; ++p) r.a[p] = *reinterpret_cast<const f64x2*>(pa + k * ldp + rbase[p]);
#pragma unroll
        for (int q = 0; q < Q; ++q) {
            r.x[q] = *reinterpret_cast<const f64x2*>(px + k * nv + cbase[q]);
            if (ps) r.s[q] = *reinterpret_cast<const f64x2*>(ps + k * nv + cbase[q]);
        }
    };
    auto multiply = [&](int t, const Raw& r) {
        const bool ok = 4 * t + k4 < K;
        double a[FM], b[FN];
#pragma unroll
        for (int p = 0; p < P; ++p) {
            a[2 * p] = ok ? (rbase[p] == m0 + 32 * p + 2 * r16 ? r.a[p].x : r.a[p].y) : 0.0;
            a[2 * p + 1] = ok ? r.a[p].y : 0.0;
        }
#pragma unroll
        for (int q = 0; q < Q; ++q) {
            const bool first = cbase[q] == v0 + 32 * q + 2 * r16;
            const double b0 = ps ? r.x[q].x * r.s[q].x : r.x[q].x, b1 = ps ? r.x[q].y * r.s[q].y : r.x[q].y;
            b[2 * q] = ok ? (first ? b0 : b1) : 0.0;
            b[2 * q + 1] = ok ? b1 : 0.0;
        }
#pragma unroll
        for (int i = 0; i < FM; ++i)
#pragma unroll
            for (int j = 0; j < FN; ++j)
                acc[i][j] = __builtin_amdgcn_mfma_f64_16x16x4f64(a[i], b[j], acc[i][j], 0, 0, 0);
    };
    constexpr int D = FM * FN >= 16 ? 4 : FN >= 4 ? 6 : 8;  // steps in flight
    if (steps > 0) {
        Raw raw[D];
        static_for<D - 1>([&](auto uc) { fetch(min(decltype(uc)::value, steps - 1), raw[decltype(uc)::value]); });
        for (int t = 0; t < steps; t += D)
            static_for<D>([&](auto uc) {
                constexpr int u = decltype(uc)::value;
                fetch(min(t + u + D - 1, steps - 1), raw[(u + D - 1) % D]);
                if (t + u < steps) multiply(t + u, raw[u]);
            });
    }
    double t8[FM][4] = {};
#pragma unroll
    for (int j = 0; j < FN; ++j) {
        const int v = v0 + 32 * (j / 2) + 2 * r16 + (j & 1);
        const double* pv = psi + (long)min(v, nv - 1) * ldp;
#pragma unroll
        for (int p = 0; p < P; ++p)
#pragma unroll
            for (int r = 0; r < 4; ++r) {
                // (a row pair past the end only reaches sums that are not
                // stored, but for the pair that the last row of an odd nmu begins)
                const int gm = m0 + 32 * p + 2 * (k4 + 4 * r), gb = min(gm, nmu - 2);
                const f64x2 w = *reinterpret_cast<const f64x2*>(pv + gb);
                t8[2 * p][r] += v < nv ? acc[2 * p][j][r] * (gm == gb ? w.x : w.y) : 0.0;
                t8[2 * p + 1][r] += v < nv ? acc[2 * p + 1][j][r] * w.y : 0.0;
            }
    }
#pragma unroll
    for (int i = 0; i < FM; ++i)
#pragma unroll
        for (int r = 0; r < 4; ++r) {
#pragma unroll
            for (int off = 8; off > 0; off >>= 1) t8[i][r] += __shfl_xor(t8[i][r], off, 64);
            if (r16 == 0) red[threadIdx.x >> 6][32 * (i / 2) + 2 * (k4 + 4 * r) + (i & 1)] = t8[i][r];
        }
    __syncthreads();
    const int gm = m0 + threadIdx.x;
    if (threadIdx.x < BM && gm < nmu) {
        double s = 0.0;
#pragma unroll
        for (int w = 0; w < OVW; ++w) s += red[w][threadIdx.x];
        part[((long)split * gridDim.y + chunk) * nmu + gm] = s;
    }
}

// x' = s o x for the large molecules' K1
__global__ void ov_scale_kernel(const double* x, const double* s, long ncv, double* xs)
{
    for (long i = blockIdx.x * (long)blockDim.x + threadIdx.x; i < ncv; i += (long)gridDim.x * blockDim.x)
        xs[i] = s[i] * x[i];
}

// PsiC(mu, c) u(mu): u goes with the operand that has fewer fragments.
struct WeightedPsiCA {
    static constexpr bool kContig = true;
    static constexpr int NRAW = 2;
    struct Handle { const double* pc; const double* u; };
    const double* psic; long ldp; const double* u; int MN;
    __device__ Handle row(int c) const { return {psic + (long)c * ldp, u}; }
    __device__ Handle shift(const Handle& h, int k) const { return {h.pc + k, h.u + k}; }
    __device__ void fetch(const Handle& h, int mu, double (&r)[2]) const
    {
        r[0] = h.pc[mu];
        r[1] = h.u[mu];
    }
    __device__ double combine(const double (&r)[2]) const { return r[0] * r[1]; }
};

// t(mu) = sum over the nparts partials, in order
__global__ void ov_sum_kernel(const double* part, int nparts, long n, double* t)
{
    for (long i = blockIdx.x * (long)blockDim.x + threadIdx.x; i < n; i += (long)gridDim.x * blockDim.x) {
        double s = 0.0;
        for (int p = 0; p < nparts; ++p) s += part[(long)p * n + i];
        t[i] = s;
    }
}

// u = M t for a small M: 16 rows per workgroup, eight waves split the
// columns (a wave reads 16 rows of four columns per load), one launch instead
// of gemv_wide's two.
constexpr int OV2W = 8;
constexpr int OV2_MAX = 960;  // at 480 rows 6.4 us against 9.0 for gemv_wide, at 1000 9.5 / 9.3, at 3000 21 / 18
__global__ __launch_bounds__(64 * OV2W) void ov_k2_kernel(const double* m, long ldm, int nmu, const double* t,
                                                          double* u)
{
    __shared__ double red[OV2W][16];
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    const int row = min((int)blockIdx.x * 16 + (lane & 15), nmu - 1);
    const int kw = (nmu + OV2W - 1) / OV2W, k0 = wave * kw, k1 = min(nmu, k0 + kw);
    constexpr int U = 8;
    double s[U] = {};
    int k = k0 + (lane >> 4);
    for (; k + 4 * (U - 1) < k1; k += 4 * U) {
        double a[U], b[U];
#pragma unroll
        for (int i = 0; i < U; ++i) {
            a[i] = m[row + (long)(k + 4 * i) * ldm];
            b[i] = t[k + 4 * i];
        }
#pragma unroll
        for (int i = 0; i < U; ++i) s[i] += a[i] * b[i];
    }
    for (; k < k1; k += 4) s[0] += m[row + (long)k * ldm] * t[k];
    double v = ((s[0] + s[1]) + (s[2] + s[3])) + ((s[4] + s[5]) + (s[6] + s[7]));
    v += __shfl_xor(v, 16, 64);
    v += __shfl_xor(v, 32, 64);
    if (lane < 16) red[wave][lane] = v;
    __syncthreads();
    const int gm = blockIdx.x * 16 + threadIdx.x;
    if (threadIdx.x < 16 && gm < nmu) {
        double o = 0.0;
#pragma unroll
        for (int w = 0; w < OV2W; ++w) o += red[w][threadIdx.x];
        u[gm] = o;
    }
}

// Y(v, c) = sum_{mu in range} PsiC(mu, c) PsiV(mu, v) u(mu): with one range the
// operator epilogue, otherwise part[split ncv + v + nv c].  The waves' tiles
// meet in LDS; wave w adds up fragments w, w + OVW, ...
template <int FN>
__global__ __launch_bounds__(64 * OVW) void ov_k3_kernel(const double* psi, long ldp, const double* u, int nmu, int nc,
                                                         int nv, int kmu, OperatorEpilogue ep, double* part)
{
    constexpr int FM = OVM / 16;
    __shared__ double red[OVW][FM * FN][4][64];
    const int m0 = blockIdx.x * OVM, v0 = blockIdx.y * 16 * FN, split = blockIdx.z;
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    int k0, K;
    ov_wave_range(min(kmu, nmu - split * kmu), k0, K);
    const long mu0 = (long)split * kmu + k0;
    AccDirect<FM, FN> acc;
    gemm_f64_direct<FM, FN, ov_depth<FN>()>(WeightedPsiCA{psi + nv * ldp + mu0, ldp, u + mu0, nc},
                                            ColMajorB{psi + mu0, ldp, nv}, m0, v0, K, acc);
#pragma unroll
    for (int i = 0; i < FM; ++i)
#pragma unroll
        for (int j = 0; j < FN; ++j)
#pragma unroll
            for (int r = 0; r < 4; ++r) red[wave][i * FN + j][r][lane] = acc.v[i][j][r];
    __syncthreads();
    const long ncv = (long)nv * nc;
    for (int f = wave; f < FM * FN; f += OVW) {
        const int v = v0 + 16 * (f % FN) + (lane & 15), c = m0 + 16 * (f / FN) + (lane >> 4);
        if (v >= nv) continue;
        OperatorEpilogue::Terms t[4];
        if (!part)
#pragma unroll
            for (int r = 0; r < 4; ++r) t[r] = ep.load(v + (long)min(c + 4 * r, nc - 1) * nv, 0);
#pragma unroll
        for (int r = 0; r < 4; ++r) {
            if (c + 4 * r >= nc) continue;
            const long idx = v + (long)(c + 4 * r) * nv;
            double y = 0.0;
#pragma unroll
            for (int w = 0; w < OVW; ++w) y += red[w][f][r][lane];
            if (part) part[split * ncv + idx] = y;
            else ep.store(idx, 0, ep.value(t[r], y));
        }
    }
}

// y(idx) = sum of the S partials (range order), then the operator epilogue
__global__ void ov_epilogue_kernel(OperatorEpilogue ep, const double* part, int S, long ncv)
{
    for (long i = blockIdx.x * (long)blockDim.x + threadIdx.x; i < ncv; i += (long)gridDim.x * blockDim.x) {
        const OperatorEpilogue::Terms t = ep.load(i, 0);
        double y = 0.0;
        for (int c = 0; c < S; ++c) y += part[(long)c * ncv + i];
        ep.store(i, 0, ep.value(t, y));
    }
}

// Ranges of a sum of length k over `wgs` row and column tiles: as many as
// leave at most `want` workgroups, each wave's part at least 64 long.
static int ov_splits(int wgs, int k, int want)
{
    return std::max(1, std::min(want / std::max(wgs, 1), k / (64 * OVW)));
}

int operator_f64_one(ngw_context* ctx, const OperatorArgs& a)
{
    hipStream_t s = ctx->stream;
    const int nmu = ctx->n_intp, nv = ctx->nval, nc = ctx->ncond;
    const long ncv = ctx->ncv, ldp = ctx->ld_psi;
    const double* psi = ctx->psi.as<double>();
    // K1: columns in chunks of 16 (nv <= 16), 32 or 64; K3: of up to 64.
    // Ranges up to one workgroup per CU (2000 x 40 x 400: K1 14.2 us, K3 16.0,
    // against 17.8 and 20.8 with two); the largest molecules take 64-row K1
    // tiles and two per CU (5000 x 100 x 1500: K1 57 us against 65 - 81 for the
    // other choices, K3 51 against 66 with one; 3000 x 64 x 700: 27 us
    // against 20 with the 32-row tiles).  Whole calls, large form / small form:
    // 3000 x 70 x 800 77 / 65 us, 3600 x 72 x 900 92 / 78, 4200 x 90 x 900
    // 99 / 101, 4000 x 100 x 1000 105 / 93, 4500 x 100 x 1200 124 / 139,
    // 5000 x 100 x 1500 145 / 184: they meet at 3.4e8 to 5e8, above the line.
    const bool big = nv > 32 && nmu > 1 && (double)nmu * nv * nc >= OV_BIG;
    const int fn1 = nv <= 16 || nmu < 2 ? 1 : nv <= 32 ? 2 : 4, nch1 = (nv + 16 * fn1 - 1) / (16 * fn1);
    const int nch3 = (nv + 63) / 64, fn3 = ((nv + nch3 - 1) / nch3 + 15) / 16;
    const int bm1 = big ? 2 * OVM : OVM;
    const int mt1 = (nmu + bm1 - 1) / bm1, mt3 = (nc + OVM - 1) / OVM;
    const int want = big ? 2 * NCU : NCU;
    int S1 = ov_splits(mt1 * nch1, nc, want), S3 = ov_splits(mt3 * nch3, nmu, want);
    const int kc = (nc + S1 - 1) / S1, kmu = (nmu + S3 - 1) / S3;
    S1 = (nc + kc - 1) / kc;
    S3 = (nmu + kmu - 1) / kmu;
    const int np1 = S1 * nch1;
    NGW_TRY(ctx->ex_t.ensure(sizeof(double) * ((size_t)np1 * nmu + 2 * (size_t)nmu)));
    if (S3 > 1) NGW_TRY(ctx->ex_s.ensure(sizeof(double) * (size_t)S3 * ncv));
    double* p1 = ctx->ex_t.as<double>();
    double* t = p1 + (size_t)np1 * nmu;
    double* u = t + nmu;
    double* p3 = S3 > 1 ? ctx->ex_s.as<double>() : nullptr;
    const double* sx = a.tda ? nullptr : ctx->sqrtr.as<double>();  // null once x is scaled
    const OperatorEpilogue ep = a.epilogue(ctx);
    const double* x = a.x;
    if (big && sx) {
        NGW_TRY(ctx->ex_x.ensure(sizeof(double) * (size_t)ncv));
        hipLaunchKernelGGL(ov_scale_kernel, dim3((unsigned)std::min<long>((ncv + 255) / 256, 2048)), dim3(256), 0, s,
                           a.x, sx, ncv, ctx->ex_x.as<double>());
        x = ctx->ex_x.as<double>();
        sx = nullptr;
    }
    {
        ProfScope ps(ctx, KC_K1);
        auto go = [&](auto kernel) {
            hipLaunchKernelGGL(kernel, dim3(mt1, nch1, S1), dim3(64 * OVW), 0, s, psi, ldp, x, sx, nmu, nc, nv, kc,
                               np1 > 1 ? p1 : t);
        };
        if (fn1 == 1) go(ov_k1_kernel<1>);
        else if (fn1 == 2) go(ov_k1_pair_kernel<2, 2>);
        else if (!big) go(ov_k1_pair_kernel<2, 4>);
        else go(ov_k1_pair_kernel<4, 4>);
        if (np1 > 1)
            hipLaunchKernelGGL(ov_sum_kernel, dim3((nmu + 255) / 256), dim3(256), 0, s, p1, np1, (long)nmu, t);
    }
    {
        ProfScope ps(ctx, KC_K2);
        if (nmu <= OV2_MAX)
            hipLaunchKernelGGL(ov_k2_kernel, dim3((nmu + 15) / 16), dim3(64 * OV2W), 0, s, ctx->mmat.as<double>(),
                               (long)ctx->ld_m, nmu, t, u);
        else
            NGW_TRY(gemv_wide(s, ctx->mmat.as<double>(), ctx->ld_m, nmu, nmu, t, u, ctx->gv_part));
    }
    {
        ProfScope ps(ctx, KC_K3);
        auto go = [&](auto kernel) {
            hipLaunchKernelGGL(kernel, dim3(mt3, nch3, S3), dim3(64 * OVW), 0, s, psi, ldp, u, nmu, nc, nv, kmu, ep,
                               p3);
        };
        if (fn3 == 1) go(ov_k3_kernel<1>);
        else if (fn3 == 2) go(ov_k3_kernel<2>);
        else if (fn3 == 3) go(ov_k3_kernel<3>);
        else go(ov_k3_kernel<4>);
        if (p3)
            hipLaunchKernelGGL(ov_epilogue_kernel, dim3((unsigned)std::min<long>((ncv + 255) / 256, 2048)), dim3(256),
                               0, s, ep, p3, S3, ncv);
    }
    NGW_HIP(hipGetLastError());
    return NGW_OK;
}

// ---------------------------------------------------------------- launchers
// Tile choice of the FP64 products.  Every form below adds each element's sum
// in the same order, so the choice changes no bit of a result.  A lone
// workgroup per CU needs 0.35 us per 16 k for a 32 x 32 tile, 0.54 us for
// 64 x 64 and 1.0 us for 128 x 64, a 16 x 16 tile per wave (no LDS) about
// 0.2 us, so few tiles go to the small forms; with every CU busy the larger
// tiles win through fewer loads per MFMA.  Measured (us, nmu x nv x nc, B):
//   K1 480x8x56, 8: 7 direct / 11.6 64x64; 731x13x129, 37: 12.4 / 15.9;
//      1000x24x250, 80: 40 / 33; 1000x24x250, 100: 42 64x64 / 51 128x64;
//      2000x40x400, 40: 77 / 73; 2000x40x400, 800: 1064 / 1056;
//      5000x100x1500, 4: 195 / 233; 5000x100x1500, 100: 2914 / 2848
//      (128 rows are 0 to 5% faster once both forms fill their rounds of
//      workgroups, and up to 17% slower where a few tiles more than a round are
//      left for the last one: that, not nc, is what parts the two, and the line
//      at nc = 1024 only keeps the largest operators on 128 rows)
//   K2 480, 256: 10 direct / 14 32x32 / 22 64x64; 5000, 40: 98 / 124 / 168;
//      2000, 200: 79 / 54 / 74; 5000, 200: 450 / 247 / 333;
//      5000, 1600: 1661 32x32 / 1278 128x64
//   K3 480x8x56, 256: 16 direct / 28 64x64 / 44 128x64; 1000x24x250, 80:
//      42 / 51 / 82; 2000x40x400, 40: 134 / 89 / 139; 2000x40x400, 200:
//      500 / 281 / 258; 5000x100x1500, 200: 5241 64x64 / 4575 128x64
constexpr int DIRECT_K1_TILES = NCU;  // 64 x 64 tiles: at most one per CU
constexpr int DIRECT_K3_TILES = NCU / 2;
constexpr int WIDE_K3_TILES = NCU;
constexpr int DIRECT_K2_WAVES = 4 * NCU;  // 16 x 16 tiles: at most one per SIMD
constexpr int WIDE_K2_TILES = 8 * NCU;    // 32 x 32 tiles
constexpr int WIDE_K1_NC = 1024;
// A launch counts its threads in 32 bits and runs only the remainder of a larger
// one, without an error (64-row K1 tiles: 4096 points and 131,072 vectors of 128
// valence states): the 128-row tiles, half as many, take such a call.
constexpr long MAX_GRID_THREADS = (1L << 32) - 1;

static bool k1_direct(int nmu, int nv, int B) { return tiles(nmu, 64, (long)nv * B, 64) <= DIRECT_K1_TILES; }

// K1 into the slot partial sums, and their sum t unless K2 adds the two slots
// itself (*pair).
static int launch_k1(ngw_context* ctx, const double* x, long ldx, const double* sx, int B, double* tpart,
                     double* t, bool* pair)
{
    const int nmu = ctx->n_intp, nv = ctx->nval, nc = ctx->ncond;
    const double* psi = ctx->psi.as<double>();
    const long ldp = ctx->ld_psi, N = (long)nv * B;
    hipStream_t s = ctx->stream;
    const ColMajorA al{psi + (long)nv * ldp, ldp, nmu};
    const XprimeB bl{x, sx, ldx, nv, nv * B};
    const bool direct = k1_direct(nmu, nv, B);
    {
        ProfScope ps(ctx, KC_K1);
        auto go = [&](auto kernel, int bm) {
            const int mt = (nmu + bm - 1) / bm, nt = (int)((N + K1N - 1) / K1N);
            hipLaunchKernelGGL(kernel, dim3(mt * nt), dim3(GNT), 0, s, al, bl, psi, ldp, nmu, nc, nv, B, tpart,
                               (long)nmu, mt, mt * nt);
        };
        if (direct && tiles(nmu, 64, N, 64) <= DIRECT_K1_TILES / 4) go(k1_direct_kernel<1, 2>, 16);
        else if (direct) go(k1_direct_kernel<2, 2>, 32);
        else if (nc < WIDE_K1_NC && tiles(nmu, 64, N, K1N) * GNT <= MAX_GRID_THREADS) go(k1_f64_kernel<64>, 64);
        else go(k1_f64_kernel<128>, 128);
        NGW_HIP(hipGetLastError());
    }
    *pair = direct && nv <= K1N;
    if (*pair) return NGW_OK;
    ProfScope ps(ctx, KC_CONVERT);
    return k1_reduce(s, tpart, (long)nmu, nmu, B, nv, t);
}

template <class BL>
static int launch_k2(ngw_context* ctx, const BL& bl, int B, double* u)
{
    const int nmu = ctx->n_intp;
    const ColMajorA al{ctx->mmat.as<double>(), ctx->ld_m, nmu};
    auto go = [&](auto kernel, int bm, int bn, int nt) {
        const int mt = (nmu + bm - 1) / bm, n = mt * ((B + bn - 1) / bn);
        hipLaunchKernelGGL(kernel, dim3(n), dim3(nt), 0, ctx->stream, al, bl, nmu, B, u, (long)nmu, mt, n);
    };
    if (tiles(nmu, 16, B, 16) <= DIRECT_K2_WAVES) go(k2_direct_kernel<1, 1, 4, BL>, 16, 16, 64);
    else if (tiles(nmu, 32, B, 32) <= WIDE_K2_TILES) go(k2_f64_kernel<32, 32, BL>, 32, 32, GNT);
    else go(k2_f64_kernel<128, 64, BL>, 128, 64, GNT);
    NGW_HIP(hipGetLastError());
    return NGW_OK;
}

static int launch_k3(ngw_context* ctx, const double* u, int B, const OperatorEpilogue& ep)
{
    const int nmu = ctx->n_intp, nv = ctx->nval, nc = ctx->ncond;
    const double* psi = ctx->psi.as<double>();
    const long ldp = ctx->ld_psi, N = (long)nv * B;
    const ColMajorAT al{psi + (long)nv * ldp, ldp, nc};
    const WeightedPsiVB bl{psi, ldp, u, (long)nmu, nv, nv * B};
    auto go = [&](auto kernel, int bm, int bn, int nt) {
        const int mt = (nc + bm - 1) / bm, n = mt * (int)((N + bn - 1) / bn);
        hipLaunchKernelGGL(kernel, dim3(n), dim3(nt), 0, ctx->stream, al, bl, nmu, nc, nv, B, ep, mt, n);
    };
    const long t64 = tiles(nc, 64, N, 64);
    if (t64 <= DIRECT_K3_TILES) {
        if (tiles(nc, 16, N, 16) <= 4 * NCU) go(k3_direct_kernel<1, 1, 4>, 16, 16, 64);
        else go(k3_direct_kernel<2, 1, 4>, 32, 16, 64);
    } else if (t64 <= WIDE_K3_TILES) {
        go(k3_f64_kernel<64, 64>, 64, 64, GNT);
    } else {
        go(k3_f64_kernel<128, 64>, 128, 64, GNT);
    }
    NGW_HIP(hipGetLastError());
    return NGW_OK;
}

int operator_f64(ngw_context* ctx, const OperatorArgs& a)
{
    const int nmu = ctx->n_intp, nv = ctx->nval, B = a.nvec;
    if (B <= 0) return NGW_OK;
    if (B == 1) return operator_f64_one(ctx, a);
    const int S = k1_slots(nv);
    NGW_TRY(ctx->tpart.ensure(sizeof(double) * ((size_t)S + 1) * B * nmu));
    NGW_TRY(ctx->ubuf.ensure(sizeof(double) * (size_t)B * nmu));
    double* tpart = ctx->tpart.as<double>();
    double* t = tpart + (size_t)S * B * nmu;
    double* u = ctx->ubuf.as<double>();
    const double* sx = a.tda ? nullptr : ctx->sqrtr.as<double>();
    bool pair = false;
    NGW_TRY(launch_k1(ctx, a.x, a.ldx, sx, B, tpart, t, &pair));
    {
        ProfScope ps(ctx, KC_K2);
        if (pair) NGW_TRY(launch_k2(ctx, SlotPairB{tpart, (long)nmu, B}, B, u));
        else NGW_TRY(launch_k2(ctx, ColMajorB{t, (long)nmu, B}, B, u));
    }
    {
        ProfScope ps(ctx, KC_K3);
        NGW_TRY(launch_k3(ctx, u, B, a.epilogue(ctx)));
    }
    return NGW_OK;
}

// P vectors: v0(:, b) = s o C^T (M c_{m_b n_b})   (s = 1 for TDA),
// SIGMA/calculate_sigma_lanczos_BLOCK.F90z:286-358.
int pvectors_f64(ngw_context* ctx, const int* d_mband, const int* d_nband, int nvec, int tda,
                 double* d_p, long ldp_out)
{
    const int nmu = ctx->n_intp;
    NGW_TRY(ctx->ubuf.ensure(sizeof(double) * (size_t)nvec * nmu));
    double* u = ctx->ubuf.as<double>();
    ProfScope ps(ctx, KC_PVEC);
    NGW_TRY(launch_k2(ctx, PairB{ctx->psi.as<double>(), ctx->ld_psi, d_mband, d_nband, nvec}, nvec, u));
    OperatorEpilogue ep{};
    ep.out = d_p;
    ep.ldo = ldp_out;
    ep.s = tda ? nullptr : ctx->sqrtr.as<double>();
    ep.beta = 1.0;
    ep.alpha = 1.0;
    return launch_k3(ctx, u, nvec, ep);
}

}  // namespace ngw
