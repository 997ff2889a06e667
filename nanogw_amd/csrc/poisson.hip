// ISDF Coulomb kernel M = (ntrans/h^3) zeta^T V zeta on the device.
//
// V zeta_mu is the isolated-system Poisson solve of NanoGW's Zpoisson
// (shared/fft_module.F90z:122-177): put the column into the FFT box at the
// integer grid coordinates, R2C FFT, multiply by the truncated Coulomb kernel
// of Zcreate_coul_0D (:628-691), C2R FFT, pick the grid points and scale by
// 1/N.  Columns are processed in batches, by dense real transforms of the
// eight parity classes on the matrix cores (below), or, for boxes too large
// for those, by one hand-written scatter kernel, one batched hipFFT D2Z, one
// kernel-multiply kernel, one batched Z2D and one gather kernel.  V zeta is kept for a group of batches (all columns when
// they fit in 16 GiB) and M(:, group) = zeta^T (V zeta_group) is one FP64
// MFMA GEMM per group (isdf_parallel_sym_UltraLowMem.F90:865-867): a GEMM
// per FFT batch (33 columns at 158^3) would give too few tiles to fill the
// GPU.

#include <hipfft/hipfft.h>

#include <algorithm>
#include <cmath>
#include <cstdlib>
#include <cstring>
#include <vector>

#include "ngw_kernels.h"

namespace ngw {

#define NGW_FFT(call)                                                                        \
    do {                                                                                     \
        hipfftResult r_ = (call);                                                            \
        if (r_ != HIPFFT_SUCCESS)                                                            \
            return ::ngw::fail(NGW_ERR_HIP, std::string(#call " -> hipfft error ") + std::to_string((int)r_)); \
    } while (0)

// Box offset of each grid point (x fastest), periodic wrap of the centred
// coordinates as in Zpoisson's fft_box%Zbox(-n/2:n/2-1, ...) layout.
__global__ void box_offsets_kernel(const int* grid, int ngrid, int n1, int n2, int n3, long* off)
{
    int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= ngrid) return;
    int x = grid[3 * i], y = grid[3 * i + 1], z = grid[3 * i + 2];
    x = ((x % n1) + n1) % n1;
    y = ((y % n2) + n2) % n2;
    z = ((z % n3) + n3) % n3;
    off[i] = ((long)z * n2 + y) * n1 + x;
}

// box[b][off[i]] = zeta(i, col0 + b); the rest of the box is zero.
__global__ void scatter_kernel(const double* zeta, long ldz, int ngrid, const long* off, long boxsz,
                               double* box, int nb)
{
    const int b = blockIdx.y;
    const double* zc = zeta + (long)b * ldz;
    double* bx = box + (long)b * boxsz;
    for (int i = blockIdx.x * blockDim.x + threadIdx.x; i < ngrid; i += gridDim.x * blockDim.x)
        bx[off[i]] = zc[i];
}

// V(G) box multiply: fbox[b][g] *= vcoul[g]
__global__ void kernel_multiply(double2* fbox, const double* vcoul, long csz, int nb)
{
    const long total = csz * nb;
    for (long t = blockIdx.x * (long)blockDim.x + threadIdx.x; t < total; t += (long)gridDim.x * blockDim.x) {
        const double v = vcoul[t % csz];
        double2 f = fbox[t];
        f.x *= v;
        f.y *= v;
        fbox[t] = f;
    }
}

// vz(i, b) = box[b][off[i]] * scale
__global__ void gather_kernel(const double* box, long boxsz, const long* off, int ngrid, double scale,
                              double* vz, long ldv)
{
    const int b = blockIdx.y;
    const double* bx = box + (long)b * boxsz;
    double* vc = vz + (long)b * ldv;
    for (int i = blockIdx.x * blockDim.x + threadIdx.x; i < ngrid; i += gridDim.x * blockDim.x)
        vc[i] = bx[off[i]] * scale;
}

// v(G) = 8 pi (1 - cos(|G| R_c)) / |G|^2,  v(0) = 8 pi R_c^2 / 2   (trunc > 0)
//      = 8 pi / |G|^2, v(0) = 0                                     (trunc <= 0)
// at G_i = 2 pi j_i / (n_i h).
__device__ double coulomb_v(int n1, int n2, int n3, int j1, int j2, int j3, double h, double trunc)
{
    const double pi = 3.1415926535897932384626433832795;
    double g1 = 2.0 * pi / (n1 * h) * j1, g2 = 2.0 * pi / (n2 * h) * j2, g3 = 2.0 * pi / (n3 * h) * j3;
    double ekin = g1 * g1 + g2 * g2 + g3 * g3;
    const double qzero = 1.0e-6;
    double v;
    if (trunc > 0.0)
        v = (ekin < qzero * qzero) ? trunc * trunc / 2.0 : (1.0 - cos(trunc * sqrt(ekin))) / ekin;
    else
        v = (ekin < qzero * qzero) ? 0.0 : 1.0 / ekin;
    return 8.0 * pi * v;
}

// v(G) on the R2C half box.
__global__ void coulomb_kernel(int n1, int n2, int n3, double h, double trunc, double* vcoul)
{
    const int h1 = n1 / 2 + 1;
    const long csz = (long)h1 * n2 * n3;
    for (long t = blockIdx.x * (long)blockDim.x + threadIdx.x; t < csz; t += (long)gridDim.x * blockDim.x) {
        int i1 = (int)(t % h1);
        int i2 = (int)((t / h1) % n2);
        int i3 = (int)(t / ((long)h1 * n2));
        vcoul[t] = coulomb_v(n1, n2, n3, i1, i2 < n2 / 2 ? i2 : i2 - n2, i3 < n3 / 2 ? i3 : i3 - n3, h, trunc);
    }
}

// ---------------------------------------------------------------- parity transforms
// The Poisson solve of a density confined to |x| <= m about the box centre (a
// sphere in the isolated-system box of four radii: m = n/4), as real
// transforms.  v(G) is even in each G_i, so along each axis the even part
// z(a) + z(-a) and the odd part z(a) - z(-a), a = 0..m, never mix: with
// h = n/2 + 1 frequencies
//   F_e(j) = sum_a z_e(a) cos(2 pi j a / n),  F_o(j) with sin,
//   out_e(a) = (1/n) sum_j w_j v F_e(j) cos(2 pi j a / n),  w = 1, 2, .., 2, 1,
//   out(+-a) = out_e(a) +- out_o(a),
// and in 3-D each of the eight parity classes goes through three small dense
// matrices, the kernel, and their transposes: 14 m^4 multiply-adds each way
// and class at h = 2 m, against a complex FFT of the (4 m)^3 box, 63/64 of
// which is empty on input and unused on output.  All products are FP64 MFMA;
// an MFMA result (row l/16 + 4 r, column l % 16 in register r) is the B
// operand of the next product's k step r as it stands, so the chain of two
// axes stays in registers.
//   pt_forward  fold one pair of planes z = +-az, transform x and y
//   pt_kernel   transform z, multiply, transform z back (in place)
//   pt_inverse  transform y and x back, unfold to the grid points
// The intermediate is 8 (m + 1) h x 16 HT doubles per column (6.9 MB at 114^3).
// Measured on 2000 columns of a 114^3 box (97,000 points): 24 ms against
// 270 ms of batched hipFFT D2Z / Z2D (Bluestein transforms for 114 = 2 3 19).
// Every matrix is padded with zeros to the kernels' 16 MT positions by 16 HT
// frequencies, so no product needs a bound.
struct PtAxis {
    int n, m, h;             // box, extent, frequencies
    const double* fwd[2];    // [16 MT][16 HT] cos / sin
    const double* inv[2];    // [16 HT][16 MT]
};
struct PtPlan {
    PtAxis x, y, z;
    int pitch;               // LDS row pitch of a plane
    long npair;              // y.h * 16 HT
    const int* map;          // grid index of (z, y, x) of the support cube, -1 where there is none
    const double* vw;        // [16 HT][npair] v(G) w / N, zero padded
};

typedef double pf64x4 __attribute__((ext_vector_type(4)));

__device__ __forceinline__ int pt_source(const PtPlan& p, int z, int y, int x)
{
    return p.map[((long)(z + p.z.m) * (2 * p.y.m + 1) + (y + p.y.m)) * (2 * p.x.m + 1) + (x + p.x.m)];
}

template <int MT, int HT>
__global__ __launch_bounds__(512) void pt_forward_kernel(PtPlan p, const double* zeta, long ldz, double* b)
{
    extern __shared__ double plane[];  // [class][ay][pitch]
    const int az = blockIdx.x;
    const double* zc = zeta + (long)blockIdx.y * ldz;
    double* bc = b + (long)blockIdx.y * 8 * (p.z.m + 1) * p.npair;
    const int ny = p.y.m + 1, nx = p.x.m + 1, psz = ny * p.pitch;
    for (int e = threadIdx.x; e < psz; e += 512) {
        const int ay = e / p.pitch, ax = e - ay * p.pitch;
        double s[8];
#pragma unroll
        for (int k = 0; k < 8; ++k) {
            const bool skip = ax >= nx || ((k & 1) && ax == 0) || ((k & 2) && ay == 0) || ((k & 4) && az == 0);
            const int i = skip ? -1 : pt_source(p, k & 4 ? -az : az, k & 2 ? -ay : ay, k & 1 ? -ax : ax);
            s[k] = i >= 0 ? zc[i] : 0.0;
        }
#pragma unroll
        for (int bit = 1; bit < 8; bit <<= 1)
#pragma unroll
            for (int k = 0; k < 8; ++k)
                if (!(k & bit)) {
                    const double u = s[k], v = s[k | bit];
                    s[k] = u + v;
                    s[k | bit] = u - v;
                }
#pragma unroll
        for (int k = 0; k < 8; ++k) plane[k * psz + e] = s[k];
    }
    __syncthreads();
    const int lane = threadIdx.x & 63, c = threadIdx.x >> 6, r16 = lane & 15, k4 = lane >> 4;
    const double* pl = plane + c * psz;
    const double* tx = p.x.fwd[c & 1] + r16;
    const double* ty = p.y.fwd[(c >> 1) & 1] + r16;
    double* out = bc + ((long)c * (p.z.m + 1) + az) * p.npair;
    constexpr int HP = 16 * HT;
    const int kx = (nx + 3) / 4;
#pragma unroll 1
    for (int j1 = 0; j1 < HP; j1 += 16) {
        pf64x4 t1[MT];
#pragma unroll
        for (int i = 0; i < MT; ++i) t1[i] = pf64x4{0.0, 0.0, 0.0, 0.0};
#pragma unroll 4
        for (int k = 0; k < kx; ++k) {
            const double w = tx[(4 * k + k4) * HP + j1];
#pragma unroll
            for (int i = 0; i < MT; ++i)
                t1[i] = __builtin_amdgcn_mfma_f64_16x16x4f64(pl[min(16 * i + r16, ny - 1) * p.pitch + 4 * k + k4], w,
                                                             t1[i], 0, 0, 0);
        }
        pf64x4 t2[HT];
#pragma unroll
        for (int j = 0; j < HT; ++j) t2[j] = pf64x4{0.0, 0.0, 0.0, 0.0};
#pragma unroll
        for (int k = 0; k < 4 * MT; ++k)
#pragma unroll
            for (int j = 0; j < HT; ++j)
                t2[j] = __builtin_amdgcn_mfma_f64_16x16x4f64(ty[(4 * k + k4) * HP + 16 * j], t1[k / 4][k % 4], t2[j], 0,
                                                             0, 0);
#pragma unroll
        for (int j = 0; j < HT; ++j)
#pragma unroll
            for (int r = 0; r < 4; ++r) {
                const int j2 = 16 * j + 4 * r + k4;
                if (j2 < p.y.h) out[j2 * HP + j1 + r16] = t2[j][r];
            }
    }
}

// One wave: 16 (j2, j1) pairs of one column, its eight classes one after the
// other with the pairs' v in registers.  The cos and sin tables serve both
// directions from LDS (row pitch 16 HT + 4 doubles: the backward product reads
// them transposed without bank conflicts); through L1, which they fill, the
// kernel took 550 us per 77 columns of the 114^3 box, now 410.
template <int MT, int HT>
__global__ __launch_bounds__(512) void pt_kernel_kernel(PtPlan p, double* b)
{
    constexpr int HP = 16 * HT, AP = 16 * MT, TP = HP + 4;
    __shared__ double tab[2][AP][TP];
    for (int e = threadIdx.x; e < 2 * AP * HP; e += 512) {
        const int par = e / (AP * HP), r = e - par * AP * HP;
        tab[par][r / HP][r % HP] = p.z.fwd[par][r];
    }
    __syncthreads();
    const int lane = threadIdx.x & 63, r16 = lane & 15, k4 = lane >> 4;
    const long pair = (blockIdx.x * 8L + (threadIdx.x >> 6)) * 16 + r16;
    if (pair - r16 >= p.npair) return;
    const int nz = p.z.m + 1;
    double* bc = b + (long)blockIdx.y * 8 * nz * p.npair + pair;
    double v[HT][4];
#pragma unroll
    for (int j = 0; j < HT; ++j)
#pragma unroll
        for (int r = 0; r < 4; ++r) v[j][r] = p.vw[(16 * j + 4 * r + k4) * p.npair + pair];
#pragma unroll 1
    for (int c = 0; c < 8; ++c) {
        double* x = bc + (long)c * nz * p.npair;
        const double* tf = &tab[c >> 2][k4][r16];
        const double* ti = &tab[c >> 2][r16][k4];
        double xv[4 * MT];
#pragma unroll
        for (int k = 0; k < 4 * MT; ++k) xv[k] = x[min(4 * k + k4, nz - 1) * p.npair];  // past the end: times zero
        pf64x4 f[HT];
#pragma unroll
        for (int j = 0; j < HT; ++j) f[j] = pf64x4{0.0, 0.0, 0.0, 0.0};
#pragma unroll
        for (int k = 0; k < 4 * MT; ++k)
#pragma unroll
            for (int j = 0; j < HT; ++j)
                f[j] = __builtin_amdgcn_mfma_f64_16x16x4f64(tf[4 * k * TP + 16 * j], xv[k], f[j], 0, 0, 0);
        pf64x4 o[MT];
#pragma unroll
        for (int i = 0; i < MT; ++i) o[i] = pf64x4{0.0, 0.0, 0.0, 0.0};
#pragma unroll
        for (int j = 0; j < HT; ++j)
#pragma unroll
            for (int r = 0; r < 4; ++r) {
                const double g = f[j][r] * v[j][r];
#pragma unroll
                for (int i = 0; i < MT; ++i)
                    o[i] = __builtin_amdgcn_mfma_f64_16x16x4f64(ti[16 * i * TP + 16 * j + 4 * r], g, o[i], 0, 0, 0);
            }
#pragma unroll
        for (int i = 0; i < MT; ++i)
#pragma unroll
            for (int r = 0; r < 4; ++r) {
                const int a = 16 * i + 4 * r + k4;
                if (a < nz) x[a * p.npair] = o[i][r];
            }
    }
}

template <int MT, int HT>
__global__ __launch_bounds__(512) void pt_inverse_kernel(PtPlan p, const double* b, double* vz, long ldv)
{
    extern __shared__ double plane[];  // [class][ay][pitch]
    const int az = blockIdx.x;
    const double* bc = b + (long)blockIdx.y * 8 * (p.z.m + 1) * p.npair;
    const int ny = p.y.m + 1, nx = p.x.m + 1, psz = ny * p.pitch;
    const int lane = threadIdx.x & 63, c = threadIdx.x >> 6, r16 = lane & 15, k4 = lane >> 4;
    double* pl = plane + c * psz;
    const double* tx = p.x.inv[c & 1] + r16;
    const double* ty = p.y.inv[(c >> 1) & 1] + r16;
    const double* in = bc + ((long)c * (p.z.m + 1) + az) * p.npair + r16;
    constexpr int HP = 16 * HT, AP = 16 * MT;
    const int k2 = (p.y.h + 3) / 4;
#pragma unroll 1
    for (int a0 = 0; a0 < ny; a0 += 16) {
        // U(j1, ay) = sum_j2 in(j2, j1) inv_y(j2, ay)
        pf64x4 u[HT];
#pragma unroll
        for (int j = 0; j < HT; ++j) u[j] = pf64x4{0.0, 0.0, 0.0, 0.0};
#pragma unroll 4
        for (int k = 0; k < k2; ++k) {
            const double w = ty[(4 * k + k4) * AP + a0];
            const double* row = in + min(4 * k + k4, p.y.h - 1) * HP;
#pragma unroll
            for (int j = 0; j < HT; ++j) u[j] = __builtin_amdgcn_mfma_f64_16x16x4f64(row[16 * j], w, u[j], 0, 0, 0);
        }
        // out(ax, ay) = sum_j1 inv_x(j1, ax) U(j1, ay)
        pf64x4 o[MT];
#pragma unroll
        for (int i = 0; i < MT; ++i) o[i] = pf64x4{0.0, 0.0, 0.0, 0.0};
#pragma unroll
        for (int j = 0; j < HT; ++j)
#pragma unroll
            for (int r = 0; r < 4; ++r)
#pragma unroll
                for (int i = 0; i < MT; ++i)
                    o[i] = __builtin_amdgcn_mfma_f64_16x16x4f64(tx[(16 * j + 4 * r + k4) * AP + 16 * i], u[j][r], o[i],
                                                                0, 0, 0);
        const int ay = a0 + r16;
#pragma unroll
        for (int i = 0; i < MT; ++i)
#pragma unroll
            for (int r = 0; r < 4; ++r) {
                const int ax = 16 * i + 4 * r + k4;
                if (ay < ny && ax < nx) pl[ay * p.pitch + ax] = o[i][r];
            }
    }
    __syncthreads();
    double* vc = vz + (long)blockIdx.y * ldv;
    for (int e = threadIdx.x; e < ny * nx; e += 512) {
        const int ay = e / nx, ax = e - ay * nx;
        double s[8];
#pragma unroll
        for (int k = 0; k < 8; ++k) s[k] = plane[k * psz + ay * p.pitch + ax];
#pragma unroll
        for (int bit = 1; bit < 8; bit <<= 1)
#pragma unroll
            for (int k = 0; k < 8; ++k)
                if (!(k & bit)) {
                    const double u = s[k], v = s[k | bit];
                    s[k] = u + v;
                    s[k | bit] = u - v;
                }
#pragma unroll
        for (int k = 0; k < 8; ++k) {
            if (((k & 1) && ax == 0) || ((k & 2) && ay == 0) || ((k & 4) && az == 0)) continue;
            const int i = pt_source(p, k & 4 ? -az : az, k & 2 ? -ay : ay, k & 1 ? -ax : ax);
            if (i >= 0) vc[i] = s[k];
        }
    }
}

// vw(j3, (j2, j1)) = v(G) w1 w2 w3 / N with v as in coulomb_kernel; zero in
// the padding.
__global__ void pt_weights_kernel(PtPlan p, int hp, double h, double trunc, double* vw)
{
    const long total = hp * p.npair;
    for (long t = blockIdx.x * (long)blockDim.x + threadIdx.x; t < total; t += (long)gridDim.x * blockDim.x) {
        const int j3 = (int)(t / p.npair);
        const long r = t - j3 * p.npair;
        const int j2 = (int)(r / hp), j1 = (int)(r - (long)j2 * hp);
        double o = 0.0;
        if (j1 < p.x.h && j3 < p.z.h) {
            const double w = (j1 == 0 || 2 * j1 == p.x.n ? 1.0 : 2.0) * (j2 == 0 || 2 * j2 == p.y.n ? 1.0 : 2.0) *
                             (j3 == 0 || 2 * j3 == p.z.n ? 1.0 : 2.0);
            o = coulomb_v(p.x.n, p.y.n, p.z.n, j1, j2, j3, h, trunc) * w /
                ((double)p.x.n * (double)p.y.n * (double)p.z.n);
        }
        vw[t] = o;
    }
}

}  // namespace ngw

using namespace ngw;

namespace {

// V zeta of `cols` columns at a time into vz(ngrid, .), by one of the two
// Poisson solvers.
struct PoissonFft {
    DevBuf box, fbox, vc, off, grid;
    hipfftHandle pf = 0, pb = 0;
    long boxsz = 0, csz = 0;
    int cols = 0;
    ~PoissonFft()
    {
        if (pf) hipfftDestroy(pf);
        if (pb) hipfftDestroy(pb);
    }
    int init(hipStream_t s, int ngrid, int n_intp, const int* hgrid, const int* nfft, double h, double trunc)
    {
        const int n1 = nfft[0], n2 = nfft[1], n3 = nfft[2];
        boxsz = (long)n1 * n2 * n3;
        csz = (long)(n1 / 2 + 1) * n2 * n3;
        // batch so that the real and complex boxes stay near 2 GiB
        cols = (int)std::max(1L, std::min((long)n_intp, (2L << 30) / (8 * boxsz + 16 * csz)));
        cols = std::min(cols, 256);
        NGW_TRY(box.ensure(sizeof(double) * (size_t)boxsz * cols));
        NGW_TRY(fbox.ensure(sizeof(double) * 2 * (size_t)csz * cols));
        NGW_TRY(vc.ensure(sizeof(double) * (size_t)csz));
        NGW_TRY(off.ensure(sizeof(long) * (size_t)ngrid));
        NGW_TRY(grid.ensure(sizeof(int) * 3 * (size_t)ngrid));
        NGW_HIP(hipMemcpyAsync(grid.ptr, hgrid, sizeof(int) * 3 * (size_t)ngrid, hipMemcpyHostToDevice, s));
        hipLaunchKernelGGL(box_offsets_kernel, dim3((ngrid + 255) / 256), dim3(256), 0, s, grid.as<int>(), ngrid, n1,
                           n2, n3, off.as<long>());
        NGW_HIP(hipGetLastError());
        hipLaunchKernelGGL(coulomb_kernel, dim3(1024), dim3(256), 0, s, n1, n2, n3, h, trunc, vc.as<double>());
        NGW_HIP(hipGetLastError());
        int dims[3] = {n3, n2, n1};
        int cdims[3] = {n3, n2, n1 / 2 + 1};
        NGW_FFT(hipfftPlanMany(&pf, 3, dims, dims, 1, (int)boxsz, cdims, 1, (int)csz, HIPFFT_D2Z, cols));
        NGW_FFT(hipfftPlanMany(&pb, 3, dims, cdims, 1, (int)csz, dims, 1, (int)boxsz, HIPFFT_Z2D, cols));
        NGW_FFT(hipfftSetStream(pf, s));
        NGW_FFT(hipfftSetStream(pb, s));
        return NGW_OK;
    }
    int run(hipStream_t s, const double* z, long ldz, int ngrid, int cb, double* vz)
    {
        NGW_HIP(hipMemsetAsync(box.ptr, 0, sizeof(double) * (size_t)boxsz * cols, s));
        hipLaunchKernelGGL(scatter_kernel, dim3(std::min((ngrid + 255) / 256, 1024), cb), dim3(256), 0, s, z, ldz,
                           ngrid, off.as<long>(), boxsz, box.as<double>(), cb);
        NGW_HIP(hipGetLastError());
        NGW_FFT(hipfftExecD2Z(pf, box.as<double>(), reinterpret_cast<hipfftDoubleComplex*>(fbox.ptr)));
        hipLaunchKernelGGL(kernel_multiply, dim3(4096), dim3(256), 0, s, fbox.as<double2>(), vc.as<double>(), csz,
                           cols);
        NGW_HIP(hipGetLastError());
        NGW_FFT(hipfftExecZ2D(pb, reinterpret_cast<hipfftDoubleComplex*>(fbox.ptr), box.as<double>()));
        hipLaunchKernelGGL(gather_kernel, dim3(std::min((ngrid + 255) / 256, 1024), cb), dim3(256), 0, s,
                           box.as<double>(), boxsz, off.as<long>(), ngrid, 1.0 / (double)boxsz, vz, (long)ngrid);
        NGW_HIP(hipGetLastError());
        return NGW_OK;
    }
};

// Launchers of the three kernels at one padding.
struct PtKernels {
    int mt, ht;
    void (*fwd)(PtPlan, const double*, long, double*);
    void (*mid)(PtPlan, double*);
    void (*inv)(PtPlan, const double*, double*, long);
};
#define PT_K(MT, HT) {MT, HT, pt_forward_kernel<MT, HT>, pt_kernel_kernel<MT, HT>, pt_inverse_kernel<MT, HT>}
// m + 1 in sixteens by n/2 + 1 in sixteens; the isolated-system box (n = 4 m)
// needs (1, 2), (2, 4), (3, 5), (3, 6)
constexpr PtKernels PT_KERNELS[] = {PT_K(1, 2), PT_K(1, 4), PT_K(2, 3), PT_K(2, 4), PT_K(3, 5),
                                    PT_K(3, 6), PT_K(2, 8), PT_K(3, 8)};

struct PoissonParity {
    DevBuf map, tab, vw, b;
    PtPlan p{};
    const PtKernels* k = nullptr;
    int cols = 0;
    size_t lds = 0;
    // Whether the support and the box fit the kernels and no two grid points
    // coincide (the map holds one); fills the map and the sizes.
    bool fits(int ngrid, const int* grid, const int* nfft, std::vector<int>& hmap)
    {
        int m[3] = {0, 0, 0};
        for (int i = 0; i < ngrid; ++i)
            for (int d = 0; d < 3; ++d) m[d] = std::max(m[d], std::abs(grid[3 * i + d]));
        PtAxis* ax[3] = {&p.x, &p.y, &p.z};
        int mt = 0, ht = 0;
        for (int d = 0; d < 3; ++d) {
            PtAxis& a = *ax[d];
            a.n = nfft[d];
            a.m = m[d];
            a.h = nfft[d] / 2 + 1;
            mt = std::max(mt, (a.m + 16) / 16);
            ht = std::max(ht, (a.h + 15) / 16);
        }
        for (const PtKernels& e : PT_KERNELS)
            if (!k && e.mt >= mt && e.ht >= ht) k = &e;
        if (!k) return false;
        p.pitch = 4 * (((p.x.m + 4) / 4) | 1);  // 4 x odd: 16 rows x 4 columns of a plane hit every bank once
        p.npair = (long)p.y.h * 16 * k->ht;
        lds = sizeof(double) * 8 * (size_t)(p.y.m + 1) * p.pitch;
        hmap.assign((size_t)(2 * m[0] + 1) * (2 * m[1] + 1) * (2 * m[2] + 1), -1);
        for (int i = 0; i < ngrid; ++i) {
            int& e = hmap[((size_t)(grid[3 * i + 2] + m[2]) * (2 * m[1] + 1) + grid[3 * i + 1] + m[1]) *
                              (2 * m[0] + 1) + grid[3 * i] + m[0]];
            if (e >= 0) return false;
            e = i;
        }
        return true;
    }
    int init(hipStream_t s, int n_intp, const std::vector<int>& hmap, double h, double trunc)
    {
        PtAxis* ax[3] = {&p.x, &p.y, &p.z};
        const int hp = 16 * k->ht, ap = 16 * k->mt;
        const size_t sz = (size_t)hp * ap;
        std::vector<double> ht(12 * sz, 0.0);
        NGW_TRY(tab.ensure(sizeof(double) * ht.size()));
        for (int d = 0; d < 3; ++d) {
            PtAxis& a = *ax[d];
            for (int par = 0; par < 2; ++par) {
                double* f = &ht[(4 * d + par) * sz];
                double* v = &ht[(4 * d + 2 + par) * sz];
                for (int j = 0; j < a.h; ++j)
                    for (int x = 0; x <= a.m; ++x) {
                        const long r = (long)j * x % a.n;
                        const long double t = 2.0L * 3.14159265358979323846264338327950288L * r / a.n;
                        double c = (double)(par ? std::sin(t) : std::cos(t));
                        if (4 * r % a.n == 0) {  // exact at the quarter turns
                            const long quarter = 4 * r / a.n;
                            c = par ? (quarter == 1) - (quarter == 3) : (quarter == 0) - (quarter == 2);
                        }
                        f[(size_t)x * hp + j] = c;
                        v[(size_t)j * ap + x] = c;
                    }
                a.fwd[par] = tab.as<double>() + (4 * d + par) * sz;
                a.inv[par] = tab.as<double>() + (4 * d + 2 + par) * sz;
            }
        }
        const size_t percol = sizeof(double) * 8 * (size_t)(p.z.m + 1) * p.npair;
        // Columns of a batch: all where 512 MiB hold their intermediate, else
        // whole rounds of the forward and inverse grids (one workgroup per plane
        // and column) over the 256 CUs.  With two and more planes per CU the
        // intermediate then stays within the 256 MiB cache between the kernels;
        // with one, few rounds fit that, and 512 MiB are faster.  114^3 (512
        // resident planes, 29 a column), 2000 columns: 34.2 - 34.7 ms for batches
        // of 34 and 35, 37.6 for 36, 36.0 for the 77 of 512 MiB; 158^3 (256 planes,
        // 40 a column), 600 columns: 29.8 ms for 12, 28.5 for 32; a 60^3 box's 400
        // columns 1.36 ms in one batch, 1.39 in two.
        const int percu = std::max<int>(1, std::min<int>(4, (int)((160 << 10) / lds)));  // 512 threads each
        const size_t most = (size_t)(512L << 20) / percol, fit = percu > 1 ? most / 2 : most;
        const size_t planes = (size_t)p.z.m + 1, round = NCU * (size_t)percu;
        const size_t whole = fit * planes / round * round / planes;
        cols = (int)std::max<size_t>(1, std::min<size_t>({(size_t)n_intp, 4096, (size_t)n_intp <= most ? most : whole ? whole : fit}));
        NGW_TRY(map.ensure(sizeof(int) * hmap.size()));
        NGW_TRY(vw.ensure(sizeof(double) * (size_t)hp * p.npair));
        NGW_TRY(b.ensure(percol * cols));
        NGW_HIP(hipMemcpyAsync(tab.ptr, ht.data(), sizeof(double) * ht.size(), hipMemcpyHostToDevice, s));
        NGW_HIP(hipMemcpyAsync(map.ptr, hmap.data(), sizeof(int) * hmap.size(), hipMemcpyHostToDevice, s));
        NGW_HIP(hipStreamSynchronize(s));
        p.map = map.as<int>();
        p.vw = vw.as<double>();
        hipLaunchKernelGGL(pt_weights_kernel, dim3(1024), dim3(256), 0, s, p, hp, h, trunc, vw.as<double>());
        NGW_HIP(hipGetLastError());
        // (the attribute belongs to the kernel, not to this call: always the
        // largest plane, so that no thread lowers another's limit)
        constexpr int LDS_MAX = 160 * 1024;
        NGW_HIP(hipFuncSetAttribute(reinterpret_cast<const void*>(k->fwd), hipFuncAttributeMaxDynamicSharedMemorySize,
                                    LDS_MAX));
        NGW_HIP(hipFuncSetAttribute(reinterpret_cast<const void*>(k->inv), hipFuncAttributeMaxDynamicSharedMemorySize,
                                    LDS_MAX));
        return NGW_OK;
    }
    int run(hipStream_t s, const double* z, long ldz, int ngrid, int cb, double* vz)
    {
        hipLaunchKernelGGL(k->fwd, dim3(p.z.m + 1, cb), dim3(512), lds, s, p, z, ldz, b.as<double>());
        hipLaunchKernelGGL(k->mid, dim3((unsigned)((p.npair + 127) / 128), cb), dim3(512), 0, s, p, b.as<double>());
        hipLaunchKernelGGL(k->inv, dim3(p.z.m + 1, cb), dim3(512), lds, s, p, b.as<double>(), vz, (long)ngrid);
        NGW_HIP(hipGetLastError());
        return NGW_OK;
    }
};

}  // namespace

// zeta_dev: zeta is a device array (ld_zeta) used in place; otherwise a host
// array copied to the device.  M is returned to the host.
static int coulomb_impl(ngw_context* ctx, int ngrid, int n_intp, const double* zeta, long ld_zeta, bool zeta_dev,
                        const int* grid, const int* nfft, double h, double trunc, double ntrans, double* mmtrx,
                        int ld_m)
{
    if (!ctx) return fail(NGW_ERR_ARG, "null context");
    if (ngrid <= 0 || n_intp <= 0 || ld_zeta < ngrid || ld_m < n_intp || !zeta || !grid || !nfft || !mmtrx)
        return fail(NGW_ERR_ARG, "bad sizes or null arrays");
    const int n1 = nfft[0], n2 = nfft[1], n3 = nfft[2];
    if (n1 <= 1 || n2 <= 1 || n3 <= 1 || (n1 % 2) || (n2 % 2) || (n3 % 2))
        return fail(NGW_ERR_ARG, "nfft must be even and > 1");
    if (!(h > 0.0)) return fail(NGW_ERR_ARG, "h must be positive");
    for (int i = 0; i < ngrid; ++i)
        for (int k = 0; k < 3; ++k) {
            int n = nfft[k], g = grid[3 * i + k];
            if (g < -n / 2 || g >= n / 2) return fail(NGW_ERR_ARG, "grid coordinate outside the FFT box");
        }
    NGW_HIP(hipSetDevice(ctx->device));
    hipStream_t s = ctx->stream;
    // the dense parity transforms where the support and the box are small
    // enough for them (isolated systems up to a box of about 186), the FFT
    // for the rest
    PoissonParity par;
    PoissonFft fft;
    std::vector<int> hmap;
    const bool parity = par.fits(ngrid, grid, nfft, hmap);
    if (parity) NGW_TRY(par.init(s, n_intp, hmap, h, trunc));
    else NGW_TRY(fft.init(s, ngrid, n_intp, grid, nfft, h, trunc));
    const int nb = parity ? par.cols : fft.cols;
    // columns of V zeta kept for one GEMM: a multiple of nb, up to 16 GiB
    const long vz_cols = std::max(1L, (16L << 30) / (8L * ngrid));
    const int grp = (int)std::min((long)n_intp, std::max((long)nb, vz_cols / nb * nb));
    DevBuf dzeta, dvz, dm, dpart;
    if (!zeta_dev) NGW_TRY(dzeta.ensure(sizeof(double) * (size_t)ngrid * n_intp));
    NGW_TRY(dvz.ensure(sizeof(double) * (size_t)ngrid * grp));
    NGW_TRY(dm.ensure(sizeof(double) * (size_t)n_intp * n_intp));
    const double* zd = zeta;  // device zeta and its leading dimension
    long ldz = ld_zeta;
    if (!zeta_dev) {
        if (ld_zeta == ngrid) {
            NGW_HIP(hipMemcpyAsync(dzeta.ptr, zeta, sizeof(double) * (size_t)ngrid * n_intp, hipMemcpyHostToDevice,
                                   s));
        } else {
            NGW_HIP(hipMemcpy2DAsync(dzeta.ptr, sizeof(double) * ngrid, zeta, sizeof(double) * ld_zeta,
                                     sizeof(double) * ngrid, n_intp, hipMemcpyHostToDevice, s));
        }
        zd = dzeta.as<double>();
        ldz = ngrid;
    }
    const double norm = ntrans / (h * h * h);
    int g0 = 0;  // first column of the current group
    for (int c0 = 0; c0 < n_intp; c0 += nb) {
        const int cb = std::min(nb, n_intp - c0);
        double* vz = dvz.as<double>() + (size_t)(c0 - g0) * ngrid;
        const double* z = zd + (size_t)c0 * ldz;
        if (parity) NGW_TRY(par.run(s, z, ldz, ngrid, cb, vz));
        else NGW_TRY(fft.run(s, z, ldz, ngrid, cb, vz));
        const int gend = c0 + cb;
        if (gend - g0 == grp || gend == n_intp) {
            // M(:, g0:gend) = norm * zeta^T vz; all columns at once: the
            // upper triangle, mirrored
            if (g0 == 0 && gend == n_intp)
                NGW_TRY(gemm_f64_tn_sym(s, n_intp, ngrid, norm, zd, ldz, dvz.as<double>(), ngrid, dm.as<double>(),
                                        n_intp, dpart));
            else
                NGW_TRY(gemm_f64_tn(s, n_intp, gend - g0, ngrid, norm, zd, ldz, dvz.as<double>(), ngrid,
                                    dm.as<double>() + (size_t)g0 * n_intp, n_intp));
            g0 = gend;
        }
    }
    // (one linear copy: a 2-D copy to pageable memory goes row by row)
    std::vector<double> hm(ld_m == n_intp ? 0 : (size_t)n_intp * n_intp);
    NGW_HIP(hipMemcpyAsync(ld_m == n_intp ? mmtrx : hm.data(), dm.ptr, sizeof(double) * (size_t)n_intp * n_intp,
                           hipMemcpyDeviceToHost, s));
    NGW_HIP(hipStreamSynchronize(s));
    if (ld_m != n_intp)
        for (int j = 0; j < n_intp; ++j)
            std::memcpy(mmtrx + (size_t)j * ld_m, &hm[(size_t)j * n_intp], sizeof(double) * n_intp);
    return NGW_OK;
}

extern "C" int ngw_isdf_coulomb_kernel(ngw_context* ctx, int ngrid, int n_intp, const double* zeta,
                                       long ld_zeta, const int* grid, const int* nfft, double h,
                                       double trunc, double ntrans, double* mmtrx, int ld_m)
{
    return coulomb_impl(ctx, ngrid, n_intp, zeta, ld_zeta, false, grid, nfft, h, trunc, ntrans, mmtrx, ld_m);
}

extern "C" int ngw_isdf_coulomb_kernel_dev(ngw_context* ctx, int ngrid, int n_intp, const double* d_zeta,
                                           long ld_zeta, const int* grid, const int* nfft, double h,
                                           double trunc, double ntrans, double* mmtrx, int ld_m)
{
    return coulomb_impl(ctx, ngrid, n_intp, d_zeta, ld_zeta, true, grid, nfft, h, trunc, ntrans, mmtrx, ld_m);
}
