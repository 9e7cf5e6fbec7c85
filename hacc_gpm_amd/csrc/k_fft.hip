// k_fft.hip — 3-D FFT passes for one transform length N (compiled once per N with
// -DHGPM_FFT_N=<N>, and once more for N = 1024 with -DHGPM_FFT_PLAN_ALT: the same
// passes over the radix order 8 x 8 x 16 instead of 16 x 8 x 8, fft_ops_1024_alt).  Replaces the cuFFT C2C/Z2Z calls of src/fft_tools/cuda/ffts.cu
// (plans :60-130, forward :244-294, inverse :397-445: unnormalised, in place,
// x-major ng^3 grids) and fuses the spectral solve of src/pm_solver/solver.cpp:145-170
// into the transform passes.
//
// Passes (grid index (x*N + y)*PZ + z, z contiguous; PZ = N for full complex grids; half
// spectra add HPAD elements after each x plane):
//   rows  : 1-D transforms along z; a workgroup loads RC whole rows (coalesced).
//   cols  : 1-D transforms along y (stride PZ) or x (stride N*PZ); a workgroup loads CC
//           adjacent z values of N rows (CC*8 contiguous bytes per row).
// The solve of a step runs on half spectra: the density and the potential are real, so
// only k_z = 0..N/2 is kept (row pitch HZ = N/2 + 16, the padding columns held at zero)
// and every pass after the first touches half the data:
//   r2c   : pairs of real rows a, b as one complex transform of a + i b, split into
//           the half spectra of a and b;
//   x_psi : forward x transform, phi^ = (g/2) rho^ (half the Green's function), inverse
//           x transform, in place;
//   c2r   : phi rows in pairs as one complex transform of the Hermitian extension of
//           phi^_a + i phi^_b.
// The initial conditions use the same passes: the noise is real and so is each
// displacement component (k_x_ic, k_y_ic, k_rows_c2r_real<KZ>).
// The reference's gradient, F_d^ = -i sin(k_d) G rho^ with G = -g, is F_d^ = i sin(k_d)
// psi^ with psi = IFFT(g rho^): the central difference F_d[n] = (psi[n + e_d] -
// psi[n - e_d]) / 2 = phi[n + e_d] - phi[n - e_d] of the real field phi = psi / 2, which
// the force gather forms (one inverse transform, not three).
#include "fft.h"
#include "internal.h"

using hgpm::IcSpectrum;

#ifndef HGPM_FFT_N
#error "compile with -DHGPM_FFT_N=<transform length>"
#endif

namespace {
constexpr int N = HGPM_FFT_N;
constexpr int NT = 256;   // rows passes
constexpr int HZ = N / 2 + 16; // half-spectrum row pitch: k_z = 0..N/2 + zero padding
static_assert(HZ % 16 == 0 && HZ <= N, "half-spectrum pitch");
// Half-spectrum x-plane pitch: N rows of HZ plus HPAD unused elements.  Without the pad
// the plane stride N HZ 8 bytes is a multiple of 2^17 (at N = 1024), so the N rows an
// x-pass tile reads (one per x) share their low address bits; the pad shifts each
// plane by one 128-byte line.  (N = 32 has no room for it: there HZ = N.)
constexpr int HPAD = N >= 64 ? 16 : 0;
constexpr size_t NPH = (size_t)N * HZ + HPAD;
static_assert(HPAD % 16 == 0 && (size_t)N * NPH <= (size_t)N * N * N, "half spectra fit a full grid");
// element offset of half-spectrum row r = (box N + x) N + y
__device__ __forceinline__ size_t hrow(size_t r) { return (r / N) * NPH + (r % N) * HZ; }

// rows per row tile / columns per column tile (FP32, FP64)
constexpr int rc32() { return N >= 768 ? 4 : (N >= 384 ? 8 : (N >= 192 ? 16 : (N >= 96 ? 32 : 64))); }
constexpr int cc32() { return N >= 768 ? 8 : (N >= 192 ? 16 : 32); }
constexpr int rc64() { return rc32() > 1 ? rc32() / 2 : 1; }
constexpr int cc64() { return N >= 768 ? 4 : (N >= 192 ? 8 : 16); }

// ------------------------------------------------------------- rows ----
template <typename V, int RC, int DIR>
__global__ __launch_bounds__(NT) void k_rows_c2c(V* __restrict d, const V* __restrict tw) {
    __shared__ V lds[lds_elems<N, RC>()];
    const size_t row0 = (size_t)blockIdx.x * RC;
    fft_tile<V, N, RC, NT, DIR, false, true>(
        [&](int, int, int n, int c) { return d[(row0 + c) * N + n]; },
        [&](int, int, int n, int c, V v) { d[(row0 + c) * N + n] = v; }, lds, tw);
}

// ------------------------------------------------------------- cols ----
// axis 1 (y): tile = (x, z-chunk), element (n=y, c) at x N^2 + n N + z0 + c
// axis 0 (x): tile = (y, z-chunk), element (n=x, c) at n N^2 + y N + z0 + c
// First element of column tile t: outer runs over (box, x) for the y pass and (box, y) for
// the x pass (a batch holds several grids of the same shape back to back).  NP: x-plane
// pitch (N pz for full grids, NPH for half spectra).
template <int CC> __device__ __forceinline__ size_t col_base(int t, int axis, int pz, size_t NP) {
    const int nzc = pz / CC, outer = t / nzc, zc = t % nzc;
    return axis == 1 ? (size_t)outer * NP + (size_t)zc * CC
                     : (size_t)(outer / N) * N * NP + (size_t)(outer % N) * pz + (size_t)zc * CC;
}
template <typename V, int CC, int NTC, int DIR>
__global__ __launch_bounds__(NTC) void k_cols_c2c(V* __restrict d, const V* __restrict tw, int axis, int pz,
                                                  size_t plane) {
    __shared__ V lds[lds_elems<N, CC>()];
    // adjacent z-chunks of one row share 128-byte lines: keep them on one XCD's L2
    const size_t base = col_base<CC>((int)xcd_remap(blockIdx.x, gridDim.x), axis, pz, plane);
    const size_t stride = axis == 1 ? (size_t)pz : plane;
    fft_tile<V, N, CC, NTC, DIR, false, false>(
        [&](int, int, int n, int c) { return d[base + n * stride + c]; },
        [&](int, int, int n, int c, V v) { d[base + n * stride + c] = v; }, lds, tw);
}

// FP64 force of one component, from the density's modes: the reference multiplies rho^ by
// the component's factor in a pass of its own and takes the real part of the inverse
// transform in another (kspace_solve_gradient, getRealGrid); here the z pass multiplies as
// it loads (rho^ stays for the next component; w may be rho^ itself for the last one: a
// workgroup has loaded its rows before it stores them) and the x pass stores the real
// part only, that of the last component (JOIN) all three a cell, as the gather reads them:
// from three grids a particle's corners are on three times the lines, and kicks of
// dispersed particles took twice as long (192^3 1.16 against 0.54 ms).  All three passes
// are bound by memory.
template <int RC>
__global__ __launch_bounds__(NT) void k_rows_force(const double2* rho, double2* w, const double2* __restrict tw,
                                                   const double2* __restrict modes, int dim) {
    __shared__ double2 lds[lds_elems<N, RC>()];
    const size_t row0 = (size_t)blockIdx.x * RC;
    fft_tile<double2, N, RC, NT, +1, false, true>(
        [&](int, int, int n, int c) {
            const size_t row = row0 + c;
            const double2 q = rho[row * N + n], X = modes[row / N], Y = modes[row % N], Z = modes[n];
            // Green's function; the mean's mode (where it is infinite) is dropped
            const double G = (0.5 / ((double)N * N * N)) / (X.x + Y.x + Z.x - 3.0);
            const double f = row + n == 0 ? 0.0 : -(dim == 0 ? X.y : dim == 1 ? Y.y : Z.y) * G;
            return row + n == 0 ? make_double2(0.0, 0.0) : make_double2(-f * q.y, f * q.x);
        },
        [&](int, int, int n, int c, double2 v) { w[(row0 + c) * N + n] = v; }, lds, tw);
}
template <int CC, int NTC, bool JOIN>
__global__ __launch_bounds__(NTC) void k_cols_force(const double2* __restrict w, double* __restrict out,
                                                    const double* __restrict fx, const double* __restrict fy,
                                                    const double2* __restrict tw) {
    __shared__ double2 lds[lds_elems<N, CC>()];
    const size_t plane = (size_t)N * N;
    const size_t base = col_base<CC>((int)xcd_remap(blockIdx.x, gridDim.x), 0, N, plane);
    fft_tile<double2, N, CC, NTC, +1, false, false>(
        [&](int, int, int n, int c) { return w[base + n * plane + c]; },
        [&](int, int, int n, int c, double2 v) {
            const size_t at = base + n * plane + c;
            if constexpr (JOIN) {
                out[3 * at] = fx[at];
                out[3 * at + 1] = fy[at];
                out[3 * at + 2] = v.x;
            } else {
                out[at] = v.x;
            }
        },
        lds, tw);
}

// Streaming: where one workgroup fills a CU (large tiles: its LDS or its registers leave no
// room for a second one) its loads, transforms and stores would follow one another.  The
// x pass of the solve, which transforms twice per tile, is then one workgroup per CU that
// walks the tiles of its XCD's contiguous range (neighbouring z-chunks at the same time
// on one L2); the next tile is loaded into registers while the current one is
// transformed, and the stores drain behind it.
constexpr int NCU = 256, NXCD = 8;
struct TileWalk {
    int t, end;
    static constexpr int step = NCU / NXCD;
    __device__ __forceinline__ TileWalk(int nt) {
        const int x = blockIdx.x % NXCD, per = nt / NXCD, rem = nt % NXCD;
        const int first = x * per + min(x, rem);
        t = first + (int)blockIdx.x / NXCD;
        end = first + per + (x < rem ? 1 : 0);
    }
};
// Opaque copy for one tile: the indices derived from it are the same for every tile, and
// kept across them they would take the registers of the next tile's elements.  (The
// twiddles lie in LDS: a global load issued behind the next tile's would wait for it, the
// vector memory counter being in order.)
__device__ __forceinline__ int opaque(int tid) {
    asm volatile("" : "+v"(tid));
    return tid;
}
// A thread's elements of a tile's stage 0.
template <int CC, int NTC> struct TileRegs {
    static constexpr int R = Plan<N>::R(0);
    typedef StageShape<N, CC, NTC, R> SS;
    static_assert(SS::TOT % NTC == 0, "whole tiles");
    float2 x[SS::NB][R];
};
// Element j + r * NBF of column c of the tile at d (uniform): a scalar base per r and one
// 32-bit byte offset per lane (j * stride * 8 < 2^32 for every plan), so an address costs
// one register.
__device__ __forceinline__ float2* tile_at(float2* d, int nbf, int r, int j, int c, size_t stride) {
    return (float2*)((char*)(d + (size_t)(r * nbf) * stride) + ((unsigned)j * (unsigned)stride + (unsigned)c) * 8u);
}
template <int CC, int NTC>
__device__ __forceinline__ void load_tile(TileRegs<CC, NTC>& X, float2* d, size_t stride, int tid) {
    typedef TileRegs<CC, NTC> T;
#pragma unroll
    for (int b = 0; b < T::SS::NB; b++) {
        const int w = tid + b * NTC, c = w % CC, j = w / CC;
#pragma unroll
        for (int r = 0; r < T::R; r++) X.x[b][r] = *tile_at(d, T::SS::NBF, r, j, c, stride);
    }
}
// The first tile's loads are waited for before the loop, so that inside it the wait for a
// tile counts the stores issued behind its loads and leaves them in flight.
__device__ __forceinline__ void wait_loads() { __builtin_amdgcn_s_waitcnt(0x0F70); } // vmcnt(0)
// ------------------------------------------------- half-spectrum solve ----
// Forward z transform of the int64 density, mean removed in FP64 (the k = 0 normalisation)
// before the FP32 rounding, for RC real rows: rows 2c and 2c+1 form the complex column c = a + i b, transformed
// once; A[k] = (C[k] + conj C[N-k]) / 2 and B[k] = (C[k] - conj C[N-k]) / 2i give the
// half spectra, k = 0..N/2, written with pitch HZ (padding written as zero).
// rhof: see fwd_z_r2c (the owner pass wrote the same FP32 values when no tile was deferred).
// REAL: the rows are those of the FP32 grid rhof (initial conditions' noise).
template <int RC, bool REAL, int NTX>
__global__ __launch_bounds__(NTX) void k_rows_r2c_density(const long long* __restrict rho,
                                                         const float* __restrict rhof,
                                                         const unsigned long long* __restrict ctl,
                                                         const unsigned long long* __restrict mass,
                                                         float2* __restrict out, const float2* __restrict tw) {
    constexpr int PC = RC / 2;
    __shared__ float2 lds[lds_elems<N, PC>()];
    float2* spec = lds; // the last stage has read all its inputs before the first output
    const size_t row0 = (size_t)blockIdx.x * RC;
    const bool f32 = REAL || (rhof != nullptr && ctl[1] == 0ull);
    // mass of this row's box (a batch holds several boxes of the same shape), from its
    // partial sums
    double mean = 0.0;
    if (!f32) {
        unsigned long long t = mass[row0 / ((size_t)N * N) * HGPM_DEP_MASS + (threadIdx.x & 63)];
        for (int off = 32; off > 0; off >>= 1) t += __shfl_xor(t, off, 64);
        mean = (double)(long long)t / ((double)N * N * N);
    }
    fft_tile<float2, N, PC, NTX, -1, false, true>(
        [&](int, int, int n, int c) {
            if (f32) return make_float2(rhof[(row0 + 2 * c) * N + n], rhof[(row0 + 2 * c + 1) * N + n]);
            const double qa = (double)rho[(row0 + 2 * c) * N + n];
            const double qb = (double)rho[(row0 + 2 * c + 1) * N + n];
            return make_float2((float)((qa - mean) * (1.0 / 16777216.0)), (float)((qb - mean) * (1.0 / 16777216.0)));
        },
        [&](int, int, int n, int c, float2 v) { spec[lds_slot<N, PC, true>(n, c)] = v; }, lds, tw);
    __syncthreads();
    for (int i = threadIdx.x; i < PC * HZ; i += NTX) {
        const int c = i / HZ, k = i % HZ;
        float2 a = make_float2(0.0f, 0.0f), b = make_float2(0.0f, 0.0f);
        if (k <= N / 2) {
            const float2 x = spec[lds_slot<N, PC, true>(k, c)];
            const float2 y = spec[lds_slot<N, PC, true>(k == 0 ? 0 : N - k, c)];
            a = make_float2(0.5f * (x.x + y.x), 0.5f * (x.y - y.y));
            b = make_float2(0.5f * (x.y + y.y), 0.5f * (y.x - x.x));
        }
        out[hrow(row0 + 2 * c) + k] = a;
        out[hrow(row0 + 2 * c + 1) + k] = b;
    }
}

// Half-spectrum x pass of the potential.  In: h1 = rho^ after the z and y forward
// passes.  Forward x transform, phi^ = (g/2) rho^ with g = (0.25/N^3)/sum_d sin^2(k_d/2),
// g(0) = 0 (gcoef = 0.125/N^3), inverse x transform, written back to h1.  The reference's Green's function
// G = (0.5/N^3)/(sum_d cos k_d - 3) = -g and gradient -i sin(k_d) (kspace_solve_gradient,
// src/pm_solver/cuda/kspace_solver.cu:55-90; calcGreens, src/pm_solver/cuda/calcGreens.hpp:11-26;
// get_gradient, src/pm_solver/kernels.hpp) give F_d^ = i sin(k_d) psi^ = 2 i sin(k_d) phi^,
// formed in real space by the gather.  hs[m] = sin^2(pi m/N).
template <int CC, int NTC>
__global__ __launch_bounds__(NTC) void k_x_psi(float2* __restrict h1, const float2* __restrict twf,
                                               const float2* __restrict twr, const float* __restrict hs,
                                               float gcoef) {
    __shared__ float2 lds[lds_elems<N, CC>()];
    const int tile = (int)xcd_remap(blockIdx.x, gridDim.x);
    const int outer = tile / (HZ / CC), zc = tile % (HZ / CC); // outer = (box, y)
    const int y = outer % N;
    const size_t NP = NPH;
    const size_t base = (size_t)(outer / N) * N * NP + (size_t)y * HZ + (size_t)zc * CC;
    typedef LastShape<N, CC, NTC> LS;
    typedef StageShape<N, CC, NTC, LS::R> SS;
    float2 R[LS::NB][LS::R];
    const int c0 = threadIdx.x % CC;
    const int z = zc * CC + c0; // < HZ <= N
    const float hyz = hs[y] + hs[z];
    fft_tile<float2, N, CC, NTC, -1, false, false>(
        [&](int, int, int n, int c) { return h1[base + n * NP + c]; },
        [&](int b, int r, int, int, float2 v) { R[b][r] = v; }, lds, twf);
    fft_tile<float2, N, CC, NTC, +1, true, false>(
        [&](int b, int r, int n, int) {
            const float ssum = hs[n] + hyz;
            // v_rcp_f32 (1 ulp) for the quotient: ssum >= sin^2(pi / N) is far from the
            // denormal range, and the solve is checked to a tolerance, not bit for bit
            const float g = (n | y | z) == 0 ? 0.0f : gcoef * __builtin_amdgcn_rcpf(ssum);
            return make_float2(g * R[b][r].x, g * R[b][r].y);
        },
        [&](int, int, int n, int c, float2 v) { h1[base + n * NP + c] = v; }, lds, twr);
}

// ------------------------------------------------- initial conditions ----
// k of mode index n along one axis (the reference's get_kmode in FP32: n, or n - N from
// N/2 on, times dk = 2 pi / rl), and -i k v.
__device__ __forceinline__ float mode_k(int n, double dk) { return (float)((double)(n > N / 2 - 1 ? n - N : n) * dk); }
__device__ __forceinline__ float2 minus_ik(float2 v, float k) { return make_float2(v.y * k, -v.x * k); }

// sqrt(P) amp / k^2 of a mode, in FP64: the .ipk log-log interpolation
// (do_pk_interpolation, src/initial_conditions/cuda/interpolation_initializer.cu:3-30,
// on k from the FP32 sum of squares), ScaleAmplitudes and the 1 / k^2 of
// transformDensityField: one logarithm and one exponential on the bin's line, or
// written out where a bin has none (an empty bin; a table with so many bins below the
// grid's largest k that the lines found no room).
__device__ __forceinline__ double ic_factor(float kx, float ky, float kz, const IcSpectrum& sp) {
#pragma clang fp contract(off)
    float s = kx * kx;
    s = s + ky * ky;
    s = s + kz * kz;
    if (s == 0.0f) return 0.0;
    const double k = sqrt((double)s), ls = log((double)s);
    if (sp.line) {
        const double2 ab = sp.line[min((int)(k / sp.k_delta), sp.nline - 1)];
        if (ab.x == ab.x) return exp(ab.x + ab.y * ls);
    }
    const int l = min((int)(k / sp.k_delta), sp.nbins - 2);
    double y = log(sp.tab[1]);
    if (l > 0) {
        const double x1 = log(sp.k_delta * (double)l), x2 = log(sp.k_delta * (double)(l + 1)), y1 = log(sp.tab[l]);
        y = y1 + (log(sp.tab[l + 1]) - y1) / (x2 - x1) * (0.5 * ls - x1);
    }
    return exp(0.5 * y - ls) * sp.amp;
}

// x pass of the initial conditions.  In: h1 = the noise after the z and y forward passes.
// Forward x transform, phi^ = amplitude * sqrt(P) / (delta k^2), and two inverse x
// transforms: of -i k_x phi^ (to h1: the x displacement's modes) and of phi^ itself (to
// h2: -i k_y and -i k_z act on the other axes, so the y and z displacements share this
// transform and take their factors in the passes along y and z).  The reference
// transforms complex grids and keeps the real part; a mode at N/2 of axis d is its own
// mirror there with the same sign of k_d, so its -i k_d part is imaginary: dropped here.
// Bound by the FP64 work of the factor (a logarithm, an exponential, a root and a
// quotient per mode) and its three transforms: 8.3 ms at 1024^3 for 13 GB.  8 columns x
// 1024 threads there: with 16 columns the modes kept between the transforms do not fit
// the registers (85 spilled, 9.5 ms).  The whole of the initial conditions at 1024^3 went
// from 131 ms on complex grids (four transforms, three displacement passes, the spectrum
// with five logarithms per mode) to 38 ms.
template <int CC, int NTC>
__global__ __launch_bounds__(NTC) void k_x_ic(float2* __restrict h1, float2* __restrict h2,
                                              const float2* __restrict twf, const float2* __restrict twr,
                                              IcSpectrum sp) {
    __shared__ float2 lds[lds_elems<N, CC>()];
    const int tile = (int)xcd_remap(blockIdx.x, gridDim.x);
    const int y = tile / (HZ / CC), zc = tile % (HZ / CC);
    const size_t base = (size_t)y * HZ + (size_t)zc * CC;
    typedef LastShape<N, CC, NTC> LS;
    float2 R[LS::NB][LS::R];
    const float ky = mode_k(y, sp.dk), kz = mode_k(zc * CC + (int)threadIdx.x % CC, sp.dk);
    fft_tile<float2, N, CC, NTC, -1, false, false>(
        [&](int, int, int n, int c) { return h1[base + n * NPH + c]; },
        [&](int b, int r, int n, int, float2 v) {
            const double f = ic_factor(mode_k(n, sp.dk), ky, kz, sp);
            R[b][r] = make_float2((float)((double)v.x * f), (float)((double)v.y * f));
        },
        lds, twf);
    fft_tile<float2, N, CC, NTC, +1, true, false>(
        [&](int b, int r, int n, int) { return minus_ik(R[b][r], n == N / 2 ? 0.0f : mode_k(n, sp.dk)); },
        [&](int, int, int n, int c, float2 v) { h1[base + n * NPH + c] = v; }, lds, twr);
    fft_tile<float2, N, CC, NTC, +1, true, false>(
        [&](int b, int r, int, int) { return R[b][r]; },
        [&](int, int, int n, int c, float2 v) { h2[base + n * NPH + c] = v; }, lds, twr);
}

// y pass of the initial conditions: inverse y transforms of phi^ (h2, in place: the z
// displacement's, its factor taken by the z pass) and of -i k_y phi^ (to h3), from one
// read of the tile (3.5 ms at 1024^3, two passes over memory and one more of writing).
template <int CC, int NTC>
__global__ __launch_bounds__(NTC) void k_y_ic(float2* __restrict h2, float2* __restrict h3,
                                              const float2* __restrict tw, double dk) {
    __shared__ float2 lds[lds_elems<N, CC>()];
    const int tile = (int)xcd_remap(blockIdx.x, gridDim.x);
    const size_t base = (size_t)(tile / (HZ / CC)) * NPH + (size_t)(tile % (HZ / CC)) * CC;
    typedef StageShape<N, CC, NTC, Plan<N>::R(0)> SS;
    float2 X[SS::NB][Plan<N>::R(0)];
    fft_tile<float2, N, CC, NTC, +1, false, false>(
        [&](int b, int r, int n, int c) { return X[b][r] = h2[base + (size_t)n * HZ + c]; },
        [&](int, int, int n, int c, float2 v) { h2[base + (size_t)n * HZ + c] = v; }, lds, tw);
    fft_tile<float2, N, CC, NTC, +1, false, false>(
        [&](int b, int r, int n, int) { return minus_ik(X[b][r], n == N / 2 ? 0.0f : mode_k(n, dk)); },
        [&](int, int, int n, int c, float2 v) { h3[base + (size_t)n * HZ + c] = v; }, lds, tw);
}

// k_x_psi as a streaming pass: the next tile is loaded once the inverse transform's first
// stage has freed the spectrum's registers.  Measured in a run, against the same shape (16
// columns x 1024 threads) with a workgroup per tile: 2.5-2.6 -> 2.25 ms at 1024, 1.12-1.15
// -> 0.86-0.90 at 768; at 512, where a tile takes half the LDS, 0.267 -> 0.25-0.31 with one or two
// workgroups per CU, so the plain form stays there.  The y passes, one transform per tile,
// gained nothing from the same treatment (1.80 / 1.67 -> 1.93 / 1.72 ms at 1024).
constexpr bool STREAM_X = N > 512;
template <int CC, int NTC>
__global__ __launch_bounds__(NTC) void k_x_psi_stream(float2* h1, const float2* __restrict twf,
                                                      const float2* __restrict twr, const float* __restrict hs,
                                                      float gcoef, int nt) {
    __shared__ float2 lds[lds_elems<N, CC>()];
    __shared__ float2 tf[tw_packed<N, false>()], tr[tw_packed<N, true>()];
    __shared__ float hl[N];
    TileWalk w(nt);
    if (w.t >= w.end) return;
    tw_pack<float2, N, false, NTC>(tf, twf);
    tw_pack<float2, N, true, NTC>(tr, twr);
    for (int i = threadIdx.x; i < N; i += NTC) hl[i] = hs[i];
    __syncthreads();
    typedef LastShape<N, CC, NTC> LS;
    constexpr int NBL = N / RevPlan<N>::R(RevPlan<N>::S - 1);
    TileRegs<CC, NTC> X;
    float2 R[LS::NB][LS::R];
    float2* at = h1 + col_base<CC>(w.t, 0, HZ, NPH);
    load_tile(X, at, NPH, (int)threadIdx.x);
    wait_loads();
    for (;;) {
        const int tid = opaque((int)threadIdx.x);
        const int tn = w.t + TileWalk::step < w.end ? w.t + TileWalk::step : w.t;
        float2* next = h1 + col_base<CC>(tn, 0, HZ, NPH);
        const int y = w.t / (HZ / CC) % N, z = w.t % (HZ / CC) * CC + tid % CC;
        const float hyz = hl[y] + hl[z];
        fft_tile<float2, N, CC, NTC, -1, false, false, true>(
            [&](int b, int r, int, int) { return X.x[b][r]; },
            [&](int b, int r, int, int, float2 v) { R[b][r] = v; }, lds, tf, Nothing(), tid);
        const int tid2 = opaque((int)threadIdx.x);
        fft_tile<float2, N, CC, NTC, +1, true, false, true>(
            [&](int b, int r, int n, int) {
                float q = hl[n] + hyz; // see k_x_psi
                asm volatile("" : "+v"(q)); // (no branch around the quotient)
                const float gq = gcoef * __builtin_amdgcn_rcpf(q);
                const float g = (n | y | z) == 0 ? 0.0f : gq;
                return make_float2(g * R[b][r].x, g * R[b][r].y);
            },
            [&](int, int r, int n, int c, float2 v) { *tile_at(at, NBL, r, n - r * NBL, c, NPH) = v; }, lds, tr,
            [&] { load_tile(X, next, NPH, tid2); }, tid2);
        if (tn == w.t) return;
        w.t = tn;
        at = next;
    }
}

// Element n of the Hermitian extension of a half-spectrum row: h[n] for n <= N/2,
// conj h[N-n] above.
__device__ __forceinline__ float2 herm(const float2* __restrict row, int n) {
    if (n <= N / 2) return row[n];
    const float2 v = row[N - n];
    return make_float2(v.x, -v.y);
}

// Inverse z transform of real rows from their half spectra, rows in pairs: the
// Hermitian extensions of a and b as one complex transform of a + i b, whose real and
// imaginary parts are the rows.  When the last stage's butterflies per row are fewer
// than a wave (N / R_last < 64: lengths with a radix-3 or radix-16 first stage, and
// N <= 256) its direct stores would scatter each wave over several rows in short
// pieces; the rows then go through LDS and are stored whole, lane after lane.
// KZ: the half spectra are multiplied by -i k_z first (k_z = m dk; zero at N/2, see k_x_ic).
template <int RC, bool KZ, int NTX>
__global__ __launch_bounds__(NTX) void k_rows_c2r_real(const float2* __restrict hz, float* __restrict out,
                                                      const float2* __restrict tw, double dk) {
    constexpr int PC = RC / 2;
    constexpr bool STAGED = N / Plan<N>::R(Plan<N>::S - 1) < 64;
    __shared__ float2 lds[lds_elems<N, PC>()];
    const size_t row0 = (size_t)blockIdx.x * RC;
    auto ld = [&](int, int, int n, int c) {
        float2 a = herm(hz + hrow(row0 + 2 * c), n), b = herm(hz + hrow(row0 + 2 * c + 1), n);
        if constexpr (KZ) {
            // conj(-i k v) = -i (-k) conj(v): the mirrored half takes its own (negative) k_z
            const float k = n == N / 2 ? 0.0f : mode_k(n, dk);
            a = minus_ik(a, k);
            b = minus_ik(b, k);
        }
        return make_float2(a.x - b.y, a.y + b.x);
    };
    if constexpr (!STAGED) {
        fft_tile<float2, N, PC, NTX, +1, false, true>(
            ld,
            [&](int, int, int n, int c, float2 v) {
                out[(row0 + 2 * c) * N + n] = v.x;
                out[(row0 + 2 * c + 1) * N + n] = v.y;
            },
            lds, tw);
    } else {
        // the last stage has read all its inputs before the first output
        fft_tile<float2, N, PC, NTX, +1, false, true>(
            ld, [&](int, int, int n, int c, float2 v) { lds[lds_slot<N, PC, true>(n, c)] = v; }, lds, tw);
        __syncthreads();
        for (int i = threadIdx.x; i < PC * N; i += NTX) {
            const int c = i / N, n = i - c * N;
            const float2 v = lds[lds_slot<N, PC, true>(n, c)];
            out[(row0 + 2 * c) * N + n] = v.x;
            out[(row0 + 2 * c + 1) * N + n] = v.y;
        }
    }
}

// --------------------------------------------------------- launchers ----
// Column-pass / x-pass variants (columns per tile, threads per workgroup):
//   0: (4, 256)  1: (4, 512)  2: (8, 512)  3: (16, 512)  4: (8, 1024)  5: (16, 1024)
// chosen per transform length by the autotuner (default VDEF).  More threads per tile
// means fewer elements, and registers, per thread: the fused x pass holds the
// spectrum between its two transforms.
template <typename V, int CC, int NTC>
void cols_launch(V* d, int axis, int dir, const V* tw, int pz, size_t plane, hipStream_t s, int nbox = 1) {
    unsigned nb = (unsigned)((size_t)nbox * N * (pz / CC));
    if (dir < 0) k_cols_c2c<V, CC, NTC, -1><<<nb, NTC, 0, s>>>(d, tw, axis, pz, plane);
    else k_cols_c2c<V, CC, NTC, +1><<<nb, NTC, 0, s>>>(d, tw, axis, pz, plane);
}
template <typename V, int RC>
void rows_launch(V* d, int dir, const V* tw, hipStream_t s) {
    unsigned nb = (unsigned)((size_t)N * N / RC);
    if (dir < 0) k_rows_c2c<V, RC, -1><<<nb, NT, 0, s>>>(d, tw);
    else k_rows_c2c<V, RC, +1><<<nb, NT, 0, s>>>(d, tw);
}
constexpr int NVAR = 6;
constexpr int cc_of(int v) { return v <= 1 ? 4 : (v == 2 || v == 4 ? 8 : 16); }
constexpr int nt_of(int v) { return v == 0 ? 256 : (v <= 3 ? 512 : 1024); }
constexpr bool variant_ok(int v) { return cc_of(v) <= N && (N % cc_of(v)) == 0 && (size_t)N * cc_of(v) * 8 <= 140000; }
constexpr unsigned variant_mask() {
    unsigned m = 0;
    for (int v = 0; v < NVAR; v++)
        if (variant_ok(v)) m |= 1u << v;
    return m;
}
// The shape a context starts with (hgpm_autotune may pick another): 16 columns, whole
// 128-byte lines, with 1024 threads from 512 on, where fewer leave too few waves per CU.
// Measured against 8 columns x 512 threads (forward y, inverse y, x pass, us): 256: 30 28 33
// against 37 29 42; 384: 92 75 99 / 118 74 100; 512: 212 216 267 / 228 226 287; 768: 802
// 761 857 / 821 775 1132; 1024: 1795 1669 2243 / 1928 1861 2832.
constexpr int VDEF = N >= 512 ? 5 : 3;
static_assert(variant_ok(VDEF), "default variant");

// Calls f(IntC<v>) for the runtime variant v when it is valid for N, else the default.
template <typename F> void with_variant(int variant, F&& f) {
    bool done = false;
    auto one = [&](auto vc) {
        constexpr int v = decltype(vc)::value;
        if constexpr (variant_ok(v)) {
            if (!done && variant == v) { f(vc); done = true; }
        }
    };
    one(IntC<0>{}); one(IntC<1>{}); one(IntC<2>{}); one(IntC<3>{}); one(IntC<4>{}); one(IntC<5>{});
    if (!done) f(IntC<VDEF>{});
}
void pass_f32(float2* d, int axis, int dir, const float2* tw, int variant, hipStream_t s) {
    if (axis == 2) { rows_launch<float2, rc32()>(d, dir, tw, s); return; }
    with_variant(variant, [&](auto vc) {
        constexpr int v = decltype(vc)::value;
        cols_launch<float2, cc_of(v), nt_of(v)>(d, axis, dir, tw, N, (size_t)N * N, s);
    });
}
void force_f64(const double2* rho, double2* w, double* out, const double* fx, const double* fy, const double2* tw,
               const double2* modes, int dim, hipStream_t s) {
    k_rows_force<rc64()><<<(unsigned)((size_t)N * N / rc64()), NT, 0, s>>>(rho, w, tw, modes, dim);
    cols_launch<double2, cc64(), 512>(w, 1, +1, tw, N, (size_t)N * N, s);
    const unsigned nb = (unsigned)((size_t)N * N / cc64());
    if (fx) k_cols_force<cc64(), 512, true><<<nb, 512, 0, s>>>(w, out, fx, fy, tw);
    else k_cols_force<cc64(), 512, false><<<nb, 512, 0, s>>>(w, out, nullptr, nullptr, tw);
}
// Column pass over nbox half-spectrum grids N x N x HZ.
void pass_half(float2* d, int axis, int dir, const float2* tw, int variant, int nbox, hipStream_t s) {
    with_variant(variant, [&](auto vc) {
        constexpr int v = decltype(vc)::value;
        cols_launch<float2, cc_of(v), nt_of(v)>(d, axis, dir, tw, HZ, NPH, s, nbox);
    });
}
void pass_f64(double2* d, int axis, int dir, const double2* tw, hipStream_t s) {
    if (axis == 2) rows_launch<double2, rc64()>(d, dir, tw, s);
    else cols_launch<double2, cc64(), 512>(d, axis, dir, tw, N, (size_t)N * N, s);
}
// Real rows: eight (four complex columns) to a workgroup of 128 threads, 256 for the
// lengths 384 and 768 (with 128: 384 c2r 115 against 107 us, 768 c2r 980 / 850, r2c 716 /
// 660).  Small workgroups fill the chip where a grid has few rows and give up their place
// sooner where it has many.  Against 8 to 128 rows (16 to 32 KB) and 256 threads, r2c and
// c2r in us: 32: 3.9 3.7 (4.5 4.3), 64: 4.2 4.2 (6.9 6.5), 96: 5.3 5.5 (6.8 8.7), 128: 6.6
// 6.2 (8.2 7.6), 192: 15.4 16.4 (16.7 17.6), 256: 29.1 28.0 (28.1 29.1), 384: 83 107 (83
// 115), 512: 192 246 (192 248), 1024: 1508 1671 (1593 1721).
constexpr int RR = 8, NTR = N % 3 == 0 && N >= 384 ? 256 : 128;
// nbox grids of the same shape back to back (rows of every box in one launch)
void fwd_z_r2c(const long long* rho, const float* rhof, const unsigned long long* ctl,
               const unsigned long long* mass, float2* out, const float2* tw, int nbox, hipStream_t s) {
    unsigned nb = (unsigned)((size_t)nbox * N * N / RR);
    k_rows_r2c_density<RR, false, NTR><<<nb, NTR, 0, s>>>(rho, rhof, ctl, mass, out, tw);
}
void fwd_z_r2c_real(const float* in, float2* out, const float2* tw, hipStream_t s) {
    k_rows_r2c_density<RR, true, NTR><<<(unsigned)((size_t)N * N / RR), NTR, 0, s>>>(nullptr, in, nullptr, nullptr, out, tw);
}
void inv_z_c2r_real(const float2* hz, float* out, const float2* tw, int nbox, hipStream_t s) {
    unsigned nb = (unsigned)((size_t)nbox * N * N / RR);
    k_rows_c2r_real<RR, false, NTR><<<nb, NTR, 0, s>>>(hz, out, tw, 0.0);
}
// The initial conditions' passes, one box: 16 columns (128-byte rows), 1024 threads where
// such a tile leaves one workgroup per CU; the x pass then 8 columns (k_x_ic).
constexpr int NT_IC = N >= 512 ? 1024 : 512;
void ic_x(float2* h1, float2* h2, const float2* twf, const float2* twr, const IcSpectrum& sp, hipStream_t s) {
    constexpr int CC = N >= 512 ? 8 : 16;
    k_x_ic<CC, NT_IC><<<N * (HZ / CC), NT_IC, 0, s>>>(h1, h2, twf, twr, sp);
}
void ic_y(float2* h2, float2* h3, const float2* tw, double dk, hipStream_t s) {
    k_y_ic<16, NT_IC><<<N * (HZ / 16), NT_IC, 0, s>>>(h2, h3, tw, dk);
}
void ic_z(const float2* hz, float* out, const float2* tw, double dk, hipStream_t s) {
    k_rows_c2r_real<RR, true, NTR><<<(unsigned)((size_t)N * N / RR), NTR, 0, s>>>(hz, out, tw, dk);
}
template <int CC, int NTC>
void x_psi_launch(float2* h1, const float2* twf, const float2* twr, const float* hs, int nbox, hipStream_t s) {
    unsigned nb = (unsigned)((size_t)nbox * N * (HZ / CC));
    const float gcoef = (float)(0.125 / ((double)N * N * N)); // g / 2: the stored field is psi / 2
    if constexpr (STREAM_X && NTC == 1024 && CC == 16)
        k_x_psi_stream<CC, NTC><<<NCU, NTC, 0, s>>>(h1, twf, twr, hs, gcoef, (int)nb);
    else k_x_psi<CC, NTC><<<nb, NTC, 0, s>>>(h1, twf, twr, hs, gcoef);
}
void x_psi(float2* h1, const float2* twf, const float2* twr, const float* hs, int variant, int nbox, hipStream_t s) {
    with_variant(variant, [&](auto vc) {
        constexpr int v = decltype(vc)::value;
        x_psi_launch<cc_of(v), nt_of(v)>(h1, twf, twr, hs, nbox, s);
    });
}
void twiddles(double* fwd, double* rev) {
    make_twiddles<N, false>(fwd);
    make_twiddles<N, true>(rev);
}
} // namespace

// The operation table holds host function pointers: host compilation pass only.
#ifndef __HIP_DEVICE_COMPILE__
namespace hgpm {
#define HGPM_CAT2(a, b) a##b
#define HGPM_CAT(a, b) HGPM_CAT2(a, b)
#if defined(HGPM_FFT_PLAN_ALT)
extern const FftOps HGPM_CAT(HGPM_CAT(fft_ops_, HGPM_FFT_N), _alt) = {
#else
extern const FftOps HGPM_CAT(fft_ops_, HGPM_FFT_N) = {
#endif
    N, Plan<N>::S, NVAR, VDEF, variant_mask(), twiddles, pass_f32, pass_f64, force_f64,
    HZ, NPH, pass_half, fwd_z_r2c, x_psi, inv_z_c2r_real, fwd_z_r2c_real, ic_x, ic_y, ic_z,
};
} // namespace hgpm
#endif
