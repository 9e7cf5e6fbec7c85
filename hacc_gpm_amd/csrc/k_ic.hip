// k_ic.hip — Zel'dovich initial conditions on the GPU (serial::GenerateDisplacementIC,
// src/initial_conditions/initializer.cpp:65-166).
//   noise        : one N(0,1) per cell.  cuRAND's curand_normal_double
//                  (src/initial_conditions/cuda/rng_initializer.cu:38-49) is replaced by
//                  Philox4x32-10 (Salmon et al., SC'11) on counter (cell index, 0, 0),
//                  key (seed, 0), and Box-Muller with a log and cos(2 pi u) evaluated by
//                  fixed-order series, so the CPU oracle draws the same bits.
//   scale        : ScaleAmplitudes x sqrt(P(k)) with the .ipk log-log interpolation
//                  (interpolation_initializer.cu:3-41, scale_initializer.cu:3-13).
//   displacement : transformDensityField (transform_density_field_initializer.cu:72-112):
//                  psi_d^ = -i k_d / k^2 * amp / delta.
//   place        : placeParticles (place_particles_initializer.cu:49-65) after the
//                  inverse transform and the 1/np^3 ScaleFFT.
// The FP32 path runs scale and displacement inside its transform passes (k_fft.hip,
// k_x_ic); the kernels here for them are the FP64 plain path's.
#include "common.h"
#include "internal.h"
#include "../../include/hgpm.h"

#include <mutex>

#pragma clang fp contract(off)

namespace {
constexpr int BS = 256;

__device__ __forceinline__ void philox(uint32_t c[4], uint32_t k0, uint32_t k1) {
#pragma unroll
    for (int r = 0; r < 10; r++) {
        uint64_t p0 = (uint64_t)0xD2511F53u * c[0];
        uint64_t p1 = (uint64_t)0xCD9E8D57u * c[2];
        uint32_t n0 = (uint32_t)(p1 >> 32) ^ c[1] ^ k0;
        uint32_t n2 = (uint32_t)(p0 >> 32) ^ c[3] ^ k1;
        c[1] = (uint32_t)p1;
        c[3] = (uint32_t)p0;
        c[0] = n0;
        c[2] = n2;
        k0 += 0x9E3779B9u;
        k1 += 0xBB67AE85u;
    }
}

// log(x), x in (0,1]: x = m 2^e, m in [sqrt(1/2), sqrt(2)], atanh series of (m-1)/(m+1).
__device__ double det_log(double x) {
    int e;
    double m = frexp(x, &e);
    m = m * 2.0;
    e = e - 1;
    if (m > 1.4142135623730951) { m = m * 0.5; e = e + 1; }
    double t = (m - 1.0) / (m + 1.0);
    double s = t * t;
    double p = 1.0 / 23.0;
    for (int k = 10; k >= 0; k--) {
        double ck = 1.0 / (double)(2 * k + 1);
        p = p * s;
        p = p + ck;
    }
    double r = 2.0 * t;
    r = r * p;
    double el = (double)e * 0.6931471805599453;
    return el + r;
}

// cos(2 pi u), u in [0,1): quadrant + Taylor series of cos/sin on [0, pi/2).
__device__ double det_cos2pi(double u) {
    double v = 4.0 * u;
    int q = (int)v;
    double r = v - (double)q;
    double phi = r * 1.5707963267948966;
    double s2 = phi * phi;
    double cc[13], sc[13];
    cc[0] = 1.0; sc[0] = 1.0;
    for (int k = 1; k < 13; k++) {
        cc[k] = cc[k - 1] / (double)((2 * k - 1) * (2 * k));
        sc[k] = sc[k - 1] / (double)((2 * k) * (2 * k + 1));
    }
    double c = cc[12], s = sc[12];
    for (int k = 11; k >= 0; k--) {
        c = c * (-s2);
        c = c + cc[k];
        s = s * (-s2);
        s = s + sc[k];
    }
    s = s * phi;
    switch (q & 3) {
    case 0: return c;
    case 1: return -s;
    case 2: return -c;
    default: return s;
    }
}

__device__ double normal_at(uint32_t seed, uint64_t idx) {
    uint32_t c[4] = {(uint32_t)idx, (uint32_t)(idx >> 32), 0u, 0u};
    philox(c, seed, 0u);
    double u1 = ((double)(c[0] >> 5) * 67108864.0 + (double)(c[1] >> 6)) * (1.0 / 9007199254740992.0);
    double u2 = ((double)(c[2] >> 5) * 67108864.0 + (double)(c[3] >> 6)) * (1.0 / 9007199254740992.0);
    double l = det_log(1.0 - u1);
    double r = sqrt(-2.0 * l);
    return r * det_cos2pi(u2);
}

__global__ void k_noise_f32(float* __restrict g, int64_t n, uint32_t seed) {
    const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (i < n) g[i] = (float)normal_at(seed, (uint64_t)i);
}
__global__ void k_noise_f64(double2* __restrict g, int64_t n, uint32_t seed) {
    const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (i < n) g[i] = make_double2(normal_at(seed, (uint64_t)i), 0.0);
}

// The .ipk table as the FP32 path's x pass interpolates it (IcSpectrum::line): log P is
// linear in log k between bins, so the factor sqrt(P) amp / k^2 of a mode of squared
// wavenumber s is exp(A + B log s) with one (A, B) per bin.
__global__ void k_ic_lines(const double* __restrict in, double2* __restrict line, int n, int nbins, double k_delta,
                           double amp) {
    const int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= n) return;
    const int l = min(i, nbins - 2);
    double m = 0.0, y = log(in[1]); // the first interval is constant
    if (l > 0) {
        const double x1 = log(k_delta * (double)l), y1 = log(in[l]);
        m = (log(in[l + 1]) - y1) / (log(k_delta * (double)(l + 1)) - x1);
        y = y1 - m * x1; // log P = y + m log k
    }
    const double A = 0.5 * y + log(amp), B = 0.25 * m - 1.0;
    // an empty bin (log 0) has no line: NaN sends its modes to the formula itself
    line[i] = isfinite(A) && isfinite(B) ? make_double2(A, B) : make_double2(__builtin_nan(""), 0.0);
}

__device__ __forceinline__ float kmode(int idx, int ng, double d) {
    float l = (float)idx;
    if (idx > ((ng / 2) - 1)) l = (float)(-(ng - idx));
    return (float)((double)l * d);
}

// do_pk_interpolation (interpolation_initializer.cu:3-30) then ScaleAmplitudes.
__global__ void k_scale_f64(double2* __restrict g, int np, const double* __restrict in, int nbins, double k_delta, double rl) {
    int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    int64_t G = (int64_t)np * np * np;
    if (i >= G) return;
    int ix = (int)(i / ((int64_t)np * np)), iy = (int)((i / np) % np), iz = (int)(i % np);
    double y = 0.0;
    if ((ix | iy | iz) != 0) {
        double d = (2 * HGPM_PI) / rl;
        float kx = kmode(ix, np, d), ky = kmode(iy, np, d), kz = kmode(iz, np, d);
        float s = kx * kx;
        s = s + ky * ky;
        s = s + kz * kz;
        double my_k = sqrt((double)s);
        int left = (int)(my_k / k_delta);
        int right = left + 1;
        double sc = ((double)G) / (rl * rl * rl);
        if (left > nbins - 2) left = nbins - 2; // range checked on the host
        if (right > nbins - 1) right = nbins - 1;
        if (left == 0) y = in[right] * sc;
        else {
            double logy1 = log(in[left]);
            double logx1 = log(k_delta * (double)left);
            double logy2 = log(in[right]);
            double logx2 = log(k_delta * (double)right);
            double logx = log(my_k);
            double logy = logy1 + ((logy2 - logy1) / (logx2 - logx1)) * (logx - logx1);
            y = exp(logy) * sc;
        }
    }
    double f = sqrt(y);
    double2 v = g[i];
    v.x *= f;
    v.y *= f;
    g[i] = v;
}

// transformDensityField for one axis.
__global__ void k_disp_f64(const double2* __restrict amp, double2* __restrict out, int np, int dim, double delta,
                           double rl) {
    int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    int64_t G = (int64_t)np * np * np;
    if (i >= G) return;
    int ix = (int)(i / ((int64_t)np * np)), iy = (int)((i / np) % np), iz = (int)(i % np);
    double d = (2 * HGPM_PI) / rl;
    int mx = ix > np / 2 - 1 ? ix - np : ix, my = iy > np / 2 - 1 ? iy - np : iy, mz = iz > np / 2 - 1 ? iz - np : iz;
    double kx = d * mx, ky = d * my, kz = d * mz;
    double k2 = kx * kx + ky * ky + kz * kz;
    double k2mul = k2 == 0 ? 0.0 : 1.0 / k2;
    double mul = (1.0 / delta) * k2mul;
    double2 c = amp[i];
    double cr = c.x * mul, ci = c.y * mul;
    double kd = dim == 0 ? kx : (dim == 1 ? ky : kz);
    out[i] = make_double2(ci * kd, -cr * kd);
}

// placeParticles: x = q ng/np + delta psi (FP64, then fixed point: rint(x 2^22) mod
// ng 2^22), v = velMul psi, the three axes of a particle together: one 12-byte store each
// of position and velocity.  A workgroup places 16 rows of 16 lattice points of one
// Lagrangian tile, so the tile's place is found by scalar divisions and a lane's by its
// bits.  Bound by memory: three 4-byte grids read in 64-byte pieces (neighbouring tiles
// share the 128-byte lines, on one XCD), 24 bytes written per particle: 7.6 ms at 1024^3,
// 5.1 TB/s (36.5 ms one axis at a time from complex grids, with 4-byte stores 12 bytes
// apart; 11.5 ms with 64-bit divisions per lane for the lattice place and the wrap).
static_assert(BS == HGPM_TL * HGPM_TL, "one x plane of a tile per workgroup");
__global__ __launch_bounds__(BS) void k_place_split(const float* __restrict sx, const float* __restrict sy,
                                                    const float* __restrict sz, PosPack* __restrict pos,
                                                    float* __restrict vel, int np, int ng, double delta,
                                                    float vel_mul) {
    const unsigned w = (unsigned)xcd_remap(blockIdx.x, gridDim.x); // tile, x plane of the tile
    const unsigned t = w / HGPM_TL, nt = (unsigned)np / HGPM_TL, tyx = t / nt;
    const unsigned l = threadIdx.x;
    const unsigned q[3] = {tyx / nt * HGPM_TL + w % HGPM_TL, tyx % nt * HGPM_TL + l / HGPM_TL,
                           t % nt * HGPM_TL + l % HGPM_TL};
    const unsigned i = (q[0] * np + q[1]) * np + q[2]; // < 2^30
    const float g[3] = {sx[i], sy[i], sz[i]};
    const double inv = 1.0 / ((double)np * np * np), step = (double)ng / (double)np;
    unsigned X[3];
    float v[3];
#pragma unroll
    for (int d = 0; d < 3; d++) {
        const float s = (float)((double)g[d] * inv);
        X[d] = fx_from_double((double)q[d] * step + delta * (double)s, ng);
        v[d] = vel_mul * s;
    }
    const int64_t j = (int64_t)w * BS + l; // internal (tile) order
    pos[j] = PosPack{X[0], X[1], X[2]};
#pragma unroll
    for (int d = 0; d < 3; d++) vel[3 * j + d] = v[d];
}

// ... FP64, one axis per call
__global__ void k_place_f64(const double2* __restrict sg, double* __restrict pos, double* __restrict vel, int np,
                            int ng, int dim, double delta, double vel_mul) {
    int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    int64_t G = (int64_t)np * np * np;
    if (i >= G) return;
    int q = dim == 0 ? (int)(i / ((int64_t)np * np)) : (dim == 1 ? (int)((i / np) % np) : (int)(i % np));
    double s = sg[i].x / (double)G;
    double x = (double)q * ((double)ng / (double)np) + delta * s;
    x = fmod(x + (double)ng, (double)ng);
    if (x < 0) x += (double)ng;
    if (x >= (double)ng) x -= (double)ng;
    pos[3 * i + dim] = x;
    vel[3 * i + dim] = vel_mul * s;
}

inline unsigned nblk(int64_t n) { return (unsigned)((n + BS - 1) / BS); }
} // namespace

namespace hgpm {
void launch_ic_noise_f32(float* g, int np, uint32_t seed, hipStream_t s) {
    const int64_t n = (int64_t)np * np * np;
    k_noise_f32<<<nblk(n), BS, 0, s>>>(g, n, seed);
}
void launch_ic_noise_f64(double2* g, int np, uint32_t seed, hipStream_t s) {
    const int64_t n = (int64_t)np * np * np;
    k_noise_f64<<<nblk(n), BS, 0, s>>>(g, n, seed);
}
void launch_ic_lines(const double* ipk, int ipk_bins, double k_delta, double amp, double2* line, int n,
                     hipStream_t s) {
    k_ic_lines<<<nblk(n), BS, 0, s>>>(ipk, line, n, ipk_bins, k_delta, amp);
}
void launch_ic_scale_f64(double2* g, int np, const double* ipk, int ipk_bins, double k_delta, double rl,
                         hipStream_t s) {
    k_scale_f64<<<nblk((int64_t)np * np * np), BS, 0, s>>>(g, np, ipk, ipk_bins, k_delta, rl);
}
void launch_ic_displacement_f64(const double2* amp, double2* out, int np, int dim, double delta, double rl,
                                hipStream_t s) {
    k_disp_f64<<<nblk((int64_t)np * np * np), BS, 0, s>>>(amp, out, np, dim, delta, rl);
}
void launch_ic_place_split(const float* sx, const float* sy, const float* sz, PosPackH* pos, float* vel, int np,
                           int ng, double delta, float vel_mul, hipStream_t s) {
    k_place_split<<<nblk((int64_t)np * np * np), BS, 0, s>>>(sx, sy, sz, (PosPack*)pos, vel, np, ng, delta, vel_mul);
}
void launch_ic_place_f64(const double2* sg, double* pos, double* vel, int np, int ng, int dim, double delta,
                         double vel_mul, hipStream_t s) {
    k_place_f64<<<nblk((int64_t)np * np * np), BS, 0, s>>>(sg, pos, vel, np, ng, dim, delta, vel_mul);
}

} // namespace hgpm

// ---- staging of the .ipk table for hgpm_generate_ic_noalloc ----
// A fixed device array in place of the table buffer hgpm_generate_ic allocates per
// call.  Each device holds its own copy from the first context created on it until the
// process ends.  Host code never passes this name to a kernel or a copy (in host code it
// is a stand-in, not a device address): it uses the address ic_static_table returns.
namespace {
__device__ __align__(256) double scratch[HGPM_IC_STATIC_BINS];

constexpr int IC_MAX_DEVICES = 64;
std::mutex g_ic_mu;
double* g_ic_ptr[IC_MAX_DEVICES] = {};
} // namespace

namespace hgpm {
// The device address of the staging array on `device`, which must be the current
// device: looked up once per device (hipGetSymbolAddress), then cached.
int ic_static_table(int device, double** ptr) {
    if (device < 0 || device >= IC_MAX_DEVICES) return -1;
    std::lock_guard<std::mutex> lock(g_ic_mu);
    if (!g_ic_ptr[device]) {
        double* p = nullptr;
        if (hipGetSymbolAddress((void**)&p, HIP_SYMBOL(scratch)) != hipSuccess || !p) return -1;
        g_ic_ptr[device] = p;
    }
    *ptr = g_ic_ptr[device];
    return 0;
}
} // namespace hgpm
