// k_fp64.hip — the plain FP64 path: every quantity in FP64 (double3 positions and
// velocities, complex128 grids).  It is the "FP64 plain GPU path" the FP32 engine is
// measured against, the serial step of the reference's default build
// (src/haccgpm.hpp:67-72) with grid_t = complex128:
//   k_drift   UpdatePosKernel       src/pm_actions/cuda/update_positions_pm.cu:3-20
//   k_cic     memset + CICKernel    src/pm_actions/cuda/cic_pm.cu:46-87,142-147
//   FftOps.force_f64 (k_rows_force, k_cols_force) kspace_solve_gradient,
//             src/pm_solver/cuda/kspace_solver.cu:55-90 (+ calcGreens), and its real part,
//             getRealGrid, src/initial_conditions/cuda/transform_density_field_initializer.cu:14-28
//   k_icic    ICICKernel            src/pm_actions/cuda/icic_pm.cu:72-127
// The last component's x pass joins the three (copyGridToFloat4,
// src/pm_solver/cuda/combine.cu:21-34).  A step of 128^3 went from 0.62 ms (a pass for each
// component's modes, one for its real part, eight atomics per particle) to 0.33 ms.
#include "common.h"
#include "internal.h"

namespace {
constexpr int BS = 256;
inline unsigned nblk(int64_t n) { return (unsigned)((n + BS - 1) / BS); }

__global__ void k_drift(double* __restrict pos, const double* __restrict vel, int64_t n, int ng, double pf) {
    int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= n) return;
    const double g = (double)ng;
#pragma unroll
    for (int d = 0; d < 3; d++) {
        double x = pos[3 * i + d] + vel[3 * i + d] * pf;
        x = fmod(x + g, g);
        if (x < 0) x += g;   // moved by more than a box in one step
        if (x >= g) x -= g;
        pos[3 * i + d] = x;
    }
}

__global__ void k_zero(double* __restrict p, size_t n) {
    size_t i = (size_t)blockIdx.x * blockDim.x + threadIdx.x;
    size_t st = (size_t)gridDim.x * blockDim.x;
    for (; i < n; i += st) p[i] = 0.0;
}

// cells per axis of the 8 corners: c[d][0] the particle's (kept in range for any input;
// positions are wrapped into [0, ng)), c[d][1] the next one, periodic
__device__ __forceinline__ void corners(double X, double Y, double Z, int ng, int c[3][2], double f[3]) {
    const double x[3] = {X, Y, Z};
#pragma unroll
    for (int d = 0; d < 3; d++) {
        int i = (int)x[d];
        f[d] = x[d] - i;
        if ((unsigned)i >= (unsigned)ng) i = ((i % ng) + ng) % ng;
        c[d][0] = i;
        c[d][1] = i + 1 == ng ? 0 : i + 1;
    }
}

// Bound by the FP64 atomics on L2 (88 G/s).  Particles are in lattice order, z fastest:
// where the next lane's particle lies in the next cell of the same row, this lane's four
// upper corners are that lane's lower ones and are added by it, four atomics per particle
// instead of eight: 0.194 -> 0.098 ms at 128^3.
__global__ __launch_bounds__(BS) void k_cic(const double* __restrict pos, int64_t n, int ng, double mass,
                                            double2* __restrict grid) {
    const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    const int lane = threadIdx.x & 63;
    const bool valid = i < n;
    const int64_t j = valid ? i : 0;
    int c[3][2];
    double f[3];
    corners(pos[3 * j], pos[3 * j + 1], pos[3 * j + 2], ng, c, f);
    // row (x, y) of the cell, < 2^20, -1 for no particle
    const int row = valid ? c[0][0] * ng + c[1][0] : -1;
    const int prow = __shfl_up(row, 1, 64), pz = __shfl_up(c[2][1], 1, 64);
    const int nrow = __shfl_down(row, 1, 64), nz = __shfl_down(c[2][0], 1, 64);
    const bool take = lane > 0 && valid && prow == row && pz == c[2][0]; // the previous lane's upper corners
    const bool give = lane < 63 && valid && nrow == row && nz == c[2][1];
#pragma unroll
    for (int x = 0; x < 2; x++)
#pragma unroll
        for (int y = 0; y < 2; y++) {
            const double dx = x ? f[0] : 1.0 - f[0];
            const double dy = y ? f[1] : 1.0 - f[1];
            double lo = dx * dy * (1.0 - f[2]) * mass;
            const double up = dx * dy * f[2] * mass;
            const double prev = __shfl_up(up, 1, 64);
            if (take) lo += prev;
            if (valid) {
                const int64_t r = gidx(ng, c[0][x], c[1][y], 0);
                unsafeAtomicAdd(&grid[r + c[2][0]].x, lo);
                if (!give) unsafeAtomicAdd(&grid[r + c[2][1]].x, up);
            }
        }
}

// Bound by the lines that the lanes' corners touch: the three components of a cell lie
// together (24 bytes), and the two corners of a row are read as one run.  Kicks of early /
// dispersed / randomly ordered particles at 192^3: 0.23 / 0.51 / 0.72 ms; from three grids
// 0.30 / 1.14 / 1.75, cell by cell 0.26 / 0.55 / 0.74.
__global__ void k_icic(const double* __restrict pos, double* __restrict vel, const double* __restrict force, int64_t n,
                       int ng, double deltaT, double fscal) {
    int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= n) return;
    int c[3][2];
    double f[3];
    corners(pos[3 * i], pos[3 * i + 1], pos[3 * i + 2], ng, c, f);
    double dv0 = 0, dv1 = 0, dv2 = 0;
    const int z = min(c[2][0], ng - 2); // both corners of a row from one run of 48 bytes ...
#pragma unroll
    for (int x = 0; x < 2; x++)
#pragma unroll
        for (int y = 0; y < 2; y++) {
            const double dx = x ? f[0] : 1.0 - f[0];
            const double dy = y ? f[1] : 1.0 - f[1];
            const double* row = force + 3 * gidx(ng, c[0][x], c[1][y], 0);
            double F[6];
#pragma unroll
            for (int k = 0; k < 6; k++) F[k] = row[3 * z + k];
            if (c[2][1] == 0) { // ... but the row's last cell and its first one
#pragma unroll
                for (int d = 0; d < 3; d++) {
                    F[d] = F[3 + d];
                    F[3 + d] = row[d];
                }
            }
            const double lo = dx * dy * (1.0 - f[2]) * deltaT * fscal, up = dx * dy * f[2] * deltaT * fscal;
            dv0 += lo * F[0];
            dv1 += lo * F[1];
            dv2 += lo * F[2];
            dv0 += up * F[3];
            dv1 += up * F[4];
            dv2 += up * F[5];
        }
    vel[3 * i] += dv0;
    vel[3 * i + 1] += dv1;
    vel[3 * i + 2] += dv2;
}

__global__ void k_fold(double* __restrict pos, int64_t n3, int ng) {
    int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= n3) return;
    double x = pos[i] / (double)ng;
    if (x >= 0.5) x -= 0.5;
    pos[i] = x * 2 * (double)ng;
}

__global__ void k_density_to_real(const double2* __restrict g, double* __restrict out, int64_t g3) {
    int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (i < g3) out[i] = g[i].x;
}
} // namespace

namespace hgpm {
void launch_f64_drift(double* pos, const double* vel, int64_t n, int ng, double pf, hipStream_t s) {
    if (n) k_drift<<<nblk(n), BS, 0, s>>>(pos, vel, n, ng, pf);
}
void launch_f64_zero(double* p, size_t n, hipStream_t s) {
    unsigned nb = nblk((int64_t)n);
    if (nb > 65536u * 8) nb = 65536u * 8;
    if (n) k_zero<<<nb, BS, 0, s>>>(p, n);
}
void launch_f64_cic(const double* pos, int64_t n, int ng, double mass, double2* grid, hipStream_t s) {
    launch_f64_zero((double*)grid, (size_t)2 * ng * ng * ng, s);
    if (n) k_cic<<<nblk(n), BS, 0, s>>>(pos, n, ng, mass, grid);
}
void launch_f64_icic(const double* pos, double* vel, const double* force, int64_t n, int ng, double deltaT,
                     double fscal, hipStream_t s) {
    if (n) k_icic<<<nblk(n), BS, 0, s>>>(pos, vel, force, n, ng, deltaT, fscal);
}
void launch_f64_fold(double* pos, int64_t n, int ng, hipStream_t s) {
    if (n) k_fold<<<nblk(3 * n), BS, 0, s>>>(pos, 3 * n, ng);
}
void launch_f64_density_to_real(const double2* grid, double* out, int64_t g3, hipStream_t s) {
    k_density_to_real<<<nblk(g3), BS, 0, s>>>(grid, out, g3);
}
} // namespace hgpm
