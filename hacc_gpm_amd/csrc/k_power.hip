// k_power.hip — P(k) shell binning with deterministic FP64 sums.
// Restates scalePower (src/power_spectrum/cuda/scale_power.cu:3-12), PkCICFilter
// (src/power_spectrum/cuda/filter_power.cu:47-61) and BinPower / calc_power_bins
// (src/power_spectrum/cuda/bin_power.cu:3-32).  The bin index follows the
// reference's FP32 formula (float k components, sqrtf, float kbin, truncation);
// the power uses FP64 and the CIC window (x/sin x)^4 per axis from an FP64 table.
//
// The bin and the window of a mode depend on |k_x|, |k_y| and |k_z| alone, and on the first
// two in either order, so the rows (+-a, +-b) and (+-b, +-a) are summed together, mode by
// mode along z, and binned once: up to eight modes of a full grid's row for one square
// root, one quotient and one addition to a bin (sixteen from half spectra, whose modes
// with 0 < k_z < N/2 stand for their mirror too).  A wave takes such an orbit of rows; its
// lanes are consecutive k_z.  The sums are ordered: each wave owns its accumulators, SLOTS
// per bin, and the lanes that share one add to it in turn (LDS instructions of a wave
// execute in order), then the partials of waves and workgroups are added in a fixed order.
// Bound by the additions and their turns where bins are many, else by the reading of the
// spectrum: at 1024^3 from half spectra 1.5 ms with 32 bins (2.9 TB/s), 2.6 ms with 221; at
// 256^3 with 221 bins 0.064 ms with the reduction.  One mode per lane of single-wave
// workgroups over full spectra, their partials added by one thread per bin, took 9.7 ms
// (1024^3, 32 bins) and 1.05 ms (256^3, 221 bins, whose private accumulators left one
// wave per CU).
#include "common.h"
#include "internal.h"

#pragma clang fp contract(off)

namespace {
constexpr int PW = 4;        // waves per workgroup
constexpr int PB = 64 * PW;
constexpr int PBLOCKS = 1024;

__device__ __forceinline__ float kmode(int idx, int ng, double d) {
    float l = (float)idx;
    if (idx > ((ng / 2) - 1)) l = (float)(-(ng - idx));
    return (float)((double)l * d);
}

// Orbit o = a (a + 1) / 2 + b, 0 <= b <= a <= N/2.
__device__ __forceinline__ void orbit_of(int o, int& a, int& b) {
    a = (int)((sqrtf(8.0f * (float)o + 1.0f) - 1.0f) * 0.5f);
    while ((a + 1) * (a + 2) / 2 <= o) a++;
    while (a * (a + 1) / 2 > o) a--;
    b = o - a * (a + 1) / 2;
}

// spec: HALF: half spectra, k_z = 0..N/2, rows of `pitch` and x planes of `plane`
// elements; else full grids.  partial: per bin, then per workgroup: the power, and behind
// all of them the modes (whole numbers).
template <typename V, bool HALF, int SLOTS>
__global__ __launch_bounds__(PB) void k_power_bins(const V* __restrict spec, int ng, int pitch, size_t plane,
                                                   double dfold, double minK, double binDelta, int nbins,
                                                   const double* __restrict win, double scale,
                                                   double* __restrict partial) {
    extern __shared__ double sh[];
    const int lane = threadIdx.x & 63, wv = threadIdx.x >> 6;
    const int per = nbins * SLOTS;
    double* acc = sh + wv * per;                 // [nbins][SLOTS] of this wave
    unsigned* cnt = (unsigned*)(sh + PW * per);  // [nbins][SLOTS], shared: whole numbers
    for (int i = threadIdx.x; i < PW * per; i += PB) sh[i] = 0.0;
    for (int i = threadIdx.x; i < per; i += PB) cnt[i] = 0u;
    __syncthreads();
    const int h = ng / 2, norb = (h + 1) * (h + 2) / 2;
    const int nz = HALF ? h + 1 : ng;
    const int slot = lane % SLOTS, turn = lane / SLOTS;
    const int nw = gridDim.x * PW;
    for (int o = (int)blockIdx.x * PW + wv; o < norb; o += nw) {
        int a, b;
        orbit_of(__builtin_amdgcn_readfirstlane(o), a, b);
        // the orbit's rows: (a, b), its mirrors, and the same with the axes swapped; an
        // index 0 or N/2 is its own mirror
        const V* row[8];
        int nr = 0;
        const int am = a == 0 || a == h ? a : ng - a, bm = b == 0 || b == h ? b : ng - b;
#pragma unroll
        for (int i = 0; i < 8; i++) {
            const int x0 = i & 2 ? am : a, y0 = i & 1 ? bm : b;
            const bool own = (!(i & 2) || am != a) && (!(i & 1) || bm != b) && (!(i & 4) || a != b);
            const int x = i & 4 ? y0 : x0, y = i & 4 ? x0 : y0;
            row[i] = own ? spec + (size_t)x * plane + (size_t)y * pitch : nullptr;
            nr += own ? 1 : 0;
        }
        const float kx = kmode(a, ng, dfold), ky = kmode(b, ng, dfold);
        const float kxy = kx * kx + ky * ky;
        const double wxy = win[a] * win[b];
        for (int z0 = 0; z0 < nz; z0 += 64) {
            const int z = z0 + lane;
            V v[8];
#pragma unroll
            for (int i = 0; i < 8; i++)
                v[i] = row[i] && z < nz ? row[i][z] : cmake<V>(0, 0);
            double p = 0.0;
#pragma unroll
            for (int i = 0; i < 8; i++) p += (double)v[i].x * (double)v[i].x + (double)v[i].y * (double)v[i].y;
            const float kz = kmode(z < nz ? z : 0, ng, dfold);
            const float s = kxy + kz * kz;
            const float kb = (float)((double)sqrtf(s) - minK);
            const int bin = (int)((double)kb / binDelta);
            const bool drop = z >= nz || (a | b | z) == 0 || (a == h && b == h && z == h) || bin < 0 || bin >= nbins;
            const int weight = HALF && z != 0 && z != h ? 2 : 1;
            const double t = (double)weight * p * scale * (wxy * win[z < nz ? z : 0]);
            const int at = drop ? 0 : bin * SLOTS + slot;
#pragma unroll
            for (int g = 0; g < 64 / SLOTS; g++)
                if (turn == g && !drop) unsafeAtomicAdd(&acc[at], t);
            if (!drop) atomicAdd(&cnt[at], (unsigned)(nr * weight));
        }
    }
    __syncthreads();
    for (int b = threadIdx.x; b < nbins; b += PB) {
        double t = 0.0;
        unsigned long long n = 0;
        for (int w = 0; w < PW; w++)
            for (int k = 0; k < SLOTS; k++) t += sh[w * per + b * SLOTS + k];
        for (int k = 0; k < SLOTS; k++) n += cnt[b * SLOTS + k];
        partial[(size_t)b * gridDim.x + blockIdx.x] = t;
        partial[(size_t)(nbins + b) * gridDim.x + blockIdx.x] = (double)n;
    }
}

// One workgroup per bin: its partials in a fixed order.
__global__ __launch_bounds__(PB) void k_power_reduce(const double* __restrict partial, int nblocks, int nbins,
                                                     double* __restrict sums, long long* __restrict counts) {
    __shared__ double s[2][PB];
    const int b = blockIdx.x, tid = threadIdx.x;
    double t = 0.0, n = 0.0;
    for (int k = tid; k < nblocks; k += PB) {
        t += partial[(size_t)b * nblocks + k];
        n += partial[(size_t)(nbins + b) * nblocks + k];
    }
    s[0][tid] = t;
    s[1][tid] = n;
    __syncthreads();
    for (int w = PB / 2; w > 0; w >>= 1) {
        if (tid < w) {
            s[0][tid] += s[0][tid + w];
            s[1][tid] += s[1][tid + w];
        }
        __syncthreads();
    }
    if (tid == 0) {
        sums[b] = s[0][0];
        counts[b] = (long long)s[1][0];
    }
}

template <typename V, bool HALF, int SLOTS>
void bins_launch(const V* spec, int ng, int pitch, size_t plane, double dfold, double minK, double binDelta, int nbins,
                 const double* win, double scale, double* partial, int nblocks, hipStream_t s) {
    const size_t shmem = (size_t)nbins * SLOTS * (PW * sizeof(double) + sizeof(unsigned));
    (void)hipFuncSetAttribute((const void*)k_power_bins<V, HALF, SLOTS>, hipFuncAttributeMaxDynamicSharedMemorySize,
                              (int)shmem);
    k_power_bins<V, HALF, SLOTS><<<nblocks, PB, shmem, s>>>(spec, ng, pitch, plane, dfold, minK, binDelta, nbins, win,
                                                            scale, partial);
}
} // namespace

namespace hgpm {
int power_partial_blocks(int ng) {
    const int h = ng / 2, norb = (h + 1) * (h + 2) / 2, nb = (norb + PW - 1) / PW;
    return nb < PBLOCKS ? nb : PBLOCKS;
}

// 16 accumulators per bin and wave (four turns) while they leave room for 16 waves a CU;
// with more bins 8 (eight turns, 73 KB a workgroup at 256 bins)
template <typename V, bool HALF>
void launch_power_bins(const V* spec, int ng, int pitch, size_t plane, double rl_fold, double minK, double binDelta,
                       int nbins, const double* win, double scale, double* partial, int nblocks, double* sums,
                       long long* counts, hipStream_t s) {
    const double dfold = (2 * HGPM_PI) / rl_fold;
    if (nbins <= 64)
        bins_launch<V, HALF, 16>(spec, ng, pitch, plane, dfold, minK, binDelta, nbins, win, scale, partial, nblocks, s);
    else
        bins_launch<V, HALF, 8>(spec, ng, pitch, plane, dfold, minK, binDelta, nbins, win, scale, partial, nblocks, s);
    k_power_reduce<<<nbins, PB, 0, s>>>(partial, nblocks, nbins, sums, counts);
}
template void launch_power_bins<float2, true>(const float2*, int, int, size_t, double, double, double, int,
                                              const double*, double, double*, int, double*, long long*, hipStream_t);
template void launch_power_bins<double2, false>(const double2*, int, int, size_t, double, double, double, int,
                                                const double*, double, double*, int, double*, long long*, hipStream_t);
} // namespace hgpm
