// Host-side check of the engine's control code (capi.cpp, hostcopy.cpp, host.cpp, compiled
// for the host) against a HIP runtime of its own: device memory is host memory, streams run
// at once, kernels are replaced by what they leave in the buffers that the control code
// relies on, and calls fail where a scenario says so.  Error paths that no call sequence
// brings about on a healthy GPU run here, without one.  runtime_check <scenario> prints
// "<cases> <bad>" after a line for each bad one.
#include "../../include/hgpm.h"
#include "hostcopy.h"
#include "internal.h"

#include <cmath>
#include <cstdio>
#include <cstdlib>
#include <cstring>
#include <functional>
#include <mutex>
#include <string>
#include <thread>
#include <vector>

// ---------------------------------------------------------------- the runtime ----
namespace fake {
std::mutex mu;
thread_local hipError_t last = hipSuccess;
constexpr int NDEV = 2;
thread_local int device = 0;
struct Handle { int device; }; // a stream or an event
hipError_t make(Handle** h) { return *h = new Handle{device}, hipSuccess; }
bool capturing = false;     // launches are recorded, not run
bool graph_fails = false;   // hipGraphLaunch
bool no_pinned = false;     // hipHostMalloc fails ...
int events_left = -1;       // ... events do, after so many (< 0: they do not)
int launch_no = 0;          // launches since the last reset ...
int launch_fails = -1;      // ... the one that fails (< 0: none)
void clear() {
    launch_no = 0;
    launch_fails = -1;
}
int memory = 0; // what a caller's buffers are: 0 unknown to the runtime, 1 unregistered, 2 page-locked
const char *lo = nullptr, *hi = nullptr; // a caller's buffer ...
int direct = 0, copies = 0;              // ... and the copies made from or to it, and in all
void moved(const void* d, const void* s) {
    std::lock_guard<std::mutex> lock(mu);
    copies++;
    for (const void* p : {d, s}) direct += p >= lo && p < hi;
}
hipError_t err(hipError_t e) { return e == hipSuccess ? e : last = e; }
// One launch: true when its effects happen.
bool launch() {
    const bool bad = launch_no++ == launch_fails;
    if (bad) last = hipErrorOutOfMemory;
    return !bad && !capturing;
}
} // namespace fake
using fake::err;

extern "C" {
hipError_t hipGetLastError() {
    const hipError_t e = fake::last;
    fake::last = hipSuccess;
    return e;
}
const char* hipGetErrorString(hipError_t e) { return e == hipSuccess ? "no error" : "error"; }
hipError_t hipGetDeviceCount(int* n) { return *n = fake::NDEV, hipSuccess; }
hipError_t hipGetDevice(int* d) { return *d = fake::device, hipSuccess; }
hipError_t hipSetDevice(int d) {
    if (d < 0 || d >= fake::NDEV) return err(hipErrorInvalidDevice);
    return fake::device = d, hipSuccess;
}
hipError_t hipMemGetInfo(size_t* f, size_t* t) { return *f = *t = (size_t)4 << 30, hipSuccess; }
hipError_t hipMalloc(void** p, size_t n) { return *p = calloc(1, n), hipSuccess; }
hipError_t hipFree(void* p) { return free(p), hipSuccess; }
hipError_t hipHostMalloc(void** p, size_t n, unsigned) {
    if (fake::no_pinned) return err(hipErrorOutOfMemory);
    return *p = malloc(n), hipSuccess;
}
hipError_t hipPointerGetAttributes(hipPointerAttribute_t* a, const void*) {
    if (fake::memory == 0) return err(hipErrorInvalidValue);
    a->type = fake::memory == 1 ? hipMemoryTypeUnregistered : hipMemoryTypeHost;
    return hipSuccess;
}
hipError_t hipHostFree(void* p) { return free(p), hipSuccess; }
hipError_t hipMemcpy(void* d, const void* s, size_t n, hipMemcpyKind) { return memcpy(d, s, n), hipSuccess; }
hipError_t hipMemcpyAsync(void* d, const void* s, size_t n, hipMemcpyKind, hipStream_t) {
    fake::moved(d, s);
    if (!fake::capturing) memcpy(d, s, n);
    return hipSuccess;
}
hipError_t hipMemset(void* d, int v, size_t n) { return memset(d, v, n), hipSuccess; }
hipError_t hipStreamCreateWithFlags(hipStream_t* s, unsigned) { return fake::make((fake::Handle**)s); }
hipError_t hipStreamDestroy(hipStream_t s) { return delete (fake::Handle*)s, hipSuccess; }
hipError_t hipStreamSynchronize(hipStream_t) { return hipSuccess; }
hipError_t hipStreamWaitEvent(hipStream_t, hipEvent_t, unsigned) { return hipSuccess; }
hipError_t hipEventCreateWithFlags(hipEvent_t* e, unsigned) {
    if (fake::events_left == 0) return err(hipErrorOutOfMemory);
    if (fake::events_left > 0) fake::events_left--;
    return fake::make((fake::Handle**)e); }
hipError_t hipEventCreate(hipEvent_t* e) { return hipEventCreateWithFlags(e, 0); }
hipError_t hipEventDestroy(hipEvent_t e) { return delete (fake::Handle*)e, hipSuccess; }
hipError_t hipEventRecord(hipEvent_t e, hipStream_t s) { // an event belongs to its stream's device
    if (!s) return hipSuccess;
    return err(((fake::Handle*)e)->device == ((fake::Handle*)s)->device ? hipSuccess : hipErrorInvalidHandle);
}
hipError_t hipEventSynchronize(hipEvent_t) { return hipSuccess; }
hipError_t hipEventQuery(hipEvent_t) { return hipSuccess; }
hipError_t hipEventElapsedTime(float* ms, hipEvent_t, hipEvent_t) { return *ms = 1.0f, hipSuccess; }
hipError_t hipStreamBeginCapture(hipStream_t, hipStreamCaptureMode) { return fake::capturing = true, hipSuccess; }
hipError_t hipStreamEndCapture(hipStream_t, hipGraph_t* g) { return fake::capturing = false, *g = nullptr, hipSuccess; }
hipError_t hipGraphInstantiate(hipGraphExec_t* e, hipGraph_t, hipGraphNode_t*, char*, size_t) {
    return *e = nullptr, hipSuccess;
}
hipError_t hipGraphLaunch(hipGraphExec_t, hipStream_t) { return err(fake::graph_fails ? hipErrorOutOfMemory : hipSuccess); }
hipError_t hipGraphDestroy(hipGraph_t) { return hipSuccess; }
hipError_t hipGraphExecDestroy(hipGraphExec_t) { return hipSuccess; }
}

// ---------------------------------------------------------------- the kernels ----
namespace hgpm {
// What the deposit's kernels rely on and leave behind: the control words and mass sums of
// their set cleared, no chunk listed; cursors, lists and sums used; the other set cleared.
int dep_stale = 0; // deposits that started from anything else
// What the grids hold: the density as its reader takes it, the potential (FP32).
bool holds_density = false, holds_potential = false;
void launch_deposit_windows(const PosPackH*, int64_t, int ng, float, const DepositBuffers& b, hipStream_t) {
    if (!fake::launch()) return;
    const int nblk = (ng / 16) * (ng / 16) * (ng / 16) * b.nbox;
    bool clean = true;
    for (int i = 0; i < b.set_words; i++) clean = clean && (i == HGPM_DEP_CTL || b.ctl[i] == 0);
    for (int i = 0; i < nblk; i++) clean = clean && b.count[i] == 0;
    dep_stale += !clean;
    b.ctl[1] += 2;
    b.ctl[4] += 100;
    for (int i = 0; i < HGPM_DEP_MASS * b.nbox; i++) b.ctl[HGPM_DEP_CTL + 1 + i] += 7;
    for (int i = 0; i < nblk; i++) b.count[i] += 3;
}
void launch_deposit_binned(const PosPackH* p, int64_t n, int ng, float m, long long*, float* rhof,
                           const DepositBuffers& b, hipStream_t s) {
    holds_density = !rhof;
    holds_potential = holds_potential && !rhof;
    launch_deposit_windows(p, n, ng, m, b, s);
    memset(b.count, 0, sizeof(unsigned) * (ng / 16) * (ng / 16) * (ng / 16) * b.nbox);
    if (fake::launch()) memset(b.next, 0, sizeof(unsigned long long) * b.set_words);
    else holds_density = false;
}
void launch_deposit_owner(int ng, long long*, float* rhof, const DepositBuffers& b, hipStream_t) {
    holds_potential = holds_potential && !rhof; // whether it runs or not
    holds_density = false;
    if (fake::launch()) memset(b.count, 0, sizeof(unsigned) * (ng / 16) * (ng / 16) * (ng / 16) * b.nbox);
    holds_density = !rhof;
}
void launch_deposit_deferred(const PosPackH*, int64_t, int, float, long long*, const DepositBuffers& b, hipStream_t) {
    if (fake::launch()) memset(b.next, 0, sizeof(unsigned long long) * b.set_words);
    else holds_density = false;
}
void launch_zero_u64(unsigned long long* p, size_t n, hipStream_t) {
    if (fake::launch()) memset(p, 0, sizeof(*p) * n);
}
#define STUB(name, ...) \
    void name(__VA_ARGS__) { (void)fake::launch(); }
STUB(launch_drift, PosPackH*, const float*, int64_t, int, float, hipStream_t)
STUB(launch_compare, const PosPackH*, const float*, const double*, const double*, const PosPackH*, const float*,
     const double*, const double*, int64_t, int, int, double*, hipStream_t)
void launch_f64_cic(const double*, int64_t, int, double, double2*, hipStream_t) { holds_density = fake::launch(); }
STUB(launch_f64_fold, double*, int64_t, int, hipStream_t)
STUB(launch_f64_icic, const double*, double*, const double*, int64_t, int, double, double, hipStream_t)
STUB(launch_f64_drift, double*, const double*, int64_t, int, double, hipStream_t)
STUB(launch_f64_density_to_real, const double2*, double*, int64_t, hipStream_t)
STUB(launch_ic_lines, const double*, int, double, double, double2*, int, hipStream_t)
STUB(launch_ic_noise_f32, float*, int, uint32_t, hipStream_t)
STUB(launch_ic_noise_f64, double2*, int, uint32_t, hipStream_t)
STUB(launch_ic_place_split, const float*, const float*, const float*, PosPackH*, float*, int, int, double, float, hipStream_t)
STUB(launch_ic_place_f64, const double2*, double*, double*, int, int, int, double, double, hipStream_t)
STUB(launch_ic_scale_f64, double2*, int, const double*, int, double, double, hipStream_t)
STUB(launch_ic_displacement_f64, const double2*, double2*, int, int, double, double, hipStream_t)
STUB(launch_gather_kick, PosPackH*, float*, int64_t, int, const float*, double, double, int, float, int, const void*, int, hipStream_t)
STUB(launch_to_internal, const PosPackH*, const float*, PosPackH*, float*, int64_t, int, hipStream_t)
STUB(launch_to_reference, const PosPackH*, const float*, PosPackH*, float*, int64_t, int, hipStream_t)
STUB(launch_split_to_f64, const PosPackH*, const float*, double*, double*, int64_t, int, hipStream_t)
STUB(launch_split_from_f64, const double*, const double*, PosPackH*, float*, int64_t, int, int, hipStream_t)
STUB(launch_split_to_float3, const PosPackH*, const float*, float*, float*, int64_t, int, hipStream_t)
STUB(launch_split_from_float3, const float*, const float*, PosPackH*, float*, int64_t, int, int, hipStream_t)
STUB(launch_force_from_psi, const float*, float*, int, hipStream_t)
int compare_partials() { return 1; }
int power_partial_blocks(int) { return 1; }
int ic_static_table(int, double** p) {
    static double t[HGPM_IC_STATIC_BINS];
    return *p = t, 0;
}
template <typename V, bool H>
void launch_power_bins(const V*, int, int, size_t, double, double, double, int, const double*, double, double*, int,
                       double*, long long*, hipStream_t) {
    (void)fake::launch();
}
template void launch_power_bins<float2, true>(const float2*, int, int, size_t, double, double, double, int,
                                              const double*, double, double*, int, double*, long long*, hipStream_t);
template void launch_power_bins<double2, false>(const double2*, int, int, size_t, double, double, double, int,
                                                const double*, double, double*, int, double*, long long*, hipStream_t);

FftOps table(int n) {
    FftOps f{};
    f.n = n;
    f.stages = 1;
    f.n_variants = f.valid_mask = 1;
    f.hz = n / 2 + 16;
    f.plane = (size_t)n * f.hz;
    f.twiddles = [](double*, double*) {};
    f.pass_f32 = [](float2*, int, int, const float2*, int, hipStream_t) { (void)fake::launch(); };
    f.pass_f64 = [](double2*, int, int, const double2*, hipStream_t) { holds_density = fake::launch() && false; };
    f.force_f64 = [](const double2*, double2*, double*, const double*, const double*, const double2*, const double2*, int, hipStream_t) { (void)fake::launch(); };
    f.pass_half = [](float2*, int, int, const float2*, int, int, hipStream_t) { (void)fake::launch(); };
    f.fwd_z_r2c = [](const long long*, const float*, const unsigned long long*, const unsigned long long*, float2*,
                     const float2*, int, hipStream_t) { (void)fake::launch(); };
    f.x_psi = [](float2*, const float2*, const float2*, const float*, int, int, hipStream_t) { (void)fake::launch(); };
    f.inv_z_c2r_real = [](const float2*, float*, const float2*, int, hipStream_t) { holds_potential = fake::launch(); };
    return f;
}
#define TABLE(n) extern const FftOps fft_ops_##n; const FftOps fft_ops_##n = table(n);
HGPM_FFT_SIZES(TABLE)
extern const FftOps fft_ops_1024_alt;
const FftOps fft_ops_1024_alt = table(1024);
} // namespace hgpm

// -------------------------------------------------------------- the scenarios ----
namespace {
int cases = 0, bad = 0;
void check(bool ok, const std::string& what) {
    cases++;
    if (!ok) {
        bad++;
        printf("bad: %s\n", what.c_str());
    }
}
hgpm_params params(int ng, int precision = HGPM_FP32) {
    hgpm_params p{};
    p.ng = p.np = ng;
    p.rl = 2.0 * ng;
    p.nsteps = 10;
    p.z_ini = 50.0;
    p.hubble = 0.7;
    p.omega_cdm = 0.25;
    p.omega_matter = p.omega_cb = 0.3;
    p.ss8 = 0.8;
    p.ns = 0.96;
    p.t_cmb = 2.7;
    p.pk_folds = 1;
    p.pk_bins = 16;
    p.precision = precision;
    return p;
}
hgpm_ctx* box(int ng, int precision = HGPM_FP32) {
    const hgpm_params p = params(ng, precision);
    hgpm_ctx* c = nullptr;
    if (hgpm_create(&p, &c)) {
        printf("hgpm_create: %s\n", hgpm_last_error(nullptr));
        exit(2);
    }
    std::vector<float> x(3 * (size_t)ng * ng * ng, 1.0f);
    if (hgpm_set_particles(c, x.data(), x.data())) exit(2);
    fake::clear();
    return c;
}
struct Spectrum {
    double k[16], pk[16];
    int64_t n[16];
    int of(hgpm_ctx* c, int fold) { return hgpm_power_spectrum(c, fold, k, pk, n); }
};

// A deposit whose launches failed, in whatever call made it: the next one starts from
// cleared control words and mass sums, and no chunk listed.
void deposit() {
    const hgpm_step_coeffs co{};
    Spectrum sp;
    const std::function<int(hgpm_ctx*)> calls[] = {
        [](hgpm_ctx* c) { return hgpm_cic(c); }, [&](hgpm_ctx* c) { return hgpm_step(c, &co); },
        [&](hgpm_ctx* c) { return sp.of(c, 0); }, [&](hgpm_ctx* c) { return sp.of(c, 1); }};
    for (int call = 0; call < 4; call++)
        for (int before = 0; before < 2; before++)  // either set of control words
            for (int at = 0; at < 4; at++)          // the launch that fails
                for (int twice = 0; twice < 2; twice++) { // and the one after it
                    hgpm_ctx* c = box(32);
                    for (int i = 0; i < before; i++) (void)hgpm_cic(c);
                    const std::string what = "call " + std::to_string(call) + " before " + std::to_string(before) +
                                             " launch " + std::to_string(at) + " twice " + std::to_string(twice);
                    hgpm::dep_stale = 0;
                    for (int i = 0; i <= twice; i++) {
                        fake::clear();
                        fake::launch_fails = at;
                        const int rc = calls[call](c);
                        check(rc == (fake::launch_no > at ? HGPM_ERR_HIP : HGPM_OK), what + ": the failure is reported");
                    }
                    fake::clear();
                    hgpm::dep_stale = 0; // (a deposit that fails may start from anything)
                    for (int i = 0; i < 3; i++) check(hgpm_cic(c) == HGPM_OK, what + ": the deposit after it");
                    check(hgpm::dep_stale == 0, what + ": stale control words");
                    int deferred = -1;
                    check(hgpm_get_tunable(c, "deposit_deferred", &deferred) == HGPM_OK && deferred == 2,
                          what + ": the last deposit's words");
                    hgpm_destroy(c);
                }
    // a graph run whose capture or launch fails, then steps one by one
    for (int how = 0; how < 2; how++)
        for (int before = 0; before < 2; before++) {
            const hgpm_params p[2] = {params(32), params(64)};
            hgpm_ensemble* e = nullptr;
            check(hgpm_ensemble_create(2, p, &e) == HGPM_OK, "ensemble");
            for (int b = 0; b < 2; b++) {
                std::vector<float> x(3 * (size_t)p[b].np * p[b].np * p[b].np, 1.0f);
                check(hgpm_ensemble_set_particles(e, b, x.data(), x.data()) == HGPM_OK, "ensemble particles");
            }
            const hgpm_step_coeffs co3[6] = {};
            fake::clear();
            for (int i = 0; i < before; i++) check(hgpm_ensemble_step(e, co3) == HGPM_OK, "ensemble step");
            fake::clear();
            if (how == 0) fake::launch_fails = 12;
            else fake::graph_fails = true;
            const std::string what = "ensemble run " + std::to_string(how) + " before " + std::to_string(before);
            check(hgpm_ensemble_run(e, 3, co3) == HGPM_ERR_HIP, what + ": the failure is reported");
            fake::clear();
            fake::graph_fails = false;
            (void)hipGetLastError();
            hgpm::dep_stale = 0;
            for (int i = 0; i < 3; i++) check(hgpm_ensemble_step(e, co3) == HGPM_OK, what + ": the steps after it");
            check(hgpm::dep_stale == 0, what + ": stale control words");
            hgpm_ensemble_destroy(e);
        }
}

// A call whose launches fail: what it has overwritten is refused afterwards, what it has
// not is still there.
void state() {
    const hgpm_step_coeffs co{};
    Spectrum sp;
    for (int prec : {HGPM_FP32, HGPM_FP64}) {
        const bool f32 = prec == HGPM_FP32;
        const size_t n = 32 * 32 * 32;
        std::vector<double> buf(3 * n);
        auto density = [&](hgpm_ctx* c) {
            return f32 ? hgpm_get_density(c, (int64_t*)buf.data()) : hgpm_get_density_f64(c, buf.data());
        };
        auto force = [&](hgpm_ctx* c) { return f32 ? hgpm_get_force(c, (float*)buf.data()) : hgpm_get_force_f64(c, buf.data()); };
        struct Call {
            const char* name;
            bool solved; // starts from a force, else from a density
            std::function<int(hgpm_ctx*)> run;
        };
        const Call calls[] = {{"P(k)", true, [&](hgpm_ctx* c) { return sp.of(c, 0); }},
                              {"folded P(k)", true, [&](hgpm_ctx* c) { return sp.of(c, 1); }},
                              {"P(k), density", false, [&](hgpm_ctx* c) { return sp.of(c, 0); }},
                              {"step", true, [&](hgpm_ctx* c) { return hgpm_step(c, &co); }},
                              {"step, density", false, [&](hgpm_ctx* c) { return hgpm_step(c, &co); }},
                              {"cic", true, [](hgpm_ctx* c) { return hgpm_cic(c); }},
                              {"fft", false, [&](hgpm_ctx* c) { return hgpm_fft_host(c, buf.data(), -1); }},
                              {"solve", false, [](hgpm_ctx* c) { return hgpm_solve_gradient(c); }},
                              {"grid P(k)", false, [&](hgpm_ctx* c) {
                                   return hgpm_power_spectrum_grid(c, 0, sp.k, sp.pk, sp.n);
                               }}};
        for (const Call& call : calls)
            for (int at = 0;; at++) {
                hgpm_ctx* c = box(32, prec);
                (void)hgpm_cic(c);
                if (call.solved) (void)hgpm_solve_gradient(c);
                fake::clear();
                fake::launch_fails = at;
                const int rc = call.run(c);
                const bool failed = fake::launch_no > at;
                const std::string name = call.name, what = std::string(f32 ? "FP32 " : "FP64 ") + name + " launch " + std::to_string(at);
                check(rc == (failed ? HGPM_ERR_HIP : HGPM_OK), what + ": reported");
                fake::clear();
                const bool has_density = hgpm::holds_density, has_force = !f32 || hgpm::holds_potential;
                const int d = density(c), f = force(c);
                check(d == HGPM_ERR_STATE || (d == HGPM_OK && has_density), what + ": density");
                check(f == HGPM_ERR_STATE || (f == HGPM_OK && has_force), what + ": force");
                check(hgpm_update_velocities(c, 0.0, 1.0) == f, what + ": kick");
                check(hgpm_kick_drift(c, 0.0, 1.0, 0.0) == f, what + ": kick and drift");
                // the transforms of these only read the int64 density
                if (failed && f32 && (name == "solve" || name == "grid P(k)") && at < 3)
                    check(d == HGPM_OK, what + ": the density is still there");
                // P(k) of FP64 leaves the force grids alone until it has its spectrum
                if (failed && !f32 && call.solved && name == "P(k)" && at == 0)
                    check(f == HGPM_OK, what + ": the force is still there");
                hgpm_destroy(c);
                if (!failed) break;
            }
    }
}

// Every host array to and from the device and back, from the calling thread.
void round_trips(int ng, hgpm_ctx* f32, hgpm_ctx* f64, const std::string& what) {
    const size_t n = (size_t)ng * ng * ng;
    std::vector<double> x(3 * n), v(3 * n), a(3 * n), b(3 * n);
    for (size_t i = 0; i < 3 * n; i++) {
        x[i] = (double)(i % (16 * ng)) / 16.0;
        v[i] = (double)i;
    }
    check(hgpm_set_particles_f64(f64, x.data(), v.data()) == HGPM_OK, what + ": set FP64 particles");
    check(hgpm_get_particles_f64(f64, a.data(), b.data()) == HGPM_OK, what + ": get FP64 particles");
    check(a == x && b == v, what + ": FP64 particles");
    std::vector<int64_t> q(n), r(n);
    for (size_t i = 0; i < n; i++) q[i] = (int64_t)i * 3 - 7;
    check(hgpm_set_density(f32, q.data()) == HGPM_OK, what + ": set density");
    check(hgpm_get_density(f32, r.data()) == HGPM_OK, what + ": get density");
    check(q == r, what + ": density");
    std::vector<float> p(3 * n, 0.5f), w(3 * n, 0.25f);
    check(hgpm_set_particles(f32, p.data(), w.data()) == HGPM_OK, what + ": set particles");
    check(hgpm_get_particles(f32, p.data(), w.data()) == HGPM_OK, what + ": get particles");
    std::vector<float> g(2 * n);
    for (size_t i = 0; i < 2 * n; i++) g[i] = (float)(i % 1000);
    const std::vector<float> g0 = g;
    check(hgpm_fft_host(f32, g.data(), -1) == HGPM_OK, what + ": host FFT");
    check(g == g0, what + ": host FFT's grid"); // (the passes here leave it as it is)
}

// Contexts of two devices, used from threads whose current device is either.
void device() {
    for (int ng : {32, 64, 96}) {
        hgpm_ctx *f32[2], *f64[2];
        for (int d = 0; d < 2; d++) {
            (void)hipSetDevice(d);
            f32[d] = box(ng);
            f64[d] = box(ng, HGPM_FP64);
        }
        auto use = [&](int current) {
            for (int i = 0; i < 4; i++) {
                (void)hipSetDevice(current);
                const std::string what = std::to_string(ng) + "^3 device " + std::to_string(i % 2) + " from " + std::to_string(current);
                round_trips(ng, f32[i % 2], f64[i % 2], what);
                check(fake::device == current, what + ": the current device is left alone");
            }
        };
        use(0);
        use(1);
        std::thread other([&] { use(1); });
        other.join();
        for (int d = 0; d < 2; d++) {
            hgpm_destroy(f32[d]);
            hgpm_destroy(f64[d]);
        }
        (void)hipSetDevice(0);
    }
}

// A host that cannot pin memory, or make events: transfers take the runtime's own copy,
// and values out of range are refused all the same.
void unpinned() {
    for (int ng : {32, 64})
        for (int how = 0; how < 3; how++) {
            hgpm_ctx *f32 = box(ng), *f64 = box(ng, HGPM_FP64);
            const hgpm_params p = params(ng);
            hgpm_destroy(f32); // (and with the last context its idle rings)
            hgpm_destroy(f64);
            fake::no_pinned = how == 0;
            fake::events_left = how == 0 ? -1 : how == 1 ? 0 : 3;
            check(hgpm_create(&p, &f32) == HGPM_OK, "create");
            const hgpm_params p64 = params(ng, HGPM_FP64);
            check(hgpm_create(&p64, &f64) == HGPM_OK, "create FP64");
            const std::string what = std::to_string(ng) + "^3, way " + std::to_string(how);
            round_trips(ng, f32, f64, what);
            check(hipGetLastError() == hipSuccess, what + ": no error left for the next launch");
            check(hgpm_cic(f32) == HGPM_OK, what + ": a deposit after it");
            const size_t n3 = 3 * (size_t)ng * ng * ng;
            for (size_t at : {(size_t)0, n3 / 2, n3 - 1})
                for (int velocity = 0; velocity < 2; velocity++) {
                    std::vector<float> x(n3, 1.0f), v(n3, 1.0f);
                    (velocity ? v : x)[at] = velocity ? INFINITY : 1073741824.0f;
                    check(hgpm_set_particles(f32, x.data(), v.data()) == HGPM_ERR_ARG, what + ": refused");
                    check(strstr(hgpm_last_error(f32), ("index " + std::to_string(at / 3)).c_str()) != nullptr,
                          what + ": its index");
                }
            hgpm_destroy(f32);
            hgpm_destroy(f64);
            fake::no_pinned = false;
            fake::events_left = -1;
        }
}

// Transfers of every size at which the route changes, in one segment and in three, with
// and without a check, memory of each kind: the bytes arrive, the route is the one of the size.
void sizes() {
    const size_t MB = (size_t)1 << 20;
    hgpm_ctx* keep = box(32);
    std::vector<size_t> list = {4, 1000, MB - 4, MB, MB + 4, 2 * MB - 4, 2 * MB, 2 * MB + 4, 4 * MB,
                                16 * MB + 8, 32 * MB - 4, 32 * MB, 32 * MB + 4, 40 * MB + 12};
    for (size_t bytes : list)
        for (int parts : {1, 3})
            for (int rule = 0; rule < 10; rule++) {
                const int memory = fake::memory = rule / 3 % 3; // rule % 3: the check
                const bool scratch = rule == 9;
                std::vector<float> a(bytes / 4), b(bytes / 4), dev(bytes / 4);
                for (size_t i = 0; i < a.size(); i++) a[i] = (float)(i % 65521);
                hgpm::HostSeg up[3], down[3];
                size_t o = 0;
                for (int k = 0; k < parts; k++) { // uneven parts, none where there are no more bytes
                    const size_t m = k == parts - 1 ? a.size() - o : a.size() / (k + 3);
                    up[k] = {a.data() + o, dev.data() + o, 4 * m, rule % 3, scratch && k == 0};
                    down[k] = {b.data() + o, dev.data() + o, 4 * m};
                    o += m;
                }
                const std::string what = std::to_string(bytes) + " bytes in " + std::to_string(parts) + " check " + std::to_string(rule);
                int out = -2;
                fake::lo = (const char*)a.data();
                fake::hi = fake::lo + bytes;
                fake::direct = fake::copies = 0;
                check(hgpm::copy_to_device(up, parts, 0, nullptr, &out) == hipSuccess && out == -1, what + ": up");
                check(dev == a, what + ": on the device");
                const bool plain = rule % 3 == 0 && (memory == 2 || (bytes > MB && (bytes <= 32 * MB || scratch)));
                check(plain ? fake::direct == fake::copies : fake::direct == 0, what + ": route up");
                fake::lo = (const char*)b.data();
                fake::hi = fake::lo + bytes;
                fake::direct = fake::copies = 0;
                check(hgpm::copy_to_host(down, parts, 0, nullptr) == hipSuccess, what + ": down");
                check(b == a && fake::direct == (memory == 2 ? fake::copies : 0), what + ": back, and its route");
                check(hipGetLastError() == hipSuccess, what + ": no error left for the next launch");
                if (rule % 3) { // a bad value anywhere names its segment
                    for (size_t at : {(size_t)0, a.size() / 2, a.size() - 1}) {
                        const float was = a[at];
                        a[at] = rule % 3 == 1 ? NAN : -1073741824.0f;
                        int seg = 0;
                        while ((char*)&a[at] >= (char*)up[seg].host + up[seg].bytes) seg++;
                        check(hgpm::copy_to_device(up, parts, 0, nullptr, &out) == hipSuccess && out == seg, what + ": bad value");
                        a[at] = was;
                    }
                }
            }
    fake::memory = 0;
    hgpm_destroy(keep);
}
} // namespace

int main(int argc, char** argv) {
    const std::string s = argc > 1 ? argv[1] : "";
    if (s == "deposit") deposit();
    else if (s == "state") state();
    else if (s == "device") device();
    else if (s == "unpinned") unpinned();
    else if (s == "sizes") sizes();
    else return 3;
    printf("%d %d\n", cases, bad);
    return 0;
}
