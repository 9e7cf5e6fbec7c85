// hostcopy.cpp — copies between pageable host memory and the device (hostcopy.h).
#include "hostcopy.h"

#include <algorithm>
#include <atomic>
#include <cmath>
#include <cstring>
#include <exception>
#include <memory>
#include <mutex>
#include <new>
#include <thread>
#include <vector>

namespace hgpm {
namespace {
struct Piece {
    char *host, *dev;
    size_t bytes;
    int seg;
};
// Whether all of n bytes of floats pass the check, copied on the way with COPY (no early
// exit: the loop vectorises).
template <bool COPY> bool checked(char* to, const char* from, size_t n, int check) {
    if (check == 0) {
        if (COPY) memcpy(to, from, n);
        return true;
    }
    const size_t m = n / sizeof(float);
    const float* f = (const float*)from;
    float* t = (float*)to;
    int bad = 0;
    if (check == 1)
        for (size_t i = 0; i < m; i++) {
            if (COPY) t[i] = f[i];
            bad |= !(std::fabs(f[i]) <= 3.402823466e38f);
        }
    else
        for (size_t i = 0; i < m; i++) {
            if (COPY) t[i] = f[i];
            bad |= !(std::fabs(f[i]) < 1073741824.0f);
        }
    return !bad;
}
// A wait of a few microseconds to a millisecond for another thread's flag.
template <typename F> void wait_for(F&& done) {
    for (int i = 0; !done(); i++)
        if (i > 64) std::this_thread::yield();
}

constexpr int SLOTS = 8;
// 2 MB pieces: a transfer of its own costs about 9 us (1 MB pieces reach 38 GB/s one after
// the other, 4 MB ones 50, whole arrays 57), and the first piece's copy starts early
constexpr size_t SLOT = (size_t)2 << 20;
constexpr size_t KEPT = 2;
// Uploads without a check from 1 to 32 MB take the runtime's own copy, which pins the
// caller's pages and leaves out the copy to a slot.  Below, a slot is filled sooner than
// the pages are pinned; above, several threads fill slots faster than one thread pins.
// Runtime's copy / ring, us, memory just written: 1 MB 49 / 44, 2 MB 78 / 91, 4 MB 133 /
// 194, 8 MB 243 / 332, 16 MB 458 / 587, 24 MB 685 / 781, 32 MB 915-928 / 988-1031, 64 MB
// 2303 / 1812.  Downloads: 2 MB 123 / 114, 16 MB 947 / 612.
constexpr size_t PLAIN_MIN = (size_t)1 << 20, PLAIN_MAX = (size_t)32 << 20;

struct Ring {
    char* pin = nullptr; // SLOTS x SLOT bytes
    hipEvent_t ev[SLOTS] = {};
    int device = 0;
    ~Ring() {
        if (pin) (void)hipHostFree(pin);
        for (hipEvent_t e : ev)
            if (e) (void)hipEventDestroy(e);
    }
};
std::mutex g_mu;
// never destroyed: a process may end with contexts alive, after the runtime's own end
std::vector<std::unique_ptr<Ring>>& g_idle = []() -> std::vector<std::unique_ptr<Ring>>& {
    auto* v = new std::vector<std::unique_ptr<Ring>>;
    v->reserve(KEPT); // a ring is put back without an allocation
    return *v;
}();
int g_owners = 0;

// The device current for a scope: a ring's events belong to the device that they are made
// on, and a context may be used from a thread whose current device is another one.
class OnDevice {
public:
    explicit OnDevice(int device) {
        if (hipGetDevice(&was_) != hipSuccess || was_ == device) was_ = -1;
        else (void)hipSetDevice(device);
    }
    ~OnDevice() {
        if (was_ >= 0) (void)hipSetDevice(was_);
    }

private:
    int was_ = -1;
};

// A ring on a device, the current one, for one transfer; put back by its destructor.
class Lease {
public:
    hipError_t take(int dev) {
        {
            std::lock_guard<std::mutex> lock(g_mu);
            for (auto& r : g_idle)
                if (r->device == dev) {
                    std::swap(r, g_idle.back());
                    ring_ = std::move(g_idle.back());
                    g_idle.pop_back();
                    return hipSuccess;
                }
        }
        ring_.reset(new (std::nothrow) Ring);
        if (!ring_) return hipErrorOutOfMemory;
        ring_->device = dev;
        hipError_t e = hipHostMalloc((void**)&ring_->pin, SLOTS * SLOT, hipHostMallocDefault);
        if (e != hipSuccess) ring_->pin = nullptr;
        for (int i = 0; i < SLOTS && e == hipSuccess; i++) {
            e = hipEventCreateWithFlags(&ring_->ev[i], hipEventDisableTiming);
            if (e != hipSuccess) ring_->ev[i] = nullptr;
        }
        if (e != hipSuccess) ring_.reset();
        return e;
    }
    ~Lease() {
        if (!ring_) return;
        std::lock_guard<std::mutex> lock(g_mu);
        if (g_owners > 0 && g_idle.size() < KEPT) g_idle.push_back(std::move(ring_));
    }
    Ring& operator*() { return *ring_; }

private:
    std::unique_ptr<Ring> ring_;
};

// The segments one after the other through the runtime's own copy.
hipError_t move_plain(const HostSeg* seg, int n, hipStream_t st, bool up, int* bad) {
    hipError_t e = hipSuccess;
    for (int k = 0; k < n && e == hipSuccess; k++) {
        if (up && bad && *bad < 0 && !checked<false>(nullptr, (const char*)seg[k].host, seg[k].bytes, seg[k].check))
            *bad = k;
        e = up ? hipMemcpyAsync(seg[k].dev, seg[k].host, seg[k].bytes, hipMemcpyHostToDevice, st)
               : hipMemcpyAsync(seg[k].host, seg[k].dev, seg[k].bytes, hipMemcpyDeviceToHost, st);
    }
    const hipError_t w = hipStreamSynchronize(st);
    return e == hipSuccess ? w : e;
}

// Memory the device reads and writes by itself: page-locked, managed or its own.
bool reachable(const void* p) {
    hipPointerAttribute_t a;
    if (hipPointerGetAttributes(&a, p) != hipSuccess) {
        (void)hipGetLastError(); // pageable, to some versions of the runtime
        return false;
    }
    return a.type != hipMemoryTypeUnregistered;
}

hipError_t move(const HostSeg* seg, int n, int device, hipStream_t st, bool up, int* bad) {
    if (bad) *bad = -1;
    size_t total = 0;
    for (int s = 0; s < n; s++) total += seg[s].bytes;
    if (!total) return hipSuccess;
    bool check = false, direct = true, scratch = false;
    for (int s = 0; s < n; s++) {
        check = check || seg[s].check;
        scratch = scratch || seg[s].scratch;
    }
    for (int s = 0; s < n && direct; s++) direct = !seg[s].bytes || reachable(seg[s].host);
    // a checked upload keeps the ring, whose threads check: 128^3 particles from page-locked
    // memory 1.4 against 2.8 ms
    // scratch: read by other cores, it would be slower to write again than the ring saves
    // (128^3 particles in the split layout: written in 9.4 and moved in 1.9 ms, through the
    // ring 11.6 and 1.5)
    if (!check && (direct || (up && total > PLAIN_MIN && (total <= PLAIN_MAX || scratch))))
        return move_plain(seg, n, st, up, bad);
    OnDevice on(device);
    Lease lease;
    hipError_t e = lease.take(device);
    if (e != hipSuccess) { // no ring to be had (a limit on pinned memory): without one
        (void)hipGetLastError();
        return move_plain(seg, n, st, up, bad);
    }
    Ring& r = *lease;
    auto slot = [&](int i) { return r.pin + (size_t)(i % SLOTS) * SLOT; };
    if (total <= SLOT) {
        // small: every segment in one slot, without threads
        const hipMemcpyKind kind = up ? hipMemcpyHostToDevice : hipMemcpyDeviceToHost;
        size_t o = 0;
        for (int k = 0; k < n && e == hipSuccess; o += seg[k++].bytes) {
            char* at = r.pin + o;
            if (up && !checked<true>(at, (const char*)seg[k].host, seg[k].bytes, seg[k].check) && bad && *bad < 0) *bad = k;
            e = up ? hipMemcpyAsync(seg[k].dev, at, seg[k].bytes, kind, st)
                   : hipMemcpyAsync(at, seg[k].dev, seg[k].bytes, kind, st);
        }
        const hipError_t w = hipStreamSynchronize(st); // nothing in flight from or to the ring
        if (e == hipSuccess) e = w;
        o = 0;
        for (int k = 0; k < n && e == hipSuccess && !up; o += seg[k++].bytes) memcpy(seg[k].host, r.pin + o, seg[k].bytes);
        return e;
    }
    std::vector<Piece> p;
    for (int s = 0; s < n; s++)
        for (size_t o = 0; o < seg[s].bytes; o += SLOT)
            p.push_back(Piece{(char*)seg[s].host + o, (char*)seg[s].dev + o,
                              seg[s].bytes - o < SLOT ? seg[s].bytes - o : SLOT, s});
    const int np = (int)p.size();
    // the calling thread queues the transfers in order; piece i uses slot i mod SLOTS
    std::vector<std::atomic<int>> copied(np); // its memory copy is done
    for (auto& c : copied) c.store(0, std::memory_order_relaxed);
    std::atomic<int> queued{0}, next{0}, first_bad{n}, failed{0};
    auto transfer = [&](int i) {
        hipError_t q = up ? hipMemcpyAsync(p[i].dev, slot(i), p[i].bytes, hipMemcpyHostToDevice, st)
                          : hipMemcpyAsync(slot(i), p[i].dev, p[i].bytes, hipMemcpyDeviceToHost, st);
        if (q == hipSuccess) q = hipEventRecord(r.ev[i % SLOTS], st);
        return q;
    };
    // the memory copy of piece i; up: once the slot's last transfer has left it, down: once
    // its own has arrived
    auto copy = [&](int i) {
        const int wait = up ? i - SLOTS : i;
        if (wait >= 0) {
            wait_for([&] { return queued.load(std::memory_order_acquire) > wait || failed.load(); });
            if (failed.load()) return;
            if (hipEventSynchronize(r.ev[i % SLOTS]) != hipSuccess) failed.store(1);
        }
        if (up) {
            if (!checked<true>(slot(i), p[i].host, p[i].bytes, seg[p[i].seg].check)) {
                int b = first_bad.load();
                while (p[i].seg < b && !first_bad.compare_exchange_weak(b, p[i].seg)) {}
            }
        } else
            memcpy(p[i].host, slot(i), p[i].bytes);
        copied[i].store(1, std::memory_order_release);
    };
    // what is queued before the transfer is waited for here, not by every thread
    if (!up && (e = hipStreamSynchronize(st)) != hipSuccess) return e;
    auto work = [&](int device) {
        (void)hipSetDevice(device);
        for (int i = next.fetch_add(1); i < np && !failed.load(); i = next.fetch_add(1)) copy(i);
    };
    // a thread per piece, as many as there are slots at most
    const unsigned hw = std::thread::hardware_concurrency();
    const int nt = std::max(1, std::min({SLOTS, np, hw ? (int)hw : 1}));
    std::vector<std::thread> team;
    team.reserve(nt);
    try {
        for (int t = 0; t < nt; t++) team.emplace_back(work, r.device);
    } catch (const std::exception&) { // no more threads: those there are do
    }
    for (int i = 0; i < np && e == hipSuccess; i++) {
        if (team.empty() && up) copy(i);
        const int need = up ? i : i - SLOTS;
        if (need >= 0) wait_for([&] { return copied[need].load(std::memory_order_acquire) || failed.load(); });
        e = failed.load() ? hipErrorUnknown : transfer(i);
        queued.store(i + 1, std::memory_order_release);
        if (team.empty() && !up && e == hipSuccess) copy(i);
    }
    if (e != hipSuccess) failed.store(1);
    for (auto& t : team) t.join();
    if (e == hipSuccess && up) e = hipStreamSynchronize(st);
    if (e == hipSuccess && failed.load()) e = hipErrorUnknown;
    if (e != hipSuccess) (void)hipStreamSynchronize(st); // nothing in flight from or to the ring
    if (bad && first_bad.load() < n) *bad = first_bad.load();
    return e;
}
} // namespace

hipError_t copy_to_host(const HostSeg* seg, int n, int device, hipStream_t st) {
    return move(seg, n, device, st, false, nullptr);
}
hipError_t copy_to_device(const HostSeg* seg, int n, int device, hipStream_t st, int* bad) {
    return move(seg, n, device, st, true, bad);
}

void host_copy_add_owner() {
    std::lock_guard<std::mutex> lock(g_mu);
    g_owners++;
}
void host_copy_release_owner() {
    std::vector<std::unique_ptr<Ring>> gone; // freed outside the lock
    std::lock_guard<std::mutex> lock(g_mu);
    if (--g_owners == 0) gone.swap(g_idle);
}
} // namespace hgpm
