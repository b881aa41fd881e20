// The read-back of fields (gf_hostio.hip) over a HIP runtime of this file's
// own: copies are noted and done only when something waits for them, and any
// call can be made to fail.  Host code only, no GPU.
#include <dlfcn.h>
#include <pthread.h>

#include <algorithm>
#include <cstdio>
#include <cstdlib>
#include <cstring>
#include <new>
#include <string>

#include "../../go-ferro_amd/csrc/gf_hostio.hip"

// ------------------------------------------------------------ the runtime
namespace {

struct Pending {
    void* dst;
    const void* src;
    size_t bytes;
};
std::mutex g_rt;
std::vector<Pending> g_queue;      // of the one stream, oldest first
size_t g_done = 0;
int g_mallocs = 0, g_frees = 0, g_events = 0;
size_t g_to_slots = 0;             // copies whose destination a slot is
hipError_t g_last = hipSuccess;
hipMemoryType g_type = hipMemoryTypeUnregistered;   // of the caller's buffer
bool g_known = true;                                // the runtime answers for it
thread_local int t_device = 0;

// The call that fails: the `at`-th of the named kind from now on, every
// later one too when `on` is set.
struct Fail {
    const char* what = "";
    int at = -1;
    bool on = false;
    hipError_t e = hipSuccess;
} g_fail;

hipError_t may_fail(const char* what) {
    if (std::strcmp(what, g_fail.what)) return hipSuccess;
    const int at = g_fail.at--;
    if (at == 0 || (at < 0 && g_fail.on)) return g_last = g_fail.e;
    return hipSuccess;
}

void finish(size_t upto) {
    for (; g_done < upto; g_done++) std::memcpy(g_queue[g_done].dst, g_queue[g_done].src, g_queue[g_done].bytes);
}

struct FakeEvent {
    size_t upto;
    int device;
};

}  // namespace

#define GF_FAKE(what)                                  \
    std::lock_guard<std::mutex> lock(g_rt);            \
    if (hipError_t e_ = may_fail(what)) return e_

extern "C" {
hipError_t hipHostMalloc(void** p, size_t n, unsigned) {
    GF_FAKE("hipHostMalloc");
    *p = std::malloc(n);
    std::memset(*p, 0xA5, n);
    g_mallocs++;
    return hipSuccess;
}
hipError_t hipHostFree(void* p) {
    std::lock_guard<std::mutex> lock(g_rt);
    std::free(p);
    g_frees++;
    return hipSuccess;
}
hipError_t hipMemcpyAsync(void* dst, const void* src, size_t n, hipMemcpyKind, hipStream_t) {
    GF_FAKE("hipMemcpyAsync");
    g_queue.push_back({dst, src, n});
    for (char* s : gf::g_slot)
        if (s && dst >= s && dst < s + gf::kSlotBytes) g_to_slots++;
    return hipSuccess;
}
hipError_t hipEventCreateWithFlags(hipEvent_t* e, unsigned) {
    GF_FAKE("hipEventCreateWithFlags");
    *e = static_cast<hipEvent_t>(std::malloc(sizeof(FakeEvent)));
    *reinterpret_cast<FakeEvent*>(*e) = {0, t_device};
    g_events++;
    return hipSuccess;
}
hipError_t hipEventDestroy(hipEvent_t e) {
    std::lock_guard<std::mutex> lock(g_rt);
    std::free(e);
    g_events--;
    return hipSuccess;
}
hipError_t hipEventRecord(hipEvent_t e, hipStream_t) {
    GF_FAKE("hipEventRecord");
    FakeEvent* f = reinterpret_cast<FakeEvent*>(e);
    if (f->device != 1) return g_last = hipErrorInvalidHandle;   // the stream is device 1's
    f->upto = g_queue.size();
    return hipSuccess;
}
hipError_t hipEventSynchronize(hipEvent_t e) {
    GF_FAKE("hipEventSynchronize");
    finish(reinterpret_cast<FakeEvent*>(e)->upto);
    return hipSuccess;
}
hipError_t hipStreamSynchronize(hipStream_t) {
    GF_FAKE("hipStreamSynchronize");
    finish(g_queue.size());
    return hipSuccess;
}
hipError_t hipPointerGetAttributes(hipPointerAttribute_t* a, const void*) {
    if (!g_known) return g_last = hipErrorInvalidValue;
    a->type = g_type;
    return hipSuccess;
}
hipError_t hipGetDevice(int* d) { *d = t_device; return hipSuccess; }
hipError_t hipSetDevice(int d) { t_device = d; return hipSuccess; }
hipError_t hipGetLastError() {
    std::lock_guard<std::mutex> lock(g_rt);
    return std::exchange(g_last, hipSuccess);
}
}

namespace gf {
gf_status set_error(gf_ctx*, gf_status code, const std::string&) { return code; }
gf_status hip_check(gf_ctx*, hipError_t e, const char*) { return e == hipSuccess ? GF_OK : GF_ERR_HIP; }
}  // namespace gf

// Allocations and threads that fail: the n-th from now on (-1: none).
static std::atomic<int> g_new_in{-1}, g_thread_in{-1};

void* operator new(size_t n) {
    int left = g_new_in.load();
    if (left >= 0 && g_new_in.fetch_sub(1) == 0) throw std::bad_alloc();
    if (void* p = std::malloc(n)) return p;
    throw std::bad_alloc();
}
void operator delete(void* p) noexcept { std::free(p); }
void operator delete(void* p, size_t) noexcept { std::free(p); }

extern "C" int pthread_create(pthread_t* t, const pthread_attr_t* a, void* (*f)(void*), void* x) {
    using Create = int (*)(pthread_t*, const pthread_attr_t*, void* (*)(void*), void*);
    static const Create real = reinterpret_cast<Create>(dlsym(RTLD_NEXT, "pthread_create"));
    return g_thread_in >= 0 && g_thread_in.fetch_sub(1) == 0 ? EAGAIN : real(t, a, f, x);
}

// ------------------------------------------------------------ the cases
namespace {

struct Field {
    std::vector<std::vector<double>> parts;
    std::vector<const double*> src;
    std::vector<int64_t> count;
    std::vector<double> want, host;
    explicit Field(std::vector<int64_t> n) : count(n) {
        double v = 0.5;
        for (int64_t k : n) {
            parts.emplace_back(static_cast<size_t>(k));
            for (double& x : parts.back()) x = v += 1.25;
        }
        for (const auto& p : parts) {
            src.push_back(p.data());
            want.insert(want.end(), p.begin(), p.end());
        }
        host.assign(want.size(), -1.);
    }
    gf_status read(gf_ctx& c) {
        std::fill(host.begin(), host.end(), -1.);
        return gf::download_parts(&c, src.data(), count.data(), static_cast<int>(src.size()), host.data());
    }
    bool whole() const { return host == want; }
};

// one double; fields below and above a slot; parts of a slot,
// of one double less and more; the threads' threshold; staggered parts; nine
const std::vector<std::vector<int64_t>> kFields = {
    {1, 1, 1}, {2730, 2731, 2730}, {2731, 2731, 2731}, {43690, 43690, 43690}, {87381, 87381, 87381},
    {87381, 87381, 87382}, {131072, 131073, 131071}, {349525, 349525, 349525}, {349526, 349525, 349526},
    {1400011, 1400009, 1400010}, {7, 140000, 900001}, {131072, 1, 131072, 1, 1, 1, 1, 1, 200000},
    {5000, 5000, 5000, 5000, 5000, 5000, 5000, 5000, 5000}};

size_t bytes_of(const std::vector<int64_t>& n) {
    size_t b = 0;
    for (int64_t k : n) b += sizeof(double) * static_cast<size_t>(k);
    return b;
}
void clear() {
    g_fail = Fail{};
    g_queue.clear();
    g_queue.reserve(4096);   // no allocation of the runtime's counts below
    g_done = 0;
    g_to_slots = 0;
    g_last = hipSuccess;
    g_new_in = -1;
    g_thread_in = -1;
    g_type = hipMemoryTypeUnregistered;
    g_known = true;
}

int bad(const char* what, const Field& f, int k) {
    std::printf("%s: field of %zu doubles, %d\n", what, f.want.size(), k);
    return 1;
}

// Reads until a read goes through the slots, and counts the reads before it.
int warm(Field& f, gf_ctx& c) {
    for (int k = 0; k < 16; k++) {
        clear();
        if (f.read(c) || !f.whole() || g_last) return -1;
        if (g_to_slots) return k;
    }
    return -1;
}

int whole() {
    for (const auto& n : kFields) {
        Field f(n);
        for (int device : {0, 1}) {   // the caller's current device, the context's or not
            gf_ctx c;
            c.device = t_device = 1;
            if (warm(f, c) < 0) return bad("no slot used", f, device);
            for (int r = 0; r < 3; r++) {
                clear();
                t_device = device;
                g_known = r != 1;
                if (f.read(c) || !f.whole() || g_last || g_done != g_queue.size()) return bad("whole", f, r);
                if (t_device != device || g_events) return bad("left behind", f, r);
                if (g_to_slots == 0) return bad("no slot used", f, device);
            }
        }
        if (g_mallocs != g_frees) return bad("slots not given back", f, g_mallocs - g_frees);
    }
    return 0;
}

// One read-back, or a few small ones, allocate nothing; the slots come when
// the rule says so, serve other contexts and go with the last one.
int pays() {
    for (const auto& n : kFields) {
        Field f(n);
        const size_t bytes = bytes_of(n);
        const int before = g_mallocs;
        {
            gf_ctx a, b;
            a.device = b.device = t_device = 1;
            const int reads = warm(f, a);
            int chunks = 0;
            for (int64_t k : n) chunks += static_cast<int>((sizeof(double) * k + gf::kSlotBytes - 1) / gf::kSlotBytes);
            const size_t slots = bytes <= gf::kSlotBytes ? 1 : std::min(bytes < gf::kThreadsFrom ? 2 : gf::kSlots, chunks);
            const int paid = static_cast<int>((slots * gf::kPays + bytes - 1) / bytes) - 1;
            const int want = slots == 1 ? std::min(paid, gf::kPaysCalls - 1) : paid;
            if (reads != want || g_mallocs - before != static_cast<int>(slots)) return bad("pays", f, reads);
            if (warm(f, b) != 0) return bad("another context", f, 0);
        }
        if (g_frees != g_mallocs) return bad("given back", f, 0);
    }
    return 0;
}

// A buffer the caller pinned, or a device's: one copy a part, straight into it.
int known() {
    for (hipMemoryType type : {hipMemoryTypeHost, hipMemoryTypeDevice, hipMemoryTypeManaged})
        for (const auto& n : kFields) {
            Field f(n);
            gf_ctx c;
            c.device = t_device = 1;
            clear();
            g_type = type;
            const int before = g_mallocs;
            if (f.read(c) || !f.whole() || g_to_slots || g_mallocs != before || g_queue.size() != n.size())
                return bad("known memory", f, type);
        }
    return 0;
}

// A slot that cannot be had: a direct copy; an event: a wait for the stream; and
// no error left.
int unavailable() {
    for (const char* what : {"hipHostMalloc", "hipEventCreateWithFlags"})
        for (const auto& n : kFields)
            for (int at = 0; at < 16; at += 5) {
                Field f(n);
                gf_ctx c;
                c.device = t_device = 1;
                for (int r = 0; r < 12; r++) {
                    clear();
                    g_fail = {what, at, true, hipErrorOutOfMemory};
                    if (f.read(c) || !f.whole() || g_last || g_events) return bad(what, f, at);
                }
            }
    return 0;
}

// A copy, a record or a wait that fails, also once: the call's error, and
// nothing on its way into a slot.
int errors() {
    for (const char* what : {"hipMemcpyAsync", "hipEventRecord", "hipEventSynchronize", "hipStreamSynchronize"})
        for (const auto& n : kFields)
            for (int at = 0; at < 40; at += 1 + at / 2) {
                Field f(n);
                gf_ctx c;
                c.device = t_device = 1;
                if (warm(f, c) < 0) return bad("no slot used", f, at);
                clear();
                g_fail = {what, at, false, hipErrorLaunchFailure};
                const gf_status st = f.read(c);
                const bool reached = g_fail.at < 0;
                if (reached != (st == GF_ERR_HIP) || (!reached && !f.whole())) return bad(what, f, at);
                if (g_events || (g_done != g_queue.size() && std::strcmp(what, "hipStreamSynchronize")))
                    return bad("left behind", f, at);
            }
    return 0;
}

// Host memory or threads that run out: no exception leaves the call.
int host_limits() {
    for (std::atomic<int>* limit : {&g_new_in, &g_thread_in})
        for (const auto& n : kFields)
            for (int at = 0; at < 12; at++) {
                Field f(n);
                gf_ctx c;
                c.device = t_device = 1;
                if (warm(f, c) < 0) return bad("no slot used", f, at);
                clear();
                *limit = at;
                const gf_status st = f.read(c);
                *limit = -1;
                if (st || !f.whole()) return bad(limit == &g_new_in ? "operator new" : "pthread_create", f, at);
            }
    return 0;
}

// The slots in another thread's hands: a direct copy at once.
int contended() {
    for (const auto& n : kFields) {
        Field f(n);
        gf_ctx c;
        c.device = t_device = 1;
        if (warm(f, c) < 0) return bad("no slot used", f, 0);
        clear();
        std::atomic<int> step{0};
        std::thread other([&] {
            std::lock_guard<std::mutex> held(gf::g_slots_lock);
            step = 1;
            while (step != 2) std::this_thread::yield();
        });
        while (step != 1) std::this_thread::yield();
        const gf_status st = f.read(c);
        step = 2;
        other.join();
        if (st || !f.whole() || g_to_slots) return bad("contended", f, 0);
    }
    return 0;
}

// Pinned sums from the fourth average on; null, with no error left, while
// they cannot be had.
int sums() {
    for (int fails = 0; fails < 3; fails++) {
        gf_ctx c;
        c.red_blocks = 7;
        clear();
        g_fail = {"hipHostMalloc", 0, true, hipErrorOutOfMemory};
        for (int call = 1; call <= 40; call++) {
            if (call == 4 * fails + 1) g_fail = Fail{};
            const double* p = gf::host_sums(&c);
            if ((p != nullptr) != (call >= 4 * (fails + 1)) || g_last) {
                std::printf("sums: call %d after %d failures\n", call, fails);
                return 1;
            }
        }
        hipHostFree(c.red_host);
    }
    return 0;
}

}  // namespace

int main(int argc, char** argv) {
    const std::string what = argc > 1 ? argv[1] : "";
    if (what == "whole") return whole();
    if (what == "pays") return pays();
    if (what == "sums") return sums();
    if (what == "known") return known();
    if (what == "unavailable") return unavailable();
    if (what == "errors") return errors();
    if (what == "host_limits") return host_limits();
    if (what == "contended") return contended();
    std::printf("unknown case %s\n", what.c_str());
    return 2;
}
