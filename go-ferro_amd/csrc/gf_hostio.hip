// gf_hostio.hip — device to host copies of a context's fields.
//
// A caller's buffer is most often ordinary memory: a direct copy into it goes
// through the runtime's own staging on one thread, and a buffer just allocated is
// faulted in page by page on that thread: 10 GB/s, 20 ms for the three
// components of a 256x256x128 field.  Here the copies land in pinned slots
// of 1 MiB, and from 8 MiB on several threads move them on, each with two
// slots of its own, so that the faults run in parallel and a slot's copy
// overlaps the move of the other: 40 steps of that film with the read-back
// 121 -> 108 ms.  A field of up to one slot takes one wait and one move where the
// direct copies wait for each part: three parts of 8 KB 46 -> 20 us, nine of 8 KB
// 139 -> 44 (16x16x8, one step with its average, whose sums go to pinned memory,
// and read-back 148 -> 107).  From 64 KiB to 2 MiB both take the same time into
// memory in use (34 and 36 us for 192 KB, 88 and 86 for 1.5 MB), but not into new
// memory: the first read-back of 96 antiferromagnets, 192 fields of 1.3 MB on
// average, makes their 100 steps 182 ms directly and 155 through the slots.
//
// The slots are shared by the process's contexts: at most kSlots of them,
// allocated when they pay and given back with the last context.  A slot takes
// about 0.1 ms to allocate and free again, and saves 26 us of a small field, 20 to
// 120 us of a MB of a larger one: a program that reads one field and ends is
// slower for it (12.6 MB: first read-back 0.79 -> 1.54 ms, end of the context 4.4
// -> 5.3 ms).  So slots come with the fourth read-back of up to a slot, or once
// kPays bytes have been read for each slot needed; what came before copied
// directly.
//
// One call holds the slots at a time.  A call that finds them held (another
// thread's) copies directly, as does one that cannot allocate one, and one into
// memory the runtime knows, which the caller pinned (201 MB in 3.6 ms, 6.6
// through the slots; 1.4 MB 53 us and 82).  What a copy, or the work queued
// before it, fails with is the call's error.
#include <algorithm>
#include <atomic>
#include <cstring>
#include <mutex>
#include <thread>

#include "gf_internal.h"

namespace gf {

namespace {

constexpr size_t kSlotBytes = size_t{1} << 20;
constexpr int kThreads = 8;
constexpr int kSlots = 2 * kThreads;
constexpr size_t kThreadsFrom = size_t{8} << 20;
constexpr int kParts = 9;         // most arrays of a field
constexpr int kPaysCalls = 4;
constexpr size_t kPays = size_t{2} << 20;

std::mutex g_slots_lock;          // held while the slots are used or freed
std::mutex g_users_lock;
int64_t g_users = 0;              // contexts alive
char* g_slot[kSlots] = {};
int g_reads = 0;                  // read-backs that found no slot since they were last given back
size_t g_bytes = 0;

// The parts of a field one after another in host memory, as chunks of at most
// a slot.
struct Chunk {
    const char* src;
    char* dst;
    size_t bytes;
};
struct Chunks {
    const double* const* src;
    const int64_t* count;
    int parts;
    double* host;
    int first[kParts + 1] = {};   // of a part; the last is the number of all

    Chunks(const double* const* s, const int64_t* n, int p, double* h) : src(s), count(n), parts(p), host(h) {
        for (int q = 0; q < p; q++) first[q + 1] = first[q] + static_cast<int>((bytes(q) + kSlotBytes - 1) / kSlotBytes);
    }
    size_t bytes(int part) const { return sizeof(double) * static_cast<size_t>(count[part]); }
    int size() const { return first[parts]; }
    Chunk operator[](int i) const {
        int q = 0;
        char* dst = reinterpret_cast<char*>(host);
        for (; i >= first[q + 1]; q++) dst += bytes(q);
        const size_t o = static_cast<size_t>(i - first[q]) * kSlotBytes;
        return {reinterpret_cast<const char*>(src[q]) + o, dst + o, std::min(kSlotBytes, bytes(q) - o)};
    }
};

// The context's device while events are made for its stream, and the
// caller's again after it.
struct OnDevice {
    int was = -1;
    explicit OnDevice(int device) {
        if (hipGetDevice(&was) != hipSuccess || was == device || hipSetDevice(device) != hipSuccess) was = -1;
    }
    ~OnDevice() {
        if (was >= 0) (void)hipSetDevice(was);
    }
};

// A point of the stream to wait for: an event, or where none can be had the
// stream's end.
struct Mark {
    hipEvent_t e = nullptr;
    hipError_t set(hipStream_t s) {
        if (!e && hipEventCreateWithFlags(&e, hipEventDisableTiming) != hipSuccess) {
            e = nullptr;
            (void)hipGetLastError();   // not the next launch's error
        }
        return e ? hipEventRecord(e, s) : hipSuccess;
    }
    hipError_t wait(hipStream_t s) const { return e ? hipEventSynchronize(e) : hipStreamSynchronize(s); }
    ~Mark() {
        if (e) (void)hipEventDestroy(e);
    }
};

// The first n slots for a field of `total` bytes, allocated where they are not
// yet; false when they do not pay yet or cannot be had.
bool have_slots(int n, size_t total) {
    if (g_slot[n - 1]) return true;
    g_reads++;
    g_bytes += total;
    if (!(n == 1 && g_reads >= kPaysCalls) && g_bytes / static_cast<size_t>(n) < kPays) return false;
    for (int i = 0; i < n; i++)
        if (!g_slot[i] && hipHostMalloc(reinterpret_cast<void**>(&g_slot[i]), kSlotBytes, hipHostMallocPortable) != hipSuccess) {
            g_slot[i] = nullptr;
            return false;
        }
    return true;
}

// Chunks w, w + workers, ... through the slots w and w + workers.
hipError_t move_chunks(const Chunks& chunks, int w, int workers, hipStream_t s) {
    Mark done[2];
    hipError_t e = hipSuccess;
    auto send = [&](int i, int b) {
        const Chunk k = chunks[i];
        e = hipMemcpyAsync(g_slot[w + b * workers], k.src, k.bytes, hipMemcpyDeviceToHost, s);
        if (e == hipSuccess) e = done[b].set(s);
    };
    const int n = chunks.size();
    for (int b = 0; b < 2 && w + b * workers < n && e == hipSuccess; b++) send(w + b * workers, b);
    int b = 0;
    for (int i = w; i < n && e == hipSuccess; i += workers, b ^= 1) {
        if ((e = done[b].wait(s)) != hipSuccess) break;
        const Chunk k = chunks[i];
        std::memcpy(k.dst, g_slot[w + b * workers], k.bytes);
        if (i + 2 * workers < n) send(i + 2 * workers, b);
    }
    // no copy into a slot is left behind when a call fails
    if (e != hipSuccess) (void)hipStreamSynchronize(s);
    return e;
}

hipError_t move_large(const Chunks& chunks, int workers, int device, hipStream_t s) {
    // the work queued before is waited for once, not by every thread
    hipError_t e = workers > 1 ? hipStreamSynchronize(s) : hipSuccess;
    if (e != hipSuccess) return e;
    std::atomic<int> failed{hipSuccess};
    auto work = [&](int w) {
        hipError_t r = w ? hipSetDevice(device) : hipSuccess;
        if (r == hipSuccess) r = move_chunks(chunks, w, workers, s);
        int none = hipSuccess;
        if (r != hipSuccess) failed.compare_exchange_strong(none, static_cast<int>(r));
    };
    std::thread pool[kThreads];
    int started = 1;
    try {
        for (; started < workers; started++) pool[started] = std::thread(work, started);
    } catch (...) {
        // no more threads: this one does what they would have
    }
    work(0);
    for (int w = started; w < workers; w++) work(w);
    for (std::thread& t : pool)
        if (t.joinable()) t.join();
    return static_cast<hipError_t>(failed.load());
}

// A field of at most one slot: its parts into it, one wait, one move.
hipError_t move_small(const Chunks& chunks, hipStream_t s) {
    char* const slot = g_slot[0];
    hipError_t e = hipSuccess;
    size_t o = 0;
    for (int i = 0; i < chunks.size() && e == hipSuccess; i++) {
        const Chunk k = chunks[i];
        e = hipMemcpyAsync(slot + o, k.src, k.bytes, hipMemcpyDeviceToHost, s);
        o += k.bytes;
    }
    const hipError_t w = hipStreamSynchronize(s);   // also after a failure: no copy into the slot is left behind
    if (e == hipSuccess) e = w;
    if (e == hipSuccess) std::memcpy(chunks.host, slot, o);   // the parts lie one after another there too
    return e;
}

// Through the slots, with the result in *e; false, with nothing copied, when
// they do not pay yet or a slot cannot be had.
bool through_slots(gf_ctx* c, const Chunks& chunks, size_t total, hipError_t* e) {
    if (total <= kSlotBytes) {
        if (!have_slots(1, total)) return false;
        *e = move_small(chunks, c->stream);
        return true;
    }
    const int workers = total < kThreadsFrom ? 1 : kThreads, slots = std::min(2 * workers, chunks.size());
    const OnDevice here(c->device);
    if (!have_slots(slots, total)) return false;
    *e = move_large(chunks, workers, c->device, c->stream);
    return true;
}

// Memory the caller pinned, or a device's: a copy engine writes to it directly.
bool known_memory(const void* p) {
    hipPointerAttribute_t a{};
    if (hipPointerGetAttributes(&a, p) == hipSuccess) return a.type != hipMemoryTypeUnregistered;
    (void)hipGetLastError();   // an address the runtime does not know
    return false;
}

}  // namespace

void host_slots_retain() {
    std::lock_guard<std::mutex> g(g_users_lock);
    g_users++;
}

void host_slots_release() {
    std::lock_guard<std::mutex> g(g_users_lock);
    if (--g_users > 0) return;
    std::lock_guard<std::mutex> h(g_slots_lock);
    for (char*& p : g_slot) {
        if (p) (void)hipHostFree(p);
        p = nullptr;
    }
    g_reads = 0;
    g_bytes = 0;
}

// A kernel's partial sums straight in pinned memory save the copy after it, 11
// us (16x16x8: 26 us an average, 15 without it), and the memory takes 25 to 190 us
// to allocate: from the fourth average on.
double* host_sums(gf_ctx* c) {
    if (c->red_host || ++c->red_calls < kPaysCalls) return c->red_host;
    c->red_calls = 0;
    if (hipHostMalloc(reinterpret_cast<void**>(&c->red_host), sizeof(double) * 3 * static_cast<size_t>(c->red_blocks),
                      hipHostMallocDefault) != hipSuccess) {
        c->red_host = nullptr;
        (void)hipGetLastError();   // not the next launch's error
    }
    return c->red_host;
}

gf_status download_parts(gf_ctx* c, const double* const* src, const int64_t* count, int parts, double* host) {
    const Chunks chunks(src, count, parts, host);
    size_t total = 0;
    for (int p = 0; p < parts; p++) total += chunks.bytes(p);
    std::unique_lock<std::mutex> held(g_slots_lock, std::defer_lock);
    if (!known_memory(host)) (void)held.try_lock();
    hipError_t e = hipSuccess;
    if (held.owns_lock()) {
        // an error of a copy or of the work before it is the call's
        if (through_slots(c, chunks, total, &e)) return hip_check(c, e, "download");
        (void)hipGetLastError();   // what made the slots unusable is not the next launch's error
    }
    double* dst = host;
    for (int p = 0; p < parts && e == hipSuccess; p++) {
        e = hipMemcpyAsync(dst, src[p], chunks.bytes(p), hipMemcpyDeviceToHost, c->stream);
        dst += count[p];
    }
    const hipError_t w = hipStreamSynchronize(c->stream);   // also after a failure: no copy into the caller's is left behind
    const gf_status st = hip_check(c, e, "download");
    return st ? st : hip_check(c, w, "download sync");
}

}  // namespace gf
