// gf_hostio.hip — device to host copies of a context's fields.
//
// A caller's buffer is ordinary memory: a direct copy into it goes through
// the runtime's own staging on one thread, and a buffer just allocated is
// faulted in page by page on that thread: 10 GB/s, 20 ms for the three
// components of a 256x256x128 field.  Here the copies land in pinned slots
// of 1 MiB, and from 8 MiB on several threads move them on, each with two
// slots of its own, so that the faults run in parallel and a slot's copy
// overlaps the move of the other: 40 steps of that film with the read-back
// 121 -> 108 ms.  A field of up to one slot takes one wait and one move where
// the direct copies wait for each component: 16x16x8, one step with its average
// (whose partial sums go to pinned memory) and read-back 148 -> 107 us; 30x20x30
// antiferromagnet, 10 steps 344 -> 335 us (369 with an event per component).
//
// The slots are shared by the process's contexts: at most kSlots of them,
// allocated when first needed and given back with the last context.  One
// call holds them at a time; a call that finds them held (another thread's)
// copies directly, as does one whose slot cannot be allocated.
#include <algorithm>
#include <atomic>
#include <cstring>
#include <mutex>
#include <system_error>
#include <thread>
#include <vector>

#include "gf_internal.h"

namespace gf {

namespace {

constexpr size_t kSlotBytes = size_t{1} << 20;
constexpr int kThreads = 8;
constexpr int kSlots = 2 * kThreads;
constexpr size_t kThreadsFrom = size_t{8} << 20;

std::mutex g_slots_lock;          // held while the slots are used or freed
std::mutex g_users_lock;
int64_t g_users = 0;              // contexts alive
char* g_slot[kSlots] = {};

struct Chunk {
    const char* src;
    char* dst;
    size_t bytes;
};

// Chunks w, w + workers, ... through the slots w, w + workers, ... below
// 2 * workers.
hipError_t move_chunks(const std::vector<Chunk>& chunks, int w, int workers, hipStream_t s) {
    hipEvent_t ev[2] = {nullptr, nullptr};
    hipError_t e = hipSuccess;
    auto send = [&](size_t i, int b) {
        char*& slot = g_slot[w + b * workers];
        if (!slot) e = hipHostMalloc(reinterpret_cast<void**>(&slot), kSlotBytes, hipHostMallocPortable);
        if (e == hipSuccess && !ev[b]) e = hipEventCreateWithFlags(&ev[b], hipEventDisableTiming);
        if (e == hipSuccess) e = hipMemcpyAsync(slot, chunks[i].src, chunks[i].bytes, hipMemcpyDeviceToHost, s);
        if (e == hipSuccess) e = hipEventRecord(ev[b], s);
    };
    const size_t n = chunks.size(), step = static_cast<size_t>(workers);
    for (int b = 0; b < 2 && e == hipSuccess; b++) {
        const size_t i = static_cast<size_t>(w) + static_cast<size_t>(b) * step;
        if (i < n) send(i, b);
    }
    int b = 0;
    for (size_t i = static_cast<size_t>(w); i < n && e == hipSuccess; i += step, b ^= 1) {
        if ((e = hipEventSynchronize(ev[b])) != hipSuccess) break;
        std::memcpy(chunks[i].dst, g_slot[w + b * workers], chunks[i].bytes);
        if (i + 2 * step < n) send(i + 2 * step, b);
    }
    // no copy into a slot is left behind when a call fails
    if (e != hipSuccess) hipStreamSynchronize(s);
    for (hipEvent_t v : ev)
        if (v) hipEventDestroy(v);
    return e;
}

hipError_t move_large(const std::vector<Chunk>& chunks, int workers, int device, hipStream_t s) {
    // the work queued before is waited for once, not by every thread
    hipError_t e = workers > 1 ? hipStreamSynchronize(s) : hipSuccess;
    if (e != hipSuccess) return e;
    std::atomic<int> failed{hipSuccess};
    std::vector<std::thread> pool;
    auto work = [&](int w) {
        hipError_t r = w ? hipSetDevice(device) : hipSuccess;
        if (r == hipSuccess) r = move_chunks(chunks, w, workers, s);
        if (r != hipSuccess) failed = static_cast<int>(r);
    };
    int started = 1;
    try {
        pool.reserve(static_cast<size_t>(workers));
        for (; started < workers; started++) pool.emplace_back(work, started);
    } catch (const std::system_error&) {
        // no more threads: this one does what they would have
    }
    work(0);
    for (int w = started; w < workers; w++) work(w);
    for (std::thread& t : pool) t.join();
    return static_cast<hipError_t>(failed.load());
}

// A field of at most one slot: its parts into it, one wait, one move.
hipError_t move_small(const std::vector<Chunk>& chunks, hipStream_t s) {
    char*& slot = g_slot[0];
    hipError_t e = hipSuccess;
    if (!slot) e = hipHostMalloc(reinterpret_cast<void**>(&slot), kSlotBytes, hipHostMallocPortable);
    size_t o = 0;
    for (const Chunk& k : chunks) {
        if (e == hipSuccess) e = hipMemcpyAsync(slot + o, k.src, k.bytes, hipMemcpyDeviceToHost, s);
        o += k.bytes;
    }
    const hipError_t w = hipStreamSynchronize(s);   // also after a failure: no copy into the slot is left behind
    if (e == hipSuccess) e = w;
    if (e == hipSuccess) std::memcpy(chunks[0].dst, slot, o);   // the parts lie one after another there too
    return e;
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
        if (p) hipHostFree(p);
        p = nullptr;
    }
}

gf_status download_parts(gf_ctx* c, const double* const* src, const int64_t* count, int parts, double* host) {
    std::unique_lock<std::mutex> held(g_slots_lock, std::try_to_lock);
    size_t total = 0;
    for (int p = 0; p < parts; p++) total += sizeof(double) * static_cast<size_t>(count[p]);
    hipError_t e = hipErrorOutOfMemory;
    if (held.owns_lock()) {
        std::vector<Chunk> chunks;
        char* dst = reinterpret_cast<char*>(host);
        for (int p = 0; p < parts; p++) {
            const char* from = reinterpret_cast<const char*>(src[p]);
            const size_t bytes = sizeof(double) * static_cast<size_t>(count[p]);
            for (size_t o = 0; o < bytes; o += kSlotBytes)
                chunks.push_back({from + o, dst + o, std::min(kSlotBytes, bytes - o)});
            dst += bytes;
        }
        e = total <= kSlotBytes ? move_small(chunks, c->stream)
                                : move_large(chunks, total < kThreadsFrom ? 1 : kThreads, c->device, c->stream);
    }
    if (e != hipSuccess) {
        double* dst = host;
        e = hipSuccess;
        hipGetLastError();   // what made the slots unusable is not the next launch's error
        for (int p = 0; p < parts && e == hipSuccess; p++) {
            e = hipMemcpyAsync(dst, src[p], sizeof(double) * static_cast<size_t>(count[p]), hipMemcpyDeviceToHost,
                               c->stream);
            dst += count[p];
        }
        const gf_status st = hip_check(c, e, "download");
        if (st) return st;
        return hip_check(c, hipStreamSynchronize(c->stream), "download sync");
    }
    return GF_OK;
}

}  // namespace gf
