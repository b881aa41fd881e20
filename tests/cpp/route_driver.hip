// The size rules that choose 32-bit offsets, against the largest offsets the
// chosen kernels form.  Host code only: the library's launches end in the
// hipLaunchKernel below, which notes the kernel instead of running it.
#include <cstdio>
#include <cstring>

#include "../../go-ferro_amd/csrc/gf_internal.h"

static const void* g_kernel = nullptr;

extern "C" hipError_t hipLaunchKernel(const void* kernel, dim3, dim3, void**, size_t, hipStream_t) {
    g_kernel = kernel;
    return hipSuccess;
}
extern "C" hipError_t hipGetLastError() { return hipSuccess; }
// what a launch does first, which would look for a device
extern "C" hipError_t __hipPushCallConfiguration(dim3, dim3, size_t, hipStream_t) { return hipSuccess; }
extern "C" hipError_t __hipPopCallConfiguration(dim3*, dim3*, size_t*, hipStream_t*) { return hipSuccess; }

namespace {

constexpr int64_t kBytes32 = int64_t{1} << 32;

// Bytes an array of count doubles spans: its largest byte offset is below it.
int64_t span(int64_t count) { return count * static_cast<int64_t>(sizeof(double)); }

int elastic_force() {
    int seen[2] = {0, 0};
    for (int64_t nz = 5; nz <= 4096; nz += nz < 32 ? 1 : nz / 3)
        for (int64_t ny : {int64_t{1}, int64_t{2}, int64_t{3}, int64_t{509}, int64_t{6689}, int64_t{6690}, int64_t{7327}})
            for (int64_t limit : {int64_t{1} << 28, (int64_t{1} << 29) * nz / 12, int64_t{1} << 29})
                for (int64_t d = -2; d <= 2; d++)
                    for (bool liao : {false, true}) {
                        const int64_t nx = limit / (ny * nz) + d;
                        if (nx < 1) continue;
                        const int64_t n = nx * ny * nz, slot = 12 * nx * ny;
                        const bool fits = span(n) <= kBytes32 / 2 - 8 && (!liao || span(slot) <= kBytes32);
                        if (gf::el_narrow(nx, ny, nz, liao) != fits) {
                            std::printf("elastic force %lld x %lld x %lld liao %d: %d\n", (long long)nx, (long long)ny,
                                        (long long)nz, liao, !fits);
                            return 1;
                        }
                        seen[fits]++;
                    }
    return seen[0] && seen[1] ? 0 : 1;
}

// The kernel a list of FM cells runs on a grid of n cells.
const void* list_kernel(int64_t n, int64_t count, bool mixed = false) {
    static const uint32_t ids = 0;
    g_kernel = nullptr;
    gf::StageArgs a{};
    a.nx = a.ny = 1;
    a.nz = n;
    a.mixed = mixed;
    return gf::launch_mag_stage(a, n, nullptr, &ids, count) == hipSuccess ? g_kernel : nullptr;
}

int magnet_list() {
    const int64_t narrow = int64_t{1} << 28;
    const void* small = list_kernel(narrow - 1, 1);
    if (!small || small != list_kernel(100, 99)) return 1;
    const void* wide = list_kernel(narrow, 1);
    if (!wide || wide == small) {
        std::printf("a grid of 2^28 cells runs the list's 32-bit kernel\n");
        return 1;
    }
    if (wide != list_kernel(2 * narrow, 2 * narrow - 1) || wide != list_kernel(16 * narrow - 1, 1)) return 1;
    const void* two = list_kernel(narrow - 1, 1, true);   // several materials: the neighbours' codes are read
    if (!two || two == small || two == wide || wide != list_kernel(narrow, 1, true)) return 1;
    return list_kernel(100, 0) || list_kernel(narrow, 0);   // no FM cell: no launch
}

// Every quotient of an index below 2^28 by an axis length: the lengths around
// powers of two and around what divides 2^28, the indices around multiples.
int cell_div() {
    const uint32_t end = 1u << 28;
    for (int b = 0; b <= 28; b++)
        for (int64_t d = (int64_t{1} << b) - 3; d <= (int64_t{1} << b) + 3; d++) {
            if (d < 1 || d >= end) continue;
            uint32_t m, s;
            gf::cell_div_one(d, m, s);
            for (int64_t k = 0; k < 4096; k++) {
                const int64_t mult = k * ((end / d) / 4096 + 1) * d;
                for (int64_t id : {mult - 1, mult, mult + d - 1, static_cast<int64_t>(end) - 1 - k})
                    if (id >= 0 && id < end && gf::cell_div_apply(static_cast<uint32_t>(id), m, s) != id / d) {
                        std::printf("%lld / %lld\n", (long long)id, (long long)d);
                        return 1;
                    }
            }
        }
    return 0;
}

}  // namespace

int main(int argc, char** argv) {
    const char* what = argc > 1 ? argv[1] : "";
    if (!std::strcmp(what, "elastic_force")) return elastic_force();
    if (!std::strcmp(what, "magnet_list")) return magnet_list();
    if (!std::strcmp(what, "cell_div")) return cell_div();
    std::printf("unknown rule %s\n", what);
    return 2;
}
