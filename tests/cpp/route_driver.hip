// The size rules that choose 32-bit offsets, against the largest offsets the
// chosen kernels form.  Host code only.
#include <cstdio>
#include <cstring>

#include "../../go-ferro_amd/csrc/gf_internal.h"

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

}  // namespace

int main(int argc, char** argv) {
    const char* what = argc > 1 ? argv[1] : "";
    if (!std::strcmp(what, "elastic_force")) return elastic_force();
    std::printf("unknown rule %s\n", what);
    return 2;
}
