// Random items of rect_step_kernel: the entries staged (step_range) fit what
// the plan requests (step_shape, step_bytes), and hold the end of every cell.
// Prints the number of items; exits with 1 at the first that fails.
#include <cstdio>
#include <random>

#include "tcw_step.h"

using namespace tcwc;

int main() {
    std::mt19937_64 rng(5);
    auto uni = [&](uint64_t lo, uint64_t hi) { return lo + rng() % (hi - lo + 1); };
    const uint32_t TAs[] = {2, 3, 7, 60, 1799, 1800, 3600};
    long items = 0, tight = 0;
    for (int trial = 0; trial < 40000; trial++) {
        const uint32_t TA = TAs[uni(0, 6)];
        // steps of an atom or more, whole and fractional
        auto step = [&](uint64_t atoms) {
            const uint64_t k = uni(1, atoms), f = uni(0, 3) ? uni(0, TA - 1) : 0;
            return (uint32_t)(k * TA + f);
        };
        const uint32_t dt0 = step(uni(0, 1) ? 2 : 12), dtau = step(uni(0, 1) ? 3 : 20);
        const uint32_t N_t0 = uni(1, 200), N_tau = uni(1, 600);
        const uint32_t t0 = uni(0, 3 * TA), tau = uni(0, 4 * TA);
        const int N = uni(1, 4000), rb = 16 * uni(1, 32), tile = 64 << uni(0, 2);
        const StepShape sh = step_shape(rb, tile, N_tau, dt0, dtau, TA);
        if (!step_in_lds(sh)) continue;
        auto end = [&](uint32_t m, uint32_t n) {  // of cell (m, n), as the reference has it
            const uint64_t j = ((uint64_t)t0 + (uint64_t)m * dt0 + tau + (uint64_t)n * dtau) / TA;
            return (int64_t)(j < 1 ? 1 : j > (uint64_t)N ? N : j);
        };
        for (uint32_t row0 = 0; row0 < N_t0; row0 += rb)
            for (uint32_t col0 = 0; col0 < N_tau; col0 += tile) {
                const uint32_t rl = row0 + rb < N_t0 ? row0 + rb - 1 : N_t0 - 1;
                const uint32_t cl = col0 + tile < N_tau ? col0 + tile - 1 : N_tau - 1;
                const StepRange r = step_range(t0 + row0 * dt0, tau + col0 * dtau, t0 + rl * dt0,
                                               tau + cl * dtau, N, [&](uint32_t x) { return x / TA; });
                const int e = r.count - 1;
                const bool fits = r.count >= 1 && r.count <= sh.entries &&
                                  (e * TCW_NCOL + (e >> sh.pad) + TCW_NCOL) * 8 <= step_bytes(sh);
                const bool holds = end(row0, col0) >= r.first && end(rl, cl) <= r.first + e;
                items++;
                tight += r.count >= sh.entries - 1;
                if (!fits || !holds) {
                    std::printf("TA %u dt0 %u dtau %u t0 %u tau %u N %d rb %d tile %d item (%u, %u): "
                                "%d of %d entries from %d, cells' %lld .. %lld\n", TA, dt0, dtau, t0,
                                tau, N, rb, tile, row0, col0, r.count, sh.entries, r.first,
                                (long long)end(row0, col0), (long long)end(rl, cl));
                    return 1;
                }
            }
    }
    std::printf("%ld items, %ld within one entry of the most\n", items, tight);
    return items > 10000 && tight > 100 ? 0 : 1;
}
