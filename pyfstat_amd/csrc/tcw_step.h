// tcw_step.h -- the prefix entries that an item of rect_step_kernel stages in LDS:
// how many there can be (the plan's layout) and which they are (the kernel).
// Host and device code, free of HIP, so that both are checked on the CPU.
// Not part of the C ABI.
#pragma once

#include <cstdint>

#include "tcw_hip.h"

#ifdef __HIPCC__
#define TCW_HD __host__ __device__ __forceinline__
#else
#define TCW_HD inline
#endif

namespace tcwc {

// Bytes of staged range per item.  The widest of 256, 128 and 64 columns whose
// range stays below the first figure (four workgroups a CU or more), else 64
// columns if that stays below the second, else 256 read from the table (128
// templates of 1000 to 4000 bins, steps of 2 and 3 bins, at 20, 28, 36 and 52 KB:
// 112, 95, 94 and 100 us).
constexpr int STEP_LDS_AIM = 36 << 10;
constexpr int STEP_LDS_MOST = 76 << 10;

struct StepShape {
    int entries;  // staged prefix entries of an item at most
    int pad;      // entry e lies at e * 7 + (e >> pad) doubles
};

// An item of rb rows and `tile` columns.  Its first and last end lie span =
// (rb - 1) dt0 + (columns - 1) dtau apart, so floor(last / TA) - floor(first / TA) is
// at most floor(span / TA) + 1, and the entries one more (room for one to spare).
TCW_HD StepShape step_shape(int rb, int tile, uint32_t N_tau, uint32_t dt0, uint32_t dtau,
                            uint32_t TA) {
    const uint32_t nc = N_tau < (uint32_t)tile ? N_tau : (uint32_t)tile;
    const uint64_t span = ((uint64_t)(rb - 1) * dt0 + (uint64_t)(nc - 1) * dtau) / TA + 3;
    StepShape sh;
    sh.entries = span < (1u << 20) ? (int)span : 1 << 20;
    const uint32_t b = dtau / TA;
    sh.pad = 31;
    if (b > 0 && b % 2 == 0 && dtau % TA == 0)
        for (sh.pad = 0; 2u << sh.pad <= b; sh.pad++) {
        }
    return sh;
}
TCW_HD int step_bytes(const StepShape &sh) {
    return (sh.entries * TCW_NCOL + (sh.entries >> sh.pad) + 1) * (int)sizeof(double);
}
TCW_HD bool step_in_lds(const StepShape &sh) { return step_bytes(sh) <= STEP_LDS_MOST; }

TCW_HD int step_clamp(int j, int N) { return j < 1 ? 1 : j > N ? N : j; }

// The entries first .. first + count - 1 that an item reads: from the end of its
// first row's (start Tr) and column's (duration xf) window to that of the last
// ones (Tl, xl), each floor((T + x) / TA) as the cells have it (the quotients of T
// and x by themselves, and a carry at either, can be one entry more than the
// shape's).  div: x / TA.
struct StepRange {
    int first, count;
};
template <typename Div>
TCW_HD StepRange step_range(uint32_t Tr, uint32_t xf, uint32_t Tl, uint32_t xl, int N, Div div) {
    const int first = step_clamp((int)div(Tr + xf), N);
    const int last = step_clamp((int)div(Tl + xl), N);
    return StepRange{first, last - first + 1};
}

}  // namespace tcwc
