// Which GEMM kernel a call of more than 4 rows takes, and how it splits k (q4_gemm.hip). Host
// arithmetic without HIP types; `cus` is the device's compute units (256 on MI355X).
#pragma once

#include <algorithm>
#include <cstddef>
#include <cstdint>

namespace hyperion::hip {

constexpr uint32_t kMaxGemmSegments = 3;

// A (possibly grouped) call: m rows, ceil(k / 128) pairs of groups, the segments' widths. A dual
// call (gate and up with the gating in the epilogue) has their two segments.
struct GemmShape {
    uint32_t m, pairs, nseg;
    uint32_t n[kMaxGemmSegments];
    bool dual;
};

// The tile kernels.
enum class GemmKernel : uint32_t {
    kGroup128 = 1,   // q4_gemm_g_kernel<8, 2, 8>: 128 x 256, group step, one per CU
    kGroup256 = 2,   // q4_gemm_g_kernel<16, 2, 8>: 256 x 256, group step, one per CU
};

struct GemmChoice {
    GemmKernel kernel;
    uint32_t ksplit;
};

// Bytes of the fixed scratch of launch_q4_gemm_noalloc.
constexpr size_t kNoAllocScratchBytes = size_t{64} << 20;

constexpr uint32_t kFewRows = 64;   // rows of the few-row kernel, at most
constexpr uint32_t kFewWaves = 8;   // waves of its workgroups

inline uint64_t row_tiles(const GemmShape& g) {   // 16-column tiles
    uint64_t t = 0;
    for (uint32_t i = 0; i < g.nseg; ++i) t += (g.n[i] + 15u) / 16u;
    return t;
}

// Whether the few-row kernel takes the call. Each wave reads its rows of X from L2, about 12 TB/s
// over the chip, so its time grows with rows x k x column tiles; the tile kernels' hardly below
// 128 rows. Measured, the tile kernels against it (us, calls among others, weights alternating):
//   gate + up [2 x 15360, 3840]  33 at 32 rows -> 27, but 36 -> 42 at 33
//   [15360, 3840]                27 -> 17 at 32, 26.9 -> 24.1 at 33, 29 -> 35 at 64
//   q/k/v [8192, 3840], o [3840, 4096]  23-25 -> 12 and 11 at 32, 19.5 and 18.3 at 64
//   [3840, 8192]                 25.7 -> 21 at 33, 26.3 -> 25.8 at 48, 27 -> 33 at 64
//   down [3840, 15360]           31 -> 31 at 32, 31 -> 37 at 33, 31 -> 45 at 48, 32 -> 58 at 64
// The last line's tile calls split k, and a split call that the host waits for pays 45-55 us more
// for its partials' allocation, which such a wait has given back: down alone 96 -> 48 at 33, 93 ->
// 58 at 48, 92 -> 70 at 64, [3840, 8192] 85 -> 44 at 64. So: always up to 32 rows, to 64 where
// the column tiles are at most two per compute unit.
inline bool few_rows(const GemmShape& g, uint64_t cus) {
    return g.m <= 32u || (g.m <= kFewRows && row_tiles(g) <= 2u * cus);
}

// As many column tiles per wave (they share its X reads) as leave 7 waves per compute unit
// with every tile's pairs over 8 waves, then the fewest waves per tile that still do; from
// 33 rows on at most 2 (registers, and the LDS of the sums). At 16 rows (us): [15360, 3840]
// 18.7, 13.2 and 12.0 with 1, 2 and 4 tiles per wave, q/k/v [8192, 3840] 10.9, 8.5 and 11.4,
// down [3840, 15360] 19.0, 21.5 and 30.1.
struct FewRowShape {
    uint32_t tiles;    // column tiles per wave
    uint32_t splits;   // waves per tile
};
inline FewRowShape few_row_shape(const GemmShape& g, uint64_t cus) {
    const uint64_t tiles = row_tiles(g);
    const uint32_t nt_max = g.m <= 32u ? 4u : 2u;
    uint32_t nt = g.dual ? 2u : 1u;
    while (nt < nt_max && tiles / (2u * nt) * kFewWaves >= 7u * cus) nt *= 2u;
    uint32_t s = 1u;
    while (s < kFewWaves && tiles / nt * s < 7u * cus && 2u * s <= g.pairs) s *= 2u;
    return {nt, s};
}

// Workgroups of one k split: (rows / tile rows) x (column tiles over the segments).
inline uint64_t gemm_tiles(const GemmShape& g, uint32_t rows, uint32_t cols) {
    uint64_t tn = 0;
    for (uint32_t i = 0; i < g.nseg; ++i) tn += (g.n[i] + cols - 1u) / cols;
    return static_cast<uint64_t>((g.m + rows - 1u) / rows) * tn;
}

// Bytes of the fp32 partial sums of `splits` k splits.
inline uint64_t partial_bytes(const GemmShape& g, uint32_t splits) {
    uint64_t n = 0;
    for (uint32_t i = 0; i < g.nseg; ++i) n += g.n[i];
    return static_cast<uint64_t>(splits) * g.m * n * sizeof(float);
}

// Smallest split (<= 4, at least 6 pairs in each) whose grid of `tiles` x split reaches
// 90% of the CUs.
inline uint32_t fill_split(const GemmShape& g, uint64_t tiles, uint64_t cus) {
    uint32_t s = 1u;
    while (s < 4u && tiles * s * 10u < cus * 9u && (g.pairs + s) / (s + 1u) >= 6u) ++s;
    return s;
}

// k splits that fill the compute units, at most 4: no choice of choose_gemm. It bounds the
// partials (larger splits only within 64 MiB), and launch_q4_gemm_noalloc refuses a call by it.
inline uint32_t filling_split(const GemmShape& g, uint64_t cus) {
    const uint64_t big = gemm_tiles(g, 256u, 256u);
    if (big * 10u >= cus * 9u) return 1u;
    if (g.pairs >= 64u) {
        const uint32_t s = fill_split(g, big, cus);
        if (big * s * 10u >= cus * 9u) return s;
    }
    const uint64_t mid = gemm_tiles(g, 128u, 256u);
    const uint32_t s = fill_split(g, mid, cus);
    if (mid * s * 10u >= cus * 6u) return s;
    return fill_split(g, gemm_tiles(g, 128u, 128u), cus);
}

// Kernel and split per call: the ones with the least estimated time,
//   10 us + rounds of one workgroup per compute unit x groups per split x time per group
//   + (split) 6.5 us + the partials' write and read at 12.5 TB/s,
// where a group (64 k) of the 128-row kernel takes 0.69 us, of the 256-row kernel 1.23 us, and up
// to 0.86 and 1.57 us as the grid goes from 60% of the compute units to all. The constants are
// fitted to a sweep of the projections and their groups (ten shapes, 20 row counts from 33 to
// 2048, both kernels, 1 to 12 splits): the estimate of the choice is 4% off on average and 17% at
// worst, and the choice 0.7% slower than the best of the sweep on average. Ragged grids are what
// it is for, where filling the compute units by splitting alone (filling_split, on 128-column
// tiles for small grids) runs into a second round. Against that rule (us): down [3840, 15360]
// 203 rows 61 -> 43, 700 rows 149 -> 93, 1111 rows 195 -> 135; q/k/v [8192, 3840] 300 rows 55 ->
// 41, 700 rows 77 -> 53; o [3840, 4096] 700 rows 59 -> 43; [15360, 3840] 300 rows 73 -> 53.
inline GemmChoice choose_gemm(const GemmShape& g, uint64_t cus) {
    constexpr uint32_t kMaxSplits = 12u;
    const uint32_t most = filling_split(g, cus);
    GemmChoice best{GemmKernel::kGroup128, 1u};
    double best_us = 1e30;
    for (const GemmKernel kernel : {GemmKernel::kGroup256, GemmKernel::kGroup128}) {
        const bool big = kernel == GemmKernel::kGroup256;
        const uint64_t tiles = gemm_tiles(g, big ? 256u : 128u, 256u);
        for (uint32_t s = 1u; s <= kMaxSplits && (g.pairs + s - 1u) / s >= 3u; ++s) {
            const uint64_t bytes = partial_bytes(g, s);
            if (s > most && bytes > kNoAllocScratchBytes) break;   // larger partials only where filling took them
            const uint64_t grid = tiles * s;
            const double full = std::max(0.0, std::min(1.0, static_cast<double>(grid) / cus) - 0.6) / 0.4;
            const double group = big ? 1.23 + 0.34 * full : 0.69 + 0.17 * full;
            double us = 10.0 + static_cast<double>((grid + cus - 1u) / cus) * (2u * ((g.pairs + s - 1u) / s)) * group;
            if (s > 1u) us += 6.5 + 2.0 * bytes / 12.5e6;
            if (us < best_us) {
                best_us = us;
                best = {kernel, s};
            }
        }
    }
    return best;
}

}  // namespace hyperion::hip
