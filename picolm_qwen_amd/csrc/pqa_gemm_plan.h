// The tile, the K slices and the slice workspace of the split GEMM (pqa_gemm.hip).
// Host code without HIP, so that the CPU tests can build it.
#pragma once

#include <algorithm>
#include <cstddef>

namespace pqa {

constexpr int kGemmBK = 32;  // k per tile of the GEMM's loop

// The workgroup tile (64 mi x 64 nj) and the number of K slices.
struct GemmPlan {
    int mi, nj, slices;
};

constexpr int kGemmMaxSlices = 16;

// Floats of workspace that the K slices of an m x n product may take: 16 results, up
// to a result of the largest tile per CU (50 MB on 256 CUs). It grows with m and n
// whatever the plan picks, so the workspace of a long prompt holds every shorter one
// (the slices themselves do not: 137 tokens of 4096 columns take 4, 138 one).
inline size_t gemm_slice_floats(int m, int n, int cu_count) {
    return std::min<size_t>((size_t)kGemmMaxSlices * m * n, (size_t)cu_count * 256 * 192);
}

// The tile and K slices with the least expected time, in us, from rates measured
// over 110 shapes (2 to 2048 rows, 896 to 6144 columns, K 896 to 4096; the pick is
// 3.5 % off the fastest of all combinations on average). A k tile takes a
// workgroup `step` when it has a CU for itself, and the chip as a whole needs
// `flow` per k tile and 32 x 32 block (operand traffic and power, 1.1-1.2 PFLOP/s
// on the two largest tiles); each round of workgroups costs a pipeline fill, and
// slices the launch that sums them and their way through memory. Against the one
// 256 x 192 tile without slices: 75 x 4096 x 2560 115 -> 17 us, 75 x 2560 x 4096
// 163 -> 16, 2048 x 4096 x 2560 138 -> 118 (256 x 128: 256 tiles on 256 CUs where
// 176 were busy), 2048 x 2560 x 4096 192 -> 129 (two slices of 112 tiles).
inline GemmPlan gemm_f16x3_plan(int m, int n, int kh, int cu_count) {
    static const struct {
        int mi, nj, occupancy;
        double step, flow;
    } tiles[] = {{4, 3, 1, 1.45, 6.2e-4}, {4, 2, 1, 1.08, 6.3e-4}, {2, 2, 2, 0.66, 6.5e-4}, {2, 1, 2, 0.35, 7.3e-4},
                 {1, 1, 2, 0.25, 8.5e-4}};
    const int ktiles = std::max(1, kh / kGemmBK);
    const double cus = cu_count;
    const size_t room = gemm_slice_floats(m, n, cu_count);
    GemmPlan best{4, 3, 1};
    double best_us = 1e30;
    for (const auto& t : tiles) {
        const long long mn = (long long)((m + 64 * t.mi - 1) / (64 * t.mi)) * ((n + 64 * t.nj - 1) / (64 * t.nj));
        for (int s = 1; s <= kGemmMaxSlices && s <= ktiles; s++) {
            const long long wgs = mn * s;
            if (s > 1 && (wgs > 4LL * cu_count || (size_t)s * m * n > room)) break;
            const double kt = (double)ktiles / s;
            const double alone = (double)((wgs + cu_count - 1) / cu_count) * kt * t.step;
            const double chip = (double)wgs * kt * t.mi * t.nj * t.flow * (256.0 / cus);
            double us = std::max(alone, chip) + std::max(1.0, (double)wgs / (cus * t.occupancy));
            if (s > 1) us += 3.0 + (2.0 * s + 1.0) * m * (double)n * 4e-6 / 5.5;
            if (us < best_us) {
                best_us = us;
                best = GemmPlan{t.mi, t.nj, s};
            }
        }
    }
    return best;
}

}  // namespace pqa
