// The choice of block shape and k slices of the many-row q-GEMMs.
#pragma once

#include "common.h"

namespace slhip {

// A block shape: its tile, the blocks a CU holds at once, and the time of one
// 128-k pass (us, MI355X) of 1, 2, ... blocks on a CU together.
struct GemmShape {
    uint32_t bm, bn, most;
    float pass[4];
};

struct GemmChoice {
    size_t shape;
    uint32_t slices;
};

// The shape and slices with the least estimated time for weights of n[0 ..
// nseg) columns, m rows and `passes` passes: each CU's blocks run in rounds of
// as many as it holds; slices add a launch (3.5 us) and the partial sums'
// traffic, written and read once (5.7 TB/s), within room_floats. allowed(z):
// whether k can be cut into z slices. A chain of more than `chain` passes counts
// 3% more: what its sums of that many roundings lose is worth a cut that costs
// nothing ([4096 x 14336] at M = 1024 in one slice 1.9e-7 from float64, in two
// 1.4e-7, at the same time).
template <size_t N, typename Allowed>
inline GemmChoice choose_gemm(const GemmShape (&shapes)[N], const uint64_t* n, uint32_t nseg, uint64_t m,
                              uint32_t passes, uint64_t room_floats, Allowed allowed,
                              uint32_t chain = UINT32_MAX) {
    const uint32_t cus = compute_units();
    uint64_t n_total = 0;
    for (uint32_t i = 0; i < nseg; ++i) n_total += n[i];
    GemmChoice best{0, 1};
    float least = INFINITY;
    for (size_t c = 0; c < N; ++c) {
        const GemmShape& x = shapes[c];
        uint64_t tiles = 0;
        for (uint32_t i = 0; i < nseg; ++i) tiles += (n[i] + x.bn - 1) / x.bn;
        tiles *= (m + x.bm - 1) / x.bm;
        for (uint32_t z = 1; z <= 8 && z <= passes; z *= 2) {
            if (z > 1 && z * m * n_total > room_floats) break;
            if (!allowed(z)) continue;
            const uint64_t per_cu = (tiles * z + cus - 1) / cus;
            const uint32_t rest = static_cast<uint32_t>(per_cu % x.most);
            float t = static_cast<float>(per_cu / x.most) * x.pass[x.most - 1] + (rest ? x.pass[rest - 1] : 0.f);
            t *= static_cast<float>((passes + z - 1) / z);
            if (z > 1) t += 3.5f + static_cast<float>(m * n_total) * static_cast<float>(2 * z + 1) * 0.7e-6f;
            if ((passes + z - 1) / z > chain) t *= 1.03f;
            if (t < least) {
                least = t;
                best = GemmChoice{c, z};
            }
        }
    }
    return best;
}

}  // namespace slhip
