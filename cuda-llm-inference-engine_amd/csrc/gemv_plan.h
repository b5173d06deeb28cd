// gemv_plan.h — how gemv_i8_any_kernel cuts a problem (host code without HIP,
// so that it can be tested by itself).
#pragma once

#include <algorithm>
#include <cstddef>

namespace ie {

constexpr size_t kLdsBytes = 160ull << 10;  // per workgroup on gfx950

struct AnyPlan {
    int ks_log, spk;    // 2^ks_log slices of K, spk 256-byte steps each (even)
    long long batches;  // of a wave's stream
    unsigned blocks;
    size_t lds;  // 0: no slicing fits
};

// The slicing (1, 2, 4 or 8 waves per 4-feature item) whose rounds x (steps per
// slice + 1) is least, the 1 for an item's reduction and store, of those whose
// activation rows fit LDS: each pads K to its own multiple (M = 14, K = 8708:
// eight slices to 12288 columns, one to 9216).  One workgroup per CU.
inline AnyPlan any_plan(int M, int N, int K, long long cus) {
    const long long items = ((long long)N + 3) / 4;
    const int steps = (K + 255) / 256;
    AnyPlan best{};
    long long cost = -1;
    for (int l = 0; l <= 3; ++l) {
        const int slots = 8 >> l, spk = ((steps + (1 << l) - 1) / (1 << l) + 1) / 2 * 2;
        const size_t lds = 2 * 8 * 64 * 4 + (size_t)M * ((size_t)(spk << l) * 256 + 64);
        if (lds > kLdsBytes) continue;
        const long long blocks = std::min((items + slots - 1) / slots, cus);
        const long long rounds = (items + blocks * slots - 1) / (blocks * slots), c = rounds * (spk + 1);
        if (cost < 0 || c < cost) {
            cost = c;
            best = {l, spk, rounds * (spk / 2), (unsigned)blocks, lds};
        }
    }
    return best;
}

}  // namespace ie
