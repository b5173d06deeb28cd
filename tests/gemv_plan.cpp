// Checks any_plan (csrc/gemv_plan.h) over problems: it finds a slicing exactly where one fits LDS, and what it returns
// covers the problem.  Prints the first fault and fails.
#include <cstdio>
#include <initializer_list>

#include "gemv_plan.h"

int main() {
    for (int cus : {256, 64, 1})
        for (int M = 1; M <= 16; ++M)
            for (int K = 16; K <= 45000; K += K < 20000 ? 4 : 52)
                for (int N : {1, 4, 500, 1024, 4096, 50257}) {
                    const ie::AnyPlan p = ie::any_plan(M, N, K, cus);
                    // one slice pads K to a multiple of 512, KS slices to one of 512 KS
                    bool fits = false;
                    for (int ks = 1; ks <= 8; ks *= 2) {
                        const long long cols = (K + 512LL * ks - 1) / (512 * ks) * (512 * ks);
                        fits |= 4096 + M * (cols + 64) <= 160 * 1024;
                    }
                    const long long slots = 8 >> p.ks_log, waves = (long long)p.blocks * slots;
                    const bool good = !p.lds ? !fits
                                             : fits && p.lds <= 160 * 1024 && p.spk % 2 == 0 &&
                                                   ((long long)p.spk << p.ks_log) * 256 >= K && p.blocks >= 1 &&
                                                   p.blocks <= (unsigned)cus && p.blocks <= (unsigned)(N + 3) / 4 &&
                                                   p.batches * 2 / p.spk * waves >= (N + 3) / 4 &&
                                                   p.lds == 4096 + (size_t)M * (((size_t)p.spk << p.ks_log) * 256 + 64);
                    if (!good) {
                        std::printf("M %d N %d K %d on %d units: lds %zu, 2^%d slices of %d steps, %u workgroups; one fits: %d\n", M,
                                    N, K, cus, p.lds, p.ks_log, p.spk, p.blocks, (int)fits);
                        return 1;
                    }
                }
    std::puts("ok");
    return 0;
}
