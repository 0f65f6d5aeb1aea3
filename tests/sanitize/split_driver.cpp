// Splits of the U/J launches against a given amount of memory (uj_split.h).
#include <cstdio>
#include <cstdlib>

#include "uj_split.h"

using namespace vpm;

#define HOLD(x)                                                                            \
    do {                                                                                   \
        if (!(x)) {                                                                        \
            std::printf("nt %lld ns %lld cap %zu: %s\n", (long long)nt, (long long)ns, cap, #x); \
            std::exit(1);                                                                  \
        }                                                                                  \
    } while (0)

int main()
{
    const int64_t sizes[] = {2048, 2049, 16384, 16421, 65536, 100003, 262144, 1 << 20, (1 << 20) + 1, 3000017, 1 << 23, 1 << 26};
    long cases = 0;
    for (const int64_t nt : sizes)
        for (const int64_t ns : sizes) {
            const int64_t bt = far_batch(nt, ns), ntile = (ns + kTile - 1) / kTile;
            const FarSplit all = far_split(bt, ns, 0);
            FarSplit one;
            one.far = one.rest = 1;
            const size_t most = far_part_bytes(bt, all), least = far_part_bytes(bt, one);
            size_t cap = 0;
            HOLD(far_scratch_bytes(bt, ns) <= ((size_t)256 << 20) + 64 * (size_t)(bt + ns) / 64 + 1024 + 4 * (size_t)ntile);
            for (cap = most; cap + 1 >= least && cap > 0; cap = cap > least ? (cap / 2 > least ? cap / 2 : least) : cap - 1) {
                FarSplit k;
                int tries = 0;
                size_t got = 0;
                const int rc = fit_far_split(bt, ns, 0, k, [&](size_t bytes) {
                    ++tries;
                    got = bytes;
                    return bytes <= cap ? VPM_OK : VPM_ENOMEM;
                });
                ++cases;
                HOLD(tries <= 16);
                HOLD(rc == (cap >= least ? VPM_OK : VPM_ENOMEM));
                if (rc) break;
                HOLD(got == far_part_bytes(bt, k) && got <= cap);
                HOLD(k.far >= 1 && k.rest >= 1 && k.far <= all.far && k.rest <= all.rest);
                HOLD(k.chunk * k.far >= ntile && k.chunk * (k.far - 1) < ntile);
                if (cap == most) HOLD(tries == 1 && k.far == all.far && k.rest == all.rest);
            }
            // another error ends the search
            FarSplit k;
            int tries = 0;
            HOLD(fit_far_split(bt, ns, 0, k, [&](size_t) { ++tries; return VPM_EDEVICE; }) == VPM_EDEVICE && tries == 1);
        }
    for (int64_t K0 : {1, 2, 3, 8, 17, 512}) {
        const int64_t nt = K0, ns = 0;
        for (size_t cap = 0; cap <= 512; ++cap) {
            int64_t K = K0;
            const int rc = fit_splits(K, [&](int64_t m) { return (size_t)m <= cap ? VPM_OK : VPM_ENOMEM; });
            HOLD(rc == (cap >= 1 ? VPM_OK : VPM_ENOMEM) && K >= 1 && K <= K0);
            if (!rc) HOLD((size_t)K <= cap && (K == K0 || 2 * K + 1 > (int64_t)cap));
            ++cases;
        }
    }
    std::printf("split_driver OK, %ld cases\n", cases);
    return 0;
}
