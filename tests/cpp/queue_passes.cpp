// Host check of the work queue's arithmetic at its sizes' ends: a launch's 32-bit position count
// never wraps (every group takes one position past the end), and each particle is at one position
// of each pass.
#include <cstdio>
#include <initializer_list>

#include "../../sph-exa-nnet_amd/csrc/nnet_layout.hpp"

using namespace nnet_amd;

int main()
{
    int n_fail = 0;
    for (uint32_t groups : {1u, 3u, 512u, 2048u, 8192u})
        for (uint64_t mid : {1ull, 512ull, 2048ull, 50021ull, 1ull << 30, 1ull << 31, (1ull << 31) + 512, 3ull << 30,
                             0ull + queue_limit(256)})
            for (int64_t d = -9000; d <= 9000; d += d > -5 && d < 5 ? 1 : 5)
                for (bool ordered : {false, true})
                {
                    const int64_t n = (int64_t)mid + d;
                    if (n < 1 || (uint64_t)n > queue_limit(256)) continue;
                    const uint32_t nq = (uint32_t)n, t = queue_passes(nq, groups, ordered);
                    const uint64_t last = (uint64_t)t * nq + groups;
                    const bool ok = (t == 1 || t == 2) && last <= 0xffffffffull && t * nq == (uint64_t)t * nq &&
                                    !(t == 2 && (ordered || nq <= groups)) &&
                                    (t == 2 || ordered || nq <= groups || 2ull * nq + groups > 0xffffffffull);
                    if (!ok && n_fail++ < 20)
                        std::printf("FAIL n %lld groups %u ordered %d passes %u\n", (long long)n, groups, ordered, t);
                }
    // dense particles first: not where more than half of the sample is idle, nor where all that burns is
    // dense or none of it is
    for (uint32_t idle = 0; idle <= PLAN_SAMPLE; ++idle)
        for (uint32_t dense = 0; idle + dense <= PLAN_SAMPLE; ++dense)
        {
            const uint32_t thin = PLAN_SAMPLE - idle - dense;
            if (dense_first_pays(idle, dense) != (idle <= PLAN_SAMPLE / 2 && dense >= 1 && thin >= 1) && n_fail++ < 20)
                std::printf("FAIL idle %u dense %u\n", idle, dense);
        }
    std::printf("%d failures\n", n_fail);
    return n_fail != 0;
}
