// Host check of the dispatch order's places: by the count's bit length, dense burning particles
// without a count first, other particles without one last (cold dense ones among them).
#include <cstdio>
#include <initializer_list>

#include "../../sph-exa-nnet_amd/csrc/nnet_layout.hpp"

using namespace nnet_amd;

int main()
{
    int n_fail = 0;
    auto check = [&](bool ok, unsigned c, bool d)
    {
        if (!ok && n_fail++ < 20) std::printf("FAIL count %u dense burning %d: %d\n", c, d, order_bucket(c, d));
    };
    check(order_bucket(0, false) == 0, 0, false);
    check(order_bucket(0, true) == NBUCKET - 1, 0, true);
    for (unsigned c = 1, b = 1; b <= 32; ++b, c = c < 0x80000000u ? 2 * c : c)
        for (unsigned x : {c, c + (c >> 1), c | (c - 1)})
            for (bool d : {false, true})
                check(order_bucket(x, d) == (int)(b < 32 ? b : 31) && order_bucket(x, d) > order_bucket(0, false), x, d);
    std::printf("%d failures\n", n_fail);
    return n_fail != 0;
}
