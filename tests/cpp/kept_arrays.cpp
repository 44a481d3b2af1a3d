// Host-side check that the arrays the next iteration may read again (binding energies, dY/dt,
// d(dY/dt)/dT, RHS correction, EOS, Jacobian) survive a solve: no factor entry that the FP64 or the
// mixed factorization stores reaches them.
#include <cstdio>

#include "../../sph-exa-nnet_amd/csrc/nnet_layout.hpp"

using namespace nnet_amd;

static int n_fail = 0;
static void below(const char* what, long i, long end)
{
    if ((i < 0 || i >= end) && n_fail++ < 50) std::printf("FAIL %s: %ld outside [0, %ld)\n", what, i, end);
}

template<int NET>
void run()
{
    using F = Lds<NET, false>;
    using M = Lds<NET, true>;
    using X = LuIdx<NET>;
    constexpr int N = X::N;
    for (int k = 0; k < N; ++k)
        for (int j = k + 1; j <= N; ++j)
        {
            below("FP64 factor entry", X::uidx(k, j), F::oBE);
            below("FP32 factor entry", X::uidx(k, j), 2L * M::oBE);
        }
    below("FP32 multiplier", M::NU + X::lrow(N - 1) + N - 2, 2L * M::oBE);
    below("FP32 pivot reciprocal", M::NU + M::NL + N - 1, 2L * M::oBE);
    below("kept arrays before the state", F::phaseEnd - 1, F::oY);
    below("kept arrays before the state", M::phaseEnd - 1, M::oY);
}

// the eight-pivot LU's publish: rows of block B, columns up to N (the last tile's padding is left out)
template<int NET>
void publish()
{
    using F = Lds<NET, false>;
    using X = Lu8Idx<NET>;
    for (int B = 0; B < X::NB; ++B)
        for (int tid = 0; tid < 256; ++tid)
            for (int tj = (8 * B >> 4) / 2; tj < Cfg<NET>::TT / 2; ++tj)
                for (int h = 0; h < 2; ++h)
                {
                    const int p0 = 8 * B, w = tid >> 6, lr = (tid & 63) >> 4, lc = tid & 15;
                    const int col = tile_col(w % 2 + 2 * tj, lc), row = p0 + lr + 4 * h;
                    const bool in = 16 * (2 * tj + 2) <= X::N + 1 || col <= X::N;
                    if (w / 2 == (p0 >> 4) % 2 && in && (tj > (p0 >> 4) / 2 || col > row))
                        below("published pivot row", X::uidx(row, col), F::oBE);
                }
}

int main()
{
    run<14>();
    run<86>();
    run<87>();
    publish<86>();
    publish<87>();
    std::printf("%d failures\n", n_fail);
    return n_fail ? 1 : 0;
}
