// Host-side check of the eight-pivot LU (PanelLU of nnet_solver.hip, net86 / net87 FP64): every
// LDS index its lanes form is inside the array it addresses, and its blocks normalise every entry
// (k, j), k < j <= N, of the upper factor exactly once, after its publish.
#include <cstdio>
#include <vector>

#include "../../sph-exa-nnet_amd/csrc/nnet_layout.hpp"

using namespace nnet_amd;

static int n_fail = 0;
static void in(const char* what, long i, long lo, long hi)
{
    if ((i < lo || i >= hi) && n_fail++ < 50) std::printf("FAIL %s: %ld outside [%ld, %ld)\n", what, i, lo, hi);
}

template<int NET>
void run()
{
    using X = Lu8Idx<NET>;
    using L = Lds<NET, false>;
    constexpr int    N = X::N, NPAD = X::NPAD, TI = Cfg<NET>::TT / 2;
    const long       uEnd = L::uWords, panEnd = L::panWords;
    std::vector<int> published(uEnd, -1), normalised(uEnd, 0);
    in("packed rows below the live arrays", uEnd, 0, L::oY + 1);
    in("panel buffers inside the allocation", L::oPan + panEnd, 0, L::total + 1);
    in("16-byte aligned panel rows", (L::oPan | PANEL8 | NPAD * PANEL8) & 1, 0, 1);
    for (int B = 0; B < X::NB; ++B)
    {
        const int p0 = 8 * B, Tp = p0 >> 4, c0 = p0 & 15, nq = N - p0 < 8 ? N - p0 : 8;
        for (int tid = 0; tid < 256; ++tid) // publish
        {
            const int lane = tid & 63, w = tid >> 6, lr = lane >> 4, lc = lane & 15, wr = w / 2, wc = w % 2;
            if (wc == Tp % 2 && (lc >> 3) == (c0 >> 3))
                for (int ti = Tp / 2; ti < TI; ++ti)
                    for (int v = 0; v < 4; ++v)
                        in("panel column", X::pcol(B, tile_row(wr + 2 * ti, lr, v), lc - c0), 0, panEnd);
            if (wr == Tp % 2)
                for (int tj = Tp / 2; tj < TI; ++tj)
                    for (int h = 0; h < 2; ++h)
                    {
                        const int col = tile_col(wc + 2 * tj, lc), row = p0 + lr + 4 * h;
                        if (tj > Tp / 2 || col > row)
                        {
                            in("strictly right of the diagonal", col, row + 1, NPAD);
                            in("pivot row", X::uidx(row, col), 0, uEnd);
                            published[X::uidx(row, col)] = B;
                        }
                    }
        }
        in("wavefronts of the trailing rows", X::rowWaves(B), 0, 3);
        in("wavefronts of the columns", X::colWaves(B), 1, 3);
        std::vector<int> rowDone(NPAD, 0);
        for (int w = 0; w < 4; ++w)
            for (int lane = 0; lane < 64; ++lane)
            {
                for (int c = 0; c < 8; ++c)
                    in("diagonal row", X::pcol(B, p0 + (lane & 7), c), 0, panEnd);
                if (w < X::rowWaves(B))
                {
                    const int i = X::row0(B) + 64 * w + lane;
                    for (int c = 0; c < 8; ++c)
                        in("trailing row", X::pcol(B, i < N ? i : N - 1, c), 0, panEnd);
                    if (i < N) ++rowDone[i];
                }
                if (w >= 2 && w - 2 < X::colWaves(B))
                {
                    const int j = X::col0(B) + 64 * (w - 2) + lane;
                    for (int q = 0; q < nq; ++q)
                    {
                        in("column entry", X::uidx(p0, j <= N ? j : N) + q, 0, uEnd);
                        if (j <= N && p0 + q < j)
                        {
                            const long u = X::uidx(p0 + q, j);
                            in("published in this block", published[u], B, B + 1);
                            ++normalised[u];
                        }
                    }
                }
                const int wr = w / 2, wc = w % 2, lr = lane >> 4, lc = lane & 15;
                for (int t = 0; t < TI && X::rowWaves(B) > 0; ++t)
                    for (int s = 0; s < 2; ++s)
                    {
                        in("A operand", X::pcol(B, 16 * (wr + 2 * t) + lc, lr + 4 * s), 0, panEnd);
                        if (t >= (Tp + (c0 ? 1 : 0)) / 2)
                            in("B operand", X::uidx(p0 + lr + 4 * s, tile_col(wc + 2 * t, lc)), 0, uEnd);
                    }
            }
        for (int i = p0 + 8; i < N; ++i)
            in("trailing row eliminated once", rowDone[i], 1, 2);
    }
    for (int k = 0; k < N; ++k)
        for (int j = k + 1; j <= N; ++j)
            in("upper entry normalised once", normalised[X::uidx(k, j)], 1, 2);
}

int main()
{
    run<86>();
    run<87>();
    std::printf("%d failures\n", n_fail);
    return n_fail ? 1 : 0;
}
