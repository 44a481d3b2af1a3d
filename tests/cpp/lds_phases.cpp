// Host-side check of LDS indices that lds_bounds.cpp does not walk: the row LU of net14, the cycle
// records, the abundance differences in the screening array, the kept assembly arrays, the
// refinement residual and the fill's running non-zero index.
#include <cstdint>
#include <cstdio>

#include "../../sph-exa-nnet_amd/csrc/nnet_image.hpp"

using namespace nnet_amd;

static int n_checks = 0, n_fail = 0;
static void in(int net, bool mix, const char* what, long i, long lo, long hi)
{
    ++n_checks;
    if ((i < lo || i >= hi) && n_fail++ < 50)
        std::printf("FAIL net%d%s %s: %ld outside [%ld, %ld)\n", net, mix ? " mixed" : "", what, i, lo, hi);
}

template<int NET, bool MIX>
void run()
{
    using C = Cfg<NET>;
    using L = Lds<NET, MIX>;
    constexpr int D = C::D, N = C::N, NT = C::NT, WR = C::WR, TI = C::TT / WR;
    auto          at = [](const char* w, long i, long lo, long hi) { in(NET, MIX, w, i, lo, hi); };

    // a record per wavefront behind the panel buffers, whole doubles, inside the allocation
    at("panel buffers end", L::oPan + L::panWords, 0, L::oCyc + 1);
    for (int w = 0; w < NT / 64; ++w)
        at("cycle record", L::oCyc + 3 * w + 2, L::oPan + L::panWords, L::total);
    // Yg - Y per species, in the screening array
    for (int s = 0; s < D; ++s)
        at("sDYg[s]", L::oMu + s, L::oMu, L::oEff);
    // the lanes' shares of the kept arrays: every word once, none outside
    constexpr int KEEP = L::phaseEnd - L::oBE, NKEEP = (KEEP + NT - 1) / NT;
    int           words = 0;
    for (int t = 0; t < NT; ++t)
        for (int q = 0; q < NKEEP; ++q)
        {
            at("kept word (selected)", L::oBE + (q * NT + t < KEEP ? q * NT + t : 0), L::oBE, L::phaseEnd);
            words += q * NT + t < KEEP;
        }
    at("kept words", words, KEEP, KEEP + 1);
    // the temperature row's operand, selected before the load
    for (int c = 0; c < 16 * C::TT; ++c)
        at("row 0 sBE", L::oBE + (c < 1 ? 0 : c < N ? c - 1 : D - 1), L::oBE, L::oDYdot);
    if (MIX)
        for (int r = 0; r < N; ++r)
            at("residual", L::oPan + r, L::oPan, L::oPan + L::panWords);
    if (NET == 14 && !MIX)
    {
        // row LU: the fill's tile into rows of 18, one row read per lane as pairs; the arrays it
        // overwrites are dead and the kept ones lie behind
        constexpr int STRIDE = 18;
        at("aligned groups", L::total % 2 + STRIDE % 2, 0, 1);
        for (int l = 0; l < 64; ++l)
            for (int v = 0; v < 4; ++v)
            {
                at("row LU store", tile_row(0, l >> 4, v) * STRIDE + (l & 15), 0, L::headEnd);
                at("row LU store below the kept arrays", tile_row(0, l >> 4, v) * STRIDE + (l & 15), 0, L::oBE);
                at("row LU load", (l & 15) * STRIDE + 4 * (l >> 4) + v, 0, L::headEnd);
            }
        at("row LU pair", (4 * STRIDE) % 2, 0, 1);
        for (int l = 0; l < N; ++l)
            at("row LU solution", L::oX + l, L::oX, L::oRow0);
    }
    // the fill's index runs through the lane's non-zeros in slot order
    HostList hl = builtin_list(NET);
    AsmImage im;
    if (!build_asm_image(NET, D, (int)hl.pb.size(), hl.rb.data(), hl.pb.data(), hl.ids.data(), hl.nums.data(), im).empty())
        at("image builds", 1, 0, 1);
    int next = 0;
    for (int t = 0; t < NT; ++t)
    {
        int nzi = (int)im.lanemap[t * 4 + 2];
        at("lane's first non-zero", nzi, next, next + 1);
        for (int slot = 0; slot < TI * TI * 4; ++slot)
        {
            const int nz = (im.lanemap[t * 4 + (slot < 32 ? 0 : 1)] >> (slot & 31)) & 1;
            at("fill sJv", nz ? nzi : 0, 0, im.nnz);
            nzi += nz;
        }
        next = nzi;
    }
    at("non-zeros placed", next, im.nnz, im.nnz + 1);
}

int main()
{
    run<14, false>();
    run<14, true>();
    run<86, false>();
    run<86, true>();
    run<87, false>();
    run<87, true>();
    std::printf("%d checks, %d failures\n", n_checks, n_fail);
    return n_fail != 0;
}
