// Kernel configuration and LDS layout of the solve kernels, plus the index functions the kernels
// use to address their LDS arrays.  Everything here is constexpr and free of HIP types, so the
// same definitions compile into the device code and into host-side checks of every LDS index
// the kernels form (clang treats constexpr functions as host and device functions).
#pragma once
#include <cstdint>

namespace nnet_amd
{
constexpr int MAXQ  = 3;  // reactant entries per reaction
constexpr int MAXSP = 88; // species + 1 of the largest network
// row stride (doubles) of the eight-pivot LU's panel columns: even, so that a row's eight entries
// are 16-byte aligned, and 20 words over 64 LDS banks spread the 16 rows of a tile evenly
constexpr int PANEL8 = 10;

// The exp / pow values of the six hand-fitted rate groups, evaluated one per lane of a wavefront and
// broadcast from there (nnet_dev_rates.hpp): NP1 pows of T, NE1 exps of T, NE2 exps of pow values.
// (No array holds them: the Jacobian's is kept for the next attempt.)
namespace spx
{
constexpr int NE1 = 36, NP1 = 13, N1 = NE1 + NP1, NE2 = 6;
}

// Rate slots written by the six hand-fitted rate groups (3-alpha forward/reverse, 12C+12C,
// 12C+16O, 16O+16O, 12C(a,g) forward/reverse, 16O(a,g) forward/reverse).
struct SpecialIdx
{
    int r3a_e, r3a_l, r24, r1216, r32, rcag_e, rcag_l, roag_e, roag_l;
};

// ---------------------------------------------------------------------------------------------
// Kernel configuration per network
// ---------------------------------------------------------------------------------------------
// NT threads per workgroup (one particle), TT x TT tiles of 16 on a WR x WR wave grid, NNZ / IMG
// capacities of the Jacobian pattern and of the LDS assembly image, WPE = waves per SIMD the
// register budget is sized for (net14: 3 measured faster than 4 (spills) and 2 (fewer particles))
template<int NET>
struct Cfg;
template<>
struct Cfg<14>
{
    static constexpr int D = 14, N = 15, NR = 29, NE = 16, NT = 64, TT = 1, WR = 1, NNZ = 72, IMG = 576, WPE = 3;
};
template<>
struct Cfg<86>
{
    static constexpr int D = 86, N = 87, NR = 309, NE = 157, NT = 256, TT = 6, WR = 2, NNZ = 800, IMG = 5248, WPE = 2;
};
template<>
struct Cfg<87>
{
    static constexpr int D = 87, N = 88, NR = 311, NE = 157, NT = 256, TT = 6, WR = 2, NNZ = 800, IMG = 5248, WPE = 2;
};

// LDS of one workgroup, in doubles (the assembly image is a separate array of IMG words)
template<int NET, bool MIX>
struct Lds
{
    using C = Cfg<NET>;
    static constexpr int D = C::D, N = C::N, NR = C::NR, NE = C::NE;
    static constexpr int NU = N * (N + 1) / 2; // packed normalised rows (columns k+1 .. N)
    static constexpr int NL = N * (N - 1) / 2; // packed multipliers (columns 0 .. k-1)
    // head: rate and mass-action arrays, dead once the Jacobian is summed (the NR words at oJok are
    // spare: a reaction without derivative holds zeros at oTr)
    static constexpr int oMu = 0, oEff = oMu + D, oDeff = oEff + NE, oL = oDeff + NE, oDl = oL + NE,
                         oRate = oDl + NE, oDrate = oRate + NR, oVal = oDrate + NR, oDval = oVal + NR,
                         oTr = oDval + NR, oJok = oTr + NR * MAXQ, headEnd = oJok + NR;
    // FP32 factors of the mixed path (U rows, multipliers, pivot reciprocals), in doubles
    static constexpr int f32Words = MIX ? (NU + NL + N + 1) / 2 : 0;
    // tail: what the matrix fill and the FP64 refinement residual read; behind the factors, because
    // the next iteration reads it again when it linearises at the same state
    static constexpr int factorEnd = MIX ? f32Words : NU;
    static constexpr int oBE = (headEnd > factorEnd ? headEnd : factorEnd), oDYdot = oBE + D, oDYdT = oDYdot + D,
                         oCorr = oDYdT + D, oEv = oCorr + D, oEos = oEv + 12, oJv = oEos + 4,
                         phaseEnd = oJv + C::NNZ;
    // the FP64 packed rows alias the head once the matrix sits in registers; the eight-pivot LU's
    // (net86 / net87, FP64) operand loads also address the tiles' padding columns behind them
    static constexpr int NPAD = 16 * C::TT;
    static constexpr bool LU8 = C::TT > 1 && !MIX;
    static constexpr int uWords = LU8 ? NPAD * (NPAD - 1) / 2 : NU;
    static constexpr int unionSize = phaseEnd > uWords ? phaseEnd : uWords;
    static constexpr int oY = unionSize, oYb = oY + D, oX = oYb + D, oRow0 = oX + N + 1;
    // LU panel buffers (two generations of: panel columns [row][4], pivot rows [column][4]); after
    // the LU they hold the refinement residual.  Eight-pivot LU: two generations of panel columns
    // [row][PANEL8] (its pivot rows go straight into the packed rows).
    static constexpr int oPan = ((oRow0 + (MIX ? N + 1 : 0)) + 3) & ~3, panWords = (LU8 ? 2 * PANEL8 : 16) * NPAD,
                         oCyc = oPan + panWords,
                         total = (oCyc + 3 * (C::NT / 64) + 1) & ~1; // a Cycle per wavefront
};

// Exact cycles of rejected attempts.  A rejected attempt restarts from the same accepted state, so
// all that follows until the next acceptance is a function of the attempt's (dt, T_buffer) alone:
// when a pair comes back bit for bit, the attempts between the two visits repeat until the
// Newton-iteration cap.  A pair that comes back at once is status STALLED; for longer periods the
// controller counts the whole periods that fit under the cap and runs only the rest, ending in the
// state and with the counts that running them all ends in.  The pair kept for comparison is
// replaced after windows of doubled length (Brent, BIT 20, 176, 1980), which finds any period
// within a few times max(period, lead-in).
struct Cycle
{
    uint64_t dt, Tb;  // bits of the kept pair
    uint32_t it, lim; // iteration at which it was kept, length of its window (0: none kept)
};
static_assert(sizeof(Cycle) == 24, "three LDS doubles");

// After a rejection at iteration `total` that leaves the pair (dt, Tb): the iterations of whole
// periods to count without running them (0: no period known).  At least one iteration is left
// to run, so the cap ends the particle as it always does.
__attribute__((always_inline)) constexpr long cycle_skip(Cycle& c, uint64_t dt, uint64_t Tb, long total, long max_iter)
{
    const uint32_t since = (uint32_t)total - c.it;
    if (c.lim != 0 && c.dt == dt && c.Tb == Tb)
    {
        const long     rem  = max_iter - 1 - total; // max_iter <= 0: no cap
        const uint32_t skip = rem > 0 ? (uint32_t)(rem < 0x7fffffffL ? rem : 0x7fffffffL) / since * since : 0;
        c.it += skip;
        return (long)skip;
    }
    if (c.lim == 0 || since >= c.lim)
    {
        c.dt  = dt;
        c.Tb  = Tb;
        c.it  = (uint32_t)total;
        c.lim = c.lim == 0 ? 1 : c.lim < 0x40000000u ? 2 * c.lim : c.lim;
    }
    return 0;
}

// The work queue of a launch is a 32-bit count of the positions taken so far; every particle group
// takes one past the end before it stops.  How often the queue runs over its nq particles in a launch
// of `groups` particle groups: twice (dense particles first, solve_particles) without an order and with
// more particles than start at once, but only where twice the count still fits.
__attribute__((always_inline)) constexpr uint32_t queue_passes(uint32_t nq, uint32_t groups, bool ordered)
{
    return !ordered && nq > groups && nq <= (0xffffffffu - groups) / 2 ? 2 : 1;
}
// A second pass takes every position again, and positions come at one atomic each (11.4 ns on one
// address, however many groups ask), so it is left out where it cannot pay: where half of the particles
// do not burn and taking positions is much of the call, and where the particles that burn are all of one
// kind.  Of PLAN_SAMPLE particles spread over the batch `idle` do not burn and `dense` burn and are
// dense.  Two passes against one: 50,021 net14 particles, all idle, 1.19 ms against 0.63; 1,000,000 of
// net86, nine in ten idle, 28.6 against 19.8; 100,000 of net86 that take two iterations each, 20 / 50 / 80%
// of them idle, 14.1 / 9.0 / 4.4 against 13.9 / 8.9 / 3.8.  What it gains with capped particles: solve_particles.
constexpr uint32_t PLAN_SAMPLE = 256;
constexpr bool     dense_first_pays(uint32_t idle, uint32_t dense)
{
    return 2 * idle <= PLAN_SAMPLE && dense > 0 && idle + dense < PLAN_SAMPLE;
}
// Particles of one launch at most, on a device of n_cu compute units (32 wavefronts each).
constexpr uint64_t queue_limit(uint32_t n_cu) { return 0xffffffffull - 32ull * n_cu; }

// Place of a particle in an ordered call, highest first: the bit length of its count (an earlier
// step's Newton iterations).  A dense particle that burns and has no count yet (a first step) goes
// first, as in a call without an order: 60,013 net86 particles, two steps at cap 2,000: 91.2 -> 86.2 ms.
// A cold one's count stays 0 in every step; it goes last, not in front of the long ones (four long net14
// particles among 1,000,000 cold dense ones: 18.8 -> 17.4 ms).
constexpr int NBUCKET = 32;
__attribute__((always_inline)) constexpr int order_bucket(uint32_t count, bool dense_burning)
{
    if (count == 0) return dense_burning ? NBUCKET - 1 : 0;
    const int b = 32 - __builtin_clz(count);
    return b < NBUCKET ? b : NBUCKET - 1;
}

// Jacobian non-zero slot (position in the image's descending-length order) that lane `tid` of a
// particle's NT lanes sums in pass `pass`, or a value >= nnz when it has none: pass p takes slot
// tid + NT p; with four wavefronts the slots beyond three full passes go to wavefront 1 (no species
// lanes, the lightest load of that phase) rather than to wavefront 0, which holds the longest lists.
constexpr int jac_slot(int tid, int pass, int NT, int nnz)
{
    int k = tid + NT * pass;
    if (NT == 256 && pass >= 3) k = (tid >> 6) == 1 ? 3 * NT + 64 * (pass - 3) + (tid - 64) : nnz;
    return k;
}

// Matrix row held by register v of lane (lr = (l & 63) >> 4, lc = l & 15) in tile row I of the
// register-resident Newton matrix, and its column in tile column J (the v_mfma_f64_16x16x4f64
// result layout).
constexpr int tile_row(int I, int lr, int v) { return 16 * I + lr + 4 * v; }
constexpr int tile_col(int J, int lc) { return 16 * J + lc; }

// Index functions of the tile LU (blocks of four pivots) and of its triangular solves.
template<int NET>
struct LuIdx
{
    using C = Cfg<NET>;
    static constexpr int N = C::N, TT = C::TT, WR = C::WR, TI = TT / WR, NPAD = 16 * TT;
    static constexpr int NS = (N + 3) / 4; // blocks of four pivots

    // normalised upper entry (k, j), k < j <= N: net86 / net87 pack it by columns (column j holds
    // rows 0 .. j-1, so the back substitution's lanes read consecutive words: measured faster),
    // net14 by rows (row k holds columns k+1 .. N: its single wavefront's LU stores are then the
    // consecutive ones, measured faster there); first packed entry of multiplier row k (columns
    // 0 .. k-1)
    static constexpr int uidx(int k, int j)
    {
        return NET == 14 ? k * N - k * (k - 1) / 2 - k - 1 + j : j * (j - 1) / 2 + k;
    }
    static constexpr int lrow(int k) { return k * (k - 1) / 2; }
    // panel buffers of block `step`: generation (step & 1) of [row][4] panel columns P, followed
    // by [column][4] pivot rows RT
    static constexpr int pan(int step) { return (step & 1) * 8 * NPAD; }
    static constexpr int pcol(int step, int row, int q) { return pan(step) + row * 4 + q; }
    static constexpr int prow(int step, int col, int q) { return pan(step) + 4 * NPAD + col * 4 + q; }
    static constexpr int trow(int I, int lr, int v) { return tile_row(I, lr, v); }
    static constexpr int tcol(int J, int lc) { return tile_col(J, lc); }
    // A-operand row m of a tile: FP64 MFMA rows come in result order; the FP32 MFMA returns row
    // 4(l>>4) + v in register v, so with the FP64 placement A-operand row m is (m>>2) + 4(m&3)
    static constexpr int arow(bool fp32, int m) { return fp32 ? (m >> 2) + 4 * (m & 3) : m; }
};

// Index functions of the eight-pivot LU (net86 / net87, FP64): block B eliminates pivots 8B ..
// 8B + 7 (B even: the first half of tile row / column B/2, B odd: the second half).
template<int NET>
struct Lu8Idx
{
    using C = Cfg<NET>;
    static constexpr int N = C::N, NPAD = 16 * C::TT;
    static constexpr int NB = (N + 7) / 8; // blocks
    // panel column q of block B in generation (B & 1) of the panel buffers
    static constexpr int pcol(int B, int row, int q) { return (B & 1) * PANEL8 * NPAD + row * PANEL8 + q; }
    // normalised upper entry (k, j), k < j < NPAD, packed by columns as LuIdx::uidx packs it
    static constexpr int uidx(int k, int j) { return j * (j - 1) / 2 + k; }
    // waves that hold trailing rows (lane row 8B + 8 + 64 w + lane) and columns (lane column 8B +
    // 1 + 64 w + lane, so that the block's own columns are normalised by the same lanes)
    static constexpr int row0(int B) { return 8 * B + 8; }
    static constexpr int col0(int B) { return 8 * B + 1; }
    static constexpr int rowWaves(int B) { return row0(B) >= N ? 0 : (N - row0(B) + 63) / 64; }
    static constexpr int colWaves(int B) { return (N + 1 - col0(B) + 63) / 64; }
};
} // namespace nnet_amd
