// Host-side check of the controller's exact-cycle rule (cycle_skip of nnet_layout.hpp): a controller
// loop over random deterministic maps, with the rule and without it, ends at every cap with the
// same status, state and counts.
#include <cstdio>
#include <random>
#include <vector>

#include "../../sph-exa-nnet_amd/csrc/nnet_layout.hpp"

using namespace nnet_amd;

// One attempt from state x takes cost[x] iterations (more than one: a rejection at a later
// iteration) and leaves the pair of state next[x]; accept[x]: the attempt ends accepted.
struct Map
{
    std::vector<int> next, cost, accept;
};
struct End
{
    int      status; // 0 all substeps accepted, 3 replay, 4 cap
    int      x, part, nsub;
    uint32_t newton;
    long     run; // iterations run
    bool     operator==(const End& o) const
    {
        return status == o.status && x == o.x && part == o.part && nsub == o.nsub && newton == o.newton;
    }
};

static End integrate(const Map& m, int x, long cap, bool rule)
{
    End   e{0, x, 0, 0, 0, 0};
    Cycle c{0, 0, 0, 0};
    long  total = 0;
    for (;;)
    {
        for (e.part = 1;; ++e.part)
        {
            ++total, ++e.newton, ++e.run;
            const int from = e.x;
            if (e.part == m.cost[from]) // the attempt ends
            {
                e.x = m.next[from];
                if (m.accept[from])
                {
                    c.lim = 0;
                    if (++e.nsub == 6) return e;
                }
                else
                {
                    if (e.x == from)
                    {
                        e.status = 3;
                        return e;
                    }
                    if (rule)
                    {
                        // the pair: two words of the state, so that either alone may repeat
                        const long s = cycle_skip(c, (uint64_t)e.x / 3, (uint64_t)e.x % 3, total, cap);
                        total += s;
                        e.newton += (uint32_t)s;
                    }
                }
            }
            if (cap > 0 && total >= cap)
            {
                e.status = 4;
                return e;
            }
            if (e.part == m.cost[from]) break;
        }
    }
}

int main()
{
    std::mt19937 g(7);
    long         bad = 0, capped = 0, run = 0, counted = 0;
    for (int trial = 0; trial < 4000; ++trial)
    {
        Map       m;
        const int n = 1 + (int)(g() % (trial % 3 == 0 ? 6 : trial % 3 == 1 ? 60 : 900));
        for (int x = 0; x < n; ++x)
        {
            m.next.push_back((int)(g() % n));
            m.cost.push_back(1 + (g() % 4 == 0 ? (int)(g() % 11) : 0));
            m.accept.push_back(g() % 40 == 0);
        }
        const int x0 = (int)(g() % n);
        for (long cap : {1L, 2L, 3L, 10L, 99L, 100L, 101L, 1999L, 2000L, 10000L + (long)(g() % 50)})
        {
            const End a = integrate(m, x0, cap, false), b = integrate(m, x0, cap, true);
            if (!(a == b) && bad++ < 20)
                std::printf("FAIL trial %d cap %ld: status %d %d state %d %d substeps %d %d newton %u %u\n", trial, cap,
                            a.status, b.status, a.x, b.x, a.nsub, b.nsub, a.newton, b.newton);
            if (a.status == 4 && cap >= 10000)
            {
                ++capped;
                counted += a.newton;
                run += b.run;
                // Brent's bound: lead-in and period are at most n attempts of at most 11 iterations
                if (b.run > 6L * 11 * n + 64 && b.run < a.run && bad++ < 20)
                    std::printf("FAIL trial %d: %ld iterations run for %d states\n", trial, b.run, n);
            }
        }
        // caps beyond 32 bits: the rule alone reaches them (the last partial period is run)
        Map       two{{1, 2, 1}, {1, 1 + (int)(g() % 3), 1}, {0, 0, 0}};
        const long far = (1L << 33) + (long)(g() % 1000);
        if (trial < 50)
        {
            const End b = integrate(two, 0, far, true);
            if (!(b.status == 4 && b.newton == (uint32_t)far) && bad++ < 20)
                std::printf("FAIL far cap: status %d newton %u\n", b.status, b.newton);
        }
    }
    std::printf("%ld failures; %ld capped runs, %ld iterations counted, %ld run\n", bad, capped, counted, run);
    return bad || capped == 0 || run * 4 > counted ? 1 : 0;
}
