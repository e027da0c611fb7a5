// Sweeps the prefill attention's plan (csrc/mg_prefill_plan.hpp) over shapes,
// windows, CU counts and workspaces: prints the number of plans, how many of
// them split the keys (windowed ones apart), and how many break a rule:
//   every tile's keys lie in its parts (a split part beyond the plan would read
//   another tile's slots), the parts' partials fit the workspace, the tiles hold
//   every pair, and the bound on a tile's reach holds.
// One argument list T nq nkv pos0 window: that shape's plan alone (256 CUs, 64 MiB).
#include "mg_prefill_plan.hpp"

#include <cstdio>
#include <cstdlib>
#include <random>

static bool bad_plan(const mg::PfArgs &a, int64_t work, int64_t D)
{
    const uint32_t PW = 1u << a.lw;
    if (int64_t(a.nqt) * PW < a.npair || int64_t(a.nqt - 1) * PW >= a.npair) return true;
    if (a.parts > 1 && (int64_t(a.nqt) * a.nkv * a.parts << a.lw) * (D + 2) * 4 > work) return true;
    const int64_t longest = mg::pf_longest(a.pos0, a.window, a.hpg, a.hw, a.npair, PW);
    for (uint32_t qt = 0; qt < a.nqt; ++qt) {
        const uint32_t pb0 = qt << a.lw, pl = (pb0 + PW < a.npair ? pb0 + PW : a.npair) - 1;
        const mg::PfSpan s = mg::pf_span(a.pos0, a.window, a.hpg, a.hw, pb0, pl);
        // rows of other tiles' windows may open the keys, but none the call does not attend
        const int64_t lo0 = a.window > 0 && a.pos0 - a.window + 1 > 0 ? a.pos0 - a.window + 1 : 0;
        if (s.klo < lo0 || (a.window > 0 && s.klo > a.pos0 + pb0 / a.hpg - a.window + 1 && s.klo > 0)) return true;
        if (s.span < 0 || s.span > longest) return true;
        if (a.parts > 1 && s.span / mg::kPfKeys >= int64_t(a.parts) * a.per) return true;
    }
    return false;
}

static mg::PfArgs plan(int64_t T, int64_t nq, int64_t nkv, int64_t pos0, int64_t window, int cus, int64_t work, int64_t D)
{
    mg::PfArgs a{};
    a.nkv = nkv;
    a.pos0 = pos0;
    a.window = window;
    a.hpg = uint32_t(nq / nkv);
    a.npair = uint32_t(T * a.hpg);
    mg::pf_plan(a, cus, work, D);
    return a;
}

int main(int argc, char **argv)
{
    long plans = 0, split = 0, wsplit = 0, bad = 0;
    auto check = [&](int64_t T, int64_t nq, int64_t nkv, int64_t pos0, int64_t window, int cus, int64_t work, int64_t D) {
        const mg::PfArgs a = plan(T, nq, nkv, pos0, window, cus, work, D);
        ++plans;
        split += a.parts > 1;
        wsplit += a.parts > 1 && window > 0;
        bad += bad_plan(a, work, D);
    };
    if (argc == 6)
        check(atoll(argv[1]), atoll(argv[2]), atoll(argv[3]), atoll(argv[4]), atoll(argv[5]), 256, int64_t(64) << 20, 128);
    else {
        std::mt19937_64 rng(7);
        auto upto = [&](int64_t n) { return int64_t(rng() % uint64_t(n)); };
        const int64_t hpgs[] = {1, 2, 3, 4, 5, 6, 7, 8, 9, 16, 40, 130, 300};
        for (long i = 0; i < 2000000; ++i) {
            const int64_t hpg = hpgs[upto(13)], nkv = int64_t(1) << upto(4);
            const int64_t T = 1 + upto(int64_t(1) << (1 + upto(12)));
            const int64_t pos0 = upto(4) == 0 ? 0 : upto(int64_t(1) << (1 + upto(15)));
            const int64_t window = upto(4) == 0 ? 0 : 1 + upto(int64_t(1) << (1 + upto(13)));
            check(T, nkv * hpg, nkv, pos0, window, upto(2) ? 256 : 1 + int(upto(304)), int64_t(4096) << upto(18),
                  upto(2) ? 128 : 64);
        }
        check(100, 40, 8, 50, INT64_MAX, 256, int64_t(64) << 20, 128); // a window no position reaches
    }
    printf("%ld %ld %ld %ld\n", plans, split, wsplit, bad);
}
