// The prefill attention's division of work (k_attn_prefill.hip): the keys a
// tile of (query row, head) pairs attends, and the tiles' width and key parts.
// Plain C++: a host test sweeps the plan over shapes, windows and CU counts.
#pragma once

#include <cmath>
#include <stdint.h>

#if defined(__HIPCC__)
#define MG_PP __host__ __device__ inline
#else
#define MG_PP inline
#endif

namespace mg
{
    constexpr int kPfKeys = 64; // keys per step

    struct PfArgs
    {
        int64_t nkv, ldq, ldo, slots, pos0, window;
        uint32_t npair, hpg, nqt; // T * hpg (row, head) pairs a kv head, heads per kv head, pair tiles
        uint32_t hw;              // heads of a row's start group (pf_span): hpg's largest divisor <= 8
        uint32_t nfirst;          // shortest tiles that start ahead of the others
        uint32_t lw;              // log2 of the pairs per tile (work-group)
        int parts, per;           // key parts per tile, steps per part
        float scale2;             // |scaling| * log2(e), 2^-126 in place of 0
        uint32_t qsign;           // 0x80008000 when scaling < 0: q enters with its sign flipped
    };

    // The keys a pair tile works over: [klo, klo + span], up to its last live
    // pair's position. With a window klo is the window start of the row that
    // opens the tile's group of 256 (row, head) pairs, `hw` heads a row: a row's
    // 64-key steps, and with them its weights' reference (k_attn_prefill), then
    // lie the same whatever tile width and key parts a call takes. (16 or 24 rows
    // ahead of the tile for 16 heads a row, 26 for 5 and 128 for one where tiles
    // are narrow: no step more of 17 at a 1024-key window, two for one head a row.)
    struct PfSpan
    {
        int64_t klo;
        int span;
    };
    MG_PP PfSpan pf_span(int64_t pos0, int64_t window, uint32_t hpg, uint32_t hw, uint32_t pb0, uint32_t pl)
    {
        const uint32_t row = pb0 / hpg, at = row * hw + (pb0 - row * hpg) % hw;
        const int64_t p0 = pos0 + (at & ~255u) / hw;
        const int64_t klo = window > 0 && p0 - window + 1 > 0 ? p0 - window + 1 : 0;
        return {klo, int(pos0 + pl / hpg - klo)};
    }

    // The most any tile of PW pairs reaches past its first key (a bound on
    // pf_span's span). Without a window that is the last position. With one, the
    // tile's rows add to the window's keys: its own PW pairs, from any pair of a
    // row on, lie in at most (PW + hpg - 2) / hpg rows past its first, and its
    // group opens less than 256 / hw rows ahead of that. (The end tiles alone do
    // not give it: the first may start before the window fills, the last may hold
    // few rows.)
    inline int64_t pf_longest(int64_t pos0, int64_t window, uint32_t hpg, uint32_t hw, uint32_t npair, uint32_t PW)
    {
        const int64_t T = int64_t(npair) / hpg, last = pos0 + T - 1;
        if (window <= 0 || window > last) return last;
        const int64_t ahead = PW == 256 && hw == hpg ? 0 : (254 + int64_t(hw)) / hw; // such tiles are the groups
        const int64_t rows = (int64_t(PW) + hpg - 2) / hpg + ahead;
        const int64_t most = window - 1 + (rows < T - 1 ? rows : T - 1);
        return most < last ? most : last;
    }

    // Pairs per tile, parts per tile and steps per part. One 256-pair
    // work-group a tile leaves CUs idle when the tiles are few: then tiles of
    // half as many pairs (four waves instead of eight, one a SIMD, a step in
    // about 0.65 of the time; only in one round, as two of them take longer
    // than one of 256 pairs) or, behind long contexts (100 tokens of 32 / 2
    // heads: 26 tiles of 142 steps), the tiles' keys in parts that a second
    // kernel merges, or both. Priced in 256-pair steps (about 1.8 us): a plan
    // runs for its longest part times the rounds of work-groups the parts
    // make; a split adds kMergeSteps for the second launch and the partials'
    // round trip (D + 2 f32 a pair and part, written and read).
    inline void pf_plan(PfArgs &a, int cus, int64_t work_bytes, int64_t D)
    {
        constexpr double kMergeSteps = 3.0, kBytesPerStep = 8.0e6, kNarrowStep = 0.65;
        a.parts = 1;
        a.per = 0;
        a.nfirst = 0;
        a.hw = a.hpg;
        while (a.hw > 8 || a.hpg % a.hw != 0) --a.hw;
        double best = 0.0;
        for (uint32_t lw = 8; lw >= 7; --lw) {
            const uint32_t PW = 1u << lw, nqt = uint32_t((int64_t(a.npair) + PW - 1) >> lw), pl = a.npair - 1;
            const int64_t tiles = int64_t(nqt) * a.nkv;
            const double step = lw == 8 ? 1.0 : kNarrowStep;
            const int64_t reach = pf_longest(a.pos0, a.window, a.hpg, a.hw, a.npair, PW);
            const int64_t longest = reach / kPfKeys + 1;
            // the tiles' steps together: from the first tile's on, a step more every
            // 64 positions until the window fills (at `reach`), the same after it
            // (from the end tiles alone 4096 tokens of 7 / 7 heads of 64 in a window of
            // 1024 took three parts a tile in two rounds, 44.3 us: 25.7 unsplit)
            const PfSpan first = pf_span(a.pos0, a.window, a.hpg, a.hw, 0, PW - 1 < pl ? PW - 1 : pl);
            const double from = double(first.span), to = double(a.pos0 + pl / a.hpg), full = double(reach);
            const double mean = to <= full || to <= from ? 0.5 * (from + (to < full ? to : full))
                                                         : full - 0.5 * (full - from) * (full - from) / (to - from);
            const double total = double(tiles) * (mean / kPfKeys + 0.75);
            const double evened = std::ceil(double(tiles) / cus) * total / double(tiles);
            const double whole = (double(longest) > evened ? double(longest) : evened) * step;
            if (lw == 8 || (whole < best && tiles <= cus)) {
                best = whole;
                a.lw = lw;
                a.nqt = nqt;
                a.parts = 1;
            }
            if (tiles >= 2 * cus) return; // the tiles fill the chip on their own
            for (int64_t parts = 2; parts <= 256 && parts <= longest; parts += parts < 16 ? 1 : parts / 8) {
                const int64_t per = (longest + parts - 1) / parts;
                const int64_t np = (longest + per - 1) / per;
                if ((tiles * np << lw) * (D + 2) * int64_t(sizeof(float)) > work_bytes) break;
                const double some = total / double(per) + 0.5 * double(tiles); // parts holding keys
                const double live = some < double(tiles * np) ? some : double(tiles * np);
                const double bytes = 2.0 * live * double(a.npair < PW ? a.npair : PW) * double(D) * 4.0;
                const double t = double(per) * std::ceil(live / cus) * step + kMergeSteps + bytes / kBytesPerStep;
                if (t < best && (lw == 8 || live <= cus)) {
                    best = t;
                    a.lw = lw;
                    a.nqt = nqt;
                    a.parts = int(np);
                    a.per = int(per);
                }
            }
        }
    }
} // namespace mg
