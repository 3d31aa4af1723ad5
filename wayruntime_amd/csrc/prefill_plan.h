// How a prefill launch is cut: chosen from the sizes alone, on the host (plain C++: tests compile it by itself).
#pragma once

#include <algorithm>
#include <cstdint>

namespace wr {

struct PrefillSizes {
    uint32_t p0, T, window;          // first position, rows, keys a row sees (0: all)
    uint32_t nq, nkv, hd;            // hd 64, 128 or 256; nq / nkv 1, 2, 4 or 8
};

// (head, 32-row block) pairs to a workgroup, position blocks and the workgroups of each, whether a workgroup has one block
// or a long and a short one, and into how many parts the blocks' keys go (one: not at all).
struct PrefillPlan {
    uint32_t np, nblk, ny, parts;
    bool single;
};

// Four pairs to a workgroup feed eight waves, two to a SIMD, from each tile: the form for launches that fill the chip.  Launches
// of fewer workgroups than CUs last as long as their longest block; with two pairs a workgroup has half the rows, a wave to
// a SIMD whose steps take 0.74 to 0.87 of the time, and there are twice as many.  A launch whose longest block is still a long chain
// is cut into parts: every part pays a block's ends (Q in, the sets' merge, rows out) and the rows go through memory once more.
// In microseconds: the ends of a block, a step (64 keys of a 32-row unit at head dims up to 128, 32 keys at 256) and the tiles' way into LDS in
// either form, the combine launch, what it takes a part and eight of them beyond the first (it asks for eight at a time: 32/8/64, 3 rows behind 4000 keys, 8 parts
// 11.0 us, 9 12.2), and the bytes it and the parts move.
// Blocks without a window, or before it is full, are of unequal length, and the long ones go first: the short ones of a second round fill in behind
// one another, so that of one to two rounds a unit's two blocks last as long as any other's.  (Counted as whole rounds of mean length, launches of a
// few more workgroups than CUs were left to four pairs: 16/8/256, 1501 rows 53 us, in twos 42; 8/8/128, 3000 rows 46 and 37; 16/8/128, 1501
// rows 29.0 and 25.2.)  At head dim 64 two workgroups of two pairs fit a CU: one that shares it takes 1.49 of a step, and 512 are a
// round (16/16/64, 1501 rows 21.9 us in fours, 18.2; 3000 39.0 and 33.7).
// Fitted to eleven shapes by thirteen row counts by nine contexts and windows, both forms, 1 to 32 parts (profiles/prefill_parts.txt has all
// of them, with what is picked and what was picked of four pairs alone): what is picked is 0.2 to 0.5 % off the best on average, 25 % at worst, and takes 0.90 (64), 0.92
// (128) and 0.91 (256) of what the parts picked for four pairs alone take; more than 2.5 % more at two sizes (8/2/256, 2048 rows of a window of 128
// behind 100 keys, 256 workgroups on 256 CUs: 18.6, 20.0; 8/4/256, 33 rows behind 16 000 keys: 31.0, 33.2).
// `parts`: most parts; `twos`: whether workgroups of two pairs are there; `room`: bytes for the parts' rows.
inline PrefillPlan prefill_plan(const PrefillSizes& a, uint32_t n_cus, bool twos, uint32_t parts, uint64_t room)
{
    constexpr uint32_t kKeys = 32;   // of a tile
    struct Cost {
        float ends[2], step[2], tile_mb[2];        // two pairs, four
        float combine, trip, part, mb_us;
        float pair;                                // saved where the second block's first loads are on their way early
        float over, tail;                          // ends of a round behind another; how much of the last round stays empty
        float shared_ends, shared_step;            // of two pairs: two workgroups on a CU
    };
    const Cost c = a.hd == 64    ? Cost{{7.69f, 8.53f}, {0.563f, 0.759f}, {0.00927f, 0.00917f}, 4.47f, 0.726f, 0.236f, 2.96f, 1.55f, 1.13f, 0.552f, 1.09f, 1.49f}
                   : a.hd == 128 ? Cost{{7.2f, 10.2f}, {0.602f, 0.693f}, {0.00964f, 0.0105f}, 2.48f, 0.8f, 0.127f, 3.3f, 2.05f, 0.9f, 0.588f, 1.f, 1.f}
                                 : Cost{{8.67f, 9.11f}, {0.828f, 1.04f}, {0.0101f, 0.00971f}, 2.14f, 0.98f, 0.281f, 4.f, 2.29f, 1.11f, 0.486f, 1.f, 1.f};
    const uint32_t group = a.nq / a.nkv, per_step = a.hd == 256 ? 1 : 2;
    const float row_mb = (float)a.T * a.nq * a.hd * 4e-6f, cus = (float)n_cus;
    const uint64_t row_bytes = (uint64_t)a.T * a.nq * (a.hd + 2) * 4;
    PrefillPlan best{};
    float least = 0.f;
    for (uint32_t np = 4; np >= (twos ? 2u : 4u); np -= 2) {
        const uint32_t Gw = std::min(group, np), BP = 32 * (np / Gw);
        const uint32_t nblk = (a.T + BP - 1) / BP, ny = a.nkv * (group / Gw);
        const float ends = c.ends[np / 4], step = c.step[np / 4];
        // tiles of the first and the last block, and of a block on average: as many as the last from where the window is full on
        const auto tiles_of = [&](uint32_t b) {
            const uint32_t lo = a.p0 + b * BP, hi = a.p0 + std::min(a.T, (b + 1) * BP);
            const uint32_t from = (a.window > 0 && lo + 1 > a.window) ? lo + 1 - a.window : 0;
            return (hi + kKeys - 1) / kKeys - from / kKeys;
        };
        const uint32_t first = tiles_of(0), longest = std::max(first, tiles_of(nblk - 1));
        const float ramp = a.window == 0 ? 1.f : a.window > a.p0 ? std::min(1.f, (float)(a.window - a.p0) / a.T) : 0.f;
        const float mean = longest - ramp * (longest - first) * 0.5f;
        const float tiles_us = c.tile_mb[np / 4] * nblk * ny * mean * a.hd * 1.28e-4f;
        // Four pairs: a long and a short block to a workgroup balance the causal triangle, but each pays its own
        // prologue and epilogue: when the pairs of blocks would not even give every CU a workgroup, one block per workgroup
        // finishes with the longest block instead of with a pair's sum plus a second prologue and epilogue.
        const uint32_t two = (nblk + 1) / 2 * ny;
        const bool single = np == 2 || two < n_cus, sharing = np == 2 && a.hd == 64;
        for (uint32_t p = 1; p <= (twos && single ? std::min(parts, longest) : 1u); p++) {
            if (p > 1 && p * row_bytes > room) break;
            // (many parts on all CUs but a few: 4/1/256, 177 rows behind 16 000 keys, 252 workgroups 40.3 us, 240 36.3)
            if (p > 16 && np == 2 && a.hd == 256 && (uint64_t)nblk * ny * p * 16 > (uint64_t)n_cus * 15) break;
            float t;
            if (!single) {
                t = ((two + n_cus - 1) / n_cus) * (2.f * ends - c.pair + step * 2.f * mean / per_step);
            } else {
                const float W = (float)((uint64_t)nblk * ny * p), round = sharing ? 2 * cus : cus;
                const float last = (float)longest / (p * per_step), less = (float)(longest - first) / (p * per_step);   // a long block's steps, how many fewer a short one's
                const float even = (1.f - ramp) * W;                   // blocks as long as the longest
                const float steps = (float)(((longest + p - 1) / p + per_step - 1) / per_step);
                const float shared = step * (sharing ? c.shared_step : 1.f);
                if (W <= cus) {
                    t = ends + step * steps;
                } else if (W <= round) {                               // the longest shares its CU with the first of the second half
                    t = ends * c.shared_ends + step * (steps + (c.shared_step - 1.f) * (last - (W > even ? std::max(0.f, (cus - even) / (W - even)) * less : 0.f)));
                } else {
                    const float over = ends * c.over;
                    if (W <= 2 * round)
                        t = 2.f * over + shared * (2.f * last - (W > even ? std::max(0.f, 2.f * (round - even) / (W - even)) * less : 0.f));
                    else
                        t = W / round * (over + shared * mean / (p * per_step)) +
                            ((float)(uint32_t)((W + round - 1.f) / round) - W / round) * (over + shared * (last - less)) * c.tail;
                    t = std::max(t, ends + step * steps);
                }
                t += tiles_us;
            }
            if (p > 1) t += c.combine + c.trip * ((p + 7) / 8 - 1) + c.part * p + 2.f * p * row_mb / c.mb_us;
            if (best.np == 0 || t < least) {
                least = t;
                best = PrefillPlan{np, nblk, ny, p, single};
            }
        }
    }
    return best;
}

}  // namespace wr
