// Reads "first rows window query-heads kv-heads head-dim" lines, writes "pairs parts" for 256 compute units: parts up to
// 32 in 128 MiB, then none.
#include "../wayruntime_amd/csrc/prefill_plan.h"
#include <cstdio>

int main()
{
    wr::PrefillSizes s;
    while (scanf("%u %u %u %u %u %u", &s.p0, &s.T, &s.window, &s.nq, &s.nkv, &s.hd) == 6) {
        const wr::PrefillPlan p = wr::prefill_plan(s, 256, true, 32, 128ull << 20), whole = wr::prefill_plan(s, 256, true, 1, 0);
        const wr::PrefillPlan fours = wr::prefill_plan(s, 256, false, 32, 128ull << 20);
        const unsigned wrong = whole.parts != 1 || fours.parts != 1 || fours.np != 4 || (p.parts > 1 && !p.single) || (p.np == 2 && !p.single) ||
                               p.nblk * (32 * (p.np / (s.nq / s.nkv < p.np ? s.nq / s.nkv : p.np))) < s.T;
        printf("%u %u %u\n", p.np, p.parts, wrong);
    }
}
