// Walks every admitted stack need and LDS stack through the rules that size the traversal's stacks
// (crt_internal.h) and prints how many break one of them.
#include <cstdio>

#include "crt_internal.h"

int main()
{
    using namespace crt;
    long bad = 0, group = 0;
    for (uint32_t need = 0; need <= kStackMax; ++need)
        for (uint32_t lds : {8u, 16u, 32u}) {
            const uint32_t spill = spill_entries(need);
            bad += spill % 32u != 0u || spill > kSpillDepth;
            // a ray per lane: whole LDS stacks spilled, and one in LDS
            bad += spill / lds * lds + lds < need;
            // eight lanes per ray: LDS alone, of a block of kTraceBlock / 8 rays
            if (group_stack_fits(need, lds)) {
                ++group;
                bad += need > lds * kTraceBlock / (kTraceBlock / 8u);
            }
        }
    std::printf("%ld %ld\n", bad, group);
    return 0;
}
