// Host-only check of the large-tile kernel's pipelined K loop with weights that last four steps (int8 x bf16): the barrier of
// step k has to guarantee the unit pair that step k + 1 reads, at most two units in flight while big_units_may_fly(k + 1) and
// none otherwise; what step k issues must not go into a slot that step k + 1 or a later one reads.  Step counts of whole
// 128-byte weight windows and of a half last one.  Exit code 0 = all hold.
#include <algorithm>
#include <cstdio>
#include <vector>

#include "../../therock_amd/csrc/common.hpp"

int main()
{
    using namespace mi355;
    constexpr int kSlots = 6;
    int failures         = 0;
    for(int kt_count = 2; kt_count <= 256; kt_count += 2)
    {
        const int units = (kt_count + 2) / 4 * 2;
        std::vector<int> slot(kSlots, -1), issued;
        auto issue = [&](int u, int k) {
            if(u >= units)
                return;
            if(slot[u % kSlots] >= big_pair_of_step(k + 1, true))
                failures += std::printf("overwritten: steps=%d step=%d unit=%d\n", kt_count, k, u) > 0;
            slot[u % kSlots] = u;
            issued.push_back(u);
        };
        for(int u = 0; u < 4; u++)
            issue(u, -1);
        int landed  = 0;
        auto needed = [&](int step, int in_flight) {
            landed = std::max(landed, (int)issued.size() - in_flight);
            for(int u : {big_pair_of_step(step, true), big_pair_of_step(step, true) + 1})
            {
                const auto at = std::find(issued.begin(), issued.end(), u);
                if(at == issued.end() || at - issued.begin() >= landed)
                    failures += std::printf("not landed: steps=%d step=%d unit=%d\n", kt_count, step, u) > 0;
            }
        };
        needed(0, units >= 4 ? 2 : 0); // the wait ahead of the loop
        for(int k = 0; k < kt_count; k++)
        {
            if(k + 1 < kt_count)
                needed(k + 1, big_units_may_fly(k + 1, kt_count, true) ? 2 : 0);
            if(k % 2 == 0)
                issue(big_unit_of_step(k, true), k);
        }
        if((int)issued.size() != units)
            failures += std::printf("units left out: steps=%d\n", kt_count) > 0;
    }
    if(failures == 0)
        std::printf("pipelined_schedule_check ok\n");
    return failures == 0 ? 0 : 1;
}
