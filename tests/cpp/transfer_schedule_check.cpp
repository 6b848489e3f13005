// Host-only check of the waits in the large-tile kernel's K loop where operands are not pipelined, the fp8 down GEMM
// (big_unit_of_step, big_pair_of_step, big_units_may_fly in therock_amd/csrc/common.hpp; pipelined_schedule_check.cpp walks
// the loop with int8 weights): the transfers of a weight-role wave land in the order they were issued, a wait for "at most n
// in flight" guarantees all but the last n, and what has landed at the barrier of a step must hold the unit pair the step
// reads; what a step issues must not go into a ring slot that is still to be read.  Exit code 0 = all hold.
#include <algorithm>
#include <cstdio>
#include <vector>

#include "../../therock_amd/csrc/common.hpp"

int main()
{
    using namespace mi355;
    constexpr int kSlots = 6, kInstructions = 4; // units in the ring, transfers per unit and wave
    int failures         = 0;
    for(int kt_count = 2; kt_count <= 256; kt_count += 2) // whole weight lines
    {
        const int units = kt_count;
        std::vector<int> slot(kSlots, -1); // unit last sent to each slot
        std::vector<int> issued;
        auto issue = [&](int u, int k) {
            if(u >= units)
                return;
            if(slot[u % kSlots] >= 0 && slot[u % kSlots] >= big_pair_of_step(k, false)) // read in this step or later
                failures += std::printf("overwritten: steps=%d step=%d unit=%d\n", kt_count, k, u) > 0;
            slot[u % kSlots] = u;
            issued.push_back(u);
        };
        for(int u = 0; u < 4; u++)
            issue(u, 0);
        int landed = 0; // of issued
        for(int k = 0; k < kt_count; k++)
        {
            const int in_flight = big_units_may_fly(k, kt_count, false) ? (k & 1 ? 12 : 8) / kInstructions : 0;
            landed              = std::max(landed, (int)issued.size() - in_flight);
            for(int u : {big_pair_of_step(k, false), big_pair_of_step(k, false) + 1})
            {
                const auto at = std::find(issued.begin(), issued.end(), u);
                if(at == issued.end() || at - issued.begin() >= landed)
                    failures += std::printf("not landed: steps=%d step=%d unit=%d\n", kt_count, k, u) > 0;
            }
            issue(big_unit_of_step(k, false), k);
        }
        if((int)issued.size() != units)
            failures += std::printf("units left out: steps=%d\n", kt_count) > 0;
    }
    if(failures == 0)
        std::printf("transfer_schedule_check ok\n");
    return failures == 0 ? 0 : 1;
}
