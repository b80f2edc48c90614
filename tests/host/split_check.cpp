// split_slice (pixienn_amd/csrc/grouped.h) on the host, over slices, channel counts and places of a stream.
#include "../../pixienn_amd/csrc/grouped.h"

#include <cstdio>

using namespace pxh;

namespace {

int failed = 0, checks = 0;

void check(bool good, const char* what, size_t items, size_t channels, uint32_t places)
{
    ++checks;
    if (!good && ++failed < 10) std::printf("%s: %zu items, %zu channels, %u places\n", what, items, channels, places);
}

}  // namespace

int main()
{
    const uint32_t per_member = kGroupItems;
    for (uint32_t places: { 0u, 2u, 8u, 16u, 64u, 510u, 512u, 608u })
        for (size_t channels: { 1, 2, 3, 5, 7, 8, 16, 31, 64, 95, 512, 1024 })
            for (size_t workgroups: { kGroupFill, static_cast<size_t>(1) })
                for (size_t items = 1; items < 2000000; items += items < 20000 ? 61 : items / 7) {
                    const GroupPlan p = split_slice(items, per_member, channels, workgroups, places);
                    if (!p.members) continue;
                    check(p.members <= kGroupMost && p.members * kGroupShare <= places, "an eighth of the places", items, channels, places);
                    check(p.span % kWave == 0 && p.span <= per_member, "a member holds its share", items, channels, places);
                    check(static_cast<size_t>(p.span) * p.members >= items, "every item has a member", items, channels, places);
                    check(static_cast<size_t>(p.span) * (p.members - 1) < items, "every member has items", items, channels, places);
                }

    uint32_t mask[4] = {};
    check(units_of_mask(mask, 4, 256) == 256, "no mask", 0, 0, 0);
    mask[0] = 0x0F0Fu;
    mask[3] = 0x80000000u;
    check(units_of_mask(mask, 4, 256) == 9, "a mask", 0, 0, 0);
    for (uint32_t& m: mask) m = ~0u;
    check(units_of_mask(mask, 4, 104) == 104, "a mask of more units than there are", 0, 0, 0);
    std::printf("%d checks, %d failed\n", checks, failed);
    return failed != 0;
}
