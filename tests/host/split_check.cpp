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

    // the splits that the shapes of tests/test_gpu_shared_slices.py are chosen for
    const struct { size_t items, channels; uint32_t per_member, members, span; } named[] = {
        { 4097, 95, kGroupItems, 2, 2112 }, { 6144, 64, kGroupItems, 3, 2048 }, { 17521, 30, kGroupItems, 8, 2240 },
        { 24579, 12, kGroupItems, 12, 2112 }, { 133120, 8, kGroupItems, 64, 2112 }, { 133120, 7, kGroupItems, 0, 0 },
        { 98304, 32, kGroupItems, 16, kGroupItems }, { 24579, 130, kGroupItems, 5, 4928 }, { 4112, 512, kGroupItems, 1, 4160 },
        { 83160, 96, 4 * kGroupItems, 6, 13888 }, { 180000, 41, 4 * kGroupItems, 13, 13888 },
        { 393215, 32, 4 * kGroupItems, 16, 4 * kGroupItems },
    };
    for (const auto& n: named) {
        const GroupPlan p = split_slice(n.items, n.per_member, n.channels, kGroupFill, 512);
        check(p.members == n.members && p.span == n.span, "the split of a named slice", n.items, n.channels, 512);
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
