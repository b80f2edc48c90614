// split_slice and group_plan (pixienn_amd/csrc/grouped.h) on the host, over slices, channel counts and places of a stream.
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
            for (size_t workgroups: { group_fill(static_cast<int>(channels)), static_cast<size_t>(1) })
                for (size_t items = 1; items < 2000000; items += items < 20000 ? 61 : items / 7) {
                    const GroupPlan p = split_slice(items, per_member, channels, workgroups, places);
                    if (!p.members) continue;
                    check(p.members <= kGroupMost && p.members * kGroupShare <= places, "an eighth of the places", items, channels, places);
                    check(p.span % kWave == 0 && p.span <= per_member, "a member holds its share", items, channels, places);
                    check(static_cast<size_t>(p.span) * p.members >= items, "every item has a member", items, channels, places);
                    check(static_cast<size_t>(p.span) * (p.members - 1) < items, "every member has items", items, channels, places);
                }

    // workgroups of a whole number of channels, as many as the device runs at once
    for (int channels = 1; channels < 1100; ++channels) {
        const size_t fill = group_fill(channels);
        check(channels > 512 ? fill == 1 : fill % channels == 0 && fill <= 512 && fill + channels > 512, "whole channels", fill, channels, 512);
    }

    // the splits that the shapes of tests/test_gpu_shared_slices.py and of tests/test_gpu_odd_planes.py are chosen for
    const struct { int batch, channels, spatial; bool vec; uint32_t items, members, span; } named[] = {
        { 1, 95, 16388, true, 4097, 2, 2112 }, { 4, 64, 6144, true, 6144, 3, 2048 }, { 7, 30, 10012, true, 17521, 8, 2240 },
        { 3, 12, 32772, true, 24579, 12, 2112 }, { 1, 8, 532480, true, 133120, 64, 2112 }, { 1, 7, 532480, true, 133120, 0, 0 },
        { 4, 32, 98304, true, 98304, 16, kGroupItems }, { 3, 130, 32772, true, 24579, 5, 4928 }, { 4, 512, 4112, true, 4112, 1, 4160 },
        { 16, 48, 10816, true, 43264, 10, 4352 },
        { 8, 96, 10395, false, 20792, 5, 4160 }, { 32, 41, 5625, false, 45024, 12, 3776 }, { 1, 32, 393215, false, 98304, 16, kGroupItems },
        { 500, 60, 45, false, 6000, 2, 3008 }, { 700, 23, 77, false, 14000, 6, 2368 }, { 2, 23, 160001, false, 80002, 22, 3648 },
    };
    for (const auto& n: named) {
        const GroupPlan p = group_plan(n.batch, n.channels, n.spatial, n.vec, group_fill(n.channels), 512);
        check(!p.members || p.items == n.items, "vectors of a named slice", n.items, n.channels, 512);
        check(p.members == n.members && p.span == n.span, "the split of a named slice", n.items, n.channels, 512);
    }

    // tensors that take groups: aligned, and odd planes
    const struct { size_t total; int spatial; bool vec; int activation; bool groups; } sizes[] = {
        { 1u << 19, 4, true, PXH_LEAKY, true }, { (1u << 19) - 1, 4, true, PXH_LEAKY, false }, { 1u << 20, 4, true, PXH_MISH, true },
        { (1u << 20) - 1, 4, true, PXH_MISH, false }, { 7u << 20, 257, false, PXH_LEAKY, true }, { (7u << 20) - 1, 257, false, PXH_LEAKY, false },
        { 7u << 20, 257, false, PXH_LOGISTIC, true }, { (7u << 20) - 1, 13, false, PXH_SWISH, false }, { 7u << 20, 13, false, PXH_TANH, true },
        { 1u << 29, 257, false, PXH_MISH, false }, { 1u << 20, 255, false, PXH_RELU, true }, { (1u << 20) - 1, 255, false, PXH_RELU, false },
        { 1u << 20, 256, false, PXH_LINEAR, false }, { 1u << 29, 3, false, PXH_LEAKY, false }, { 1u << 29, 3, false, PXH_LOGISTIC, false },
    };
    for (const auto& n: sizes)
        check(enough_for_groups(n.total, n.spatial, n.vec, n.activation) == n.groups, "a tensor large enough", n.total, n.spatial, 0);

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
