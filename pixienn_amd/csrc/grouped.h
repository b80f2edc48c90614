// The one-launch training passes for slices that one workgroup of 1024 lanes cannot hold: a channel's slice is shared by the
// workgroups of a group, which exchange their sums inside the launch.  (Groups of one workgroup: where grouped_backward says.)
#pragma once

#include "resident.h"

namespace pxh {

constexpr int kGroupThreads = 512;

// What a member leaves for the others: up to four doubles, read as soon as they are there.  A word that is not there yet
// holds kNotThere, a NaN that no sum comes out as (canonical_word below); a launch in front puts it there.
constexpr uint64_t kNotThere = ~0ull;
constexpr int kFirstWords = 4;      // sums A and B, the squares, the largest magnitude
constexpr int kSumWords = 2;

// Next numbers of the first launch and of the second, and whether a wait of the first gave up (in a cache line that no
// number is taken from: 2 x 64 x 160^2 with one channel beyond the clamp 37 us in the same line, 34 so).
constexpr int kLost = 32, kTickets = kLost + 1;

struct GroupGeom {
    ResidentGeom g;
    uint32_t items;         // vectors of a channel's slice
    uint32_t span;          // of a member: a whole number of wavefronts
    uint32_t members;       // of a channel
    uint32_t image_skip;    // values between the end of a channel's plane and its plane in the next image
    FastDiv by_members;
    uint64_t* words;        // [channel][member][kFirstWords or kSumWords]; null with one member
    uint64_t* redo_words;   // [channel][member][kSumWords], of a clipped backward's second launch
    uint32_t* tickets;      // [kTickets]
    uint32_t looks;         // at a word that is not there yet, before a member goes on without it
};

__device__ __forceinline__ float* at_byte(float* p, uint32_t bytes)
{
    return reinterpret_cast<float*>(reinterpret_cast<char*>(p) + bytes);
}

__device__ __forceinline__ const float* at_byte(const float* p, uint32_t bytes)
{
    return reinterpret_cast<const float*>(reinterpret_cast<const char*>(p) + bytes);
}

// The workgroups of a launch take numbers, and a channel's members have consecutive ones.  A workgroup waits only for
// members of its own channel.  Those with lower numbers are running; of those with higher ones some may still have to
// start, in the one channel whose numbers are not all taken.  Every workgroup of another channel finishes without them and
// gives up its place, so they start as long as the stream has more places than waiting members hold.  A launch has fewer
// waiting members than kGroupShare's part of the places (an eighth), so that up to eight launches may run at once on the
// units of a stream's mask, beside anything that ends by itself.  More of them than that, less than that left by a kernel
// that stays for seconds, units that the environment takes away without the runtime's knowledge, or two launches at once on
// one workspace, which the interface forbids: there a wait may reach its bound (kLooks below).
__device__ __forceinline__ uint32_t take_ticket(uint32_t* counter, uint32_t& shared)
{
    __syncthreads();
    if (threadIdx.x == 0) shared = atomicAdd(counter, 1u);
    __syncthreads();
    return shared;
}

// A workgroup's way through the shares, from number to number below `all`, as one of its threads sees it.  `wg` is that
// thread's side of the workgroup: sync() is its barrier, ask() has one thread take the next number into the word that next()
// reads.  share(number) answers whether it has asked already, behind barriers of its own that follow the reading of
// `number`; where it has not, a wave may still have to read the word, and only a barrier tells that none has.
template<typename Workgroup, typename Share>
__host__ __device__ __forceinline__ void walk_shares(Workgroup& wg, uint32_t number, uint32_t all, Share&& share)
{
    while (number < all) {
        if (!share(number)) {
            wg.sync();
            wg.ask();
        }
        wg.sync();       // the number is there; and the next share reuses the workgroup's LDS
        number = wg.next();
    }
}

__device__ __forceinline__ uint64_t canonical_word(double v)
{
    const uint64_t bits = __double_as_longlong(v);
    return bits == kNotThere ? 0x7FF8000000000000ull : bits;
}

// About the time in which one half of the machine loads its shares (16 x 64 x 152^2: 62 us with it, 67 without, 64 with twice
// as long; 16 x 128 x 152^2: 120, 123, 122).
__device__ __forceinline__ void head_start() { __builtin_amdgcn_s_sleep(127); }

// Leaves a member's figures for the others (every thread calls it with the same ones).
template<int WORDS>
__device__ __forceinline__ void leave_figures(uint64_t* channel_words, uint32_t member, const double (&figures)[WORDS])
{
    if (threadIdx.x == 0) {
#pragma unroll
        for (int w = 0; w < WORDS; ++w)
            __hip_atomic_store(channel_words + member * WORDS + w, canonical_word(figures[w]), __ATOMIC_RELAXED,
                               __HIP_MEMORY_SCOPE_AGENT);
    }
}

// The figures of all members in every thread, added up in an order of the members alone (the last of four: the largest).
// The bound on the looks makes the exit unconditional (kLooks: seconds).  Where it was reached, what is missing was never
// formed: every figure is a NaN and the answer is false, in every thread.
template<int WORDS>
__device__ __forceinline__ bool collect_figures(const uint64_t* channel_words, uint32_t members, uint32_t most_looks,
                                                double (&figures)[WORDS])
{
    __shared__ double theirs[kGroupThreads];
    const uint32_t t = threadIdx.x;
    if (t < members * WORDS) {
        uint64_t word = __hip_atomic_load(channel_words + t, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        for (uint32_t looks = most_looks; word == kNotThere && looks; --looks) {
            __builtin_amdgcn_s_sleep(1);
            word = __hip_atomic_load(channel_words + t, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        }
        theirs[t] = __longlong_as_double(static_cast<long long>(word));
    }
    __syncthreads();
    // a lane per member in every wave
    const uint32_t lane = t & (kWave - 1);
    bool missing = false;
#pragma unroll
    for (int w = 0; w < WORDS; ++w) {
        const double v = lane < members ? theirs[lane * WORDS + w] : 0.0;
        missing = missing || static_cast<uint64_t>(__double_as_longlong(v)) == kNotThere;
        if (w < 3) figures[w] = wave_sum(v);
        else figures[w] = static_cast<double>(wave_max(static_cast<float>(v)));
    }
    if (!__any(missing)) return true;
#pragma unroll
    for (int w = 0; w < WORDS; ++w) figures[w] = __longlong_as_double(0x7FF8000000000000ll);
    return false;
}

// ---- the rules
// Members at most: a lane each, and their words a thread each.
constexpr uint32_t kGroupMost = kWave;
static_assert(kGroupMost * kFirstWords <= kGroupThreads, "a thread per word");
constexpr uint32_t kGroupShare = 8;

constexpr uint32_t kGroupItems = 12 * kGroupThreads;      // vectors that a member holds

// Workgroups that slices are split for: as many as the device runs at once, in a whole number of channels: a few more run in a
// second round (8 x 96 x 135 x 77 in 576 and in 480: 33.6 -> 26.4 us, 64 x 200 x 25^2 600 and 400: 34.5 -> 28.8,
// 9 x 20 x 203 x 251 520 and 500: 37.0 -> 29.3).
constexpr size_t kGroupFill = 512;
inline size_t group_fill(int channels)
{
    const size_t whole = kGroupFill / channels * channels;
    return whole > 0 ? whole : 1;
}

// Whether a tensor is large enough for groups.
//
// Small tensors (which the caches hold for the launches that read them twice) stay with those launches: a group's second one
// costs them more where it has something to do.  Three or five launches -> groups, us: plain; clipped with nothing to change,
// rescaled, and clamped throughout:
//   2 x 16 x 104^2  leaky 12.0 -> 11.4; 17.6 -> 15.3, 17.6 -> 19.3, 20.1 -> 22.9   mish 16.1 -> 18.0; 21.4 -> 22.1, 21.5 -> 26.2, 27.2 -> 36.2
//   2 x 16 x 160^2        13.5 -> 12.1; 18.8 -> 16.0, 18.8 -> 20.1, 21.7 -> 24.3        18.2 -> 18.8; 23.3 -> 23.1, 23.3 -> 27.3, 29.1 -> 37.7
//   1 x 32 x 208^2        16.1 -> 12.9; 21.5 -> 16.8, 21.5 -> 21.2, 24.4 -> 25.7        22.0 -> 20.1; 27.2 -> 23.9, 27.3 -> 28.6, 33.8 -> 39.9
//   4 x 32 x 208^2        28.2 -> 23.8; 34.9 -> 28.1, 35.0 -> 36.7, 42.8 -> 45.0        39.7 -> 34.9; 46.7 -> 40.0, 46.8 -> 48.6, 63.6 -> 69.2
// From there on the usual call gains a tenth to a quarter; one that clamps gains from 16 x 64 x 152^2 on (121 -> 107).
//
// Odd planes, whose several launches leave less to gain: planes of 256 values and more from 7 M values on, below which two launches
// that finish the channels serve a plain call better and a clipped one loses wherever something changes; smaller ones, of which the
// launches give each a wave, from 1 M on where the gradient is a select.  Not mish, whose gradient wants more registers than a
// lane of these has: there the calls that find nothing to change gain a twentieth, and those that rescale or clamp lose a fifth.
//   2 x 16 x 151^2      leaky  9.6 -> 11.9; 17.9 -> 16.0, 17.9 -> 20.3, 20.1 -> 24.1
//   6 x 72 x 135 x 77         20.7 -> 23.1; 35.0 -> 27.9, 35.4 -> 35.8, 41.8 -> 43.9
//   8 x 96 x 135 x 77         36.1 -> 26.4; 43.7 -> 31.7, 44.0 -> 43.7, 56.8 -> 52.4   mish 47.4 -> 46.8; 55.5 -> 53.4, 56.5 -> 65.8, 78.9 -> 97.8
//   16 x 64 x 151^2           88.5 -> 66.0; 95.4 -> 72.4, 95.4 -> 105,  123  -> 119         95.8 -> 92.3; 105 -> 103, 106 -> 136, 158 -> 185
//   16 x 90 x 151^2           123  -> 85.5; 130  -> 89.6, 129  -> 134,  169  -> 149         133  -> 113;  144 -> 131, 144 -> 178, 202 -> 235
//   8 x 96 x 135 x 77, logistic 40.5 -> 30.7; 48.5 -> 35.4, 48.4 -> 47.2, 64.7 -> 58.6       tanh 41.9 -> 31.2; 49.7 -> 37.6, 49.9 -> 49.6, 67.0 -> 66.8
//   16 x 64 x 151^2, logistic   89.7 -> 69.7; 103 -> 76.3,  103  -> 109,  137  -> 127
//   200 x 16 x 13^2           12.4 -> 12.3; 18.3 -> 16.3, 18.6 -> 20.1, 21.1 -> 24.0
//   400 x 16 x 13^2           16.6 -> 14.0; 23.7 -> 18.0, 24.1 -> 22.3, 27.5 -> 26.2
//   3000 x 40 x 5^2           36.4 -> 25.6; 46.5 -> 30.1, 47.3 -> 37.4, 61.7 -> 47.5
constexpr size_t kGroupFewest = 1u << 19, kGroupFewestSmooth = 1u << 20, kGroupFewestOdd = 7u << 20, kGroupFewestOddSmall = 1u << 20;
constexpr int kGroupOddSmall = 256;

inline bool enough_for_groups(size_t total, int spatial, bool vec, int activation)
{
    const bool light = selects(activation);
    if (vec) return total >= (light ? kGroupFewest : kGroupFewestSmooth);
    if (spatial < kOddSpatial || activation == PXH_MISH) return false;
    return total >= (light && spatial < kGroupOddSmall ? kGroupFewestOddSmall : kGroupFewestOdd);
}

constexpr uint32_t kLooks = 1u << 22;
uint32_t group_looks();      // kLooks, or what a test has set

// Compute units of a stream: those of its mask (a bit each), or all of the device's where it has none.
inline uint32_t units_of_mask(const uint32_t* mask, int words, uint32_t units)
{
    uint32_t enabled = 0;
    for (int w = 0; w < words; ++w) enabled += static_cast<uint32_t>(__builtin_popcount(mask[w]));
    return enabled && enabled < units ? enabled : units;
}

// Workgroups of these launches that the current device runs at once for a stream.
uint32_t group_places(hipStream_t s);

struct GroupPlan {
    uint32_t items, span, members;      // members 0: another form takes the call
    uint32_t places;
};

// How a slice is split over workgroups that hold `per_member` vectors each, on a stream of `places`: into as many
// members as make `workgroups` of them, none of fewer than four vectors a lane.  Where those would be more than kGroupMost
// (up to seven channels) the launches that wait for nothing keep the slice.  64 members would serve it where nothing is rescaled
// and lose where something is or is clamped: 4 x 6 x 512^2 36.5 -> 30.6, 36.5 -> 40.5 and 46 -> 49 us, 8 x 4 x 304^2 26 -> 22.8,
// 26 -> 28 and 30 -> 34.5, 16 x 2 x 208^2 20.3 -> 19.7, 20.2 -> 24 and 23.6 -> 29.7.
inline GroupPlan split_slice(size_t items, uint32_t per_member, size_t channels, size_t workgroups, uint32_t places)
{
    size_t least = (items + per_member - 1) / per_member;
    const size_t fill = (workgroups + channels - 1) / channels, shortest = items / (4 * kGroupThreads);
    const size_t more = fill < shortest ? fill : shortest;
    if (least < more) least = more;
    const size_t span = ((items + least - 1) / least + kWave - 1) / kWave * kWave;
    const size_t members = (items + span - 1) / span;
    if (members > kGroupMost || members * kGroupShare > places) return GroupPlan{};
    return GroupPlan{ static_cast<uint32_t>(items), static_cast<uint32_t>(span), static_cast<uint32_t>(members), places };
}

inline GroupPlan group_plan(int batch, int channels, int spatial, bool vec, size_t workgroups, uint32_t places)
{
    const size_t per_channel = static_cast<size_t>(batch) * spatial;
    if (per_channel * channels >= 1ull << 30) return GroupPlan{};      // places are 32-bit byte offsets
    const size_t items = vec ? per_channel / 4 : static_cast<size_t>(batch) * ((spatial + 3) / 4);      // vectors, as odd_slice
    return split_slice(items, kGroupItems, channels, workgroups, places);
}

inline GroupGeom group_geom(const GroupPlan& p, int batch, int channels, int spatial)
{
    return GroupGeom{ resident_geom(batch, channels, spatial), p.items, p.span, p.members,
                      static_cast<uint32_t>(channels - 1) * static_cast<uint32_t>(spatial), FastDiv(p.members), nullptr, nullptr,
                      nullptr, group_looks() };
}

// Bytes of the words of `count` members, and of everything a launch (with `redo`: and the one behind it) exchanges.
constexpr size_t group_align(size_t b) { return (b + 255) & ~static_cast<size_t>(255); }
inline size_t group_bytes(uint32_t channels, uint32_t members, int words, bool redo)
{
    const size_t count = static_cast<size_t>(channels) * members;
    return group_align(count * words * 8) + (redo ? group_align(count * kSumWords * 8) : 0) + 256;
}

constexpr size_t kGroupLdsBytes = 64u << 10;

// Places GroupGeom's buffers in `at` and queues the launch that empties them.
int start_exchange(const char* who, GroupGeom& g, void* at, int words, bool redo, hipStream_t s);

int launch_grouped_backward(const char* who, const ResidentBwdArgs& r, const GroupGeom& g, uint32_t places, bool clipped,
                            bool vec, int activation, hipStream_t s);

}  // namespace pxh
