// Non-maximum suppression of detection records on the device, for gfx950.
//
// The reference runs nms (src/Box.cpp:56-147) on the host over records it copied back: a stable
// sort by probability, a pass that drops near-identical boxes of different classes, a greedy
// pass inside every (image, class) group, each of them a sequential loop.  Here the number of
// records stays on the device, so every launch is sized for the capacity and the workgroups past
// the live count leave at once.  Lists of at most 512 records take one workgroup, lists of ordinary length go
// image by image (both further down); the steps for the longest ones:
//   1. LSD radix sort (8-bit digits) of (probability descending, emission order) -> global rank;
//   2. two to four more stable passes on (image, class) -> groups contiguous, rank order inside;
//   3. duplicate pass as a fixed point: a record is decided once every conflicting record of
//      lower rank is; sweeps over all undecided records in parallel, states only ever move from
//      undecided to kept/dropped, so any schedule ends in the sequential loop's answer;
//   4. the greedy pass the same way, one workgroup per group, states in LDS;
//   5. compaction of the kept records in rank order.
#include "common.h"
#include "pixienn_hip_test.h"

#include <algorithm>
#include <atomic>
#include <type_traits>

namespace pxh {
namespace {

constexpr int kSortTile = 4096;                       // keys per workgroup and pass
constexpr int kSortRounds = kSortTile / kBlock;
constexpr int kDigits = 256;
constexpr int kWide = 1024;                           // workgroup of the single-workgroup kernels
constexpr int kGroupVisit = 1024;                     // maxCandidatesPerGroup, src/Box.cpp:105
constexpr float kDuplicateOverlap = 0.9f;             // crossClassDuplicateIoU, src/Box.cpp:71

static_assert(kDigits == kBlock, "one bin per lane of the sorting workgroups");

enum : uint32_t { kUndecided = 0, kKept = 1, kDropped = 2, kAbsent = 3 };

__device__ __forceinline__ uint32_t live_count(const int* count, int capacity)
{
    const int n = *count;
    return n < 0 ? 0u : static_cast<uint32_t>(n > capacity ? capacity : n);
}

// States are written by one lane and read by lanes of other workgroups while a kernel runs:
// both sides go to the device-coherent level.
__device__ __forceinline__ uint32_t load_state(const uint32_t* p)
{
    return __hip_atomic_load(p, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}
__device__ __forceinline__ void store_state(uint32_t* p, uint32_t v)
{
    __hip_atomic_store(p, v, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}

// Exclusive prefix sum of one value per lane over a kWide-lane workgroup; `total` in every lane.
__device__ __forceinline__ uint32_t wide_exclusive_scan(uint32_t v, uint32_t* lds /* kWide / kWave + 1 */,
                                                        uint32_t& total)
{
    const int lane = threadIdx.x & (kWave - 1);
    const int wave = threadIdx.x / kWave;
    uint32_t incl = v;
#pragma unroll
    for (int off = 1; off < kWave; off <<= 1) {
        const uint32_t up = __shfl_up(incl, off, kWave);
        if (lane >= off) incl += up;
    }
    __syncthreads();
    if (lane == kWave - 1) lds[wave] = incl;
    __syncthreads();
    if (threadIdx.x == 0) {
        uint32_t run = 0;
        for (int w = 0; w < kWide / kWave; ++w) {
            const uint32_t t = lds[w];
            lds[w] = run;
            run += t;
        }
        lds[kWide / kWave] = run;
    }
    __syncthreads();
    total = lds[kWide / kWave];
    return lds[wave] + incl - v;
}

// ---------------------------------------------------------------- radix sort passes
struct SortArgs {
    const uint64_t* keys_in;
    const uint32_t* vals_in;
    uint64_t* keys_out;
    uint32_t* vals_out;
    uint32_t* hist;          // [digit][live tiles]
    const int* count;
    int capacity;
    int shift;
};

__device__ __forceinline__ uint32_t live_tiles(uint32_t n) { return (n + kSortTile - 1) / kSortTile; }

__global__ __launch_bounds__(kBlock) void sort_histogram_kernel(SortArgs a)
{
    __shared__ uint32_t bins[kDigits];
    const uint32_t n = live_count(a.count, a.capacity);
    const uint32_t tiles = live_tiles(n);
    if (blockIdx.x >= tiles) return;
    bins[threadIdx.x] = 0;
    __syncthreads();
    const uint32_t first = blockIdx.x * kSortTile;
    for (int r = 0; r < kSortRounds; ++r) {
        const uint32_t i = first + r * kBlock + threadIdx.x;
        if (i < n) atomicAdd(&bins[(a.keys_in[i] >> a.shift) & (kDigits - 1)], 1u);
    }
    __syncthreads();
    a.hist[threadIdx.x * tiles + blockIdx.x] = bins[threadIdx.x];
}

// In-place exclusive prefix sum over `per_tile` * (live tiles) counters by ONE workgroup; the sum of
// all of them goes to *total_out when given.
__global__ __launch_bounds__(kWide) void scan_counters_kernel(uint32_t* counters, const int* count, int capacity,
                                                              uint32_t per_tile, int* total_out)
{
    __shared__ uint32_t lds[kWide / kWave + 1];
    const uint32_t n = live_count(count, capacity);
    const uint32_t entries = per_tile * live_tiles(n);
    const uint32_t per = (entries + kWide - 1) / kWide;
    const uint32_t lo = min(threadIdx.x * per, entries);
    const uint32_t hi = min(lo + per, entries);
    uint32_t sum = 0;
    for (uint32_t i = lo; i < hi; ++i) sum += counters[i];
    uint32_t total;
    uint32_t run = wide_exclusive_scan(sum, lds, total);
    for (uint32_t i = lo; i < hi; ++i) {
        const uint32_t c = counters[i];
        counters[i] = run;
        run += c;
    }
    if (total_out && threadIdx.x == 0) *total_out = static_cast<int>(total);
}

__global__ __launch_bounds__(kBlock) void sort_scatter_kernel(SortArgs a)
{
    __shared__ uint32_t base[kDigits];
    __shared__ uint32_t wave_count[kBlock / kWave][kDigits];
    const uint32_t n = live_count(a.count, a.capacity);
    const uint32_t tiles = live_tiles(n);
    if (blockIdx.x >= tiles) return;
    base[threadIdx.x] = a.hist[threadIdx.x * tiles + blockIdx.x];
#pragma unroll
    for (int w = 0; w < kBlock / kWave; ++w) wave_count[w][threadIdx.x] = 0;
    __syncthreads();
    const int lane = threadIdx.x & (kWave - 1);
    const int wave = threadIdx.x / kWave;
    const uint64_t below = (1ull << lane) - 1ull;
    const uint32_t first = blockIdx.x * kSortTile;
    for (int r = 0; r < kSortRounds; ++r) {
        if (first + r * kBlock >= n) break;                               // the same for every lane
        const uint32_t i = first + r * kBlock + threadIdx.x;
        const bool valid = i < n;
        const uint64_t key = valid ? a.keys_in[i] : 0ull;
        const uint32_t val = valid ? a.vals_in[i] : 0u;
        const uint32_t digit = static_cast<uint32_t>(key >> a.shift) & (kDigits - 1);
        // lanes of this wave that hold the same digit
        uint64_t peers = __ballot(valid);
#pragma unroll
        for (int bit = 0; bit < 8; ++bit) {
            const bool set = (digit >> bit) & 1u;
            const uint64_t with = __ballot(set);
            peers &= set ? with : ~with;
        }
        const uint32_t rank = __popcll(peers & below);
        if (valid && rank == 0) wave_count[wave][digit] = __popcll(peers);
        __syncthreads();
        if (valid) {
            uint32_t at = base[digit] + rank;
            for (int w = 0; w < wave; ++w) at += wave_count[w][digit];
            a.keys_out[at] = key;
            a.vals_out[at] = val;
        }
        __syncthreads();
        uint32_t add = 0;
#pragma unroll
        for (int w = 0; w < kBlock / kWave; ++w) {
            add += wave_count[w][threadIdx.x];
            wave_count[w][threadIdx.x] = 0;
        }
        base[threadIdx.x] += add;
        __syncthreads();
    }
}

// ---------------------------------------------------------------- keys
// Ascending key order = descending probability, then ascending emission order.
__device__ __forceinline__ uint32_t descending_bits(float v)
{
    const uint32_t u = __float_as_uint(v);
    const uint32_t ascending = (u & 0x80000000u) ? ~u : (u | 0x80000000u);
    return ~ascending;
}

__global__ __launch_bounds__(kBlock) void nms_rank_keys_kernel(const pxh_detection* records, const int* count,
                                                               int capacity, uint64_t* keys, uint32_t* vals,
                                                               uint32_t* counters)
{
    const uint32_t n = live_count(count, capacity);
    const uint32_t i = blockIdx.x * kBlock + threadIdx.x;
    if (blockIdx.x == 0 && threadIdx.x < 8) counters[threadIdx.x] = 0;
    if (i >= n) return;
    const pxh_detection d = records[i];
    keys[i] = (static_cast<uint64_t>(descending_bits(d.prob)) << 32) | d.order;
    vals[i] = i;
}

// sorted[r] = input index of the record of rank r  ->  perm, and the keys of the second sort
// An image or class number outside [0, batch) x [0, classes) is clamped into it for the grouping,
// so that the groups stay contiguous whatever the records hold.
__global__ __launch_bounds__(kBlock) void nms_group_keys_kernel(const pxh_detection* records, const int* count,
                                                                int capacity, const uint32_t* sorted, uint32_t* perm,
                                                                uint64_t* keys, uint32_t* vals, int batch, int classes)
{
    const uint32_t n = live_count(count, capacity);
    const uint32_t r = blockIdx.x * kBlock + threadIdx.x;
    if (r >= n) return;
    const uint32_t at = sorted[r];
    perm[r] = at;
    const pxh_detection d = records[at];
    const uint32_t image = static_cast<uint32_t>(min(max(d.batch, 0), batch - 1));
    const uint32_t cls = static_cast<uint32_t>(min(max(d.class_index, 0), classes - 1));
    keys[r] = (static_cast<uint64_t>(image) << 32) | cls;
    vals[r] = r;
}

__device__ __forceinline__ uint32_t lower_bound(const uint64_t* keys, uint32_t n, uint64_t key)
{
    uint32_t lo = 0, hi = n;
    while (lo < hi) {
        const uint32_t mid = lo + (hi - lo) / 2;
        if (keys[mid] < key) lo = mid + 1;
        else hi = mid;
    }
    return lo;
}

// ---------------------------------------------------------------- boxes
// normalizedRect, src/Box.cpp:47-54: (x1, y1, w, h)
__device__ __forceinline__ float4 normalized_rect(const pxh_detection& d)
{
    const float xe = d.x + d.w, ye = d.y + d.h;
    const float x1 = fminf(d.x, xe), y1 = fminf(d.y, ye);
    const float x2 = fmaxf(d.x, xe), y2 = fmaxf(d.y, ye);
    return make_float4(x1, y1, fmaxf(0.0f, x2 - x1), fmaxf(0.0f, y2 - y1));
}

// boxIoU(a, b) > threshold, src/Box.cpp:25-45, with cv::Rect2f's operator& (OpenCV >= 4.5.4): an
// empty operand or a non-positive extent gives no overlap; the extent along an axis is
// min(lo.size - (hi.origin - lo.origin), hi.size) with lo/hi ordered by origin.  threshold >= 0, so
// no overlap can never be above it; and the union is at least the larger area, so an overlap well
// below threshold * that area is decided without the division (the margin of a tenth is far more
// than all rounding involved).  Everything else takes the reference's own operations.
__device__ __forceinline__ bool overlaps_above(const float4 a, const float4 b, float threshold)
{
    if (a.z <= 0.0f || a.w <= 0.0f || b.z <= 0.0f || b.w <= 0.0f) return false;
    const bool ax = a.x < b.x, ay = a.y < b.y;
    const float xlo = ax ? a.x : b.x, xlo_w = ax ? a.z : b.z, xhi = ax ? b.x : a.x, xhi_w = ax ? b.z : a.z;
    const float ylo = ay ? a.y : b.y, ylo_h = ay ? a.w : b.w, yhi = ay ? b.y : a.y, yhi_h = ay ? b.w : a.w;
    if ((xlo < 0.0f && xlo + xlo_w < xhi) || (ylo < 0.0f && ylo + ylo_h < yhi)) return false;
    const float iw = fminf(xlo_w - (xhi - xlo), xhi_w);
    const float ih = fminf(ylo_h - (yhi - ylo), yhi_h);
    if (!(iw > 0.0f && ih > 0.0f)) return false;
    const float inter = iw * ih;
    const float area_a = a.z * a.w, area_b = b.z * b.w;
    if (inter < 0.9f * threshold * fmaxf(area_a, area_b)) return false;
    float uni = area_a + area_b - inter;
    if (!(0.0f < uni)) uni = 0.0f;
    const float q = inter / uni;
    if (isnan(q) || isinf(q)) return false;          // counts as no overlap: 0 > threshold is false
    return q > threshold;
}

struct Segments {
    uint32_t image_begin, image_end, group_begin, group_end;
};

struct NmsArgs {
    const pxh_detection* records;
    const int* count;
    int capacity;
    const uint32_t* perm;      // rank -> input index
    const uint64_t* group_key; // per place (sorted by image, class, rank)
    const uint32_t* rank;      // per place
    float4* box;               // per place
    Segments* seg;             // per place
    uint32_t* state;           // per place, duplicate pass
    uint32_t* keep;            // per rank
    uint32_t* resume;          // per place: where the next sweep of the duplicate pass continues
    uint32_t* counters;        // [k] != 0: sweep k left records undecided
    uint32_t waves;            // waves of a duplicate sweep's grid
};

__global__ __launch_bounds__(kBlock) void nms_gather_kernel(NmsArgs a)
{
    const uint32_t n = live_count(a.count, a.capacity);
    const uint32_t p = blockIdx.x * kBlock + threadIdx.x;
    if (p >= n) return;
    a.box[p] = normalized_rect(a.records[a.perm[a.rank[p]]]);
    const uint64_t key = a.group_key[p];
    const uint64_t image = key & 0xFFFFFFFF00000000ull;
    Segments s;
    s.image_begin = lower_bound(a.group_key, n, image);
    s.image_end = lower_bound(a.group_key, n, image + 0x100000000ull);
    s.group_begin = lower_bound(a.group_key, n, key);
    s.group_end = lower_bound(a.group_key, n, key + 1ull);
    a.seg[p] = s;
    a.state[p] = kUndecided;
    a.resume[p] = s.image_begin;
}

// ---------------------------------------------------------------- duplicate pass
// src/Box.cpp:65-88: a record is dropped when an earlier KEPT record of the same image and another
// class overlaps it by more than 0.9.  One WAVE per undecided record, its lanes side by side over
// the other places of the image (the record's own class group is stepped over).  Outcome for the
// record at place p: 1 = dropped, 0 = kept, 2 = still waiting for an undecided earlier record, in
// which case resume[p] is the first such place: everything before it that conflicts is dropped for
// good and need not be looked at again.
__device__ __forceinline__ int duplicate_scan(const NmsArgs& a, uint32_t p, int lane)
{
    const Segments s = a.seg[p];
    const float4 box = a.box[p];
    const uint32_t rank = a.rank[p];
    uint32_t first_pending = 0xFFFFFFFFu;
    uint32_t q0 = a.resume[p];
    while (q0 < s.image_end) {
        if (q0 >= s.group_begin && q0 < s.group_end) {          // the same class: not compared
            q0 = s.group_end;
            continue;
        }
        const uint32_t stop = q0 < s.group_begin ? s.group_begin : s.image_end;
        const uint32_t q = q0 + lane;
        bool kept_hit = false, waiting = false;
        if (q < stop && a.rank[q] < rank) {
            const uint32_t st = load_state(a.state + q);
            if (st != kDropped && overlaps_above(box, a.box[q], kDuplicateOverlap)) {
                kept_hit = st == kKept;
                waiting = st == kUndecided;
            }
        }
        if (__ballot(kept_hit)) return 1;
        const uint64_t w = __ballot(waiting);
        if (w && first_pending == 0xFFFFFFFFu) first_pending = q0 + __builtin_ctzll(w);
        q0 = min(q0 + kWave, stop);
    }
    if (first_pending == 0xFFFFFFFFu) return 0;
    if (lane == 0) a.resume[p] = first_pending;
    return 2;
}

__global__ __launch_bounds__(kBlock) void nms_duplicate_sweep_kernel(NmsArgs a, int sweep)
{
    const uint32_t n = live_count(a.count, a.capacity);
    if (sweep > 0 && a.counters[sweep - 1] == 0) return;
    const int lane = threadIdx.x & (kWave - 1);
    const uint32_t wave = (blockIdx.x * kBlock + threadIdx.x) / kWave;
    bool left = false;
    for (uint32_t p = wave; p < n; p += a.waves) {
        if (load_state(a.state + p) != kUndecided) continue;
        const int outcome = duplicate_scan(a, p, lane);
        if (outcome == 2) left = true;
        else if (lane == 0) store_state(a.state + p, outcome == 1 ? kDropped : kKept);
    }
    if (left && lane == 0) store_state(a.counters + sweep, 1u);
}

// What the sweeps left undecided (long chains of conflicts): one workgroup per image repeats the
// sweep over its own records until none is left.  Every repetition decides at least the undecided
// record of lowest rank, so the loop ends.
__global__ __launch_bounds__(kWide) void nms_duplicate_finish_kernel(NmsArgs a, int last_sweep)
{
    if (a.counters[last_sweep] == 0) return;
    const uint32_t n = live_count(a.count, a.capacity);
    const uint64_t image = static_cast<uint64_t>(blockIdx.x) << 32;
    const uint32_t begin = lower_bound(a.group_key, n, image);
    const uint32_t end = lower_bound(a.group_key, n, image + 0x100000000ull);
    const int lane = threadIdx.x & (kWave - 1);
    const uint32_t wave = threadIdx.x / kWave;
    // one repetition per record is the most the argument above allows; the bound makes the exit
    // unconditional
    for (uint32_t repetition = 0; repetition <= end - begin; ++repetition) {
        int left = 0;
        for (uint32_t p = begin + wave; p < end; p += kWide / kWave) {
            if (load_state(a.state + p) != kUndecided) continue;
            const int outcome = duplicate_scan(a, p, lane);
            if (outcome == 2) left = 1;
            else if (lane == 0) store_state(a.state + p, outcome == 1 ? kDropped : kKept);
        }
        __threadfence();
        if (__syncthreads_or(left) == 0) break;
    }
}

// ---------------------------------------------------------------- greedy pass inside a group
// src/Box.cpp:104-136: the first 1024 places of the group in rank order; a record the duplicate
// pass dropped is skipped; a record is suppressed when an earlier KEPT one overlaps it by more than
// the threshold.  One workgroup per (image, class), one lane per place, states in LDS.
__global__ __launch_bounds__(kWide) void nms_group_kernel(NmsArgs a, float threshold, FastDiv by_classes)
{
    __shared__ float4 group_box[kGroupVisit];
    __shared__ uint32_t group_state[kGroupVisit];
    const uint32_t n = live_count(a.count, a.capacity);
    if (n == 0) return;
    uint32_t image, cls;
    by_classes.divmod(blockIdx.x, image, cls);
    const uint64_t key = (static_cast<uint64_t>(image) << 32) | cls;
    const uint32_t begin = lower_bound(a.group_key, n, key);
    const uint32_t end = lower_bound(a.group_key, n, key + 1ull);
    if (begin == end) return;
    const uint32_t visit = min(end - begin, static_cast<uint32_t>(kGroupVisit));
    const uint32_t t = threadIdx.x;
    const bool active = t < visit;
    float4 box = make_float4(0, 0, 0, 0);
    bool decided = true;
    if (active) {
        box = a.box[begin + t];
        const bool alive = load_state(a.state + begin + t) == kKept;
        group_box[t] = box;
        group_state[t] = alive ? kUndecided : kAbsent;
        decided = !alive;
    }
    __syncthreads();
    const volatile uint32_t* states = group_state;
    uint32_t from = 0;
    // each repetition decides at least the undecided place of lowest rank: at most `visit` of them
    for (uint32_t repetition = 0; repetition <= visit; ++repetition) {
        if (!decided) {
            bool drop = false, pending = false;
            uint32_t first_pending = t;
            for (uint32_t j = from; j < t; ++j) {
                const uint32_t st = states[j];
                if (st == kAbsent || st == kDropped) continue;
                if (overlaps_above(box, group_box[j], threshold)) {
                    if (st == kKept) {
                        drop = true;
                        break;
                    }
                    if (!pending) {
                        pending = true;
                        first_pending = j;
                    }
                }
            }
            if (drop) {
                group_state[t] = kDropped;
                decided = true;
            } else if (!pending) {
                group_state[t] = kKept;
                decided = true;
            } else {
                from = first_pending;      // everything before it that overlaps is dropped for good
            }
        }
        if (__syncthreads_count(!decided) == 0) break;
    }
    if (active) a.keep[a.rank[begin + t]] = group_state[t] == kKept ? 1u : 0u;
    // places past the first 1024 are never visited: they stay unless the duplicate pass dropped them
    for (uint32_t p = begin + kGroupVisit + t; p < end; p += kWide)
        a.keep[a.rank[p]] = load_state(a.state + p) == kKept ? 1u : 0u;
}

// ---------------------------------------------------------------- compaction in rank order
__global__ __launch_bounds__(kBlock) void nms_count_kept_kernel(NmsArgs a, uint32_t* tile_kept)
{
    __shared__ uint32_t sum;
    const uint32_t n = live_count(a.count, a.capacity);
    if (blockIdx.x >= live_tiles(n)) return;
    if (threadIdx.x == 0) sum = 0;
    __syncthreads();
    uint32_t mine = 0;
    const uint32_t first = blockIdx.x * kSortTile;
    for (int r = 0; r < kSortRounds; ++r) {
        const uint32_t i = first + r * kBlock + threadIdx.x;
        if (i < n) mine += a.keep[i];
    }
    if (mine) atomicAdd(&sum, mine);
    __syncthreads();
    if (threadIdx.x == 0) tile_kept[blockIdx.x] = sum;
}

__global__ __launch_bounds__(kBlock) void nms_write_kept_kernel(NmsArgs a, const uint32_t* tile_first,
                                                                pxh_detection* kept)
{
    __shared__ uint32_t wave_kept[kBlock / kWave];
    const uint32_t n = live_count(a.count, a.capacity);
    if (blockIdx.x >= live_tiles(n)) return;
    const int lane = threadIdx.x & (kWave - 1);
    const int wave = threadIdx.x / kWave;
    const uint64_t below = (1ull << lane) - 1ull;
    uint32_t base = tile_first[blockIdx.x];
    const uint32_t first = blockIdx.x * kSortTile;
    for (int r = 0; r < kSortRounds; ++r) {
        if (first + r * kBlock >= n) break;                               // the same for every lane
        const uint32_t i = first + r * kBlock + threadIdx.x;
        const bool take = i < n && a.keep[i] != 0;
        const uint64_t takers = __ballot(take);
        if (lane == 0) wave_kept[wave] = __popcll(takers);
        __syncthreads();
        uint32_t at = base + __popcll(takers & below);
        uint32_t all = 0;
#pragma unroll
        for (int w = 0; w < kBlock / kWave; ++w) {
            const uint32_t c = wave_kept[w];
            if (w < wave) at += c;
            all += c;
        }
        if (take) kept[at] = a.records[a.perm[i]];
        base += all;
        __syncthreads();
    }
}

// ---------------------------------------------------------------- short lists in one workgroup
// Up to 512 records (what an inference pass leaves): everything above in ONE launch, with the
// records in LDS.  Ranks come from counting the smaller keys.  Both passes take one wave per record,
// lanes side by side over the records of lower rank, and the waves walk the ranks in ascending
// order, so nearly every record finds the ones it depends on already decided; the few that do not
// are taken again.  No group can reach the 1024-place limit.
constexpr int kSmall = 512;

// One pass over the ranks: `same_class` false = duplicates across classes (src/Box.cpp:65-88), true =
// greedy suppression inside (image, class) (src/Box.cpp:104-136).
__device__ __forceinline__ void small_pass(uint32_t n, bool same_class, float threshold, const float4* ranked_box,
                                           const uint2* ranked_group, uint32_t* state)
{
    const volatile uint32_t* states = state;
    const int lane = threadIdx.x & (kWave - 1);
    const uint32_t wave = threadIdx.x / kWave;
    // a repetition decides at least the undecided record of lowest rank; the bound makes the exit
    // unconditional
    for (uint32_t repetition = 0; repetition <= n; ++repetition) {
        int left = 0;
        for (uint32_t t = wave; t < n; t += kWide / kWave) {
            if (states[t] != kUndecided) continue;
            const float4 box = ranked_box[t];
            const uint2 group = ranked_group[t];
            bool drop = false, pending = false;
            for (uint32_t j0 = 0; j0 < t && !drop; j0 += kWave) {
                const uint32_t j = j0 + lane;
                bool hit = false, wait = false;
                if (j < t) {
                    const uint2 other = ranked_group[j];
                    if (other.x == group.x && (other.y == group.y) == same_class) {
                        const uint32_t st = states[j];
                        if ((st == kKept || st == kUndecided) && overlaps_above(box, ranked_box[j], threshold)) {
                            hit = st == kKept;
                            wait = st == kUndecided;
                        }
                    }
                }
                drop = __ballot(hit) != 0;
                pending = pending || __ballot(wait) != 0;
            }
            if (drop || !pending) {
                if (lane == 0) state[t] = drop ? kDropped : kKept;
            } else {
                left = 1;
            }
        }
        if (__syncthreads_or(left) == 0) break;
    }
}

__global__ __launch_bounds__(kWide) void nms_small_kernel(const pxh_detection* records, const int* count, int capacity,
                                                          int batch, int classes, float threshold,
                                                          pxh_detection* kept, int* kept_count)
{
    __shared__ uint64_t key[kSmall];
    __shared__ float4 ranked_box[kSmall];
    __shared__ uint2 ranked_group[kSmall];       // image, class
    __shared__ uint32_t source[kSmall];
    __shared__ uint32_t state[kSmall];
    __shared__ uint32_t scan_lds[kWide / kWave + 1];
    const uint32_t n = live_count(count, capacity);
    const uint32_t t = threadIdx.x;
    const bool valid = t < n;
    pxh_detection d{};
    if (valid) {
        d = records[t];
        key[t] = (static_cast<uint64_t>(descending_bits(d.prob)) << 32) | d.order;
    }
    __syncthreads();
    if (valid) {
        const uint64_t mine = key[t];
        uint32_t rank = 0;
        for (uint32_t j = 0; j < n; ++j) {
            const uint64_t k = key[j];
            rank += (k < mine || (k == mine && j < t)) ? 1u : 0u;
        }
        ranked_box[rank] = normalized_rect(d);
        ranked_group[rank] = make_uint2(static_cast<uint32_t>(min(max(d.batch, 0), batch - 1)),
                                        static_cast<uint32_t>(min(max(d.class_index, 0), classes - 1)));
        source[rank] = t;
        state[rank] = kUndecided;
    }
    __syncthreads();
    small_pass(n, false, kDuplicateOverlap, ranked_box, ranked_group, state);
    // survivors of the first pass enter the second; the dropped ones are absent from it
    if (valid) state[t] = state[t] == kKept ? kUndecided : kAbsent;
    __syncthreads();
    small_pass(n, true, threshold, ranked_box, ranked_group, state);
    const bool take = valid && state[t] == kKept;
    uint32_t total;
    const uint32_t at = wide_exclusive_scan(take ? 1u : 0u, scan_lds, total);
    if (take) kept[at] = records[source[t]];
    if (t == 0) *kept_count = static_cast<int>(total);
}

// ---------------------------------------------------------------- lists of ordinary length
// Every decision of nms is taken inside one image, so the records are grouped by image first and
// nothing is sorted: six launches in place of the sorting path's forty-five, whose cost at the few
// thousand records of a validation batch is the launches and the latency of short dependent steps
// (7126 records of 16 images in a list for 32768: 440 us in kernels, here 39).
//   1. images are counted per tile of 1024 records, 2. the records' keys are laid out image by image,
//      in any order inside one;
//   3. a record's place in its image is the number of smaller keys there, counted directly: n^2 of the
//      cheapest comparisons per image, all independent, where a radix sort is a chain of thirty launches;
//   4. every pair of an image is looked at once, 64 pairs per step of a wave: bit masks of the earlier
//      records that conflict, one for each of the two passes (other class and overlap above 0.9, same
//      class and overlap above the threshold);
//   5. one workgroup per image settles both passes on the masks alone, the states as bit sets in LDS;
//   6. a survivor's place in the whole list is the number of survivors before it in each image, found
//      by a search of a few lanes per image.
// A mask has 16 words, a bit to a place, of which as many that are not empty are stored as 10 MB hold for the whole
// list (all of them up to 36408 records, eight for 65536), so that the longest list fits the library's first workspace.
// Step 5 looks at the pairs of a further one again.
// An image of more than 1024 places has no masks, and more pairs than one workgroup should settle: further workgroups of
// step 5 settle it block by block, 64 places each, the blocks' pairs all over the chip at once and only the decisions
// one after the other (further down).
constexpr int kImageCapacity = 65536;                 // longest list
constexpr int kImageBatch = kWide;                    // most images: one lane each
constexpr int kMaskWords = 16;
// Places of an image; larger ones are settled block by block.  Masks against blocks, us: one image of 1100 around 6
// places 117 -> 78, around 100 80 -> 73; 4000 of one class 243 -> 130; 16 images of 1250 around 100 places 128 -> 132 and
// 32 of 1875 around 20 304 -> 308; but 64 of 625 around 20 163 -> 235 with the line at 512.
constexpr uint32_t kLargeImage = 64 * kMaskWords;
static_assert(kLargeImage <= kGroupVisit, "no place of an image with masks is past those that are visited");
static_assert(kLargeImage == kWide, "a lane to a place where one workgroup settles an image, a wave to a word of the masks");
// What a settled block leaves for those behind it: the places that the first pass kept, the kept places of the second
// that can still suppress one (two words each), the survivors of the image so far.
constexpr uint32_t kSettledWords = 5, kSettledStride = 8;
constexpr unsigned kSettleWorkgroups = 256;           // one to a compute unit
constexpr size_t kMaskBytes = 10u << 20;

// words of one pass's masks for the whole list, each with the byte that says which one it is
constexpr size_t kMaskListWords = kMaskBytes / (2 * 9);
static_assert(kMaskListWords / kImageCapacity >= 8, "the longest list stores some");

// words of a mask that are stored
int mask_slots(int capacity)
{
    const size_t fit = kMaskListWords / static_cast<size_t>(capacity);
    return fit > kMaskWords ? kMaskWords : static_cast<int>(fit);
}

// 64 places of one image
struct PlaceBlock {
    uint32_t image_begin, image_end, first, image;
};

struct ImageArgs {
    const pxh_detection* records;
    const int* count;
    int capacity, batch, classes;
    float threshold;
    uint32_t* tile_images;    // [tile][image] records
    uint32_t* image_begin;    // [batch + 1]
    uint32_t* block_count;
    PlaceBlock* blocks;
    uint64_t* loose_key;      // image by image, unordered
    uint32_t* loose_source;
    uint64_t* key;            // image by image, in rank order; from here on by place
    uint32_t* source;
    float4* box;
    uint32_t* cls;
    int mask_slots;
    uint32_t* slots;          // stored words of a place's masks: [0] other classes, [1] same class << 8
    uint8_t* ids[2];          // [slot][place]: which word it is
    uint64_t* masks[2];       // [slot][place]
    uint64_t* beyond[2];      // words that are not empty and not stored
    uint32_t* first_block;    // of each image
    uint32_t* ticket;         // large images: the next block to be settled,
    uint64_t* settled;        // and what each left for the blocks behind it, [block][kSettledStride]
    uint64_t* kept_key;       // survivors, image by image, in rank order
    uint32_t* kept_source;
    uint32_t* kept_images;    // survivors per image
};

__device__ __forceinline__ uint32_t image_of(const pxh_detection& d, int batch)
{
    return static_cast<uint32_t>(min(max(d.batch, 0), batch - 1));
}

__global__ __launch_bounds__(kWide) void nms_count_images_kernel(ImageArgs a)
{
    __shared__ uint32_t bins[kImageBatch];
    const uint32_t n = live_count(a.count, a.capacity);
    if (blockIdx.x * kWide >= n) return;
    const uint32_t t = threadIdx.x;
    bins[t] = 0;
    __syncthreads();
    const uint32_t i = blockIdx.x * kWide + t;
    if (i < n) atomicAdd(&bins[image_of(a.records[i], a.batch)], 1u);
    __syncthreads();
    if (t < static_cast<uint32_t>(a.batch)) a.tile_images[blockIdx.x * a.batch + t] = bins[t];
}

// Every workgroup works out where each image begins for itself; the first also writes it down, with the
// blocks of 64 places of all images.
__global__ __launch_bounds__(kWide) void nms_group_images_kernel(ImageArgs a)
{
    __shared__ uint32_t scan_lds[kWide / kWave + 1];
    __shared__ uint32_t cursor[kImageBatch];
    const uint32_t n = live_count(a.count, a.capacity);
    const uint32_t t = threadIdx.x;
    if (blockIdx.x * kWide >= n && blockIdx.x != 0) return;
    const uint32_t tiles = (n + kWide - 1) / kWide;
    uint32_t before = 0, all = 0;
    if (t < static_cast<uint32_t>(a.batch)) {
        for (uint32_t tile = 0; tile < tiles; ++tile) {
            const uint32_t c = a.tile_images[tile * a.batch + t];
            if (tile < blockIdx.x) before += c;
            all += c;
        }
    }
    uint32_t total;
    const uint32_t begin = wide_exclusive_scan(all, scan_lds, total);
    cursor[t] = begin + before;
    __syncthreads();
    if (blockIdx.x == 0) {
        const uint32_t mine = (all + 63) / 64;
        const uint32_t first_block = wide_exclusive_scan(mine, scan_lds, total);
        if (t <= static_cast<uint32_t>(a.batch) && t < kWide) a.image_begin[t] = begin;
        if (t < static_cast<uint32_t>(a.batch)) {
            a.first_block[t] = first_block;
            a.ticket[t] = 0;
        }
        if (t == 0) {
            *a.block_count = total;
            a.image_begin[a.batch] = n;
        }
        for (uint32_t k = 0; k < mine; ++k) a.blocks[first_block + k] = PlaceBlock{ begin, begin + all, begin + 64 * k, t };
    }
    const uint32_t i = blockIdx.x * kWide + t;
    if (i >= n) return;
    const pxh_detection d = a.records[i];
    const uint32_t at = atomicAdd(&cursor[image_of(d, a.batch)], 1u);
    a.loose_key[at] = (static_cast<uint64_t>(descending_bits(d.prob)) << 32) | d.order;
    a.loose_source[at] = i;
}

__device__ __forceinline__ uint64_t key_of_lane(uint64_t key, int lane)
{
    const uint32_t lo = __builtin_amdgcn_readlane(static_cast<uint32_t>(key), lane);
    const uint32_t hi = __builtin_amdgcn_readlane(static_cast<uint32_t>(key >> 32), lane);
    return (static_cast<uint64_t>(hi) << 32) | lo;
}

// Block `at` of 64 places; false where there are no more.  (With no records there are none: the group launch
// writes that down too.  Both loads are on their way at once: of the steps of these launches, which are short, a trip to
// memory is the longest.)
__device__ __forceinline__ bool find_block(const ImageArgs& a, uint32_t at, PlaceBlock& b)
{
    const uint32_t blocks = *a.block_count;
    b = a.blocks[at];
    return at < blocks;
}

// The two launches below take blocks by quarters.  Those are few where a list is long and nearly empty, and a workgroup for each that
// the list could have takes a place for a trip to memory: there are kTurnWorkgroups at most, which take the quarters in turns, every
// other turn in the opposite order, since a quarter costs more the further back its block lies in its image.  (A workgroup to a
// quarter, no records in a list for 40000 17.2 us, so 12.7, 3 records 19.5 and 17.2; 28160 of 64 images 72.9 and 75.5.)
constexpr uint32_t kQuarters = 4, kTurnWorkgroups = 1024;

// Calls body(block, its number, quarter) for the quarters of a workgroup; `all`: those that the list could have.  (With no records
// there are none: the group launch writes that down too.  How many there are and the first one are on their way at once: of the
// steps of these launches, which are short, a trip to memory is the longest.)  FIRST: the first quarters of all blocks before the
// others, for more images than a wave has lanes, most of whose quarters behind the first are empty (6000 records of 300 images
// 61 -> 51 us, 600 of 200 28 -> 26).
template<bool FIRST, typename Body>
__device__ __forceinline__ void in_turns(const ImageArgs& a, uint32_t all, Body&& body)
{
    uint32_t at = blockIdx.x;
    const uint32_t blocks = *a.block_count;
    PlaceBlock b = a.blocks[FIRST ? min(at, all / kQuarters - 1) : at / kQuarters];
    all = min(all, blocks * kQuarters);
    const auto block_of = [&](uint32_t n) { return FIRST ? n % blocks : n / kQuarters; };
    if (FIRST && at >= blocks && at < all) b = a.blocks[block_of(at)];
    for (uint32_t turn = 0; at < all;) {
        body(b, block_of(at), FIRST ? at / blocks : at % kQuarters);
        ++turn;
        at = turn * gridDim.x + (turn & 1 ? gridDim.x - 1 - blockIdx.x : blockIdx.x);
        if (at < all) b = a.blocks[block_of(at)];
    }
}

// One workgroup per 64 records, a lane per record in each of its 16 waves, the waves side by side over
// the image's keys.  Records of equal key keep their input order; a record's own key does not count as one (going over its
// 64 keys again for it, a trip to memory each, was half the launch: 7000 records of 16 images 14.9 -> 7.1 us).
__global__ __launch_bounds__(kWide) void nms_place_kernel(ImageArgs a)
{
    __shared__ uint32_t smaller[kWave];
    PlaceBlock b;
    if (!find_block(a, blockIdx.x, b)) return;
    const uint32_t lane = threadIdx.x & (kWave - 1);
    const uint32_t wave = threadIdx.x / kWave;
    if (threadIdx.x < kWave) smaller[threadIdx.x] = 0;
    __syncthreads();
    const bool live = b.first + lane < b.image_end;
    const uint32_t p = live ? b.first + lane : b.first;
    const uint64_t mine = a.loose_key[p];
    const uint32_t source = a.loose_source[p];
    uint32_t rank = 0;
    for (uint32_t q0 = b.image_begin + wave * kWave; q0 < b.image_end; q0 += kWide) {
        const uint32_t here = min(static_cast<uint32_t>(kWave), b.image_end - q0);
        // lanes past the end carry the largest key: none is smaller than any record's
        const uint64_t keys = lane < here ? a.loose_key[q0 + lane] : ~0ull;
        const uint32_t own = p - q0;       // beyond any lane where the record's key is not among these
        bool equal = false;
#pragma unroll 16
        for (uint32_t j = 0; j < kWave; ++j) {
            const uint64_t k = key_of_lane(keys, static_cast<int>(j));
            rank += k < mine ? 1u : 0u;
            equal |= k == mine && j != own;
        }
        if (__ballot(equal)) {
            const uint32_t sources = a.loose_source[min(q0 + lane, b.image_end - 1)];
            for (uint32_t j = 0; j < here; ++j)
                if (key_of_lane(keys, static_cast<int>(j)) == mine && static_cast<uint32_t>(__builtin_amdgcn_readlane(sources, j)) < source)
                    ++rank;
        }
    }
    if (rank) atomicAdd(&smaller[lane], rank);
    __syncthreads();
    if (wave != 0 || !live) return;
    const uint32_t place = b.image_begin + smaller[lane];
    const pxh_detection d = a.records[source];
    a.key[place] = mine;
    a.source[place] = source;
    a.box[place] = normalized_rect(d);
    a.cls[place] = static_cast<uint32_t>(min(max(d.class_index, 0), a.classes - 1));
}

// A quarter of a block of 64 places to a workgroup, 16 places: a wave holds them four times over, and its quarters and
// the 16 waves share out the places in front of them (and the block's own) evenly, from LDS; what they find is put together
// in the words it belongs to, and a lane per word and place stores them.  A pair is some 90 instructions, the whole overlap
// test for nearly every step of a wave, so what bounds the launch is how evenly the pairs lie on the compute units: 64
// places to a workgroup and a wave to a word, 7000 records of 16 images took 26 us, with a word's places shared out over
// the waves 20, now 8.0.
constexpr uint32_t kConflictPlaces = kWave / kQuarters;

template<bool FIRST>
__global__ __launch_bounds__(kWide) void nms_conflicts_kernel(ImageArgs a, uint32_t all)
{
    __shared__ float4 boxes[kLargeImage];
    __shared__ uint32_t classes[kLargeImage];
    __shared__ unsigned long long found[2][kMaskWords][kConflictPlaces];
    __shared__ uint64_t beyond[2][kConflictPlaces];
    __shared__ uint32_t slots[2][kConflictPlaces];
    const uint32_t t = threadIdx.x;
    // one part of a block; all lanes end it together
    const auto look = [&](const PlaceBlock& b, uint32_t block, uint32_t part) {
        if (b.image_end - b.image_begin > kLargeImage) {
            if (part == 0 && t < kSettledWords) a.settled[block * kSettledStride + t] = 0;
            return;
        }
        const uint32_t first = b.first + part * kConflictPlaces;
        if (first >= b.image_end) return;
        // places of the image from here on: this workgroup's are from `first_place` to `length`
        const uint32_t first_place = first - b.image_begin;
        const uint32_t length = min(first + kConflictPlaces, b.image_end) - b.image_begin;
        if (t < length) {
            boxes[t] = a.box[b.image_begin + t];
            classes[t] = a.cls[b.image_begin + t];
        }
        if (t < 2 * kMaskWords * kConflictPlaces) (&found[0][0][0])[t] = 0;
        if (t < 2 * kConflictPlaces) {
            (&beyond[0][0])[t] = 0;
            (&slots[0][0])[t] = 0;
        }
        __syncthreads();
        constexpr uint32_t kTeams = kWide / kConflictPlaces;
        const uint32_t column = t % kConflictPlaces;
        const uint32_t place = first_place + column;
        const bool live = place < length;
        const uint32_t share = (length + kTeams - 1) / kTeams;       // 16 at most
        const uint32_t q_first = t / kConflictPlaces * share, q_last = min(q_first + share, live ? place : 0u);
        const float4 box = boxes[live ? place : first_place];
        const uint32_t cls = classes[live ? place : first_place];
        uint32_t hits[2] = { 0, 0 };       // bit j: place q_first + j
        for (uint32_t q = q_first; q < q_last; ++q) {
            const bool same = classes[q] == cls;
            if (overlaps_above(box, boxes[q], same ? a.threshold : kDuplicateOverlap)) hits[same ? 1 : 0] |= 1u << (q - q_first);
        }
        // a share begins anywhere in a word and may end in the next
        const uint32_t word = q_first >> 6, shift = q_first & 63;
#pragma unroll
        for (int pass = 0; pass < 2; ++pass) {
            if (!hits[pass]) continue;
            const uint64_t low = static_cast<uint64_t>(hits[pass]) << shift;
            const uint64_t high = shift ? static_cast<uint64_t>(hits[pass]) >> (64 - shift) : 0ull;
            if (low) atomicOr(&found[pass][word][column], static_cast<unsigned long long>(low));
            if (high) atomicOr(&found[pass][word + 1][column], static_cast<unsigned long long>(high));
        }
        __syncthreads();
        const uint32_t most = a.mask_slots;
        if (t < kMaskWords * kConflictPlaces && live) {
            const uint32_t mine = t / kConflictPlaces;       // the word; `column` and `place` are those of above
#pragma unroll
            for (int pass = 0; pass < 2; ++pass) {
                const uint64_t mask = found[pass][mine][column];
                if (!mask) continue;
                const uint32_t slot = atomicAdd(&slots[pass][column], 1u);
                if (slot < most) {
                    const size_t at = static_cast<size_t>(slot) * a.capacity + b.image_begin + place;
                    a.masks[pass][at] = mask;
                    a.ids[pass][at] = static_cast<uint8_t>(mine);
                } else {
                    atomicOr(reinterpret_cast<unsigned long long*>(&beyond[pass][column]), 1ull << mine);
                }
            }
        }
        __syncthreads();
        if (t >= kConflictPlaces || !live) return;
        for (int pass = 0; pass < 2; ++pass) a.beyond[pass][b.image_begin + place] = beyond[pass][column];
        a.slots[b.image_begin + place] = min(slots[0][column], most) | min(slots[1][column], most) << 8;
    };
    in_turns<FIRST>(a, all, [&](const PlaceBlock& b, uint32_t block, uint32_t part) {
        __syncthreads();       // (a part reuses the workgroup's LDS)
        look(b, block, part);
    });
}

__device__ __forceinline__ uint64_t load_bits(const uint64_t* set, uint32_t word)
{
    return __hip_atomic_load(set + word, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
}

__device__ __forceinline__ void set_bit(uint64_t* set, uint32_t at)
{
    atomicOr(reinterpret_cast<unsigned long long*>(set + (at >> 6)), 1ull << (at & 63));
}

// What the records of lower rank say about place p (places are relative to the image here): 1 = a kept
// one conflicts, 2 = none does but one that may is undecided, 0 = neither.
struct Standing {
    int pass;
    uint32_t image_begin, p;
    const uint64_t* kept;
    const uint64_t* gone;
};

// The same for the places of one word of the bit sets, pair by pair.
__device__ __forceinline__ int recheck(const ImageArgs& a, const Standing& s, uint32_t word, const float4& box, uint32_t cls)
{
    // `kept` is read first: a bit that is set in between shows up as undecided, never as absent
    const uint64_t kept = load_bits(s.kept, word);
    uint64_t bits = kept | ~load_bits(s.gone, word);
    if (word == s.p >> 6) bits &= (1ull << (s.p & 63)) - 1;
    bool pending = false;
    for (; bits; bits &= bits - 1) {
        const int bit = __builtin_ctzll(bits);
        const uint32_t q = s.image_begin + word * 64 + bit;
        if ((a.cls[q] == cls) != (s.pass == 1)) continue;
        if (!overlaps_above(box, a.box[q], s.pass == 0 ? kDuplicateOverlap : a.threshold)) continue;
        if ((kept >> bit) & 1) return 1;
        pending = true;
    }
    return pending ? 2 : 0;
}

// The first stored words of a place's mask, which a lane keeps from round to round: read again in each, the rounds of 16
// images around 445 places took 11.4 us, now 9.4.
constexpr int kHeldWords = 4;

struct HeldMask {
    int stored;
    uint32_t word[kHeldWords];
    uint64_t mask[kHeldWords];
};

__device__ __forceinline__ HeldMask held_mask(const ImageArgs& a, uint32_t place, int pass, uint32_t slots)
{
    HeldMask h;
    h.stored = (slots >> (8 * pass)) & 0xFF;
#pragma unroll
    for (int slot = 0; slot < kHeldWords; ++slot) {
        const bool there = slot < h.stored;
        const size_t at = static_cast<size_t>(there ? slot : 0) * a.capacity + place;
        h.word[slot] = there ? a.ids[pass][at] : 0;
        h.mask[slot] = there ? a.masks[pass][at] : 0ull;
    }
    return h;
}

__device__ __forceinline__ int conflict_state(const ImageArgs& a, const Standing& s, const HeldMask& h)
{
    const uint32_t place = s.image_begin + s.p;
    const int stored = h.stored;
    if (stored == 0) return 0;                      // nothing is kept beyond the stored words either
    uint64_t beyond = stored == a.mask_slots ? a.beyond[s.pass][place] : 0ull;
    bool pending = false;
    float4 box = make_float4(0, 0, 0, 0);
    uint32_t cls = 0;
    if (beyond) {
        box = a.box[place];
        cls = a.cls[place];
    }
#pragma unroll
    for (int slot = 0; slot < kHeldWords; ++slot) {
        if (h.mask[slot] & load_bits(s.kept, h.word[slot])) return 1;
        pending = pending || (h.mask[slot] & ~load_bits(s.gone, h.word[slot])) != 0;
    }
    for (int slot = kHeldWords; slot < stored; ++slot) {
        const size_t at = static_cast<size_t>(slot) * a.capacity + place;
        const uint32_t word = a.ids[s.pass][at];
        const uint64_t mask = a.masks[s.pass][at];
        if (mask & load_bits(s.kept, word)) return 1;
        pending = pending || (mask & ~load_bits(s.gone, word)) != 0;
    }
    for (; beyond; beyond &= beyond - 1) {          // words that were not stored: all of their places
        const int state = recheck(a, s, static_cast<uint32_t>(__builtin_ctzll(beyond)), box, cls);
        if (state == 1) return 1;
        pending = pending || state == 2;
    }
    return pending ? 2 : 0;
}

// ---- large images, block by block
// A word that a block of 64 places leaves behind: 32 bits, and above them a tag that says they are there, so that they
// arrive with the look that finds them.
constexpr uint64_t kSettledTag = 1ull << 32;

// The words of block `at`, one in each of the first lanes (the others hold a tag and nothing).
__device__ __forceinline__ uint64_t look_at_block(const ImageArgs& a, uint32_t at, uint32_t lane)
{
    return lane < kSettledWords ? __hip_atomic_load(a.settled + at * kSettledStride + lane, __ATOMIC_RELAXED,
                                                    __HIP_MEMORY_SCOPE_AGENT)
                                : kSettledTag;
}

__device__ __forceinline__ bool block_is_there(uint64_t words) { return __ballot(words < kSettledTag) == 0; }

__device__ __forceinline__ uint64_t two_words(uint64_t words, int first)
{
    const uint32_t lo = __builtin_amdgcn_readlane(static_cast<uint32_t>(words), first);
    const uint32_t hi = __builtin_amdgcn_readlane(static_cast<uint32_t>(words), first + 1);
    return (static_cast<uint64_t>(hi) << 32) | lo;
}

// The lanes of `open` that are kept: a lane whose `mask` (bits of lower lanes) meets a kept one is not.  A round decides
// at least the lowest of them.
__device__ __forceinline__ uint64_t settle_lanes(uint64_t kept, uint64_t open, uint64_t mask, uint32_t lane)
{
    while (open) {
        const bool mine = (open >> lane) & 1;
        const uint64_t keep = __ballot(mine && !(mask & (kept | open)));
        const uint64_t drop = __ballot(mine && (mask & kept));
        kept |= keep;
        open &= ~(keep | drop);
    }
    return kept;
}

// A workgroup takes the next block of 64 places, a lane per place in each of its 16 waves, and goes over the blocks
// before it in the image, the waves side by side: conflicts with the places of a settled block that were kept, or, with
// one that is not settled yet, with all of its places while it is waited for.  Then the block's own places, and its
// words for the blocks behind it.  What bounds it is the chain of decisions, one and a half to two microseconds from
// block to block, and the ranking in front of it (30000 records of one image around 20 places: 1.2 ms, 11.1 on masks in
// one workgroup, 7.4 on the sorting path; 60000: 2.9, 104 and 18.5).
// An image's blocks are taken in order and a block waits only for blocks that were taken before it, whose workgroups
// therefore run: the first that is not settled never waits, so every wait ends.  (The bound on the looks makes the exit
// unconditional; it is seconds.)
__device__ void settle_blocks(const ImageArgs& a, uint32_t worker)
{
    __shared__ uint64_t dropped[2];            // by earlier blocks, a bit per lane
    __shared__ uint64_t inner[2][kWave];       // conflicts inside the block: bits of lower lanes
    __shared__ uint32_t index[kWave];          // earlier records of the same class
    __shared__ uint32_t large[kImageCapacity / kLargeImage];
    __shared__ uint32_t scan_lds[kWide / kWave + 1];
    __shared__ uint32_t taken, before;
    const uint32_t lane = threadIdx.x & (kWave - 1);
    const uint32_t wave = threadIdx.x / kWave;
    constexpr uint32_t kWaves = kWide / kWave;
    constexpr int kOwn = kWave / kWaves;       // of the block's own places, to a wave
    const bool is_large = threadIdx.x < static_cast<uint32_t>(a.batch) &&
                          a.image_begin[threadIdx.x + 1] - a.image_begin[threadIdx.x] > kLargeImage;
    uint32_t images;
    const uint32_t nth = wide_exclusive_scan(is_large ? 1u : 0u, scan_lds, images);
    if (images == 0) return;
    if (is_large) large[nth] = threadIdx.x;
    uint32_t looks_left = 1u << 22;
    for (uint32_t turn = 0; turn < images;) {
        __syncthreads();
        // the workgroups spread over the images, and move on to the next when one has no more blocks
        const uint32_t image = large[(worker + turn) % images];
        if (threadIdx.x == 0) taken = atomicAdd(a.ticket + image, 1u);
        __syncthreads();
        const uint32_t earlier = taken;
        const uint32_t at = a.first_block[image] + earlier;
        const uint32_t image_begin = a.image_begin[image], image_end = a.image_begin[image + 1];
        const uint32_t block_begin = image_begin + earlier * kWave;
        if (block_begin >= image_end) {
            ++turn;
            continue;
        }
        if (threadIdx.x < kWave) {
            inner[0][lane] = inner[1][lane] = 0;
            index[lane] = 0;
        }
        if (threadIdx.x < 2) dropped[threadIdx.x] = 0;
        if (threadIdx.x == 0) before = 0;
        __syncthreads();
        const bool live = block_begin + lane < image_end;
        const uint32_t p = live ? block_begin + lane : block_begin;
        const float4 box = a.box[p];
        const uint32_t cls = a.cls[p];
        // the block's own pairs, and how far down its group each place is: nothing suppresses one past those that are visited
        uint32_t same_before = 0;
        for (uint32_t i = wave; i < earlier; i += kWaves) {
            const int their_class = static_cast<int>(a.cls[image_begin + i * kWave + lane]);
#pragma unroll 16
            for (int j = 0; j < static_cast<int>(kWave); ++j)
                same_before += static_cast<uint32_t>(__builtin_amdgcn_readlane(their_class, j)) == cls ? 1u : 0u;
        }
#pragma unroll
        for (int u = 0; u < kOwn; ++u) {
            const int j = static_cast<int>(wave) * kOwn + u;
            const bool same = static_cast<uint32_t>(__builtin_amdgcn_readlane(static_cast<int>(cls), j)) == cls;
            const float4 other = make_float4(from_lane(box.x, j), from_lane(box.y, j), from_lane(box.z, j), from_lane(box.w, j));
            same_before += same && static_cast<uint32_t>(j) < lane ? 1u : 0u;
            if (static_cast<uint32_t>(j) < lane && overlaps_above(box, other, same ? a.threshold : kDuplicateOverlap))
                atomicOr(reinterpret_cast<unsigned long long*>(&inner[same ? 1 : 0][lane]), 1ull << j);
        }
        if (same_before) atomicAdd(&index[lane], same_before);
        __syncthreads();
        const bool visited = index[lane] < static_cast<uint32_t>(kGroupVisit);
        bool drop0 = false, drop1 = false;
        for (uint32_t i = wave; i < earlier; i += kWaves) {
            const uint32_t q = image_begin + i * kWave + lane;
            const float4 their_box = a.box[q];
            const int their_class = static_cast<int>(a.cls[q]);
            uint64_t words = look_at_block(a, at - earlier + i, lane);
            const bool there = block_is_there(words);
            const uint64_t in_first = there ? two_words(words, 0) : ~0ull, in_second = there ? two_words(words, 2) : ~0ull;
            uint64_t found[2] = { 0, 0 };
            for (uint64_t bits = in_first; bits; bits &= bits - 1) {
                const int j = __builtin_ctzll(bits);
                const bool same = static_cast<uint32_t>(__builtin_amdgcn_readlane(their_class, j)) == cls;
                const bool suppresses = (in_second >> j) & 1;
                if (!__ballot(!same || (suppresses && visited))) continue;
                const float4 other = make_float4(from_lane(their_box.x, j), from_lane(their_box.y, j),
                                                 from_lane(their_box.z, j), from_lane(their_box.w, j));
                if (overlaps_above(box, other, same ? a.threshold : kDuplicateOverlap)) {
                    if (same) found[1] |= 1ull << j;
                    else found[0] |= 1ull << j;
                }
            }
            for (; !block_is_there(words) && looks_left; --looks_left) {
                __builtin_amdgcn_s_sleep(1);
                words = look_at_block(a, at - earlier + i, lane);
            }
            drop0 = drop0 || (found[0] & two_words(words, 0));
            drop1 = drop1 || (found[1] & two_words(words, 2));
            const uint32_t survivors = __builtin_amdgcn_readlane(static_cast<uint32_t>(words), 4);
            if (i + 1 == earlier && lane == 0) before = survivors;
        }
        const uint64_t all0 = __ballot(drop0), all1 = __ballot(drop1);
        if (lane == 0) {
            if (all0) atomicOr(reinterpret_cast<unsigned long long*>(&dropped[0]), all0);
            if (all1) atomicOr(reinterpret_cast<unsigned long long*>(&dropped[1]), all1);
        }
        __syncthreads();
        if (wave != 0) continue;
        const uint64_t first = settle_lanes(0, __ballot(live) & ~dropped[0], inner[0][lane], lane);
        // the second pass knows only what the first kept; places past the first 1024 of a group are never visited and stay
        const uint64_t reached = __ballot(visited);
        const uint64_t second = settle_lanes(first & ~reached, first & reached & ~dropped[1], inner[1][lane], lane);
        const uint32_t upto = before + static_cast<uint32_t>(__popcll(second));
        if (lane < kSettledWords) {
            const uint64_t bits = lane < 2 ? first : second & reached;
            const uint32_t word = lane == 4 ? upto : static_cast<uint32_t>(bits >> (32 * (lane & 1)));
            __hip_atomic_store(a.settled + at * kSettledStride + lane, kSettledTag | word, __ATOMIC_RELAXED,
                               __HIP_MEMORY_SCOPE_AGENT);
        }
        if ((second >> lane) & 1) {
            const uint32_t to = image_begin + before + __popcll(second & ((1ull << lane) - 1));
            a.kept_key[to] = a.key[p];
            a.kept_source[to] = a.source[p];
        }
        if (block_begin + kWave >= image_end && lane == 0) a.kept_images[image] = upto;
    }
}

// One workgroup per image, a lane per place; those behind them settle the large images.  Rounds until each place is
// decided: a round decides at least the undecided place of lowest rank; the bound makes the exit unconditional.
__global__ __launch_bounds__(kWide) void nms_settle_kernel(ImageArgs a)
{
    __shared__ uint64_t kept[kMaskWords], gone[kMaskWords];
    __shared__ uint32_t scan_lds[kWide / kWave + 1];
    const uint32_t t = threadIdx.x;
    if (blockIdx.x >= static_cast<uint32_t>(a.batch)) {
        settle_blocks(a, blockIdx.x - static_cast<uint32_t>(a.batch));
        return;
    }
    const uint32_t begin = a.image_begin[blockIdx.x];
    const uint32_t places = a.image_begin[blockIdx.x + 1] - begin;
    if (places > kLargeImage) return;
    if (places == 0) {
        if (t == 0) a.kept_images[blockIdx.x] = 0;
        return;
    }
    const uint32_t slots = t < places ? a.slots[begin + t] : 0;
    if (t < kMaskWords) gone[t] = 0;
    Standing s{};
    s.image_begin = begin;
    s.p = t;
    s.kept = kept;
    s.gone = gone;
    for (s.pass = 0; s.pass < 2; ++s.pass) {
        // the second pass starts from what the first dropped: absent there
        if (t < kMaskWords) kept[t] = 0;
        __syncthreads();
        bool undecided = t < places;
        const HeldMask held = held_mask(a, begin + (undecided ? t : 0), s.pass, undecided ? slots : 0);
        if (undecided && s.pass == 1) undecided = !((load_bits(gone, t >> 6) >> (t & 63)) & 1);
        for (uint32_t round = 0; round <= kWide; ++round) {
            if (undecided) {
                const int state = conflict_state(a, s, held);
                if (state != 2) {
                    set_bit(state == 1 ? gone : kept, t);
                    undecided = false;
                }
            }
            if (__syncthreads_or(undecided) == 0) break;
        }
    }
    const bool survives = t < places && ((kept[t >> 6] >> (t & 63)) & 1);
    uint32_t total;
    const uint32_t nth = wide_exclusive_scan(survives ? 1u : 0u, scan_lds, total);
    if (survives) {
        a.kept_key[begin + nth] = a.key[begin + t];
        a.kept_source[begin + nth] = a.source[begin + t];
    }
    if (t == 0) a.kept_images[blockIdx.x] = total;
}

// One wave per survivor, a quarter of a block of 64 to a workgroup: how many of each other image's survivors come before it.  A power of two of lanes share an image
// (batches of up to 64; else images take turns): they look at as many places that split what is left evenly, and the part
// between the last that comes before and the first that does not is what is left of it.  The looks of a step are on their way at
// once, so that a step costs one trip to memory: with four lanes four steps for 440 survivors, where halving takes nine
// (7000 records of 16 images, the launch, with four waves to a wave's survivors: 13.7 -> 5.9 us).
static_assert(kQuarters * (kWide / kWave) == kWave, "a wave to a survivor");

template<bool FIRST>
__global__ __launch_bounds__(kWide) void nms_merge_images_kernel(ImageArgs a, pxh_detection* kept, int* kept_count, uint32_t lanes,
                                                                 FastDiv by_parts, uint32_t all)
{
    const uint32_t lane = threadIdx.x & (kWave - 1);
    const uint32_t wave = threadIdx.x / kWave;
    const uint32_t images = static_cast<uint32_t>(a.batch);
    if (blockIdx.x == 0 && wave == 0) {
        uint32_t sum = 0;
        for (uint32_t i = lane; i < images; i += kWave) sum += a.kept_images[i];
#pragma unroll
        for (int off = kWave / 2; off > 0; off >>= 1) sum += __shfl_xor(sum, off, kWave);
        if (lane == 0) *kept_count = static_cast<int>(sum);
    }
    const uint32_t part = lane & (lanes - 1), per_round = kWave / lanes;
    const uint64_t team = ((1ull << lanes) - 1) << (lane & ~(lanes - 1));
    // the first images' tables on their way beside the block
    const uint32_t nearest = min(lane / lanes, images - 1);
    const uint32_t near_begin = a.image_begin[nearest], near_kept = a.kept_images[nearest];
    const auto place = [&](const PlaceBlock& b, uint32_t, uint32_t nth) {
        const uint32_t at = b.first + nth * (kWide / kWave) + wave;
        const uint32_t end = min(b.first + kWave, b.image_begin + a.kept_images[b.image]);
        if (at >= end) return;
        const uint64_t key = a.kept_key[at];
        const uint32_t source = a.kept_source[at];
        constexpr uint32_t kRecordWords = sizeof(pxh_detection) / 4;
        const uint32_t record = reinterpret_cast<const uint32_t*>(a.records + source)[lane % kRecordWords];
        uint32_t before = 0;
        for (uint32_t i0 = 0; i0 < images; i0 += per_round) {
            const uint32_t i = i0 + lane / lanes;
            uint32_t lo = 0, hi = 0;
            if (i < images) {
                lo = i0 ? a.image_begin[i] : near_begin;
                hi = lo + (i0 ? a.kept_images[i] : near_kept);
            }
            const uint32_t first = lo;
            if (i == b.image) lo = hi = at;       // the survivors of its own image: those in front of it
            while (__ballot(lo < hi)) {
                // lane `part` looks at place lo + length * (part + 1) / (lanes + 1): below hi, and in order
                const uint32_t length = hi - lo;
                const auto look = [&](uint32_t step) { return lo + by_parts.div(length * step); };       // length is kImageCapacity at most
                const uint32_t middle = look(part + 1);
                bool less = false;
                if (length) {
                    const uint64_t k = a.kept_key[middle];
                    less = k < key || (k == key && a.kept_source[middle] < source);
                }
                // places that come before are the first ones: as many lanes as say so
                const uint32_t count = static_cast<uint32_t>(__popcll(__ballot(less) & team));
                if (length) {
                    const uint32_t from = count == 0 ? lo : look(count) + 1;
                    const uint32_t to = count == lanes ? hi : look(count + 1);
                    lo = from;
                    hi = to;
                }
            }
            if (part == 0 && i < images) before += lo - first;
        }
#pragma unroll
        for (int off = kWave / 2; off > 0; off >>= 1) before += __shfl_xor(before, off, kWave);
        if (lane < kRecordWords) reinterpret_cast<uint32_t*>(kept + before)[lane] = record;
    };
    in_turns<FIRST>(a, all, place);
}

size_t align256(size_t b) { return (b + 255) & ~static_cast<size_t>(255); }

struct Workspace {
    uint64_t* keys[2];
    uint32_t* vals[2];
    uint32_t* perm;
    float4* box;
    Segments* seg;
    uint32_t* state;
    uint32_t* keep;
    uint32_t* resume;
    uint32_t* hist;
    uint32_t* tile_kept;
    uint32_t* counters;
    size_t bytes;
};

Workspace carve(void* base, int capacity)
{
    const size_t cap = static_cast<size_t>(capacity > 0 ? capacity : 1);
    const size_t tiles = (cap + kSortTile - 1) / kSortTile;
    char* p = static_cast<char*>(base);
    size_t at = 0;
    auto take = [&](size_t bytes) {
        char* r = p ? p + at : nullptr;
        at += align256(bytes);
        return r;
    };
    Workspace w{};
    w.keys[0] = reinterpret_cast<uint64_t*>(take(cap * 8));
    w.keys[1] = reinterpret_cast<uint64_t*>(take(cap * 8));
    w.vals[0] = reinterpret_cast<uint32_t*>(take(cap * 4));
    w.vals[1] = reinterpret_cast<uint32_t*>(take(cap * 4));
    w.perm = reinterpret_cast<uint32_t*>(take(cap * 4));
    w.box = reinterpret_cast<float4*>(take(cap * 16));
    w.seg = reinterpret_cast<Segments*>(take(cap * sizeof(Segments)));
    w.state = reinterpret_cast<uint32_t*>(take(cap * 4));
    w.keep = reinterpret_cast<uint32_t*>(take(cap * 4));
    w.resume = reinterpret_cast<uint32_t*>(take(cap * 4));
    w.hist = reinterpret_cast<uint32_t*>(take(tiles * kDigits * 4));
    w.tile_kept = reinterpret_cast<uint32_t*>(take(tiles * 4));
    w.counters = reinterpret_cast<uint32_t*>(take(8 * 4));
    w.bytes = at;
    return w;
}

// Which lists go by image: those whose images have a lane each and whose masks and blocks fit the library's first
// workspace.  Measured on both paths, us sorted -> by image: 600 records of 64 images 161 -> 33, 7000 of 16 400 -> 76,
// 60000 of 32 1220 -> 308, of 4 4900 -> 990, of 1 18500 -> 2900; 600 of one image in a list for 65536 163 -> 69, 4000
// 930 -> 205.  One class has no pairs for the duplicate pass, and 1024 places that are visited: a long list of it stays
// with the sorting path where the batch is too small to spread it (30000 of one image 1800 -> 786, but 60000 2060 -> 2290).
bool by_image(int capacity, int batch, int classes)
{
    return batch <= kImageBatch && capacity <= kImageCapacity && (classes > 1 || capacity <= 32768 || capacity / 2048 <= batch);
}

// The same for the launches by image; `args` gets every pointer.  `mask_words`: of one pass's masks.
size_t carve_images(void* base, int capacity, int batch, size_t mask_words, ImageArgs& args)
{
    const size_t cap = static_cast<size_t>(capacity);
    const size_t tiles = (cap + kWide - 1) / kWide, images = static_cast<size_t>(batch);
    args.mask_slots = mask_slots(capacity);
    char* p = static_cast<char*>(base);
    size_t at = 0;
    auto take = [&](auto*& out, size_t count) {
        using T = std::remove_reference_t<decltype(*out)>;
        out = p ? reinterpret_cast<T*>(p + at) : nullptr;
        at += align256(count * sizeof(T));
    };
    take(args.tile_images, tiles * images);
    take(args.image_begin, images + 1);
    take(args.block_count, 1);
    take(args.blocks, cap / 64 + images + 1);
    take(args.loose_key, cap);
    take(args.loose_source, cap);
    take(args.key, cap);
    take(args.source, cap);
    take(args.box, cap);
    take(args.cls, cap);
    take(args.slots, cap);
    for (int k = 0; k < 2; ++k) {
        take(args.ids[k], mask_words);
        take(args.beyond[k], cap);
        take(args.masks[k], mask_words);
    }
    take(args.first_block, images);
    take(args.ticket, images);
    take(args.settled, (cap / 64 + images + 1) * kSettledStride);
    take(args.kept_key, cap);
    take(args.kept_source, cap);
    take(args.kept_images, images);
    return at;
}

size_t carve_images(void* base, int capacity, int batch, ImageArgs& args)
{
    return carve_images(base, capacity, batch, static_cast<size_t>(capacity) * mask_slots(capacity), args);
}

std::atomic<int> g_sweeps{ 6 };      // parallel sweeps of the duplicate pass before the per-image loop takes over

}  // namespace
}  // namespace pxh

using namespace pxh;

extern "C" {

size_t pxh_nms_workspace_bytes(int capacity)
{
    if (capacity <= 0) return 0;
    const size_t sorted = carve(nullptr, capacity).bytes;
    if (capacity <= kSmall) return sorted;
    // The most that any batch and any shorter list ask for, so that a longer list's bytes serve every shorter one:
    // a list whose records store fewer mask words can need less than a shorter one, but none more than fills kMaskBytes.
    const int most = capacity < kImageCapacity ? capacity : kImageCapacity;
    const size_t every_word = static_cast<size_t>(most) * kMaskWords;
    ImageArgs args{};
    const size_t by_image = carve_images(nullptr, most, kImageBatch, every_word < kMaskListWords ? every_word : kMaskListWords, args);
    return by_image > sorted ? by_image : sorted;
}

int pxh_debug_nms_sweeps(int sweeps)
{
    if (sweeps >= 1 && sweeps <= 6) return g_sweeps.exchange(sweeps);
    return g_sweeps.load();
}

int pxh_nms(const pxh_detection* records, const int* count, int capacity, int batch, int classes, float threshold,
            pxh_detection* kept, int* kept_count, void* workspace, size_t workspace_bytes, void* stream)
{
    if (!count || !kept_count || (capacity > 0 && (!records || !kept))) return fail_invalid("pxh_nms: null pointer");
    if (capacity < 0 || batch <= 0 || classes <= 0)
        return fail_invalid("pxh_nms: capacity must not be negative, batch and classes must be positive");
    if (!(threshold >= 0.0f)) return fail_invalid("pxh_nms: the threshold must not be negative");
    if (1ull * batch * classes >= (1ull << 31)) {
        set_error("pxh_nms: batch * classes of 2^31 or more is not supported");
        return PXH_ERR_UNSUPPORTED;
    }
    if (records == kept && capacity > 0) return fail_invalid("pxh_nms: records and kept must be distinct buffers");
    if (capacity == 0) return pxh_fill_i32(kept_count, 1, 0, stream);
    if (capacity <= kSmall) {
        hipLaunchKernelGGL(nms_small_kernel, dim3(1), dim3(kWide), 0, as_stream(stream), records, count, capacity,
                           batch, classes, threshold, kept, kept_count);
        return check_launch("pxh_nms");
    }
    void* ws;
    if (by_image(capacity, batch, classes)) {
        ImageArgs a{};
        int rc = resolve_workspace(workspace, workspace_bytes, carve_images(nullptr, capacity, batch, a), &ws,
                                   as_stream(stream));
        if (rc) return rc;
        carve_images(ws, capacity, batch, a);
        a.records = records; a.count = count; a.capacity = capacity; a.batch = batch; a.classes = classes;
        a.threshold = threshold;
        hipStream_t s = as_stream(stream);
        const dim3 wide(kWide), per_tile(grid_for(capacity, kWide));
        // blocks of 64 places: every image but the last may leave one of them partly empty
        const int images = batch < capacity ? batch : capacity;
        const dim3 per_block(static_cast<unsigned>(capacity / 64 + images));
        hipLaunchKernelGGL(nms_count_images_kernel, per_tile, wide, 0, s, a);
        hipLaunchKernelGGL(nms_group_images_kernel, per_tile, wide, 0, s, a);
        hipLaunchKernelGGL(nms_place_kernel, per_block, wide, 0, s, a);
        const uint32_t quarters = per_block.x * kQuarters;
        const dim3 in_turns(std::min(quarters, kTurnWorkgroups));
        const bool many = batch > kWave;
        hipLaunchKernelGGL(many ? nms_conflicts_kernel<true> : nms_conflicts_kernel<false>, in_turns, wide, 0, s, a, quarters);
        const unsigned helpers = static_cast<uint32_t>(capacity) > kLargeImage ? kSettleWorkgroups : 0;
        hipLaunchKernelGGL(nms_settle_kernel, dim3(batch + helpers), wide, 0, s, a);
        // as many lanes to an image as leave one for each, sixteen at most: further ones save no step worth a division
        uint32_t lanes = 1;
        while (lanes < 16 && 2 * lanes * static_cast<uint32_t>(batch) <= static_cast<uint32_t>(kWave)) lanes *= 2;
        hipLaunchKernelGGL(many ? nms_merge_images_kernel<true> : nms_merge_images_kernel<false>, in_turns, wide, 0, s, a, kept, kept_count, lanes, FastDiv(lanes + 1), quarters);
        return check_launch("pxh_nms");
    }
    int rc = resolve_workspace(workspace, workspace_bytes, carve(nullptr, capacity).bytes, &ws, as_stream(stream));
    if (rc) return rc;
    const Workspace w = carve(ws, capacity);
    hipStream_t s = as_stream(stream);
    const dim3 per_record(grid_for(capacity, kBlock)), per_tile(grid_for(capacity, kSortTile));
    const dim3 lanes(kBlock), wide(kWide);

    hipLaunchKernelGGL(nms_rank_keys_kernel, per_record, lanes, 0, s, records, count, capacity, w.keys[0], w.vals[0],
                       w.counters);
    int from = 0;
    auto sort_pass = [&](int shift) {
        SortArgs a{ w.keys[from], w.vals[from], w.keys[1 - from], w.vals[1 - from], w.hist, count, capacity, shift };
        hipLaunchKernelGGL(sort_histogram_kernel, per_tile, lanes, 0, s, a);
        hipLaunchKernelGGL(scan_counters_kernel, dim3(1), wide, 0, s, w.hist, count, capacity,
                           static_cast<uint32_t>(kDigits), static_cast<int*>(nullptr));
        hipLaunchKernelGGL(sort_scatter_kernel, per_tile, lanes, 0, s, a);
        from = 1 - from;
    };
    for (int shift = 0; shift < 64; shift += 8) sort_pass(shift);
    // keys of the second sort go to the other buffer pair; vals[from] still holds rank -> input index
    hipLaunchKernelGGL(nms_group_keys_kernel, per_record, lanes, 0, s, records, count, capacity, w.vals[from], w.perm,
                       w.keys[1 - from], w.vals[1 - from], batch, classes);
    from = 1 - from;
    for (int shift = 0; ((classes - 1) >> shift) > 0; shift += 8) sort_pass(shift);
    for (int shift = 0; ((batch - 1) >> shift) > 0; shift += 8) sort_pass(32 + shift);

    NmsArgs a{};
    a.records = records; a.count = count; a.capacity = capacity; a.perm = w.perm;
    a.group_key = w.keys[from]; a.rank = w.vals[from];
    a.box = w.box; a.seg = w.seg; a.state = w.state; a.keep = w.keep; a.resume = w.resume; a.counters = w.counters;
    hipLaunchKernelGGL(nms_gather_kernel, per_record, lanes, 0, s, a);
    const int sweeps = g_sweeps.load();      // read once: a call never sees it change
    // one wave per record, at most 64 Ki workgroups (the rest of a longer list comes round again)
    const unsigned sweep_blocks = grid_for(capacity, kBlock / kWave) < 65536u ? grid_for(capacity, kBlock / kWave) : 65536u;
    a.waves = sweep_blocks * (kBlock / kWave);
    for (int k = 0; k < sweeps; ++k)
        hipLaunchKernelGGL(nms_duplicate_sweep_kernel, dim3(sweep_blocks), lanes, 0, s, a, k);
    hipLaunchKernelGGL(nms_duplicate_finish_kernel, dim3(batch), wide, 0, s, a, sweeps - 1);
    hipLaunchKernelGGL(nms_group_kernel, dim3(static_cast<unsigned>(batch) * classes), wide, 0, s, a, threshold,
                       FastDiv(classes));
    hipLaunchKernelGGL(nms_count_kept_kernel, per_tile, lanes, 0, s, a, w.tile_kept);
    hipLaunchKernelGGL(scan_counters_kernel, dim3(1), wide, 0, s, w.tile_kept, count, capacity, 1u, kept_count);
    hipLaunchKernelGGL(nms_write_kept_kernel, per_tile, lanes, 0, s, a, w.tile_kept, kept);
    return check_launch("pxh_nms");
}

}
