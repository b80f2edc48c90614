// Batch-norm training backward in one launch where a group of workgroups shares a channel's slice.
#include "grouped.h"
#include "pixienn_hip_test.h"

#include <atomic>

namespace pxh {
namespace {

template<bool RAGGED>
__device__ __forceinline__ Pack<4> load(const float* p)
{
    if constexpr (RAGGED) return ld_word<true>(p);
    else return ld<4, true>(p, 0);
}

// What bounds these launches is memory: x and the delta are read once and the delta written once, where the three launches
// read both twice and a workgroup that holds a channel alone reads x twice.  Two workgroups to a compute unit (128
// registers a lane, 64 KB of LDS each) hold 24 vectors a lane between them; rounds of load, sums, exchange and store cost
// 7 us more than their bytes.  Against three launches, us, plain and with rescale + clip in front, leaky then mish:
//   16 x 128 x 152^2   156 -> 120   161 -> 125      220 -> 168   214 -> 169
//   16 x 64 x 304^2    298 -> 242   308 -> 260      398 -> 311   399 -> 338
//   16 x 64 x 152^2     85 ->  62    93 ->  67      112 ->  80   116 ->  87
//   4 x 16 x 416^2      52 ->  33    59 ->  38       65 ->  48    72 ->  54
//   2 x 32 x 320^2      33 ->  25    40 ->  30       44 ->  37    50 ->  43
//   2 x 32 x 160^2      17 ->  13    23 ->  17       24 ->  19    29 ->  24
// and, a group of one member, against one workgroup of 1024 lanes a channel (the limits are grouped_backward's):
//   16 x 512 x 38^2     29 ->  27    34 ->  31       37 ->  41    45 ->  46
// Loads kept in flight over fewer than two steps, or over four (spills), are slower.
//
// One member's share of channel c; `factor` and `limit` are the plan's (kRedo only).  It keeps d' = delta * act'(pre) in
// R steps of a lane and x beside it, the first R - L steps in registers and L in LDS, so that each tensor is read once.
template<int ACT, bool RAGGED, int R, int L, int MODE>
__device__ __forceinline__ void grouped_bwd_member(const ResidentBwdArgs& a, const GroupGeom& gg, const uint32_t c,
                                                   const uint32_t member, uint32_t& next_ticket,
                                                   [[maybe_unused]] const float factor, [[maybe_unused]] const float limit)
{
    constexpr int T = kGroupThreads, V = 4;
    constexpr int X = R - L;
    extern __shared__ __align__(16) float grouped_lds[];
    __shared__ double slots[MODE == kFirst ? 3 : 2][T / kWave];
    __shared__ DxCoef shared_coef;
    Pack<V>* const lds = reinterpret_cast<Pack<V>*>(grouped_lds) + threadIdx.x;
    uint32_t lane = threadIdx.x;
    const uint32_t begin = member * gg.span;
    const uint32_t end = min(gg.items, begin + gg.span);
    const uint32_t channel_at = c * static_cast<uint32_t>(gg.g.spatial);
    const auto item = [&](int r) { return begin + static_cast<uint32_t>(r * T) + lane; };
    // bytes to vector i of the slice (a tensor of these launches has fewer than 2^32: no 64-bit multiplies)
    const auto place = [&](uint32_t i) {
        if constexpr (RAGGED) {
            uint32_t n, j;
            gg.g.by_row.divmod(i, n, j);
            return (n * (gg.image_skip + gg.g.spatial) + channel_at + min(j * V, gg.g.spatial - static_cast<uint32_t>(V))) * 4u;
        } else {
            const uint32_t e = i * V;
            return (e + channel_at + gg.g.by_spatial.div(e) * gg.image_skip) * 4u;
        }
    };
    // values of vector i that the one in front holds too: they stay out of the sums, and are not written (the vector in front
    // may be another member's)
    const auto held = [&](uint32_t i) {
        uint32_t n, j;
        gg.g.by_row.divmod(i, n, j);
        const int beyond = static_cast<int>(j) * V + V - gg.g.spatial;
        return beyond > 0 ? beyond : 0;
    };
    // kStep steps at a time, a group's loads in flight while the sums pass over the group before it; the LDS part first:
    // its registers are free again after that.  Groups past the end of the share are left out, and in the one that holds
    // the end a lane past it reads the share's first vector and adds nothing: no branch around a load.
    constexpr int kStep = 2;
    static_assert(R % kStep == 0 && L % kStep == 0, "steps come in whole groups");
    const auto any = [&](int top) { return begin + static_cast<uint32_t>((top - kStep + 1) * T) < end; };
    Pack<V> d[R], x[R];
    const auto fetch = [&](int top) {
#pragma unroll
        for (int i = 0; i < kStep; ++i) {
            const uint32_t at = item(top - i);
            const uint32_t where = place(at < end ? at : begin);
            d[top - i] = load<RAGGED>(at_byte(a.b.delta, where));
            x[top - i] = load<RAGGED>(at_byte(a.b.x, where));
        }
    };
    if (any(R - 1)) fetch(R - 1);
    const FoldCoef k = make_coef(a.b.mean[c], a.b.var[c], a.b.scale[c], a.b.bias[c]);
    const float bias_updates_in = a.bias_updates[c], scale_updates_in = a.scale_updates[c], var_in = a.b.var[c];
    VarianceTerms terms{};
    const auto early_terms = [&] { if (threadIdx.x < kWave) terms = variance_terms(var_in); };
    double figures[MODE == kFirst ? kFirstWords : kSumWords] = {};
    float peak = 0.0f;
    // a vector in fp32, vectors in doubles, as in the small forms; on odd planes every value, as there
    const auto take = [&](int r) {
        const int own = item(r) >= end ? V : RAGGED ? held(item(r)) : 0;
        float va = 0.0f, vb = 0.0f, vq = 0.0f;
#pragma unroll
        for (int q = 0; q < V; ++q) {
            float t = q >= own ? d[r].v[q] : 0.0f;
            if constexpr (MODE == kFirst) {
                if constexpr (RAGGED) figures[2] += static_cast<double>(t * t);
                else vq += t * t;
                peak = fmaxf(peak, fabsf(t));
            }
            if constexpr (MODE == kRedo) t = rescaled_clipped(t, factor, limit);
            d[r].v[q] = t;
        }
        if constexpr (ACT != PXH_LINEAR) {
            float pre[V];
#pragma unroll
            for (int q = 0; q < V; ++q) pre[q] = affine(normalize(x[r].v[q], k), k);
            times_grad<ACT>(d[r].v, pre);
        }
#pragma unroll
        for (int q = 0; q < V; ++q) {
            const float t = ACT == PXH_LINEAR || q >= own ? d[r].v[q] : 0.0f;
            d[r].v[q] = t;
            const float u = q >= own ? t * (x[r].v[q] - k.mean) : 0.0f;
            if constexpr (RAGGED) {
                figures[0] += static_cast<double>(t);
                figures[1] += static_cast<double>(u);
            } else {
                va += t;
                vb += u;
            }
        }
        if constexpr (!RAGGED) {
            figures[0] += static_cast<double>(va);
            figures[1] += static_cast<double>(vb);
            if constexpr (MODE == kFirst) figures[2] += static_cast<double>(vq);
        }
        if (r >= X) lds[(r - X) * T] = x[r];
        __builtin_amdgcn_sched_barrier(0);
    };
#pragma unroll
    for (int top = R - 1; top >= 0; top -= kStep) {
        if (top >= kStep && any(top - kStep)) fetch(top - kStep);
        __builtin_amdgcn_sched_barrier(0);
        if (!any(top)) continue;
#pragma unroll
        for (int i = 0; i < kStep; ++i) take(top - i);
        // the sums as they stand: put off, every group's values would be kept until then
        asm volatile("" : "+v"(figures[0]), "+v"(figures[1]), "+v"(peak));
        if constexpr (MODE == kFirst) asm volatile("" : "+v"(figures[2]));
        __builtin_amdgcn_sched_barrier(0);
    }
    if constexpr (MODE == kFirst) {
        __shared__ float tops[T / kWave];
        resident_sum3_max<T>(figures[0], figures[1], figures[2], peak, slots, tops);
        figures[3] = static_cast<double>(peak);
    } else {
        resident_sum2<T>(figures[0], figures[1], slots);
    }
    // what the finish takes from the variance is formed while the others' figures are on their way
    constexpr int kWords = MODE == kFirst ? kFirstWords : kSumWords;
    uint64_t* const words = (MODE == kRedo ? gg.redo_words : gg.words) + static_cast<size_t>(c) * gg.members * kWords;
    if (gg.members > 1) leave_figures<kWords>(words, member, figures);
    early_terms();
    bool whole = true;
    if (gg.members > 1) {
        whole = collect_figures<kWords>(words, gg.members, gg.looks, figures);
        // The next share's number, by a thread that does not finish the channel.  Not before the others' figures are
        // there: until then it could be the number of a member that this one waits for.
        if (threadIdx.x == T - 1) next_ticket = atomicAdd(gg.tickets + (MODE == kRedo ? 1 : 0), 1u);
    }
    bool within = true;
    if constexpr (MODE == kFirst) {
        if (!whole) {
            // (not NaNs into the share, as in the other passes: the clamp of the second launch would make numbers of them)
            if (threadIdx.x == 0) __hip_atomic_store(gg.tickets + kLost, 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
            return;
        }
        const float lim = a.clip.clip;
        within = !(lim > 0.0f) || (figures[3] <= static_cast<double>(lim) && figures[2] == figures[2]);
    }
    if (threadIdx.x == 0) {
        const FinishedChannel r = finished_channel<true>(figures[0], figures[1], static_cast<int>(gg.g.per_channel), k, terms,
                                                         k.scale);
        shared_coef = r.k;
        if (member == 0 && within) {
            a.bias_updates[c] = bias_updates_in + r.bias_add;
            a.scale_updates[c] = scale_updates_in + r.scale_add;
            if (a.mean_delta) a.mean_delta[c] = r.mean_delta;
            if (a.var_delta) a.var_delta[c] = r.var_delta;
            if constexpr (MODE == kFirst) a.channel_before[c] = make_float2(bias_updates_in, scale_updates_in);
        }
        if constexpr (MODE == kFirst) {
            if (member == 0) {
                a.channel_norm[c] = make_double2(figures[2], figures[3]);
                if (gg.members == 1) a.channel_sums[c] = make_double2(figures[0], figures[1]);
                a.channel_done[c] = within ? 1 : 0;
            }
        }
    }
    if (!within) return;
    __syncthreads();
    const DxCoef kd = shared_coef;
    asm volatile("" : "+v"(lane));      // addresses formed again, not kept from the loads
    const auto leave = [&](int r) {
        const Pack<V> xv = r < X ? x[r] : lds[(r - X) * T];
        Pack<V> out;
#pragma unroll
        for (int q = 0; q < V; ++q) out.v[q] = dx_value(d[r].v[q], xv.v[q], kd);
        return out;
    };
#pragma unroll
    for (int r = 0; r < R; ++r) {
        if (r % kStep == 0 && !any(r + kStep - 1)) break;
        const Pack<V> out = leave(r);
        if (item(r) < end) {
            float* const to = at_byte(a.b.delta, place(item(r)));
            if constexpr (RAGGED) st_own(to, out, held(item(r)));
            else st<V, true>(to, 0, out);
        }
    }
}

// What a finished channel left beside its dx, rescaled; by the whole workgroup.
__device__ __forceinline__ void grouped_rescale_updates(const ResidentBwdArgs& a, const GroupGeom& gg, uint32_t c, float factor)
{
    double figures[kFirstWords];
    if (gg.members > 1) {
        __syncthreads();       // the figures of the channel before have been read
        collect_figures<kFirstWords>(gg.words + static_cast<size_t>(c) * gg.members * kFirstWords, gg.members, gg.looks,
                                     figures);
    } else {
        const double2 sums = a.channel_sums[c];
        figures[0] = sums.x;
        figures[1] = sums.y;
    }
    if (threadIdx.x == 0)
        rescale_finished_channel(figures[0], figures[1], static_cast<double>(factor), a.channel_before[c], c, a.b.var,
                                 a.b.scale, a.scale_updates, a.bias_updates, a.mean_delta, a.var_delta);
}

// A member's share of a finished channel where others have to be gone over again.
template<bool RAGGED>
__device__ __forceinline__ void grouped_rescale_member(const ResidentBwdArgs& a, const GroupGeom& gg, uint32_t c,
                                                       uint32_t member, float factor)
{
    const uint32_t begin = member * gg.span;
    const uint32_t end = min(gg.items, begin + gg.span);
#pragma unroll 1
    for (uint32_t i = begin + threadIdx.x; i < end; i += kGroupThreads) {
        const Step p = step_of<4, RAGGED>(gg.g, c, i);
        Pack<4> t = ld_step<4, true, RAGGED>(a.b.delta, p);
#pragma unroll
        for (int q = 0; q < 4; ++q) t.v[q] = factor * t.v[q];
        st_step<4, RAGGED, true>(a.b.delta, p, t);
    }
    if (member == 0) grouped_rescale_updates(a, gg, c, factor);
}

// Where every channel is finished, the tensor is rescaled as it lies, the next batch of a lane on its way while one is
// written.  Share by share with a number taken for each, 16 x 128 x 152^2 rescaled 202 -> 191 us, 16 x 64 x 152^2 108 -> 99,
// 4 x 16 x 416^2 60 -> 53.  (Five launches that read both tensors twice: 164, 91 and 51, but 164, 91 and 51 also where nothing
// is rescaled, 127, 67 and 38 here; the bytes are the same, and theirs come in one stream.)
template<bool RAGGED>
__device__ __forceinline__ void grouped_rescale_all(const ResidentBwdArgs& a, const GroupGeom& gg, float factor)
{
    constexpr int kLoads = 6;
    const uint32_t values = static_cast<uint32_t>(gg.g.channels) * gg.g.per_channel;
    const uint32_t items = values / 4;      // the values of an odd tensor's end one by one, below
    const uint32_t step = gridDim.x * (kLoads * kGroupThreads);
    const auto at = [&](uint32_t first, int u) { return first + static_cast<uint32_t>(u * kGroupThreads) + threadIdx.x; };
    Pack<4> t[2][kLoads];
    const auto fetch = [&](Pack<4> (&p)[kLoads], uint32_t first) {
#pragma unroll
        for (int u = 0; u < kLoads; ++u) {
            const uint32_t i = at(first, u);
            p[u] = load<RAGGED>(a.b.delta + static_cast<size_t>(i < items ? i : 0) * 4);
        }
    };
    const auto leave = [&](Pack<4> (&p)[kLoads], uint32_t first) {
#pragma unroll
        for (int u = 0; u < kLoads; ++u) {
            const uint32_t i = at(first, u);
#pragma unroll
            for (int q = 0; q < 4; ++q) p[u].v[q] = factor * p[u].v[q];
            float* const to = a.b.delta + static_cast<size_t>(i) * 4;
            if (i < items) {
                if constexpr (RAGGED) st_word(to, p[u]);
                else st<4, true>(to, 0, p[u]);
            }
        }
    };
    uint32_t first = blockIdx.x * (kLoads * kGroupThreads);
    if (first < items) fetch(t[0], first);
    while (first < items) {
        const uint32_t second = first + step;
        if (second < items) fetch(t[1], second);
        leave(t[0], first);
        if (second >= items) break;
        first = second + step;
        if (first < items) fetch(t[0], first);
        leave(t[1], second);
    }
    if (RAGGED && blockIdx.x == 0 && threadIdx.x < values - 4 * items) {
        float* const last = a.b.delta + 4 * static_cast<size_t>(items) + threadIdx.x;
        *last = factor * *last;
    }
    for (uint32_t c = blockIdx.x; c < static_cast<uint32_t>(gg.g.channels); c += gridDim.x)
        grouped_rescale_updates(a, gg, c, factor);
}

// What the second launch leaves where a wait of the first gave up: NaNs everywhere.  By one workgroup.
template<bool RAGGED>
__device__ __forceinline__ void leave_lost(const ResidentBwdArgs& a, const GroupGeom& gg, uint32_t all)
{
    const float nan = __int_as_float(0x7FC00000);
    if (threadIdx.x == 0 && a.clip.norm_out) *a.clip.norm_out = nan;
    const Pack<4> nans{ { nan, nan, nan, nan } };
    for (uint32_t number = 0; number < all; ++number) {
        uint32_t c, member;
        gg.by_members.divmod(number, c, member);
        const uint32_t begin = member * gg.span, end = min(gg.items, begin + gg.span);
        for (uint32_t i = begin + threadIdx.x; i < end; i += kGroupThreads)
            st_step<4, RAGGED>(a.b.delta, step_of<4, RAGGED>(gg.g, c, i), nans);
        if (member == 0 && threadIdx.x == 0) {
            a.bias_updates[c] = a.scale_updates[c] = nan;
            if (a.mean_delta) a.mean_delta[c] = nan;
            if (a.var_delta) a.var_delta[c] = nan;
        }
    }
}

// The numbers of a workgroup (walk_shares): taken one by one, or, where a channel has one member and nobody waits, a grid
// apart.
struct ShareNumbers {
    uint32_t* counter;      // null: a grid apart
    uint32_t& taken;
    uint32_t number;
    __device__ __forceinline__ void sync() const { __syncthreads(); }
    __device__ __forceinline__ void ask() const { if (counter && threadIdx.x == 0) taken = atomicAdd(counter, 1u); }
    __device__ __forceinline__ uint32_t next() { return number = counter ? taken : number + gridDim.x; }
};

// The first launch of a clipped backward and the one behind it share the work as those of resident_bwd.hip do.
template<int ACT, bool RAGGED, int R, int L, int MODE>
__global__ __launch_bounds__(kGroupThreads, 4) void bn_grouped_bwd_kernel(ResidentBwdArgs a, GroupGeom gg)
{
    // two workgroups to a compute unit, which group_places() counts on: 128 registers a lane, and this LDS
    static_assert(static_cast<size_t>(L) * 16 * kGroupThreads == kGroupLdsBytes);
    __shared__ uint32_t taken;
    float factor = 1.0f, limit = 0.0f;
    const uint32_t all = static_cast<uint32_t>(gg.g.channels) * gg.members;
    if constexpr (MODE == kRedo) {
        const ClipPlan plan = clip_plan_from<kGroupThreads>(a.channel_norm, gg.g.channels, a.clip.threshold, a.clip.clip);
        if (blockIdx.x == 0 && threadIdx.x == 0) {
            *a.clip.plan = plan;
            if (a.clip.norm_out) *a.clip.norm_out = plan.norm;
        }
        // (one workgroup sees to what never happens: the others leave in the usual case with nothing more to look at)
        if ((plan.work || blockIdx.x == 0) && gg.members > 1 && gg.tickets[kLost]) {
            if (blockIdx.x == 0) leave_lost<RAGGED>(a, gg, all);
            return;
        }
        if (!plan.work) return;
        factor = plan.factor;
        limit = plan.clip;
        if (!(plan.work & kBeyond)) return grouped_rescale_all<RAGGED>(a, gg, factor);
    }
    uint32_t* const tickets = gg.tickets + (MODE == kRedo ? 1 : 0);
    uint32_t number = blockIdx.x;
    if (gg.members > 1) {
        // the workgroups that come second to a compute unit start when the first ones have their slices: one half of the
        // machine then loads while the other waits for its sums
        if (all >= 2 * gridDim.x && blockIdx.x >= gridDim.x / 2) head_start();
        number = take_ticket(tickets, taken);
    }
    const auto share = [&](uint32_t mine) {
        uint32_t c, member;
        gg.by_members.divmod(__builtin_amdgcn_readfirstlane(mine), c, member);      // the same in every lane
        if (MODE != kRedo || !a.channel_done[c]) {
            grouped_bwd_member<ACT, RAGGED, R, L, MODE>(a, gg, c, member, taken, factor, limit);
            return true;
        }
        if (factor != 1.0f) grouped_rescale_member<RAGGED>(a, gg, c, member, factor);
        return false;
    };
    ShareNumbers numbers{ gg.members > 1 ? tickets : nullptr, taken, number };
    walk_shares(numbers, number, all, share);
}

std::atomic<uint32_t> looks_of_a_wait{ kLooks };

__global__ __launch_bounds__(kBlock) void empty_words_kernel(uint64_t* words, uint32_t count, uint32_t* tickets)
{
    const uint32_t i = blockIdx.x * kBlock + threadIdx.x;
    if (i < count) words[i] = kNotThere;
    if (i < kTickets) tickets[i] = 0;
}

}  // namespace

uint32_t group_places(hipStream_t s)
{
    // two to a compute unit (their LDS and registers); the device's units are asked for once, a stream's mask each time
    static std::atomic<uint32_t> known[16];
    int device = 0, count = 0;
    if (hipGetDevice(&device) != hipSuccess || device < 0 || device >= 16) return 0;
    uint32_t units = known[device].load(std::memory_order_relaxed);
    if (units == 0) {
        if (hipDeviceGetAttribute(&count, hipDeviceAttributeMultiprocessorCount, device) != hipSuccess || count <= 0) return 0;
        units = static_cast<uint32_t>(count);
        known[device].store(units, std::memory_order_relaxed);
    }
    constexpr int kWords = 32;
    uint32_t mask[kWords] = {};
    if (hipExtStreamGetCUMask(s, kWords, mask) != hipSuccess) (void) hipGetLastError();
    return 2 * units_of_mask(mask, kWords, units);
}

uint32_t group_looks() { return looks_of_a_wait.load(std::memory_order_relaxed); }

int start_exchange(const char* who, GroupGeom& g, void* at, int words, bool redo, hipStream_t s)
{
    const size_t count = static_cast<size_t>(g.g.channels) * g.members;
    const size_t first = group_align(count * words * 8), second = redo ? group_align(count * kSumWords * 8) : 0;
    char* base = static_cast<char*>(at);
    g.words = reinterpret_cast<uint64_t*>(base);
    g.redo_words = redo ? reinterpret_cast<uint64_t*>(base + first) : nullptr;
    g.tickets = reinterpret_cast<uint32_t*>(base + first + second);
    const uint32_t all = static_cast<uint32_t>((first + second) / 8);
    hipLaunchKernelGGL(empty_words_kernel, dim3(grid_for(all, kBlock)), dim3(kBlock), 0, s, g.words, all, g.tickets);
    return check_launch(who);
}

int launch_grouped_backward(const char* who, const ResidentBwdArgs& r, const GroupGeom& g, uint32_t places, bool clipped,
                            bool vec, int activation, hipStream_t s)
{
    const uint32_t all = static_cast<uint32_t>(g.g.channels) * g.members;
    int rc = PXH_OK;
    const auto launch = [&]<int ACT, int MODE>() {
        const dim3 grid(all < places ? all : places), block(kGroupThreads);
        const auto kernel = vec ? bn_grouped_bwd_kernel<ACT, false, 12, 8, MODE> : bn_grouped_bwd_kernel<ACT, true, 12, 8, MODE>;
        if (!rc) rc = allow_large_lds(reinterpret_cast<const void*>(kernel));
        if (!rc) hipLaunchKernelGGL(kernel, grid, block, kGroupLdsBytes, s, r, g);
    };
    const bool known = dispatch_activation(activation, [&]<int ACT>() {
        if (!clipped) {
            launch.template operator()<ACT, kPlain>();
        } else {
            launch.template operator()<ACT, kFirst>();
            launch.template operator()<ACT, kRedo>();
        }
    });
    if (!known) return fail_invalid("%s: unknown activation %d", who, activation);
    if (rc) return rc;
    return check_launch(who);
}

}  // namespace pxh

extern "C" unsigned pxh_debug_group_looks(unsigned looks) { return pxh::looks_of_a_wait.exchange(looks); }

extern "C" unsigned pxh_debug_group_places(void* stream) { return pxh::group_places(pxh::as_stream(stream)); }
