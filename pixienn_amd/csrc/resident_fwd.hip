// Batch-norm training forward in one launch: a workgroup holds a channel's whole slice.
#include "resident.h"

#include <mutex>
#include <vector>

namespace pxh {
namespace {

// Steps of the shortcut's source that a lane of the large form asks for before the reduction.  (The form with
// eight 128-bit vectors in registers and two workgroups per compute unit has no register to spare for any:
// 16 x 512 x 38^2 takes 32.9 us with four steps ahead against 31.0 us with none.)
constexpr int kResidualAhead = 4;

// Waves per SIMD that the registers are held to: a vector a step, two with a shortcut.
template<int V, int R, int L, int T, bool RES, bool RAGGED>
constexpr int kFwdWaves = RAGGED || kSmallSlice<V, R, L, T> ? (RAGGED && T == kResidentThreads ? (RES ? 4 : 8) : V * R >= 32 ? 2 : RES && V * R >= 12 ? 4 : 8)
                          : L == 0 && V * R <= (V == 1 ? (RES ? 8 : 16) : 32) ? 8 : 4;

// V = 4 needs spatial % 4 == 0 and 16-byte aligned tensors, RAGGED (odd planes) neither.  R + L vectors per thread at most.
template<int ACT, int V, int R, int L, int T = kResidentThreads, bool RES = false, bool RAGGED = false>
__global__ __launch_bounds__(T, (kFwdWaves<V, R, L, T, RES, RAGGED>)) void bn_resident_fwd_kernel(ResidentFwdArgs a)
{
    static_assert(L == 0 || T == kResidentThreads, "the LDS part is laid out for the full workgroup");
    extern __shared__ __align__(16) float resident_lds[];
    // The 128-bit form with workgroups of half the size adds a channel up exactly as the full workgroups do,
    // so that a layer gives the same statistics to the bit with and without a shortcut riding on it: thread t
    // keeps the sums of the full form's threads t (even steps) and t + T (odd steps) apart.
    constexpr bool kSmall = RAGGED || kSmallSlice<V, R, L, T>;
    constexpr bool kTwin = V == 4 && T < kResidentThreads && !kSmall;
    static_assert(!kTwin || 2 * T == kResidentThreads, "half the size");
    __shared__ double slots[2][(kTwin ? 2 : 1) * T / kWave];
    __shared__ FoldCoef shared_coef;
    const uint32_t c = blockIdx.x;
    const float shift = a.x[static_cast<size_t>(c) * a.g.spatial];
    // issued now, needed after the reduction
    const float rm_in = a.rolling_mean[c], rv_in = a.rolling_var[c], scale_in = a.scale[c], bias_in = a.bias[c];
    Pack<V> v[R];
    float a1 = 0.0f, a2 = 0.0f;
    [[maybe_unused]] float b1 = 0.0f, b2 = 0.0f;
    // Every tensor here is touched once and goes past the caches (non-temporal: with the whole slice
    // of every channel asked for at once, cached reads run at two thirds of the rate; the backward
    // kernel keeps x cached, which it reads twice).
    // No branch around a load: a lane past the end of the slice reads the slice's first vector and
    // adds nothing, so that the loads of a lane are in flight together (behind a branch each one is
    // waited for before the next is issued, and a wave then has one kilobyte on its way at a time).
    uint32_t lane = threadIdx.x;
    const auto element = [&](int r) { return (static_cast<uint32_t>(r * T) + lane) * V; };
    const auto step = [&](int r) { return step_of<V, RAGGED>(a.g, c, static_cast<uint32_t>(r * T) + lane); };
    const auto fetch = [&](int r) { return ld_step<V, true, RAGGED>(a.x, step(r)); };
    const auto ride = [&](int r) {
        if constexpr (RAGGED) return ld_step<V, true, RAGGED>(a.residual, step(r));
        const uint32_t e = element(r);
        return ld<V, true>(a.residual, a.g.at(c, e < a.g.per_channel ? e : 0u));
    };
    const auto add = [&](int r, const Pack<V>& t) {
        const bool valid = element(r) < a.g.per_channel;
        const bool second = kTwin && (r & 1);
#pragma unroll
        for (int k = 0; k < V; ++k) {
            const float d = t.v[k] - shift;
            if (second) {
                b1 += valid ? d : 0.0f;
                b2 += valid ? d * d : 0.0f;
            } else {
                a1 += valid ? d : 0.0f;
                a2 += valid ? d * d : 0.0f;
            }
        }
    };
    // the LDS part first, all of it at once: its registers are free again before the register part
    // is loaded, which lands where it stays
    if constexpr (L > 0) {
        Pack<V> stage[L];
#pragma unroll
        for (int r = R + L - 1; r >= R; --r) stage[r - R] = fetch(r);
#pragma unroll
        for (int r = R + L - 1; r >= R; --r) {
            add(r, stage[r - R]);
            *resident_lds_slot<V, R>(resident_lds, r) = stage[r - R];
        }
        // the sums as they stand, before the registers are handed to the second part
        asm volatile("" : "+v"(a1), "+v"(a2));
    }
#pragma unroll
    for (int r = R - 1; r >= 0; --r) v[r] = fetch(r);
    // The shortcut's source does not wait for the statistics: its first steps are asked for now, behind the
    // slice's own loads, and arrive while the sums are formed -- all of them where a lane holds few values
    // (16 x 1024 x 19^2: 19.9 us against 25.6 us with every step's load behind the reduction).
    // (the half-size workgroups of the 128-bit form have 128 registers: eight of twelve steps, four of sixteen)
    constexpr int kAhead = !RES ? 0 : kSmall || V * (R + L) <= 8 ? R + L : L > 0 ? kResidualAhead
                                : T < kResidentThreads ? (R <= 12 ? 8 : 4) : V == 1 ? 4 : 0;
    [[maybe_unused]] Pack<V> ahead[kAhead > 0 ? kAhead : 1];
    if constexpr (RES) {
#pragma unroll
        for (int i = 0; i < kAhead; ++i) ahead[i] = ride(i);
    }
    double t1, t2;
    if constexpr (RAGGED) {
        t1 = t2 = 0.0;
#pragma unroll
        for (int r = R - 1; r >= 0; --r) {
            const Step p = step(r);
            const int first = p.valid ? p.held : V;
#pragma unroll
            for (int k = 0; k < V; ++k) {
                const float d = k >= first ? v[r].v[k] - shift : 0.0f;
                t1 += static_cast<double>(d);
                t2 += static_cast<double>(d * d);
            }
        }
    } else if constexpr (kSmall || V == 1) {
        t1 = t2 = 0.0;
#pragma unroll
        for (int r = R - 1; r >= 0; --r) {
            const bool valid = element(r) < a.g.per_channel;
            float p1 = 0.0f, p2 = 0.0f;
#pragma unroll
            for (int k = 0; k < V; ++k) {
                const float d = valid ? v[r].v[k] - shift : 0.0f;
                p1 += d;
                p2 += d * d;
            }
            t1 += static_cast<double>(p1);
            t2 += static_cast<double>(p2);
        }
    } else {
#pragma unroll
        for (int r = R - 1; r >= 0; --r) add(r, v[r]);
        t1 = static_cast<double>(a1);
        t2 = static_cast<double>(a2);
    }
    if constexpr (kTwin) resident_sum2_twin<T>(t1, t2, static_cast<double>(b1), static_cast<double>(b2), slots);
    else resident_sum2<T>(t1, t2, slots);
    if (threadIdx.x == 0) {
        const ChannelStats st = channel_stats(t1, t2, shift, static_cast<double>(a.g.per_channel), rm_in, rv_in);
        a.mean[c] = st.mean;
        a.var[c] = st.var;
        a.rolling_mean[c] = st.rolling_mean;
        a.rolling_var[c] = st.rolling_var;
        shared_coef = make_coef(st.mean, st.var, scale_in, bias_in);
    }
    __syncthreads();
    const FoldCoef k = shared_coef;
    if constexpr (RES && (L > 0 || R > 16)) asm volatile("" : "+v"(lane));      // addresses formed again, not kept: they would spill
    const auto apply = [&](int r, [[maybe_unused]] const Pack<V>& from) {
        const uint32_t e = element(r);
        const Step kept = RAGGED ? step(r) : Step{ 0, e < a.g.per_channel, 0 };
        if (kept.valid) {
            // (not the load's place: it is formed again, not kept)
            const Step p = RAGGED ? kept : Step{ a.g.at(c, e), true, 0 };
            const Pack<V> t = r < R ? v[r < R ? r : 0] : *resident_lds_slot<V, R>(resident_lds, r);
            Pack<V> xn, pre, out;
#pragma unroll
            for (int q = 0; q < V; ++q) {
                xn.v[q] = normalize(t.v[q], k);
                pre.v[q] = affine(xn.v[q], k);
                out.v[q] = act_apply<ACT>(pre.v[q]);
                if constexpr (RES) out.v[q] = with_residual(out.v[q], from.v[q], a.res_alpha, a.res_beta);
            }
            if (a.x_saved) st_step<V, RAGGED>(a.x_saved, p, t);
            if (a.x_norm) st_step<V, RAGGED>(a.x_norm, p, xn);
            if (a.pre) st_step<V, RAGGED>(a.pre, p, pre);
            // (the shortcut's source may be y itself, whose loads nothing here waits for: a value two lanes hold is written
            // by the one that owns it)
            st_step<V, RAGGED, RES>(a.y, p, out);
        }
    };
    if constexpr (RES) {
        // the rest of the shortcut's source four steps at a time, no branch around its loads (see above)
        constexpr int kGroup = kSmall ? R : 4;
        static_assert((R + L) % kGroup == 0 && kAhead % kGroup == 0, "steps come in whole groups");
#pragma unroll
        for (int first = 0; first < R + L; first += kGroup) {
            Pack<V> from[kGroup];
#pragma unroll
            for (int i = 0; i < kGroup; ++i) {
                if (first + i < kAhead) {
                    from[i] = ahead[first + i < kAhead ? first + i : 0];
                } else {
                    from[i] = ride(first + i);
                }
            }
#pragma unroll
            for (int i = 0; i < kGroup; ++i) apply(first + i, from[i]);
        }
    } else {
#pragma unroll
        for (int r = 0; r < R + L; ++r) apply(r, Pack<V>{});
    }
}

}  // namespace

int allow_large_lds(const void* kernel)
{
    static std::mutex mutex;
    static std::vector<const void*> allowed;
    std::lock_guard<std::mutex> lock(mutex);
    for (const void* k: allowed)
        if (k == kernel) return PXH_OK;
    const hipError_t e = hipFuncSetAttribute(kernel, hipFuncAttributeMaxDynamicSharedMemorySize,
                                             static_cast<int>(kResidentLargeLdsBytes));
    if (e != hipSuccess) {
        set_error("hipFuncSetAttribute(max dynamic LDS %zu): %s", kResidentLargeLdsBytes, hipGetErrorString(e));
        return static_cast<int>(e);
    }
    allowed.push_back(kernel);
    return PXH_OK;
}

int launch_resident_forward(const char* who, const ResidentFwdArgs& r, const ResidentForm& form, int activation, hipStream_t s)
{
    const dim3 grid(r.g.channels), block(kResidentThreads);
    int large_lds_rc = PXH_OK;
    const auto launch = [&]<int ACT, bool RES>() {
        constexpr int kT = kResidentThreads;
        if (form.odd) {
            dispatch_odd_form<kOddOneStep<ACT, false>>(form.odd, r.g, [&]<int V, int R, int T>() {
                hipLaunchKernelGGL((bn_resident_fwd_kernel<ACT, V, R, 0, T, RES, V == 4>), grid, dim3(T), 0, s, r);
            });
            return;
        }
        if (form.small) {
            dispatch_small_form(form.small, [&]<int R, int T>() {
                hipLaunchKernelGGL((bn_resident_fwd_kernel<ACT, 4, R, 0, T, RES>), grid, dim3(T), 0, s, r);
            });
            return;
        }
        if (form.per_thread > kResidentVectors) {
            auto kernel = bn_resident_fwd_kernel<ACT, 4, kResidentLargeRegs, kResidentLargeLds, kT, RES>;
            large_lds_rc = allow_large_lds(reinterpret_cast<const void*>(kernel));
            if (large_lds_rc == PXH_OK)
                hipLaunchKernelGGL(kernel, grid, block, kResidentLargeLdsBytes, s, r);
        } else if constexpr (RES) {
            // The 128-bit form with the shortcut's source on top of eight vectors of the slice spills at
            // 64 registers: half-size workgroups with twice the vectors per lane and twice the registers
            // keep the same two workgroups per compute unit (16 x 512 x 38^2: 26.2 against 30.9 us).
            const size_t vectors = (static_cast<size_t>(r.g.per_channel) + 3) / 4;
            const dim3 half(kResidentNarrowThreads);
            if (vectors <= 12u * kResidentNarrowThreads)
                hipLaunchKernelGGL((bn_resident_fwd_kernel<ACT, 4, 12, 0, kResidentNarrowThreads, true>), grid,
                                   half, 0, s, r);
            else
                hipLaunchKernelGGL((bn_resident_fwd_kernel<ACT, 4, 16, 0, kResidentNarrowThreads, true>), grid,
                                   half, 0, s, r);
        } else {
            hipLaunchKernelGGL((bn_resident_fwd_kernel<ACT, 4, kResidentVectors, 0, kT, RES>), grid, block, 0, s, r);
        }
    };
    const bool known = dispatch_activation(activation, [&]<int ACT>() {
        if (r.residual) launch.template operator()<ACT, true>();
        else launch.template operator()<ACT, false>();
    });
    if (!known) return fail_invalid("%s: unknown activation %d", who, activation);
    if (large_lds_rc) return large_lds_rc;
    return check_launch(who);
}

}  // namespace pxh
