// Batch-norm training backward in one launch, plain or with the gradient rescale + clip in front.
#include "resident.h"

namespace pxh {
namespace {

// The workgroup keeps d' = delta * act'(pre) (registers + LDS); x is read again for the dx phase
// (it is still in the cache: one channel's slice is a few hundred KB).
//
// With Layer::backward's rescale + clip in front (kFirst, then a kRedo launch of the same shape): the
// first launch also adds up the channel's squares and finds its largest magnitude.  The norm that
// decides the rescale is the whole tensor's and is not known inside the launch; but the factor is at
// most 1, so a channel whose own largest magnitude is within the clamp cannot be clamped whatever the
// factor turns out to be, and all it leaves is linear in its delta: it is finished as if nothing had
// to change.  A channel above the clamp is left untouched.  The kRedo launch forms the plan from the
// per-channel figures and leaves at once in the usual case (nothing to change); else a finished
// channel is scaled by the factor, and an untouched one runs the whole pass on the rescaled and
// clamped delta.
// Channel c of a backward whose first launch finished it with the sums of its unscaled delta, scaled
// by the factor the plan arrived at.
template<int V, int R, int L, int T, bool RAGGED>
__device__ __forceinline__ void resident_rescale_channel(const ResidentBwdArgs& a, uint32_t c, float factor)
{
    // The steps' loads in flight together where a lane has the registers beside the full pass: one after the other they are
    // most of a channel's time (16 x 512 x 19^2 rescaled 29.3 -> 22.0 us, 1 x 1024 x 13^2 16.1 -> 14.4, 64 x 1024 x 13^2 91 -> 77; the
    // 128-bit forms of 1024 lanes spill with eight of them, 16 x 256 x 38^2 28.9 -> 38.6).
    constexpr bool kTogether = V == 1 || RAGGED || kSmallSlice<V, R, L, T>;
    constexpr int kLoads = !kTogether ? 1 : (R + L) % 12 == 0 ? 12 : (R + L) % 8 == 0 ? 8 : R + L;
    static_assert((R + L) % kLoads == 0, "steps come in whole groups");
#pragma unroll 1
    for (int first = 0; first < R + L; first += kLoads) {
        Pack<V> t[kLoads];
        const auto step = [&](int u) { return step_of<V, RAGGED>(a.g, c, static_cast<uint32_t>((first + u) * T + threadIdx.x)); };
        if (!kTogether && !step(0).valid) break;
#pragma unroll
        for (int u = 0; u < kLoads; ++u) t[u] = ld_step<V, true, RAGGED>(a.b.delta, step(u));
#pragma unroll
        for (int u = 0; u < kLoads; ++u) {
            const Step p = step(u);
#pragma unroll
            for (int q = 0; q < V; ++q) t[u].v[q] = factor * t[u].v[q];
            // (no barrier between a lane's loads and another's stores: only what is its own)
            if (p.valid) st_step<V, RAGGED, true>(a.b.delta, p, t[u]);
        }
    }
    if (threadIdx.x == 0) {
        const double2 sums = a.channel_sums[c];
        rescale_finished_channel(sums.x, sums.y, static_cast<double>(factor), a.channel_before[c], c, a.b.var, a.b.scale, a.scale_updates,
                                 a.bias_updates, a.mean_delta, a.var_delta);
    }
}

// Channel c by the whole workgroup; `factor` and `limit` are the plan's (kRedo only).
template<int ACT, int V, int R, int L, int MODE, int T, bool RAGGED>
__device__ __forceinline__ void resident_bwd_channel(const ResidentBwdArgs& a, const uint32_t c,
                                                     [[maybe_unused]] const float factor,
                                                     [[maybe_unused]] const float limit)
{
    extern __shared__ __align__(16) float resident_lds[];
    constexpr bool kSmall = RAGGED || kSmallSlice<V, R, L, T>;
    __shared__ double slots[MODE == kFirst ? 3 : 2][T / kWave];
    __shared__ DxCoef shared_coef;
    const FoldCoef k = make_coef(a.b.mean[c], a.b.var[c], a.b.scale[c], a.b.bias[c]);
    // The whole workgroup waits for the one thread that finishes the channel, so that thread's loads all
    // come before its first store (a load issued behind a store waits for that store too: one counter,
    // in order); the forms that run the short launches ask for them before the first pass, the large
    // form, which has no register to spare, when the sums are there.
    constexpr bool kEarly = L == 0;
    [[maybe_unused]] float early[3] = {};
    if constexpr (kEarly) {
        early[0] = a.bias_updates[c];
        early[1] = a.scale_updates[c];
        early[2] = a.b.var[c];
    }
    // the small forms, whose time is one chain, also form what the finish takes from the variance while the slice is on
    // its way (the first wave: it is the one that finishes the channel)
    [[maybe_unused]] VarianceTerms terms{};
    const auto early_terms = [&] { if (threadIdx.x < kWave) terms = variance_terms(early[2]); };
    const auto finish = [&](double sa, double sb) {
        const float bias_updates_in = kEarly ? early[0] : a.bias_updates[c];
        const float scale_updates_in = kEarly ? early[1] : a.scale_updates[c];
        const float var_in = kEarly ? early[2] : a.b.var[c];
        const FinishedChannel r = finished_channel<true>(sa, sb, static_cast<int>(a.g.per_channel), k,
                                                         kSmall ? terms : variance_terms(var_in), k.scale);
        a.bias_updates[c] = bias_updates_in + r.bias_add;
        a.scale_updates[c] = scale_updates_in + r.scale_add;
        if (a.mean_delta) a.mean_delta[c] = r.mean_delta;
        if (a.var_delta) a.var_delta[c] = r.var_delta;
        if constexpr (MODE == kFirst) a.channel_before[c] = make_float2(bias_updates_in, scale_updates_in);
        return r.k;
    };
    const bool recompute = a.b.pre == nullptr;
    Pack<V> d[R];
    std::conditional_t<kSmall || V == 1, double, float> fa = 0, fb = 0;
    [[maybe_unused]] std::conditional_t<kSmall || V == 1, double, float> fq = 0;
    [[maybe_unused]] float peak = 0.0f;
    // Two shapes of the first pass.  Grouped: no branch around the loads (see the forward kernel), lanes
    // past the end read the first vector; kGroup steps at a time, their loads go out together, then each
    // is used as it arrives.  The large form (part of the slice in LDS) is bound by its loads and takes
    // them so in groups of four; the form with one value a step (planes below four values) in groups of eight (behind a
    // branch a lane waits for each step's loads before it asks for the next).  The 128-bit form without an LDS part is held to 64
    // registers, where a group of two already spills (18.3 against 16.4 us at 16 x 256 x 38^2): it skips a step
    // past the end of the slice outright, as every form does in the second pass, which finds x in the cache.
    constexpr int kGroup = L > 0 ? 4 : 8;
    constexpr bool kGrouped = !kSmall && (L > 0 || V == 1);
    [[maybe_unused]] Pack<V> kept[kSmall ? R : 1];       // x, which the small forms hold on to
    static_assert(!kGrouped || (R % kGroup == 0 && L % kGroup == 0), "steps come in whole groups");
    // `lane` is the thread index; the second pass takes it through an empty asm statement, so that
    // its addresses are formed again there instead of being held in registers (48 of them) from the first
    [[maybe_unused]] uint32_t lane = threadIdx.x;
    [[maybe_unused]] const auto element = [&](int r) { return (static_cast<uint32_t>(r * T) + lane) * V; };
    const auto step = [&](int r) { return step_of<V, RAGGED>(a.g, c, static_cast<uint32_t>(r * T) + lane); };
    [[maybe_unused]] const auto place = [&](int r) {
        const uint32_t e = element(r);
        return a.g.at(c, e < a.g.per_channel ? e : 0u);
    };
    // a vector of the delta on its way to d': the norm's share of it first (kFirst), or the plan's
    // rescale + clamp (kRedo), then the activation's gradient
    const auto prepare = [&](Pack<V>& t, const Pack<V>& pre, bool valid) {
#pragma unroll
        for (int q = 0; q < V; ++q) {
            if constexpr (MODE == kFirst) {
                if constexpr (!kSmall) fq += valid ? t.v[q] * t.v[q] : 0.0f;
                peak = fmaxf(peak, valid ? fabsf(t.v[q]) : 0.0f);
            }
            if constexpr (MODE == kRedo) t.v[q] = rescaled_clipped(t.v[q], factor, limit);
        }
        times_grad<ACT>(t.v, pre.v);
    };
    if constexpr (kSmall) {
        // every load of the slice at once, no branch around them; the pre-activations four steps at a time
#pragma unroll
        for (int r = 0; r < R; ++r) {
            const Step p = step(r);
            d[r] = ld_step<V, true, RAGGED>(a.b.delta, p);
            kept[r] = ld_step<V, false, RAGGED>(a.b.x, p);
        }
        early_terms();
        constexpr int kFour = R < 4 ? R : R % 4 == 0 ? 4 : 3;
        static_assert(R % kFour == 0, "steps come in whole groups");
#pragma unroll
        for (int first = 0; first < R; first += kFour) {
            Pack<V> pv[kFour];
            if constexpr (ACT != PXH_LINEAR) {
                if (!recompute) {
#pragma unroll
                    for (int i = 0; i < kFour; ++i) pv[i] = ld_step<V, true, RAGGED>(a.b.pre, step(first + i));
                } else {
#pragma unroll
                    for (int i = 0; i < kFour; ++i) {
#pragma unroll
                        for (int q = 0; q < V; ++q) pv[i].v[q] = affine(normalize(kept[first + i].v[q], k), k);
                    }
                }
            }
#pragma unroll
            for (int i = 0; i < kFour; ++i) {
                const int r = first + i;
                if constexpr (RAGGED) {
                    // every value into a double of its own, and those that the vector in front holds too stay out of the sums
                    const Step p = step(r);
                    const int own = p.valid ? p.held : V;
                    if constexpr (MODE == kFirst) {
#pragma unroll
                        for (int q = 0; q < V; ++q) {
                            const float t = q >= own ? d[r].v[q] : 0.0f;
                            fq += static_cast<double>(t * t);
                        }
                    }
                    prepare(d[r], pv[i], p.valid);
#pragma unroll
                    for (int q = 0; q < V; ++q) {
                        const float t = d[r].v[q];
                        fa += static_cast<double>(q >= own ? t : 0.0f);
                        fb += static_cast<double>(q >= own ? t * (kept[r].v[q] - k.mean) : 0.0f);
                    }
                    continue;
                }
                // (a step that the slice does not reach has nothing to compute, in any lane: mish, 2 x 583 x 25 x 28 9.7 -> 7.9 us)
                if (r > 0 && static_cast<uint32_t>(r * T) >= a.g.per_channel / V) continue;
                const bool valid = element(r) < a.g.per_channel;
                float va = 0.0f, vb = 0.0f, vq = 0.0f;
#pragma unroll
                for (int q = 0; q < V; ++q) {
                    d[r].v[q] = valid ? d[r].v[q] : 0.0f;
                    vq += d[r].v[q] * d[r].v[q];
                }
                prepare(d[r], pv[i], valid);
#pragma unroll
                for (int q = 0; q < V; ++q) {
                    const float t = valid ? d[r].v[q] : 0.0f;
                    d[r].v[q] = t;
                    va += t;
                    vb += valid ? t * (kept[r].v[q] - k.mean) : 0.0f;
                }
                fa += static_cast<double>(va);
                fb += static_cast<double>(vb);
                if constexpr (MODE == kFirst) fq += static_cast<double>(vq);
            }
        }
    } else if constexpr (kGrouped) {
        // delta * f'(pre) in dv, and the step's share of the sums
        const auto take = [&](int r, Pack<V>& dv, const Pack<V>& xv, const Pack<V>& pv) {
            const bool valid = element(r) < a.g.per_channel;
            prepare(dv, pv, valid);
#pragma unroll
            for (int q = 0; q < V; ++q) {
                fa += valid ? dv.v[q] : 0.0f;
                fb += valid ? dv.v[q] * (xv.v[q] - k.mean) : 0.0f;
            }
        };
#pragma unroll
        for (int top = R + L - 1; top >= 0; top -= kGroup) {
            Pack<V> dv[kGroup], xv[kGroup], pv[kGroup];
            size_t where[kGroup];
#pragma unroll
            for (int i = 0; i < kGroup; ++i) {
                where[i] = place(top - i);
                dv[i] = ld<V, true>(a.b.delta, where[i]);
                xv[i] = ld<V, false>(a.b.x, where[i]);
            }
            // the pre-activation: the saved one, or formed again from x (one decision per group)
            if constexpr (ACT != PXH_LINEAR) {
                if (!recompute) {
#pragma unroll
                    for (int i = 0; i < kGroup; ++i) pv[i] = ld<V, true>(a.b.pre, where[i]);
                } else {
#pragma unroll
                    for (int i = 0; i < kGroup; ++i) {
#pragma unroll
                        for (int q = 0; q < V; ++q) pv[i].v[q] = affine(normalize(xv[i].v[q], k), k);
                    }
                }
            }
#pragma unroll
            for (int i = 0; i < kGroup; ++i) {
                const int r = top - i;
                take(r, dv[i], xv[i], pv[i]);
                if (r < R) d[r < R ? r : 0] = dv[i];
                else *resident_lds_slot<V, R>(resident_lds, r) = dv[i];
            }
            // The group ends here for the compiler too: the sums are taken as they stand (otherwise it
            // puts the additions off to the end of the pass and keeps every group's values until then),
            // and the next group's loads stay behind this one's arithmetic -- either would need more
            // registers than a lane has.
            if constexpr (MODE == kFirst) asm volatile("" : "+v"(fa), "+v"(fb), "+v"(fq), "+v"(peak));
            else asm volatile("" : "+v"(fa), "+v"(fb));
            __builtin_amdgcn_sched_barrier(0);
        }
    } else {
#pragma unroll
        for (int r = R + L - 1; r >= 0; --r) {
            const uint32_t e = (r * T + lane) * V;
            if (e < a.g.per_channel) {
                const size_t where = a.g.at(c, e);
                Pack<V> dv = ld<V, true>(a.b.delta, where);
                const Pack<V> xv = ld<V, false>(a.b.x, where);
                Pack<V> pv;
                if constexpr (ACT != PXH_LINEAR) {
                    if (!recompute) {
                        pv = ld<V, true>(a.b.pre, where);
                    } else {
#pragma unroll
                        for (int q = 0; q < V; ++q) pv.v[q] = affine(normalize(xv.v[q], k), k);
                    }
                }
                prepare(dv, pv, true);
#pragma unroll
                for (int q = 0; q < V; ++q) {
                    fa += dv.v[q];
                    fb += dv.v[q] * (xv.v[q] - k.mean);
                }
                if (r < R) d[r < R ? r : 0] = dv;
                else *resident_lds_slot<V, R>(resident_lds, r) = dv;
            }
        }
    }
    double sa = static_cast<double>(fa), sb = static_cast<double>(fb);
    if constexpr (MODE == kFirst) {
        __shared__ float tops[T / kWave];
        __shared__ int finished;
        double sq = static_cast<double>(fq);
        resident_sum3_max<T>(sa, sb, sq, peak, slots, tops);
        if (threadIdx.x == 0) {
            const float lim = a.clip.clip;
            const bool within = !(lim > 0.0f) || (peak <= lim && sq == sq);
            finished = within ? 1 : 0;
            if (within) shared_coef = finish(sa, sb);
            a.channel_norm[c] = make_double2(sq, static_cast<double>(peak));
            a.channel_sums[c] = make_double2(sa, sb);
            a.channel_done[c] = within ? 1 : 0;
        }
        __syncthreads();
        if (!finished) return;
    } else {
        resident_sum2<T>(sa, sb, slots);
        if (threadIdx.x == 0) shared_coef = finish(sa, sb);
        __syncthreads();
    }
    const DxCoef kd = shared_coef;
    if constexpr (L > 0) {
        asm volatile("" : "+v"(lane));
#pragma unroll
        for (int first = 0; first < R + L; first += kGroup) {
            Pack<V> xv[kGroup];
#pragma unroll
            for (int i = 0; i < kGroup; ++i) xv[i] = ld<V, false>(a.b.x, place(first + i));
#pragma unroll
            for (int i = 0; i < kGroup; ++i) {
                const int r = first + i;
                const Pack<V> dv = r < R ? d[r < R ? r : 0] : *resident_lds_slot<V, R>(resident_lds, r);
                Pack<V> out;
#pragma unroll
                for (int q = 0; q < V; ++q) out.v[q] = dx_value(dv.v[q], xv[i].v[q], kd);
                if (element(r) < a.g.per_channel) st<V, true>(a.b.delta, place(r), out);
            }
            __builtin_amdgcn_sched_barrier(0);
        }
    } else {
        asm volatile("" : "+v"(lane));      // addresses formed again, not kept from the first pass
#pragma unroll
        for (int r = 0; r < R + L; ++r) {
            const Step p = step(r);
            if (p.valid) {
                Pack<V> xv;
                if constexpr (kSmall) xv = kept[r];
                else xv = ld<V, false>(a.b.x, p.at);
                const Pack<V> dv = r < R ? d[r < R ? r : 0] : *resident_lds_slot<V, R>(resident_lds, r);
                Pack<V> out;
#pragma unroll
                for (int q = 0; q < V; ++q) out.v[q] = dx_value(dv.v[q], xv.v[q], kd);
                // (a value that two lanes hold is written by both, the same: every delta was read before the sums)
                st_step<V, RAGGED>(a.b.delta, p, out);
            }
        }
    }
}

// Waves per SIMD that the registers are held to.
template<int V, int R, int L, int MODE, int T, bool RAGGED>
constexpr int kBwdWaves = RAGGED && T == kResidentThreads ? 4 : RAGGED || kSmallSlice<V, R, L, T> ? (MODE == kRedo || V * R >= 32 ? 2 : V * R >= 12 ? 4 : V * R == 8 ? 6 : 8)
                          : L == 0 && MODE != kRedo && !(V == 1 && R > 16) ? 8 : 4;

// One workgroup per channel.  (The forms of 1024 lanes without an LDS part are held to 64 registers, two workgroups
// per compute unit: they run the 19 x 19 and 38 x 38 layers, whose launches are too short to fill the
// machine with one.)  The workgroups of the kRedo launch form the plan from the per-channel figures of
// the first launch and leave at once when nothing has to change; the forms without an LDS part run it
// as a capped grid that walks the channels otherwise.
template<int ACT, int V, int R, int L, int MODE = kPlain, int T = kResidentThreads, bool RAGGED = false>
__global__ __launch_bounds__(T, (kBwdWaves<V, R, L, MODE, T, RAGGED>)) void bn_resident_bwd_kernel(ResidentBwdArgs a)
{
    static_assert(L == 0 || T == kResidentThreads, "the LDS part is laid out for the full workgroup");
    if constexpr (MODE == kRedo) {
        const ClipPlan plan = clip_plan_from<T>(a.channel_norm, a.g.channels, a.clip.threshold,
                                                               a.clip.clip);
        if (blockIdx.x == 0 && threadIdx.x == 0) {
            *a.clip.plan = plan;
            if (a.clip.norm_out) *a.clip.norm_out = plan.norm;
        }
        if (!plan.work) return;
        if constexpr (L > 0) {
            // (one workgroup per channel: walking several costs the large form 450 bytes of spills per lane)
            const uint32_t c = blockIdx.x;
            if (!a.channel_done[c]) resident_bwd_channel<ACT, V, R, L, kRedo, T, RAGGED>(a, c, plan.factor, plan.clip);
            else if (plan.factor != 1.0f) resident_rescale_channel<V, R, L, T, RAGGED>(a, c, plan.factor);
        } else {
            for (uint32_t c = blockIdx.x; c < static_cast<uint32_t>(a.g.channels); c += gridDim.x) {
                if (!a.channel_done[c]) resident_bwd_channel<ACT, V, R, L, kRedo, T, RAGGED>(a, c, plan.factor, plan.clip);
                else if (plan.factor != 1.0f) resident_rescale_channel<V, R, L, T, RAGGED>(a, c, plan.factor);
                __syncthreads();       // the next channel reuses the workgroup's LDS
            }
        }
    } else {
        resident_bwd_channel<ACT, V, R, L, MODE, T, RAGGED>(a, blockIdx.x, 1.0f, 0.0f);
    }
}

}  // namespace

int launch_resident_backward(const char* who, const ResidentBwdArgs& r, bool clipped, const ResidentForm& form, int activation,
                             hipStream_t s)
{
    const dim3 block(kResidentThreads);
    int large_lds_rc = PXH_OK;
    const auto launch = [&]<int ACT, int MODE>() {
        // the launch that follows the plan: one workgroup per compute unit at most, each walks channels
        const bool large = !form.odd && !form.small && form.per_thread > kResidentVectors;
        const bool walks = MODE == kRedo && !large && r.g.channels > kRedoWorkgroups;
        const dim3 grid(walks ? kRedoWorkgroups : r.g.channels);
        if (form.odd) {
            dispatch_odd_form<kOddOneStep<ACT, true>>(form.odd, r.g, [&]<int V, int R, int T>() {
                hipLaunchKernelGGL((bn_resident_bwd_kernel<ACT, V, R, 0, MODE, T, V == 4>), grid, dim3(T), 0, s, r);
            });
        } else if (form.small) {
            dispatch_small_form(form.small, [&]<int R, int T>() {
                hipLaunchKernelGGL((bn_resident_bwd_kernel<ACT, 4, R, 0, MODE, T>), grid, dim3(T), 0, s, r);
            });
        } else if (large) {
            auto kernel = bn_resident_bwd_kernel<ACT, 4, kResidentLargeRegs, kResidentLargeLds, MODE>;
            large_lds_rc = allow_large_lds(reinterpret_cast<const void*>(kernel));
            if (large_lds_rc == PXH_OK) hipLaunchKernelGGL(kernel, grid, block, kResidentLargeLdsBytes, s, r);
        } else {
            hipLaunchKernelGGL((bn_resident_bwd_kernel<ACT, 4, kResidentVectors, 0, MODE>), grid, block, 0, s, r);
        }
    };
    const bool known = dispatch_activation(activation, [&]<int ACT>() {
        if (!clipped) {
            launch.template operator()<ACT, kPlain>();
        } else {
            launch.template operator()<ACT, kFirst>();
            if (large_lds_rc == PXH_OK) launch.template operator()<ACT, kRedo>();
        }
    });
    if (!known) return fail_invalid("%s: unknown activation %d", who, activation);
    if (large_lds_rc) return large_lds_rc;
    return check_launch(who);
}

}  // namespace pxh
