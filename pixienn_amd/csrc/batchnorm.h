// Device code shared by the batch-norm passes of several launches (epilogue.hip) and those of one
// (resident_fwd.hip, resident_bwd.hip).
//
// Numerics follow the CPU layer (src/BatchNorm.cpp, src/CpuUtil.cpp:248-342 of the reference):
//   x_hat = float( double(x - mean) / (sqrt(double(var)) + 1e-5f) )     eps OUTSIDE the root
//   pre   = float(float(x_hat * scale) + bias)                           two fp32 roundings
// The per-channel reciprocal R = 1 / (sqrt(double(var)) + eps) is formed once per channel in
// fp64 and kept as two floats (hi + lo); x_hat = fma(t, hi, t * lo) then rounds t * R once, which
// equals the rounded double quotient except in about 1e-7 of the elements (1 ulp there).
#pragma once

#include "stream.h"

#include <type_traits>

namespace pxh {

constexpr float kEps = .00001f;

// Folded per-channel constants of the forward pass (32 bytes: two 128-bit loads).
struct __attribute__((aligned(16))) FoldCoef {
    float mean, r_hi, r_lo, scale;
    float bias, pad0, pad1, pad2;
};

__device__ __forceinline__ FoldCoef make_coef(float mean, float var, float scale, float bias)
{
    const double r = 1.0 / (sqrt(static_cast<double>(var)) + static_cast<double>(kEps));
    FoldCoef k;
    k.mean = mean;
    k.r_hi = static_cast<float>(r);
    k.r_lo = static_cast<float>(r - static_cast<double>(k.r_hi));
    k.scale = scale;
    k.bias = bias;
    k.pad0 = k.pad1 = k.pad2 = 0.0f;
    return k;
}

__device__ __forceinline__ float normalize(float x, const FoldCoef& k)
{
    const float t = x - k.mean;
    return fmaf(t, k.r_hi, t * k.r_lo);
}

// pre-activation from x_hat: scale then bias, each rounded
__device__ __forceinline__ float affine(float xn, const FoldCoef& k)
{
    const float s = xn * k.scale;
    return s + k.bias;
}

// The linear shortcut on top of an activation's result (cuda/ShortcutLayer.h:23-37 with a linear
// activation: alpha * input + beta * from).
__device__ __forceinline__ float with_residual(float y, float from, float alpha, float beta)
{
    const float pa = alpha * y;
    const float pb = beta * from;
    return pa + pb;
}

// Mean / variance from the shifted sums S1 = sum(x - K), S2 = sum((x - K)^2) over `count` values,
// and the rolling statistics moved towards them.
struct ChannelStats { float mean, var, rolling_mean, rolling_var; };

__device__ __forceinline__ ChannelStats channel_stats(double s1, double s2, float shift_value, double count,
                                                      float rolling_mean, float rolling_var)
{
    const double shift = static_cast<double>(shift_value);
    const double m = s1 / count;
    double v = (s2 - s1 * m) / count;
    if (v < 0.0) v = 0.0;
    ChannelStats st;
    st.mean = static_cast<float>(shift + m);
    st.var = static_cast<float>(v);
    // sscal then saxpy: two fp32 roundings each (src/BatchNorm.cpp:53-56)
    float r = 0.99f * rolling_mean;
    st.rolling_mean = r + .01f * st.mean;
    r = 0.99f * rolling_var;
    st.rolling_var = r + .01f * st.var;
    return st;
}

// ---- Layer::backward's gradient rescale + clip in front of the backward sums ----
// The layer's backward opens with the norm of its delta, a rescale when the norm is beyond a threshold
// and a clamp (include/Layer.h:385-397, 479-499), and only then runs the activation gradient and the
// batch-norm backward (include/ConvLayer.h:238-252).  The first pass over the delta can carry the sum
// of squares and the largest magnitude along with its own sums, which saves the read that the norm
// alone would cost; the decision is formed on the device (ClipPlan) and the later kernels follow it.
struct __attribute__((aligned(16))) ClipPlan {
    float norm, factor, clip;
    int work;       // 0: no value of the delta changes; kChanges: some do; | kClamps: and the clamp may move one
                    // | kBeyond: and some were beyond the clamp as they came (in the channels that a first launch left)
};
enum { kChanges = 1, kClamps = 2, kBeyond = 4 };

// The plan from `count` partial (sum of squares, largest magnitude) pairs, added in an order that
// depends on THREADS alone: every workgroup that forms it arrives at the same one.  All THREADS
// threads of the workgroup call it; every one returns the plan.
template<int THREADS>
__device__ __forceinline__ ClipPlan clip_plan_from(const double2* part, int count, float threshold, float clip)
{
    __shared__ double plan_sums[THREADS / kWave];
    __shared__ float plan_tops[THREADS / kWave];
    double s = 0.0;
    float top = 0.0f;
    // kPlanLoads partials per thread and round, their loads in flight together (one after the other each
    // costs a trip to memory: 45 of them per thread at 16 x 32 x 608^2 with 256 threads)
    constexpr int kPlanLoads = 8;
    if (count <= THREADS) {
        // the one-launch backward's per-channel figures: one load per thread, the same sum
        const bool valid = static_cast<int>(threadIdx.x) < count;
        const double2 p = part[valid ? threadIdx.x : 0];
        s = valid ? p.x : 0.0;
        top = valid ? static_cast<float>(p.y) : 0.0f;
    } else for (int base = 0; base < count; base += THREADS * kPlanLoads) {
        double2 p[kPlanLoads];
#pragma unroll
        for (int u = 0; u < kPlanLoads; ++u) {
            const int j = base + u * THREADS + static_cast<int>(threadIdx.x);
            p[u] = part[j < count ? j : 0];
        }
#pragma unroll
        for (int u = 0; u < kPlanLoads; ++u) {
            const bool valid = base + u * THREADS + static_cast<int>(threadIdx.x) < count;
            s += valid ? p[u].x : 0.0;
            top = fmaxf(top, valid ? static_cast<float>(p[u].y) : 0.0f);
        }
    }
    s = wave_sum(s);
    top = wave_max(top);
    __syncthreads();       // the arrays may still be read from an earlier call
    if ((threadIdx.x & (kWave - 1)) == 0) {
        plan_sums[threadIdx.x / kWave] = s;
        plan_tops[threadIdx.x / kWave] = top;
    }
    __syncthreads();
    double total = 0.0;
    float peak = 0.0f;
#pragma unroll
    for (int w = 0; w < THREADS / kWave; ++w) {
        total += plan_sums[w];
        peak = fmaxf(peak, plan_tops[w]);
    }
    const RescalePlan r = plan_from_totals(total, peak, threshold, clip);
    const bool beyond = clip > 0.0f && (!(peak <= clip) || total != total);
    return ClipPlan{ r.norm, r.factor, clip, (r.work ? kChanges : 0) | (r.clamps ? kClamps : 0) | (r.work && beyond ? kBeyond : 0) };
}

// What the clipped forms add to a launch: where the first pass leaves its norm partials, and the
// plan that the finish kernel of the first pass writes and everything after it reads.
struct ClipArgs {
    double2* norm_partial;     // [workgroups of the first pass]
    ClipPlan* plan;
    float threshold, clip;
    float* norm_out;           // nullable
};

constexpr int kPlanThreads = 1024;
constexpr int kRedoWorkgroups = 256;      // of the one-launch form's second launch

// The passes of a backward:  kPlain -- no rescale + clip in front;  kFirst -- the sums as if nothing
// had to change, plus the norm partials;  kRedo -- after the plan: leaves at once when the sums of the
// first pass still serve, else forms them again from the rescaled and clamped delta.
// The sums of the first pass serve when nothing changes, and for the batch-norm backward also when the
// delta is only rescaled (the clamp moves no value): they are linear in the delta, so the finish
// kernel multiplies them by the factor and the dx pass applies the factor to the delta it reads.
enum { kPlain = 0, kFirst = 1, kRedo = 2 };

// ---- backward sums: A = sum d', B = sum d' * (x - mean), d' = delta * act'(pre) ----
struct BackwardArgs {
    float* delta;
    const float* x;          // saved conv output (BN) or nullptr (bias only)
    const float* pre;        // nullable when BN: recomputed from x
    const float* mean;
    const float* var;
    const float* scale;
    const float* bias;
};

// Per-channel constants of the dx pass, produced by the finish kernel (64 bytes).
struct __attribute__((aligned(16))) DxCoef {
    FoldCoef f;
    double rroot;     // 1 / sqrt(float(var + eps))
    double c2;        // var_delta * 2 / count
    double md_term;   // float(mean_delta / float(count))
    double pad;
};

// What the sums A = sum d' and B = sum d' * (x - mean) of a channel amount to: the additions to its two
// parameter updates, its mean and variance deltas, and the constants of the dx pass.  Arithmetic only.
struct FinishedChannel {
    DxCoef k;
    float bias_add, scale_add, mean_delta, var_delta;
};

// What the finish takes from the variance alone.
struct VarianceTerms {
    double denom, mean_factor, rroot;
    float power;
};

__device__ __forceinline__ VarianceTerms variance_terms(float v)
{
    const float ve = v + kEps;
    VarianceTerms t;
    t.denom = sqrt(static_cast<double>(v)) + static_cast<double>(kEps);
    t.mean_factor = -1. / static_cast<double>(sqrtf(ve));
    t.rroot = 1.0 / sqrt(static_cast<double>(ve));
    t.power = -.5f * powf(ve, -3.0f / 2.0f);
    return t;
}

template<bool BN>
__device__ __forceinline__ FinishedChannel finished_channel(double sa, double sb, int count, const FoldCoef& f,
                                                            const VarianceTerms& t, float s)
{
    FinishedChannel r{};
    r.bias_add = static_cast<float>(sa);
    if constexpr (BN) {
        // sum d' * x_hat with x_hat = (x - mean) / (sqrt(var) + eps)
        r.scale_add = static_cast<float>(sb / t.denom);
        // sums of d'' = d' * scale
        const float sum_dd = static_cast<float>(sa * static_cast<double>(s));
        const float sum_ddx = static_cast<float>(sb * static_cast<double>(s));
        r.mean_delta = static_cast<float>(static_cast<double>(sum_dd) * t.mean_factor);
        r.var_delta = sum_ddx * t.power;
        r.k.f = f;
        r.k.rroot = t.rroot;
        r.k.c2 = static_cast<double>(r.var_delta) * 2. / static_cast<double>(count);
        r.k.md_term = static_cast<double>(r.mean_delta / static_cast<float>(count));
        r.k.pad = 0.0;
    }
    return r;
}

// A channel that was finished with the sums (sa, sb) of its unscaled delta, after the plan turned out
// to rescale by `factor` (and its clamp to move nothing in this channel): everything the backward left
// is linear in the delta, so the accumulated updates are formed again from what they were `before` (bias,
// scale), with one rounding as everywhere, and so are the two per-channel deltas.  The dx values are scaled
// by the caller.
__device__ __forceinline__ void rescale_finished_channel(double sa, double sb, double factor, float2 before, int c,
                                                         const float* var, const float* scale, float* scale_updates,
                                                         float* bias_updates, float* mean_delta, float* var_delta)
{
    bias_updates[c] = before.x + static_cast<float>(factor * sa);
    const float v = var[c];
    const float s = scale[c];
    const double denom = sqrt(static_cast<double>(v)) + static_cast<double>(kEps);
    scale_updates[c] = before.y + static_cast<float>(factor * sb / denom);
    const float sum_dd = static_cast<float>(factor * sa * static_cast<double>(s));
    const float sum_ddx = static_cast<float>(factor * sb * static_cast<double>(s));
    const float ve = v + kEps;
    if (mean_delta) mean_delta[c] = static_cast<float>(static_cast<double>(sum_dd) * (-1. / static_cast<double>(sqrtf(ve))));
    if (var_delta) var_delta[c] = sum_ddx * (-.5f * powf(ve, -3.0f / 2.0f));
}

// dx from d' = delta * act'(pre)
__device__ __forceinline__ float dx_value(float d, float x, const DxCoef& k)
{
    const float dd = d * k.f.scale;
    const float xm = x - k.f.mean;
    // src/CpuUtil.cpp:336-338 evaluated in double, stored as float
    const double v = static_cast<double>(dd) * k.rroot + k.c2 * static_cast<double>(xm) + k.md_term;
    return static_cast<float>(v);
}

// ... and from the delta itself
template<int ACT>
__device__ __forceinline__ float dx_of_delta(float d, float x, float pre_in, bool recompute, const DxCoef& k)
{
    if constexpr (ACT != PXH_LINEAR) {
        float pre = pre_in;
        if (recompute) pre = affine(normalize(x, k.f), k.f);
        d = d * act_grad<ACT>(pre);
    }
    return dx_value(d, x, k);
}

}  // namespace pxh
