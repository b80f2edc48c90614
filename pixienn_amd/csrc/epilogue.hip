// Conv-layer epilogue for gfx950: batch-norm (inference and training) + bias + activation,
// forward and backward, as one-pass NCHW streaming kernels and per-channel reductions.
#include "grouped.h"

#include <mutex>

// Device memory for pxh_bn_train_act_forward_static, the entry point for callers that must not
// allocate: the partial sums and per-channel constants its kernels pass from one launch to the next.
// Every GPU the library runs on holds its own copy until the process ends.  In host code the name is
// only a handle for hipGetSymbolAddress; kernels are given the address that call returns.
constexpr size_t kStaticScratchBytes = PXH_BN_STATIC_SCRATCH_BYTES;
static __device__ __align__(256) unsigned char scratch[kStaticScratchBytes];

namespace pxh {
namespace {

// The device address of `scratch` on the current device, looked up once per device.
int static_scratch(const char* who, void** out)
{
    constexpr int kDevices = 64;
    static std::mutex mutex;
    static void* address[kDevices] = {};
    int dev = 0;
    hipError_t e = hipGetDevice(&dev);
    if (e != hipSuccess) {
        set_error("%s: hipGetDevice: %s", who, hipGetErrorString(e));
        return static_cast<int>(e);
    }
    if (dev < 0 || dev >= kDevices) {
        set_error("%s: device %d is beyond the %d devices the library keeps scratch addresses for", who, dev,
                  kDevices);
        return PXH_ERR_UNSUPPORTED;
    }
    std::lock_guard<std::mutex> lock(mutex);
    if (!address[dev]) {
        void* p = nullptr;
        e = hipGetSymbolAddress(&p, HIP_SYMBOL(scratch));
        if (e != hipSuccess || !p) {
            set_error("%s: hipGetSymbolAddress(scratch) on device %d: %s", who, dev, hipGetErrorString(e));
            return e != hipSuccess ? static_cast<int>(e) : PXH_ERR_WORKSPACE;
        }
        address[dev] = p;
    }
    *out = address[dev];
    return PXH_OK;
}

__global__ __launch_bounds__(kBlock) void bn_fold_kernel(const float* mean, const float* var, const float* scale,
                                                         const float* bias, int channels, FoldCoef* table)
{
    const int c = blockIdx.x * kBlock + threadIdx.x;
    if (c < channels) table[c] = make_coef(mean[c], var[c], scale[c], bias[c]);
}

struct EpilogueArgs {
    const float* x;
    float* y;
    float* pre;        // nullable
    float* x_saved;    // nullable
    float* x_norm;     // nullable
    const FoldCoef* table;   // BN
    const float* bias;       // bias only
    FastDiv by_spatial;
    FastDiv by_channels;
    uint32_t total;
    // the shortcut that follows the layer, taken into the same pass (else null): what is stored in y is
    // res_alpha * act(pre) + res_beta * residual, the two products and the sum each rounded
    const float* residual;
    float res_alpha, res_beta;
};

template<bool BN>
__device__ __forceinline__ FoldCoef fetch_coef(const EpilogueArgs& a, uint32_t c)
{
    if constexpr (BN) {
        return a.table[c];
    } else {
        FoldCoef k;
        k.bias = a.bias[c];
        return k;
    }
}

template<bool BN>
__device__ __forceinline__ float pre_value(float x, const FoldCoef& k, float& xn)
{
    if constexpr (BN) {
        xn = normalize(x, k);
        return affine(xn, k);
    } else {
        xn = 0.0f;
        return x + k.bias;
    }
}

// One 128-bit vector per lane over the flat tensor.  A lane finds its plane with one
// multiply-high division and loads that channel's folded constants (a 32-byte, cache-resident
// broadcast); the rare vector that straddles two planes loads the next channel's as well.
template<int ACT, bool BN, bool NT, bool RES>
__device__ __forceinline__ void epilogue_fwd_body(const EpilogueArgs& a)
{
    const uint32_t e = (blockIdx.x * static_cast<uint32_t>(kBlock) + threadIdx.x) * 4;
    if (e >= a.total) return;
    const bool full = e + 3 < a.total;
    Pack<4> xin;
    [[maybe_unused]] Pack<4> rin;
    if (full) {
        xin = ld<4, NT>(a.x, e);
        if constexpr (RES) rin = ld<4, NT>(a.residual, e);
    } else {
#pragma unroll
        for (int k = 0; k < 4; ++k) {
            xin.v[k] = (e + k < a.total) ? a.x[e + k] : 0.0f;
            if constexpr (RES) rin.v[k] = (e + k < a.total) ? a.residual[e + k] : 0.0f;
        }
    }
    const uint32_t hw = a.by_spatial.d;
    uint32_t plane, r, q, c;
    a.by_spatial.divmod(e, plane, r);
    a.by_channels.divmod(plane, q, c);
    const FoldCoef k0 = fetch_coef<BN>(a, c);
    Pack<4> yo, po, no;
    const bool crosses = !(r + 3 < hw);
    if (!__ballot(crosses)) {
        // no lane of the wave touches a plane boundary (the common case for large planes)
#pragma unroll
        for (int j = 0; j < 4; ++j) po.v[j] = pre_value<BN>(xin.v[j], k0, no.v[j]);
        act_apply_n<ACT>(po.v, yo.v);
    } else if (hw >= 4) {
        // some lane's vector runs into the next plane (at most one boundary per vector): the
        // elements past it take the next channel's constants.  Selecting the constants per element
        // keeps ONE copy of the arithmetic for the whole wave; a per-lane branch would make a wave
        // that holds a boundary (every wave, for a 13 x 13 plane) run the activation twice.
        FoldCoef k1 = k0;
        if (crosses) k1 = fetch_coef<BN>(a, c + 1 == a.by_channels.d ? 0 : c + 1);
#pragma unroll
        for (int j = 0; j < 4; ++j) {
            const bool here = r + j < hw;
            FoldCoef k;
            k.mean = here ? k0.mean : k1.mean;
            k.r_hi = here ? k0.r_hi : k1.r_hi;
            k.r_lo = here ? k0.r_lo : k1.r_lo;
            k.scale = here ? k0.scale : k1.scale;
            k.bias = here ? k0.bias : k1.bias;
            po.v[j] = pre_value<BN>(xin.v[j], k, no.v[j]);
        }
        act_apply_n<ACT>(po.v, yo.v);
    } else {
        // planes of fewer than 4 elements: several boundaries per vector, walk element by element
        FoldCoef k = k0;
        uint32_t rr = r, cc = c;
#pragma unroll
        for (int j = 0; j < 4; ++j) {
            if (rr == hw) {
                rr = 0;
                cc = cc + 1 == a.by_channels.d ? 0 : cc + 1;
                k = fetch_coef<BN>(a, cc);
            }
            po.v[j] = pre_value<BN>(xin.v[j], k, no.v[j]);
            yo.v[j] = act_apply<ACT>(po.v[j]);
            ++rr;
        }
    }
    if constexpr (RES) {
#pragma unroll
        for (int j = 0; j < 4; ++j) yo.v[j] = with_residual(yo.v[j], rin.v[j], a.res_alpha, a.res_beta);
    }
    if (full) {
        if (a.x_saved) st<4, NT>(a.x_saved, e, xin);
        if (BN && a.x_norm) st<4, NT>(a.x_norm, e, no);
        if (a.pre) st<4, NT>(a.pre, e, po);
        st<4, NT>(a.y, e, yo);
    } else {
        for (int j = 0; j < 4 && e + j < a.total; ++j) {
            if (a.x_saved) a.x_saved[e + j] = xin.v[j];
            if (BN && a.x_norm) a.x_norm[e + j] = no.v[j];
            if (a.pre) a.pre[e + j] = po.v[j];
            a.y[e + j] = yo.v[j];
        }
    }
}

template<int ACT, bool BN, bool NT>
__global__ __launch_bounds__(kBlock) void epilogue_fwd_kernel(EpilogueArgs a)
{
    epilogue_fwd_body<ACT, BN, NT, false>(a);
}

// The same pass with the shortcut that follows the layer: one more stream read, no tensor in between.
template<int ACT, bool BN, bool NT>
__global__ __launch_bounds__(kBlock) void epilogue_shortcut_fwd_kernel(EpilogueArgs a)
{
    epilogue_fwd_body<ACT, BN, NT, true>(a);
}

// Pointers that are not 16-byte aligned: one element per lane.
template<int ACT, bool BN>
__global__ __launch_bounds__(kBlock) void epilogue_fwd_scalar_kernel(EpilogueArgs a)
{
    const uint32_t e = blockIdx.x * kBlock + threadIdx.x;
    if (e >= a.total) return;
    uint32_t plane, r, q, c;
    a.by_spatial.divmod(e, plane, r);
    a.by_channels.divmod(plane, q, c);
    const FoldCoef k = fetch_coef<BN>(a, c);
    const float x = a.x[e];
    float xn;
    const float pre = pre_value<BN>(x, k, xn);
    if (a.x_saved) a.x_saved[e] = x;
    if (BN && a.x_norm) a.x_norm[e] = xn;
    if (a.pre) a.pre[e] = pre;
    float y = act_apply<ACT>(pre);
    if (a.residual) y = with_residual(y, a.residual[e], a.res_alpha, a.res_beta);
    a.y[e] = y;
}

// ---- the inference epilogue with the 2 x 2, stride 2 max-pool that follows the layer ----
// A lane takes VX consecutive outputs of one output row: 2 * VX inputs of each of two input rows (one
// plane, so one channel's constants), applies the epilogue to them and keeps the largest of each window,
// compared in the order the pool's own kernel compares them.  The layer's own output is written only when
// something else reads it.
struct EpiloguePoolArgs {
    const float* x;
    float* y;             // nullable: the layer's own output
    float* pooled;
    const FoldCoef* table;
    uint32_t units;       // lanes with work
    uint32_t iw, ow;
    FastDiv by_owv;       // ow / VX
    FastDiv by_oh;
    FastDiv by_channels;
};

template<int ACT, int VX, bool NT>
__global__ __launch_bounds__(kBlock) void epilogue_pool2_fwd_kernel(EpiloguePoolArgs a)
{
    const uint32_t t = blockIdx.x * static_cast<uint32_t>(kBlock) + threadIdx.x;
    if (t >= a.units) return;
    uint32_t rows, oxv, plane, oy, q, c;
    a.by_owv.divmod(t, rows, oxv);
    a.by_oh.divmod(rows, plane, oy);
    a.by_channels.divmod(plane, q, c);
    const uint32_t ih = a.by_oh.d * 2;
    const uint32_t in0 = (plane * ih + 2 * oy) * a.iw + 2 * oxv * VX;      // < 2^31 checked by the host
    const Pack<2 * VX> r0 = ld<2 * VX, NT>(a.x, in0);
    const Pack<2 * VX> r1 = ld<2 * VX, NT>(a.x, in0 + a.iw);
    const FoldCoef k = a.table[c];
    Pack<2 * VX> y0, y1;
    float pre[2 * VX], xn;
#pragma unroll
    for (int j = 0; j < 2 * VX; ++j) pre[j] = pre_value<true>(r0.v[j], k, xn);
    act_apply_n<ACT>(pre, y0.v);
#pragma unroll
    for (int j = 0; j < 2 * VX; ++j) pre[j] = pre_value<true>(r1.v[j], k, xn);
    act_apply_n<ACT>(pre, y1.v);
    if (a.y) {
        st<2 * VX, NT>(a.y, in0, y0);
        st<2 * VX, NT>(a.y, in0 + a.iw, y1);
    }
    Pack<VX> best;
#pragma unroll
    for (int j = 0; j < VX; ++j) {
        float b = y0.v[2 * j];
        if (y0.v[2 * j + 1] > b) b = y0.v[2 * j + 1];
        if (y1.v[2 * j] > b) b = y1.v[2 * j];
        if (y1.v[2 * j + 1] > b) b = y1.v[2 * j + 1];
        best.v[j] = b;
    }
    st<VX, NT>(a.pooled, (plane * a.by_oh.d + oy) * a.ow + oxv * VX, best);
}

int check_shape(const char* who, int batch, int channels, int spatial, uint32_t* total)
{
    if (batch <= 0 || channels <= 0 || spatial <= 0)
        return fail_invalid("%s: batch, channels and spatial must be positive (%d, %d, %d)", who, batch, channels,
                            spatial);
    const unsigned long long t = 1ull * batch * channels * spatial;
    if (t >= (1ull << 31)) {
        set_error("%s: %llu elements; tensors of 2^31 elements or more are not supported", who, t);
        return PXH_ERR_UNSUPPORTED;
    }
    *total = static_cast<uint32_t>(t);
    return PXH_OK;
}

template<bool BN>
int launch_epilogue_fwd(const char* who, EpilogueArgs a, int activation, hipStream_t stream)
{
    // the walk across a plane boundary handles any plane size, including single elements
    const bool vec = aligned16(a.x) && aligned16(a.y) && aligned16(a.pre) && aligned16(a.x_saved) &&
                     aligned16(a.x_norm) && aligned16(a.residual);
    // bytes this launch moves: x in, y out, plus each materialised extra output and the shortcut's source
    const size_t streams = 2 + (a.pre ? 1 : 0) + (a.x_saved ? 1 : 0) + (a.x_norm ? 1 : 0) + (a.residual ? 1 : 0);
    const bool nt = static_cast<size_t>(a.total) * 4 * streams >= kStreamingBytes;
    const bool known = dispatch_activation(activation, [&]<int ACT>() {
        if (vec) {
            const dim3 grid(grid_for(a.total, static_cast<size_t>(kBlock) * 4));
            if (a.residual) {
                if (nt) hipLaunchKernelGGL((epilogue_shortcut_fwd_kernel<ACT, BN, true>), grid, dim3(kBlock), 0, stream, a);
                else hipLaunchKernelGGL((epilogue_shortcut_fwd_kernel<ACT, BN, false>), grid, dim3(kBlock), 0, stream, a);
            } else if (nt) hipLaunchKernelGGL((epilogue_fwd_kernel<ACT, BN, true>), grid, dim3(kBlock), 0, stream, a);
            else hipLaunchKernelGGL((epilogue_fwd_kernel<ACT, BN, false>), grid, dim3(kBlock), 0, stream, a);
        } else {
            hipLaunchKernelGGL((epilogue_fwd_scalar_kernel<ACT, BN>), dim3(grid_for(a.total, kBlock)),
                               dim3(kBlock), 0, stream, a);
        }
    });
    if (!known) return fail_invalid("%s: unknown activation %d", who, activation);
    return check_launch(who);
}

// ------------------------------------------------------------------------------------------
// Per-channel reductions.
//
// Channel c owns `batch` planes of `spatial` contiguous floats.  A plane is cut into segments of
// kSeg floats; the (image, segment) items of a channel are dealt ReduceGeom::per_block to a workgroup,
// one item per wavefront at a time (64 lanes x 128-bit x 4 loads = one segment).  Lanes sum a
// segment in fp32, carry across segments in double; the workgroup's pair of sums goes to
// partial[c][j] and a second kernel adds the partials of a channel in a fixed order.
// ------------------------------------------------------------------------------------------
constexpr int kSegLoads = 4;                  // 128-bit loads in flight per lane
constexpr int kSeg = kWave * 4 * kSegLoads;   // 1024 floats
// Items of a workgroup: as many as kItemsPerBlock, four to a wavefront, where that leaves kFillBlocks workgroups
// (four to a compute unit); fewer, down to one a wavefront, where it does not.  A wavefront takes its items one
// after the other, so a small grid is bound by that chain and not by memory.  Sixteen items everywhere against this
// rule, backward, us: 6 x 72 x 135 x 77 (360 workgroups) leaky 26.1 -> 24.2, mish 42.1 -> 33.7; 64 x 64 x 13^2 (256)
// mish 18.6 -> 15.3; 64 x 96 x 19^2 (384) mish 27.4 -> 23.8.  The forward's sums gain 1 us.  A full grid keeps sixteen:
// more workgroups there only add partials to finish.
constexpr int kItemsPerBlock = 16;
constexpr int kFillBlocks = 1024;

struct ReduceGeom {
    int channels, spatial, parts, items, per_block, blocks;
    FastDiv by_parts;
    FastDiv by_blocks;
};

ReduceGeom make_geom(int batch, int channels, int spatial)
{
    ReduceGeom g;
    g.channels = channels;
    g.spatial = spatial;
    g.parts = (spatial + kSeg - 1) / kSeg;
    g.items = batch * g.parts;
    g.per_block = kItemsPerBlock;
    const auto blocks = [&] { return (g.items + g.per_block - 1) / g.per_block; };
    while (g.per_block > kBlock / kWave && static_cast<long long>(channels) * blocks() < kFillBlocks) g.per_block /= 2;
    g.blocks = blocks();
    g.by_parts = FastDiv(static_cast<uint32_t>(g.parts));
    g.by_blocks = FastDiv(static_cast<uint32_t>(g.blocks));
    return g;
}

// Calls body(base, seg0, seg1, lane) for every item of workgroup (c, j): `base` is the offset of
// the item's plane, [seg0, seg1) its segment inside the plane.
template<typename Body>
__device__ __forceinline__ void for_each_item(const ReduceGeom& g, uint32_t c, uint32_t j, Body&& body)
{
    const int lane = threadIdx.x & (kWave - 1);
    const int wave = threadIdx.x / kWave;
    const int first = j * g.per_block;
    const int last = min(first + g.per_block, g.items);
    for (int it = first + wave; it < last; it += kBlock / kWave) {
        uint32_t n, part;
        g.by_parts.divmod(static_cast<uint32_t>(it), n, part);
        const size_t base = (static_cast<size_t>(n) * g.channels + c) * g.spatial;
        const int seg0 = part * kSeg;
        const int seg1 = min(g.spatial, seg0 + kSeg);
        body(base, seg0, seg1, lane);
    }
}

// Odd planes: the vector at `off` of a plane, the last one moved back to end with it.  The values that it shares with the one
// in front (of the segment in front, even) stay out of the sums and are not written; every value goes into a double of
// its own.
template<bool RAGGED>
__device__ __forceinline__ int ragged_start(int off, int spatial)
{
    return RAGGED && off + 4 > spatial ? spatial - 4 : off;
}

template<int V, bool NT, bool RAGGED>
__device__ __forceinline__ Pack<V> ld_at(const float* p, size_t e)
{
    if constexpr (RAGGED) return ld_word<NT>(p + e);
    else return ld<V, NT>(p, e);
}

// ---- statistics: S1 = sum(x - K), S2 = sum((x - K)^2), K = first element of the channel ----
template<int V, bool NT, bool RAGGED = false>
__global__ __launch_bounds__(kBlock) void bn_stats_partial_kernel(const float* x, ReduceGeom g, double2* partial, float* shifts)
{
    __shared__ double slots[2][kBlock / kWave];
    uint32_t c, j;
    g.by_blocks.divmod(blockIdx.x, c, j);
    const float shift = x[static_cast<size_t>(c) * g.spatial];
    double s1 = 0.0, s2 = 0.0;
    for_each_item(g, c, j, [&](size_t base, int seg0, int seg1, int lane) {
        constexpr int kLoads = V == 1 ? kValueSteps : kSegLoads;
        Pack<V> v[kLoads];
#pragma unroll
        for (int u = 0; u < kLoads; ++u) {
            const int off = seg0 + (u * kWave + lane) * V;
            if (off < seg1) v[u] = ld_at<V, NT, RAGGED>(x, base + ragged_start<RAGGED>(off, g.spatial));
        }
        if constexpr (RAGGED || V == 1) {
#pragma unroll
            for (int u = 0; u < kLoads; ++u) {
                const int off = seg0 + (u * kWave + lane) * V;
                if (off >= seg1) break;
                const int own = off - ragged_start<RAGGED>(off, g.spatial);
#pragma unroll
                for (int k = 0; k < V; ++k) {
                    const float d = k >= own ? v[u].v[k] - shift : 0.0f;
                    s1 += static_cast<double>(d);
                    s2 += static_cast<double>(d * d);
                }
            }
            return;
        }
        float a1 = 0.0f, a2 = 0.0f;
#pragma unroll
        for (int u = 0; u < kLoads; ++u) {
            const int off = seg0 + (u * kWave + lane) * V;
            if (off < seg1) {
#pragma unroll
                for (int k = 0; k < V; ++k) {
                    const float d = v[u].v[k] - shift;
                    a1 += d;
                    a2 += d * d;
                }
            }
        }
        s1 += static_cast<double>(a1);
        s2 += static_cast<double>(a2);
    });
    const double t1 = block_sum(s1, slots[0]);
    const double t2 = block_sum(s2, slots[1]);
    if (threadIdx.x == 0) {
        partial[blockIdx.x] = make_double2(t1, t2);
        if (shifts && j == 0) shifts[c] = shift;
    }
}

// The same for channel c of the tensors: writes the statistics and folds the constants the apply
// pass needs.
__device__ __forceinline__ FoldCoef finish_stats(double s1, double s2, float shift_value, double count, int c,
                                                 float* mean, float* var, float* rolling_mean, float* rolling_var,
                                                 const float* scale, const float* bias)
{
    const ChannelStats st = channel_stats(s1, s2, shift_value, count, rolling_mean ? rolling_mean[c] : 0.0f,
                                          rolling_var ? rolling_var[c] : 0.0f);
    mean[c] = st.mean;
    var[c] = st.var;
    if (rolling_mean) {
        rolling_mean[c] = st.rolling_mean;
        rolling_var[c] = st.rolling_var;
    }
    return make_coef(st.mean, st.var, scale ? scale[c] : 1.0f, bias ? bias[c] : 0.0f);
}

// One wavefront per channel adds the channel's partials and finishes the statistics.
__global__ __launch_bounds__(kBlock) void bn_stats_finish_kernel(const float* x, const double2* partial, int channels,
                                                                 int spatial, int blocks, double count, float* mean,
                                                                 float* var, float* rolling_mean, float* rolling_var,
                                                                 const float* scale, const float* bias,
                                                                 FoldCoef* table)
{
    const int lane = threadIdx.x & (kWave - 1);
    const int c = blockIdx.x * (kBlock / kWave) + threadIdx.x / kWave;
    if (c >= channels) return;
    double s1 = 0.0, s2 = 0.0;
    for (int j = lane; j < blocks; j += kWave) {
        const double2 p = partial[static_cast<size_t>(c) * blocks + j];
        s1 += p.x;
        s2 += p.y;
    }
    s1 = wave_sum(s1);
    s2 = wave_sum(s2);
    if (lane == 0) {
        const FoldCoef k = finish_stats(s1, s2, x[static_cast<size_t>(c) * spatial], count, c, mean, var, rolling_mean,
                                        rolling_var, scale, bias);
        if (table) table[c] = k;
    }
}

// WRITE (the bias-only layer, which has no dx pass): d' goes back into delta.  With kFirst nothing is
// written (the delta is still needed as it came); with kRedo the pass also runs, writing, when nothing
// has to change but the activation has a gradient to apply.
template<int ACT, bool BN, bool WRITE, int V, bool NT, int MODE = kPlain, bool RAGGED = false>
__global__ __launch_bounds__(kBlock) void bwd_partial_kernel(BackwardArgs a, ReduceGeom g, double2* partial,
                                                             ClipArgs clip = ClipArgs{})
{
    static_assert(!(WRITE && MODE == kFirst), "the first pass of a clipped backward leaves the delta alone");
    __shared__ double slots[2][kBlock / kWave];
    [[maybe_unused]] float factor = 1.0f, limit = 0.0f;
    [[maybe_unused]] bool changes = false;
    if constexpr (MODE == kRedo) {
        const ClipPlan plan = *clip.plan;
        changes = plan.work != 0;
        // the writing form has the delta to rewrite whenever a value changes; the other only its sums to
        // form again, and only when the clamp takes part
        const bool again = WRITE ? changes : (plan.work & kClamps) != 0;
        if (!again && !(WRITE && ACT != PXH_LINEAR)) return;
        factor = changes ? plan.factor : 1.0f;
        limit = changes ? plan.clip : 0.0f;
    }
    uint32_t c, j;
    g.by_blocks.divmod(blockIdx.x, c, j);
    FoldCoef k;
    if constexpr (BN) k = make_coef(a.mean[c], a.var[c], a.scale[c], a.bias[c]);
    const bool recompute = BN && a.pre == nullptr;
    double sa = 0.0, sb = 0.0;
    [[maybe_unused]] double sq = 0.0;
    [[maybe_unused]] float peak = 0.0f;
    for_each_item(g, c, j, [&](size_t base, int seg0, int seg1, int lane) {
        constexpr int kLoads = V == 1 ? kValueSteps : kSegLoads;
        constexpr bool kEach = RAGGED || V == 1;
        Pack<V> d[kLoads], xv[kLoads], pv[kLoads];
#pragma unroll
        for (int u = 0; u < kLoads; ++u) {
            const int off = seg0 + (u * kWave + lane) * V;
            if (off < seg1) {
                const size_t at = base + ragged_start<RAGGED>(off, g.spatial);
                d[u] = ld_at<V, NT, RAGGED>(a.delta, at);
                if constexpr (BN) xv[u] = ld_at<V, NT, RAGGED>(a.x, at);
                if constexpr (ACT != PXH_LINEAR) {
                    if (!recompute) pv[u] = ld_at<V, NT, RAGGED>(a.pre, at);
                }
            }
        }
        [[maybe_unused]] float fa = 0.0f, fb = 0.0f, fq = 0.0f;
#pragma unroll
        for (int u = 0; u < kLoads; ++u) {
            const int off = seg0 + (u * kWave + lane) * V;
            if (off < seg1) {
                const int start = ragged_start<RAGGED>(off, g.spatial);
                if constexpr (MODE != kPlain) {
#pragma unroll
                    for (int q = 0; q < V; ++q) {
                        const float dv = d[u].v[q];
                        if constexpr (MODE == kFirst) {
                            if constexpr (kEach) sq += static_cast<double>(q >= off - start ? dv * dv : 0.0f);
                            else fq += dv * dv;
                            peak = fmaxf(peak, fabsf(dv));
                        } else {
                            d[u].v[q] = rescaled_clipped(dv, factor, limit);
                        }
                    }
                }
                if constexpr (ACT != PXH_LINEAR) {
                    if (recompute) {
#pragma unroll
                        for (int q = 0; q < V; ++q) pv[u].v[q] = affine(normalize(xv[u].v[q], k), k);
                    }
                    times_grad<ACT>(d[u].v, pv[u].v);
                }
#pragma unroll
                for (int q = 0; q < V; ++q) {
                    if constexpr (kEach) {
                        const float t = d[u].v[q];
                        sa += static_cast<double>(q >= off - start ? t : 0.0f);
                        if constexpr (BN) sb += static_cast<double>(q >= off - start ? t * (xv[u].v[q] - k.mean) : 0.0f);
                    } else {
                        fa += d[u].v[q];
                        if constexpr (BN) fb += d[u].v[q] * (xv[u].v[q] - k.mean);
                    }
                }
                if constexpr (WRITE && (ACT != PXH_LINEAR || MODE == kRedo)) {
                    if (ACT != PXH_LINEAR || changes) {
                        if constexpr (RAGGED) st_own(a.delta + base + start, d[u], off - start);
                        else st<V, NT>(a.delta, base + off, d[u]);
                    }
                }
            }
        }
        if constexpr (!kEach) {
            sa += static_cast<double>(fa);
            sb += static_cast<double>(fb);
            if constexpr (MODE == kFirst) sq += static_cast<double>(fq);
        }
    });
    const double ta = block_sum(sa, slots[0]);
    const double tb = block_sum(sb, slots[1]);
    if (threadIdx.x == 0) partial[blockIdx.x] = make_double2(ta, tb);
    if constexpr (MODE == kFirst) {
        __shared__ float peaks[kBlock / kWave];
        const double tq = block_sum(sq, slots[0]);      // synchronises before it reuses the slots
        peak = wave_max(peak);
        if ((threadIdx.x & (kWave - 1)) == 0) peaks[threadIdx.x / kWave] = peak;
        __syncthreads();
        if (threadIdx.x == 0) {
            float top = peaks[0];
#pragma unroll
            for (int w = 1; w < kBlock / kWave; ++w) top = fmaxf(top, peaks[w]);
            clip.norm_partial[blockIdx.x] = make_double2(tq, static_cast<double>(top));
        }
    }
}

// Channel c from its sums: accumulates the parameter updates and returns the constants of the dx pass.
template<bool BN>
__device__ __forceinline__ DxCoef finish_backward(double sa, double sb, int c, int count, const float* mean,
                                                  const float* var, const float* scale, const float* bias,
                                                  float* scale_updates, float* bias_updates, float* mean_delta,
                                                  float* var_delta)
{
    // every load before the first store: a load behind a store waits for that store as well
    FoldCoef f{};
    float v = 0.0f, s = 0.0f, scale_updates_in = 0.0f;
    const float bias_updates_in = bias_updates[c];
    if constexpr (BN) {
        scale_updates_in = scale_updates[c];
        v = var[c];
        s = scale[c];
        f = make_coef(mean[c], v, s, bias[c]);
    }
    const FinishedChannel r = finished_channel<BN>(sa, sb, count, f, BN ? variance_terms(v) : VarianceTerms{}, s);
    bias_updates[c] = bias_updates_in + r.bias_add;
    if constexpr (BN) {
        scale_updates[c] = scale_updates_in + r.scale_add;
        if (mean_delta) mean_delta[c] = r.mean_delta;
        if (var_delta) var_delta[c] = r.var_delta;
    }
    return r.k;
}

// kFirst (workgroups of kPlanThreads): every workgroup forms the plan from all norm partials of the first
// pass (the same additions in the same order everywhere), the first one records it, and the channels
// are finished only when nothing has to change; kRedo: finishes them from the second pass's sums when
// something had to.
template<bool BN, int MODE = kPlain, int THREADS = kBlock>
__global__ __launch_bounds__(THREADS) void bwd_finish_kernel(const double2* partial, int channels, int blocks, int count,
                                                             const float* mean, const float* var, const float* scale,
                                                             const float* bias, float* scale_updates,
                                                             float* bias_updates, float* mean_delta, float* var_delta,
                                                             DxCoef* coef, ClipArgs clip = ClipArgs{})
{
    [[maybe_unused]] double sums_factor = 1.0;
    if constexpr (MODE == kFirst) {
        const ClipPlan plan = clip_plan_from<THREADS>(clip.norm_partial, channels * blocks, clip.threshold, clip.clip);
        if (blockIdx.x == 0 && threadIdx.x == 0) {
            *clip.plan = plan;
            if (clip.norm_out) *clip.norm_out = plan.norm;
        }
        // with batch-norm the sums serve unless the clamp takes part; a bias-only layer's delta is
        // rewritten by the second pass whenever a value changes, and that pass leaves exact sums
        if (BN ? (plan.work & kClamps) != 0 : plan.work != 0) return;
        sums_factor = static_cast<double>(plan.factor);
    }
    if constexpr (MODE == kRedo) {
        const int work = clip.plan->work;
        if (BN ? (work & kClamps) == 0 : work == 0) return;
    }
    const int lane = threadIdx.x & (kWave - 1);
    const int c = blockIdx.x * (THREADS / kWave) + threadIdx.x / kWave;
    if (c >= channels) return;
    double sa = 0.0, sb = 0.0;
    for (int j = lane; j < blocks; j += kWave) {
        const double2 p = partial[static_cast<size_t>(c) * blocks + j];
        sa += p.x;
        sb += p.y;
    }
    sa = wave_sum(sa);
    sb = wave_sum(sb);
    if constexpr (MODE == kFirst) {
        if (sums_factor != 1.0) {
            sa *= sums_factor;
            sb *= sums_factor;
        }
    }
    if (lane == 0) {
        const DxCoef k = finish_backward<BN>(sa, sb, c, count, mean, var, scale, bias, scale_updates, bias_updates,
                                             mean_delta, var_delta);
        if constexpr (BN) coef[c] = k;
    }
}

struct DxArgs {
    float* delta;
    const float* x;
    const float* pre;   // nullable: recomputed
    const DxCoef* coef;
    FastDiv by_spatial;
    FastDiv by_channels;
    uint32_t total;
    const ClipPlan* plan;     // the clipped form: the delta goes through the plan's rescale + clamp first
};

// The delta as the sums saw it: through the plan when there is one and it changes anything.
template<bool CLIPPED, int V>
__device__ __forceinline__ void apply_plan(const DxArgs& a, Pack<V>& d)
{
    if constexpr (CLIPPED) {
        const ClipPlan plan = *a.plan;
        if (plan.work) {
#pragma unroll
            for (int k = 0; k < V; ++k) d.v[k] = rescaled_clipped(d.v[k], plan.factor, plan.clip);
        }
    }
}

template<int ACT, bool NT, bool CLIPPED = false>
__global__ __launch_bounds__(kBlock) void bn_dx_kernel(DxArgs a)
{
    const uint32_t e = (blockIdx.x * static_cast<uint32_t>(kBlock) + threadIdx.x) * 4;
    if (e >= a.total) return;
    const bool full = e + 3 < a.total;
    const bool recompute = a.pre == nullptr;
    Pack<4> din, xin, pin;
    if (full) {
        din = ld<4, NT>(a.delta, e);
        xin = ld<4, NT>(a.x, e);
        if (ACT != PXH_LINEAR && !recompute) pin = ld<4, NT>(a.pre, e);
    } else {
#pragma unroll
        for (int k = 0; k < 4; ++k) {
            const bool ok = e + k < a.total;
            din.v[k] = ok ? a.delta[e + k] : 0.0f;
            xin.v[k] = ok ? a.x[e + k] : 0.0f;
            pin.v[k] = (ok && ACT != PXH_LINEAR && !recompute) ? a.pre[e + k] : 0.0f;
        }
    }
    apply_plan<CLIPPED, 4>(a, din);
    const uint32_t hw = a.by_spatial.d;
    uint32_t plane, r, q, c;
    a.by_spatial.divmod(e, plane, r);
    a.by_channels.divmod(plane, q, c);
    Pack<4> out;
    const bool crosses = !(r + 3 < hw);
    if (!__ballot(crosses)) {
        const DxCoef k = a.coef[c];
        if constexpr (ACT != PXH_LINEAR) {
            if (recompute) {
#pragma unroll
                for (int j = 0; j < 4; ++j) pin.v[j] = affine(normalize(xin.v[j], k.f), k.f);
            }
            times_grad<ACT>(din.v, pin.v);
        }
#pragma unroll
        for (int j = 0; j < 4; ++j) out.v[j] = dx_value(din.v[j], xin.v[j], k);
    } else if (hw >= 4) {
        // one boundary per vector at most: constants selected per element, one copy of the arithmetic
        // for the wave (see epilogue_fwd_kernel)
        const DxCoef k0 = a.coef[c];
        DxCoef k1 = k0;
        if (crosses) k1 = a.coef[c + 1 == a.by_channels.d ? 0 : c + 1];
        const auto constants = [&](int j) {
            const bool here = r + j < hw;
            DxCoef k;
            k.f.mean = here ? k0.f.mean : k1.f.mean;
            k.f.r_hi = here ? k0.f.r_hi : k1.f.r_hi;
            k.f.r_lo = here ? k0.f.r_lo : k1.f.r_lo;
            k.f.scale = here ? k0.f.scale : k1.f.scale;
            k.f.bias = here ? k0.f.bias : k1.f.bias;
            k.rroot = here ? k0.rroot : k1.rroot;
            k.c2 = here ? k0.c2 : k1.c2;
            k.md_term = here ? k0.md_term : k1.md_term;
            return k;
        };
        if constexpr (ACT != PXH_LINEAR) {
            if (recompute) {
#pragma unroll
                for (int j = 0; j < 4; ++j) {
                    const DxCoef k = constants(j);
                    pin.v[j] = affine(normalize(xin.v[j], k.f), k.f);
                }
            }
            times_grad<ACT>(din.v, pin.v);
        }
#pragma unroll
        for (int j = 0; j < 4; ++j) out.v[j] = dx_value(din.v[j], xin.v[j], constants(j));
    } else {
        uint32_t rr = r, cc = c;
#pragma unroll
        for (int j = 0; j < 4; ++j) {
            if (rr == hw) {
                rr = 0;
                cc = cc + 1 == a.by_channels.d ? 0 : cc + 1;
            }
            out.v[j] = dx_of_delta<ACT>(din.v[j], xin.v[j], pin.v[j], recompute, a.coef[cc]);
            ++rr;
        }
    }
    if (full) {
        st<4, NT>(a.delta, e, out);
    } else {
        for (int j = 0; j < 4 && e + j < a.total; ++j) a.delta[e + j] = out.v[j];
    }
}

template<int ACT, bool CLIPPED = false>
__global__ __launch_bounds__(kBlock) void bn_dx_scalar_kernel(DxArgs a)
{
    const uint32_t e = blockIdx.x * kBlock + threadIdx.x;
    if (e >= a.total) return;
    uint32_t plane, r, q, c;
    a.by_spatial.divmod(e, plane, r);
    a.by_channels.divmod(plane, q, c);
    const bool recompute = a.pre == nullptr;
    const float pre = (ACT != PXH_LINEAR && !recompute) ? a.pre[e] : 0.0f;
    Pack<1> d;
    d.v[0] = a.delta[e];
    apply_plan<CLIPPED, 1>(a, d);
    a.delta[e] = dx_of_delta<ACT>(d.v[0], a.x[e], pre, recompute, a.coef[c]);
}

// ------------------------------------------------------------------------------------------
// The pass behind the partial sums with the finish of the channels inside: a workgroup goes over the same items of a channel
// as one of the sums' does, its first wave adds the channel's partials up and forms the constants while the loads of the
// first items are on their way, and the channel's first workgroup writes what is left of it.  A launch that does only that
// is 4 us, whatever the size: a chain of trips to memory and double-precision roots.  Past a size the flat pass is ahead by
// more, whose lanes take one vector each and past the caches.  Three launches -> two, us, leaky and mish: forward,
// + shortcut, backward with the pre-activation kept (one without takes groups where planes are aligned)
//   2 x 16 x 160^2       9.7 ->  7.8    9.9 ->  7.8   14.4 ->  9.7   10.2 ->  8.7   10.4 ->  8.6   18.9 -> 12.2
//   4 x 64 x 104^2      13.9 -> 10.7   14.5 -> 11.1   23.2 -> 18.0   14.3 -> 12.2   14.7 -> 12.7   29.0 -> 22.6
//   6 x 72 x 135 x 77   17.4 -> 13.1   19.8 -> 13.8   32.6 -> 28.0   17.6 -> 14.3   20.1 -> 15.5   40.0 -> 33.7
//   4 x 32 x 208^2      18.6 -> 14.2   21.4 -> 16.9   37.0 -> 33.1   19.0 -> 17.1   22.0 -> 19.3   43.0 -> 39.2
//   9 x 20 x 203 x 251  26.4 -> 22.3   31.9 -> 26.7   48.6 -> 51.3   27.2 -> 23.7   32.6 -> 27.6   58.6 -> 61.3
//   4 x 16 x 416^2      29.0 -> 27.4   35.9 -> 33.1   56.0 -> 60.2   29.3 -> 29.7   36.3 -> 37.9   66.0 -> 69.8
//   8 x 16 x 416^2      47.0 -> 45.8   60.2 -> 69.2   104  -> 123    47.1 -> 49.6   61.6 -> 77.8   122  -> 136
// (6 x 72 x 135 x 77, mish, without the pre-activation: 31.5 -> 28.4.)  The forward's line lies lower where the
// exponential is followed by a logarithm, and for mish on aligned planes with no shortcut on top: softplus 8 x 80 x 104^2 21.4 -> 21.2, but
// 16 x 48 x 104^2 24.0 -> 26.0, 4 x 16 x 392^2 26.1 -> 29.2, 38 x 69 x 47 x 85 28.5 -> 35.8, with a shortcut 33.9 -> 39.4; mish 8 x 80 x 104^2
// 20.9 -> 19.3, 16 x 48 x 104^2 23.7 -> 25.0, 4 x 16 x 392^2 26.2 -> 27.3, with a shortcut 28.3 -> 26.2 and 31.2 -> 29.6, odd planes
// (8 x 60 x 133^2) 24.5 -> 22.1, with one 28.5 -> 26.7; logistic 22.7 -> 19.4 and 25.2 -> 22.9.
// ------------------------------------------------------------------------------------------
constexpr int kFusedPartials = 4 * kWave;      // of a channel: a lane of the first wave takes four
constexpr uint32_t kFusedForward = 10u << 20, kFusedForwardChain = 7u << 20, kFusedBackward = 6u << 20;      // values of a tensor
constexpr int kFusedSpatial = 4 * kWave;       // a wave's step; planes below leave most of its lanes without a vector

__device__ __forceinline__ double2 channel_sums(const double2* partial, uint32_t c, int blocks)
{
    const int lane = threadIdx.x & (kWave - 1);
    double s1 = 0.0, s2 = 0.0;
    for (int j = lane; j < blocks; j += kWave) {
        const double2 p = partial[static_cast<size_t>(c) * blocks + j];
        s1 += p.x;
        s2 += p.y;
    }
    return make_double2(wave_sum(s1), wave_sum(s2));
}

// The items of a wave, one after the other, and their vectors.
template<bool RAGGED>
struct WaveItems {
    const ReduceGeom& g;
    uint32_t c;
    int it, last;
    size_t base = 0;
    int seg0 = 0, seg1 = 0;
    __device__ __forceinline__ WaveItems(const ReduceGeom& geom, uint32_t channel, uint32_t j)
        : g(geom), c(channel), it(j * geom.per_block + threadIdx.x / kWave), last(min(static_cast<int>((j + 1) * geom.per_block), geom.items))
    {
        place();
    }
    __device__ __forceinline__ void place()
    {
        uint32_t n, part;
        g.by_parts.divmod(static_cast<uint32_t>(it < last ? it : 0), n, part);
        base = (static_cast<size_t>(n) * g.channels + c) * g.spatial;
        seg0 = part * kSeg;
        seg1 = min(g.spatial, seg0 + kSeg);
    }
    __device__ __forceinline__ bool more() const { return it < last; }
    __device__ __forceinline__ void next()
    {
        it += kBlock / kWave;
        place();
    }
    // vector u of the lane: where it begins in its plane, and whether it is one of the item's
    __device__ __forceinline__ int offset(int u) const { return seg0 + (u * kWave + static_cast<int>(threadIdx.x & (kWave - 1))) * 4; }
    __device__ __forceinline__ bool has(int u) const { return more() && offset(u) < seg1; }
    __device__ __forceinline__ size_t at(int u) const { return base + ragged_start<RAGGED>(offset(u), g.spatial); }
    __device__ __forceinline__ int held(int u) const { return offset(u) - ragged_start<RAGGED>(offset(u), g.spatial); }
};

// Odd planes: past the caches, but for what is written beside the output.  us, all past the caches, all cached, and so: the forward
// alone 19.0, 20.3, 19.1, with the pre-activation kept 29.0, 25.2, 24.8, and with a pass behind it that reads the output 32.0, 31.6,
// 32.2 (8 x 60 x 133^2, leaky); 14.0, 15.9, 14.0, then 17.0, 17.3, and 23.3, 25.6 (6 x 72 x 135 x 77, mish; its backward 33.8, 34.4).
template<bool RAGGED, bool NT>
__device__ __forceinline__ void st_item(float* p, size_t at, const Pack<4>& v, int held)
{
    if constexpr (RAGGED) st_own<NT>(p + at, v, held);
    else st<4, false>(p, at, v);
}

struct StatsFinish {
    const double2* partial;
    const float* shifts;
    double count;
    float *mean, *var, *rolling_mean, *rolling_var;
    const float *scale, *bias;
};

template<int ACT, bool RES, bool RAGGED>
__global__ __launch_bounds__(kBlock) void bn_finish_apply_kernel(EpilogueArgs a, ReduceGeom g, StatsFinish f)
{
    __shared__ FoldCoef shared_coef;
    uint32_t c, j;
    g.by_blocks.divmod(blockIdx.x, c, j);
    WaveItems<RAGGED> item(g, c, j);
    Pack<4> x[kSegLoads], r[kSegLoads];
    const auto fetch = [&] {
#pragma unroll
        for (int u = 0; u < kSegLoads; ++u) {
            if (!item.has(u)) continue;
            x[u] = ld_at<4, false, RAGGED>(a.x, item.at(u));
            if constexpr (RES) r[u] = ld_at<4, false, RAGGED>(a.residual, item.at(u));
        }
    };
    fetch();
    if (threadIdx.x < kWave) {
        const float shift = f.shifts[c], scale = f.scale[c], bias = f.bias[c];
        const float rolling_mean = j == 0 ? f.rolling_mean[c] : 0.0f, rolling_var = j == 0 ? f.rolling_var[c] : 0.0f;
        const double2 sums = channel_sums(f.partial, c, g.blocks);
        const ChannelStats st = channel_stats(sums.x, sums.y, shift, f.count, rolling_mean, rolling_var);
        if (threadIdx.x == 0) {
            shared_coef = make_coef(st.mean, st.var, scale, bias);
            if (j == 0) {
                f.mean[c] = st.mean;
                f.var[c] = st.var;
                f.rolling_mean[c] = st.rolling_mean;
                f.rolling_var[c] = st.rolling_var;
            }
        }
    }
    __syncthreads();
    const FoldCoef k = shared_coef;
    while (item.more()) {
#pragma unroll
        for (int u = 0; u < kSegLoads; ++u) {
            if (!item.has(u)) continue;
            Pack<4> yo, po, no;
#pragma unroll
            for (int q = 0; q < 4; ++q) po.v[q] = pre_value<true>(x[u].v[q], k, no.v[q]);
            act_apply_n<ACT>(po.v, yo.v);
            if constexpr (RES) {
#pragma unroll
                for (int q = 0; q < 4; ++q) yo.v[q] = with_residual(yo.v[q], r[u].v[q], a.res_alpha, a.res_beta);
            }
            const size_t at = item.at(u);
            const int held = item.held(u);
            if (a.x_saved) st_item<RAGGED, false>(a.x_saved, at, x[u], held);
            if (a.x_norm) st_item<RAGGED, false>(a.x_norm, at, no, held);
            if (a.pre) st_item<RAGGED, false>(a.pre, at, po, held);
            st_item<RAGGED, true>(a.y, at, yo, held);
        }
        item.next();
        fetch();
    }
}

struct BackwardFinish {
    const double2* partial;
    float *scale_updates, *bias_updates, *mean_delta, *var_delta;
    int count;
};

template<int ACT, bool RAGGED>
__global__ __launch_bounds__(kBlock) void bn_finish_dx_kernel(BackwardArgs a, ReduceGeom g, BackwardFinish f)
{
    __shared__ DxCoef shared_coef;
    uint32_t c, j;
    g.by_blocks.divmod(blockIdx.x, c, j);
    WaveItems<RAGGED> item(g, c, j);
    const bool recompute = a.pre == nullptr;
    Pack<4> d[kSegLoads], x[kSegLoads], pre[kSegLoads];
    const auto fetch = [&] {
#pragma unroll
        for (int u = 0; u < kSegLoads; ++u) {
            if (!item.has(u)) continue;
            d[u] = ld_at<4, false, RAGGED>(a.delta, item.at(u));
            x[u] = ld_at<4, false, RAGGED>(a.x, item.at(u));
            if constexpr (ACT != PXH_LINEAR) {
                if (!recompute) pre[u] = ld_at<4, false, RAGGED>(a.pre, item.at(u));
            }
        }
    };
    fetch();
    if (threadIdx.x < kWave) {
        const double2 sums = channel_sums(f.partial, c, g.blocks);
        if (threadIdx.x == 0) {
            if (j == 0) {
                shared_coef = finish_backward<true>(sums.x, sums.y, c, f.count, a.mean, a.var, a.scale, a.bias, f.scale_updates,
                                                    f.bias_updates, f.mean_delta, f.var_delta);
            } else {
                const float v = a.var[c], s = a.scale[c];
                shared_coef = finished_channel<true>(sums.x, sums.y, f.count, make_coef(a.mean[c], v, s, a.bias[c]), variance_terms(v), s).k;
            }
        }
    }
    __syncthreads();
    const DxCoef k = shared_coef;
    while (item.more()) {
#pragma unroll
        for (int u = 0; u < kSegLoads; ++u) {
            if (!item.has(u)) continue;
            if constexpr (ACT != PXH_LINEAR) {
                if (recompute) {
#pragma unroll
                    for (int q = 0; q < 4; ++q) pre[u].v[q] = affine(normalize(x[u].v[q], k.f), k.f);
                }
                times_grad<ACT>(d[u].v, pre[u].v);
            }
            Pack<4> out;
#pragma unroll
            for (int q = 0; q < 4; ++q) out.v[q] = dx_value(d[u].v[q], x[u].v[q], k);
            st_item<RAGGED, true>(a.delta, item.at(u), out, item.held(u));
        }
        item.next();
        fetch();
    }
}

constexpr size_t align256(size_t b) { return (b + 255) & ~static_cast<size_t>(255); }

// workspace: [partial sums][per-channel constants]
size_t partial_bytes(int batch, int channels, int spatial)
{
    const ReduceGeom g = make_geom(batch, channels, spatial);
    return align256(static_cast<size_t>(channels) * g.blocks * sizeof(double2));
}

// The most that partial_bytes() comes to for any shape up to this one: what the size functions report, so that a
// workspace sized once for the largest batch or plane serves every smaller one (the last, shorter batch of an epoch).
// partial_bytes() itself steps up where a smaller grid is split more finely: by halves of kItemsPerBlock, each time from
// fewer than kFillBlocks workgroups to less than twice as many, and never beyond one item to a wavefront.
size_t partial_bytes_up_to(int batch, int channels, int spatial)
{
    const ReduceGeom g = make_geom(batch, channels, spatial);
    const size_t c = static_cast<size_t>(channels), items = static_cast<size_t>(g.items);
    const auto blocks = [&](size_t per_block) { return c * ((items + per_block - 1) / per_block); };
    const size_t full = blocks(kItemsPerBlock), finest = blocks(kBlock / kWave);
    constexpr size_t kMostSplit = 2 * (kFillBlocks - 1);
    const size_t split = finest < kMostSplit ? finest : kMostSplit;
    return align256((full > split ? full : split) * sizeof(double2));
}

size_t workspace_bytes_with(size_t partial, int channels)
{
    return partial + static_cast<size_t>(channels) * sizeof(DxCoef);
}

size_t workspace_bytes(int batch, int channels, int spatial)
{
    return workspace_bytes_with(partial_bytes(batch, channels, spatial), channels);
}

void* coef_region(void* ws, int batch, int channels, int spatial)
{
    return static_cast<char*>(ws) + partial_bytes(batch, channels, spatial);
}

// The clipped backward: [partial sums][per-channel constants][norm partials][plan] for the three
// launches, [per-channel norm figures][per-channel sums][updates before][per-channel flags][plan] for the one-launch form.
struct ClippedRegions {
    double2* partial;
    DxCoef* coef;
    double2* norm_partial;
    double2* channel_norm;
    double2* channel_sums;
    float2* channel_before;
    int* channel_done;
    ClipPlan* plan;
};

// per-channel norm figures, sums, updates before and flags of the one-launch clipped backward
size_t figure_bytes(int channels)
{
    const size_t c = static_cast<size_t>(channels);
    return 2 * align256(c * sizeof(double2)) + align256(c * (sizeof(float2) + sizeof(int)));
}

// the same of a group: its members' words hold the sums
size_t group_figure_bytes(int channels)
{
    const size_t c = static_cast<size_t>(channels);
    return align256(c * sizeof(double2)) + align256(c * (sizeof(float2) + sizeof(int)));
}

size_t clipped_workspace_bytes_with(size_t partial, int channels)
{
    const size_t c = static_cast<size_t>(channels);
    const size_t three = 2 * partial + align256(c * sizeof(DxCoef)) + 256;
    const size_t one = figure_bytes(channels) + 256;
    return three > one ? three : one;
}

size_t clipped_workspace_bytes(int batch, int channels, int spatial)
{
    return clipped_workspace_bytes_with(partial_bytes(batch, channels, spatial), channels);
}

ClippedRegions clipped_regions(void* ws, int batch, int channels, int spatial)
{
    const size_t c = static_cast<size_t>(channels);
    char* base = static_cast<char*>(ws);
    ClippedRegions r;
    r.partial = reinterpret_cast<double2*>(base);
    r.coef = reinterpret_cast<DxCoef*>(base + partial_bytes(batch, channels, spatial));
    r.norm_partial = reinterpret_cast<double2*>(reinterpret_cast<char*>(r.coef) + align256(c * sizeof(DxCoef)));
    r.channel_norm = reinterpret_cast<double2*>(base);
    r.channel_sums = reinterpret_cast<double2*>(base + align256(c * sizeof(double2)));
    r.channel_before = reinterpret_cast<float2*>(base + 2 * align256(c * sizeof(double2)));
    r.channel_done = reinterpret_cast<int*>(base + 2 * align256(c * sizeof(double2)) + c * sizeof(float2));
    r.plan = reinterpret_cast<ClipPlan*>(base + clipped_workspace_bytes(batch, channels, spatial) - 256);
    return r;
}

constexpr int kGroupAlone = 512;

// The groups of a backward (members 0: none).  A plain call and a clipped one take the same form, so that they agree to
// the bit where nothing is rescaled or clamped, and what they exchange has to fit the workspaces they ask for.
//
// `per_thread` is what a workgroup of 1024 lanes would hold of a channel (0: more than it can).  Where it can, a plain call
// needs no workspace, and callers on several streams may pass none: groups that exchange something are not for those slices
// (16 x 128 x 76^2: 37 us where groups would take 33, mish 66 and 47).  A group of one member exchanges nothing, and from
// kGroupAlone channels on, two to a compute unit, it is ahead (16 x 512 x 38^2: 29 -> 27 us; 16 x 384 x 38^2 22.3, 22.6), except
// where an exponential has to be computed (37 -> 41).
GroupPlan grouped_backward(int batch, int channels, int spatial, bool vec, int per_thread, int activation, hipStream_t s)
{
    if (!enough_for_groups(static_cast<size_t>(batch) * channels * spatial, spatial, vec, activation)) return GroupPlan{};
    if (per_thread && (!selects(activation) || channels < kGroupAlone)) return GroupPlan{};
    const uint32_t places = group_places(s);
    // (as few members as hold the slice where the words of more would not fit: up to three channels of a few thousand vectors)
    for (const size_t workgroups: { group_fill(channels), static_cast<size_t>(1) }) {
        const GroupPlan p = group_plan(batch, channels, spatial, vec, workgroups, places);
        if (per_thread && p.members > 1) return GroupPlan{};
        if (p.members <= 1 ||
            (group_bytes(channels, p.members, kSumWords, false) <= workspace_bytes(batch, channels, spatial) &&
             group_figure_bytes(channels) + group_bytes(channels, p.members, kFirstWords, true) + 256 <=
                 clipped_workspace_bytes(batch, channels, spatial)))
            return p;
    }
    return GroupPlan{};
}

// A tensor this large cannot stay in the last-level cache between two passes over it.
bool streams_past_cache(uint32_t total, int tensors)
{
    return static_cast<size_t>(total) * 4 * tensors >= kStreamingBytes;
}

int launch_stats_partial(const float* x, const ReduceGeom& g, double2* partial, float* shifts, uint32_t total, hipStream_t stream)
{
    const dim3 grid(static_cast<unsigned>(g.channels) * g.blocks);
    const bool nt = streams_past_cache(total, 1);
    if (g.spatial % 4 == 0 && aligned16(x)) {
        if (nt) hipLaunchKernelGGL((bn_stats_partial_kernel<4, true>), grid, dim3(kBlock), 0, stream, x, g, partial, shifts);
        else hipLaunchKernelGGL((bn_stats_partial_kernel<4, false>), grid, dim3(kBlock), 0, stream, x, g, partial, shifts);
    } else if (sums_in_vectors(g.spatial)) {
        hipLaunchKernelGGL((bn_stats_partial_kernel<4, false, true>), grid, dim3(kBlock), 0, stream, x, g, partial, shifts);
    } else {
        hipLaunchKernelGGL((bn_stats_partial_kernel<1, false>), grid, dim3(kBlock), 0, stream, x, g, partial, shifts);
    }
    return check_launch("bn_stats_partial");
}

int launch_stats(const float* x, float* mean, float* var, float* rolling_mean, float* rolling_var, const float* scale,
                 const float* bias, FoldCoef* table, int batch, int channels, int spatial, uint32_t total, void* ws,
                 hipStream_t stream)
{
    const ReduceGeom g = make_geom(batch, channels, spatial);
    double2* partial = static_cast<double2*>(ws);
    const int rc = launch_stats_partial(x, g, partial, nullptr, total, stream);
    if (rc) return rc;
    hipLaunchKernelGGL(bn_stats_finish_kernel, dim3(grid_for(channels, kBlock / kWave)), dim3(kBlock), 0, stream, x,
                       partial, channels, spatial, g.blocks, static_cast<double>(batch) * spatial, mean, var,
                       rolling_mean, rolling_var, scale, bias, table);
    return check_launch("bn_stats_finish");
}

// Whether the pass behind the partial sums finishes the channels itself.
bool finishes_inside(const ReduceGeom& g, uint32_t total, uint32_t most)
{
    return total <= most && g.blocks <= kFusedPartials && g.spatial >= kFusedSpatial;
}

// The linear shortcut taken into a forward pass (from == nullptr: none).
struct Residual {
    const float* from = nullptr;
    float alpha = 1.0f, beta = 1.0f;
};

// BN training forward + activation.  `get_workspace(need, &ws)` is asked for the `need` bytes of the three-launch form
// where the shape takes that, and where it takes a one-launch form whose limits may move (asks_for_workspace).
template<typename GetWorkspace>
int bn_train_forward(const char* who, const float* x, float* y, float* pre_activation, float* x_saved, float* x_norm,
                     float* mean, float* var, float* rolling_mean, float* rolling_var, const float* scale,
                     const float* bias, int batch, int channels, int spatial, int activation,
                     GetWorkspace&& get_workspace, void* stream, const Residual& res = Residual{})
{
    if (!x || !y || !mean || !var || !rolling_mean || !rolling_var || !scale || !bias)
        return fail_invalid("%s: null pointer", who);
    if (x_saved == x) return fail_invalid("%s: x_saved must not alias x", who);
    EpilogueArgs a{};
    int rc = check_shape(who, batch, channels, spatial, &a.total);
    if (rc) return rc;
    hipStream_t s = as_stream(stream);
    const bool vec = spatial % 4 == 0 && aligned16(x) && aligned16(y) && aligned16(pre_activation) &&
                     aligned16(x_saved) && aligned16(x_norm) && aligned16(res.from);
    {
        if (const ResidentForm form = resident_form(batch, channels, spatial, vec, activation, false)) {
            const ResidentFwdArgs r{ x, y, pre_activation, x_saved, x_norm, mean, var, rolling_mean, rolling_var,
                                     scale, bias, resident_geom(batch, channels, spatial), res.from, res.alpha, res.beta };
            if (asks_for_workspace(batch, channels, spatial, vec)) {
                // not used, but still the caller's part of this shape (see above)
                void* unused;
                rc = get_workspace(workspace_bytes(batch, channels, spatial), &unused);
                if (rc) return rc;
            }
            return launch_resident_forward(who, r, form, activation, s);
        }
    }
    void* ws;
    rc = get_workspace(workspace_bytes(batch, channels, spatial), &ws);
    if (rc) return rc;
    a.x = x; a.y = y; a.pre = pre_activation; a.x_saved = x_saved; a.x_norm = x_norm;
    a.residual = res.from; a.res_alpha = res.alpha; a.res_beta = res.beta;
    const ReduceGeom g = make_geom(batch, channels, spatial);
    const bool chain = activation == PXH_SOFTPLUS || (activation == PXH_MISH && vec && !res.from);
    if (finishes_inside(g, a.total, chain ? kFusedForwardChain : kFusedForward)) {
        // (the first value of a channel, which its sums are relative to, is kept: y may be x)
        float* const shifts = static_cast<float*>(coef_region(ws, batch, channels, spatial));
        double2* const partial = static_cast<double2*>(ws);
        rc = launch_stats_partial(x, g, partial, shifts, a.total, s);
        if (rc) return rc;
        const StatsFinish f{ partial, shifts, static_cast<double>(batch) * spatial, mean, var, rolling_mean, rolling_var, scale, bias };
        const dim3 grid(static_cast<unsigned>(channels) * g.blocks);
        const auto launch = [&]<int ACT, bool RES>() {
            if (vec) hipLaunchKernelGGL((bn_finish_apply_kernel<ACT, RES, false>), grid, dim3(kBlock), 0, s, a, g, f);
            else hipLaunchKernelGGL((bn_finish_apply_kernel<ACT, RES, true>), grid, dim3(kBlock), 0, s, a, g, f);
        };
        const bool known = dispatch_activation(activation, [&]<int ACT>() {
            if (res.from) launch.template operator()<ACT, true>();
            else launch.template operator()<ACT, false>();
        });
        if (!known) return fail_invalid("%s: unknown activation %d", who, activation);
        return check_launch(who);
    }
    FoldCoef* table = static_cast<FoldCoef*>(coef_region(ws, batch, channels, spatial));
    rc = launch_stats(x, mean, var, rolling_mean, rolling_var, scale, bias, table, batch, channels, spatial, a.total,
                      ws, s);
    if (rc) return rc;
    a.table = table;
    a.by_spatial = FastDiv(spatial); a.by_channels = FastDiv(channels);
    return launch_epilogue_fwd<true>(who, a, activation, s);
}

}  // namespace
}  // namespace pxh

using namespace pxh;

extern "C" {

size_t pxh_bn_workspace_bytes(int batch, int channels, int spatial)
{
    if (batch <= 0 || channels <= 0 || spatial <= 0) return 0;
    return workspace_bytes_with(partial_bytes_up_to(batch, channels, spatial), channels);
}

size_t pxh_bn_folded_bytes(int channels)
{
    return channels > 0 ? static_cast<size_t>(channels) * sizeof(FoldCoef) : 0;
}

int pxh_bn_fold(const float* rolling_mean, const float* rolling_var, const float* scale, const float* bias,
                int channels, void* folded, void* stream)
{
    if (!rolling_mean || !rolling_var || !scale || !bias || !folded) return fail_invalid("pxh_bn_fold: null pointer");
    if (channels <= 0) return fail_invalid("pxh_bn_fold: channels must be positive");
    if (!aligned16(folded)) return fail_invalid("pxh_bn_fold: folded must be 16-byte aligned");
    hipLaunchKernelGGL(bn_fold_kernel, dim3(grid_for(channels, kBlock)), dim3(kBlock), 0, as_stream(stream),
                       rolling_mean, rolling_var, scale, bias, channels, static_cast<FoldCoef*>(folded));
    return check_launch("pxh_bn_fold");
}

int pxh_bn_folded_act_forward(const float* x, float* y, float* pre_activation, const void* folded, int batch,
                              int channels, int spatial, int activation, void* stream)
{
    if (!x || !y || !folded) return fail_invalid("pxh_bn_folded_act_forward: null pointer");
    if (!aligned16(folded)) return fail_invalid("pxh_bn_folded_act_forward: folded must be 16-byte aligned");
    EpilogueArgs a{};
    int rc = check_shape("pxh_bn_folded_act_forward", batch, channels, spatial, &a.total);
    if (rc) return rc;
    a.x = x; a.y = y; a.pre = pre_activation;
    a.table = static_cast<const FoldCoef*>(folded);
    a.by_spatial = FastDiv(spatial); a.by_channels = FastDiv(channels);
    return launch_epilogue_fwd<true>("pxh_bn_folded_act_forward", a, activation, as_stream(stream));
}

int pxh_bn_infer_act_forward(const float* x, float* y, float* pre_activation, const float* rolling_mean,
                             const float* rolling_var, const float* scale, const float* bias, int batch,
                             int channels, int spatial, int activation, void* workspace,
                             size_t workspace_bytes_given, void* stream)
{
    if (!x || !y || !rolling_mean || !rolling_var || !scale || !bias)
        return fail_invalid("pxh_bn_infer_act_forward: null pointer");
    uint32_t total;
    int rc = check_shape("pxh_bn_infer_act_forward", batch, channels, spatial, &total);
    if (rc) return rc;
    void* ws;
    rc = resolve_workspace(workspace, workspace_bytes_given, pxh_bn_folded_bytes(channels), &ws, as_stream(stream));
    if (rc) return rc;
    rc = pxh_bn_fold(rolling_mean, rolling_var, scale, bias, channels, ws, stream);
    if (rc) return rc;
    return pxh_bn_folded_act_forward(x, y, pre_activation, ws, batch, channels, spatial, activation, stream);
}

int pxh_bias_act_forward(const float* x, float* y, float* pre_activation, const float* bias, int batch,
                         int channels, int spatial, int activation, void* stream)
{
    if (!x || !y || !bias) return fail_invalid("pxh_bias_act_forward: null pointer");
    EpilogueArgs a{};
    int rc = check_shape("pxh_bias_act_forward", batch, channels, spatial, &a.total);
    if (rc) return rc;
    a.x = x; a.y = y; a.pre = pre_activation; a.bias = bias;
    a.by_spatial = FastDiv(spatial); a.by_channels = FastDiv(channels);
    return launch_epilogue_fwd<false>("pxh_bias_act_forward", a, activation, as_stream(stream));
}

int pxh_add_bias(float* output, const float* bias, int batch, int n, int size, void* stream)
{
    return pxh_bias_act_forward(output, output, nullptr, bias, batch, n, size, PXH_LINEAR, stream);
}

int pxh_bn_stats(const float* x, float* mean, float* var, int batch, int channels, int spatial, void* workspace,
                 size_t workspace_bytes_given, void* stream)
{
    if (!x || !mean || !var) return fail_invalid("pxh_bn_stats: null pointer");
    uint32_t total;
    int rc = check_shape("pxh_bn_stats", batch, channels, spatial, &total);
    if (rc) return rc;
    void* ws;
    rc = resolve_workspace(workspace, workspace_bytes_given, workspace_bytes(batch, channels, spatial), &ws, as_stream(stream));
    if (rc) return rc;
    return launch_stats(x, mean, var, nullptr, nullptr, nullptr, nullptr, nullptr, batch, channels, spatial, total,
                        ws, as_stream(stream));
}

int pxh_bn_train_act_forward(const float* x, float* y, float* pre_activation, float* x_saved, float* x_norm,
                             float* mean, float* var, float* rolling_mean, float* rolling_var, const float* scale,
                             const float* bias, int batch, int channels, int spatial, int activation,
                             void* workspace, size_t workspace_bytes_given, void* stream)
{
    return bn_train_forward(
        "pxh_bn_train_act_forward", x, y, pre_activation, x_saved, x_norm, mean, var, rolling_mean, rolling_var,
        scale, bias, batch, channels, spatial, activation,
        [&](size_t need, void** ws) { return resolve_workspace(workspace, workspace_bytes_given, need, ws, as_stream(stream)); }, stream);
}

int pxh_bn_train_act_shortcut_forward(const float* x, float* y, float* pre_activation, float* x_saved, float* x_norm,
                                      float* mean, float* var, float* rolling_mean, float* rolling_var,
                                      const float* scale, const float* bias, const float* from, float alpha, float beta,
                                      int batch, int channels, int spatial, int activation, void* workspace,
                                      size_t workspace_bytes_given, void* stream)
{
    const char* who = "pxh_bn_train_act_shortcut_forward";
    if (!from) return fail_invalid("%s: null pointer (from)", who);
    if (from == x_saved || from == x_norm || from == pre_activation)
        return fail_invalid("%s: from must not alias an output other than y", who);
    return bn_train_forward(
        who, x, y, pre_activation, x_saved, x_norm, mean, var, rolling_mean, rolling_var, scale, bias, batch, channels,
        spatial, activation,
        [&](size_t need, void** ws) { return resolve_workspace(workspace, workspace_bytes_given, need, ws, as_stream(stream)); },
        stream, Residual{ from, alpha, beta });
}

int pxh_bn_folded_act_shortcut_forward(const float* x, float* y, float* pre_activation, const void* folded,
                                       const float* from, float alpha, float beta, int batch, int channels,
                                       int spatial, int activation, void* stream)
{
    const char* who = "pxh_bn_folded_act_shortcut_forward";
    if (!x || !y || !folded || !from) return fail_invalid("%s: null pointer", who);
    if (!aligned16(folded)) return fail_invalid("%s: folded must be 16-byte aligned", who);
    if (from == pre_activation) return fail_invalid("%s: from must not alias an output other than y", who);
    EpilogueArgs a{};
    int rc = check_shape(who, batch, channels, spatial, &a.total);
    if (rc) return rc;
    a.x = x; a.y = y; a.pre = pre_activation;
    a.table = static_cast<const FoldCoef*>(folded);
    a.by_spatial = FastDiv(spatial); a.by_channels = FastDiv(channels);
    a.residual = from; a.res_alpha = alpha; a.res_beta = beta;
    return launch_epilogue_fwd<true>(who, a, activation, as_stream(stream));
}

int pxh_bn_folded_act_maxpool_forward(const float* x, float* y, float* pooled, const void* folded, int batch,
                                      int channels, int height, int width, int activation, void* stream)
{
    const char* who = "pxh_bn_folded_act_maxpool_forward";
    if (!x || !pooled || !folded) return fail_invalid("%s: null pointer", who);
    if (!aligned16(folded)) return fail_invalid("%s: folded must be 16-byte aligned", who);
    if (height <= 0 || width <= 0) return fail_invalid("%s: height and width must be positive", who);
    if (pooled == x || pooled == y) return fail_invalid("%s: the pooled output must be a tensor of its own", who);
    uint32_t total;
    int rc = check_shape(who, batch, channels, height * width, &total);
    if (rc) return rc;
    if (height % 2 || width % 2 || !aligned16(x) || !aligned16(y) || !aligned16(pooled)) {
        set_error("%s: windows that do not tile the plane (%d x %d) or tensors off a 16-byte boundary take the two "
                  "calls (pxh_bn_folded_act_forward, pxh_maxpool_forward)", who, height, width);
        return PXH_ERR_UNSUPPORTED;
    }
    const uint32_t oh = height / 2, ow = width / 2;
    EpiloguePoolArgs a{};
    a.x = x; a.y = y; a.pooled = pooled;
    a.table = static_cast<const FoldCoef*>(folded);
    a.iw = width; a.ow = ow;
    a.by_oh = FastDiv(oh); a.by_channels = FastDiv(channels);
    const uint32_t outputs = total / 4;
    // x in, the pooled quarter out, the layer's own output when asked for
    const bool nt = static_cast<size_t>(total) * (y ? 9 : 5) >= kStreamingBytes;
    hipStream_t s = as_stream(stream);
    const auto launch = [&]<int ACT, int VX>() {
        a.units = outputs / VX;
        a.by_owv = FastDiv(ow / VX);
        const dim3 grid(grid_for(a.units, kBlock));
        if (nt) hipLaunchKernelGGL((epilogue_pool2_fwd_kernel<ACT, VX, true>), grid, dim3(kBlock), 0, s, a);
        else hipLaunchKernelGGL((epilogue_pool2_fwd_kernel<ACT, VX, false>), grid, dim3(kBlock), 0, s, a);
    };
    const bool known = dispatch_activation(activation, [&]<int ACT>() {
        if (width % 8 == 0) launch.template operator()<ACT, 4>();
        else if (width % 4 == 0) launch.template operator()<ACT, 2>();
        else launch.template operator()<ACT, 1>();
    });
    if (!known) return fail_invalid("%s: unknown activation %d", who, activation);
    return check_launch(who);
}

int pxh_bn_train_act_forward_static(const float* x, float* y, float* pre_activation, float* x_saved, float* x_norm,
                                    float* mean, float* var, float* rolling_mean, float* rolling_var,
                                    const float* scale, const float* bias, int batch, int channels, int spatial,
                                    int activation, void* stream)
{
    const char* who = "pxh_bn_train_act_forward_static";
    return bn_train_forward(
        who, x, y, pre_activation, x_saved, x_norm, mean, var, rolling_mean, rolling_var, scale, bias, batch,
        channels, spatial, activation,
        [&](size_t need, void** ws) {
            if (need > kStaticScratchBytes) {
                set_error("%s: batch %d x channels %d x spatial %d needs %zu bytes of scratch, the built-in buffer "
                          "holds %zu; use pxh_bn_train_act_forward with a workspace of pxh_bn_workspace_bytes()",
                          who, batch, channels, spatial, need, kStaticScratchBytes);
                return PXH_ERR_WORKSPACE;
            }
            return static_scratch(who, ws);
        },
        stream);
}

// The rescale + clip in front of a backward, or none.
struct ClipSpec {
    bool on;
    float threshold, clip;
    float* norm_out;
};

static int bn_backward(const char* who, float* delta, const float* x, const float* pre_activation, const float* mean,
                       const float* var, const float* scale, const float* bias, float* scale_updates,
                       float* bias_updates, float* mean_delta, float* var_delta, int batch, int channels, int spatial,
                       int activation, const ClipSpec& cs, void* workspace, size_t workspace_bytes_given, void* stream)
{
    if (!delta || !x || !mean || !var || !scale || !bias || !scale_updates || !bias_updates)
        return fail_invalid("%s: null pointer", who);
    uint32_t total;
    int rc = check_shape(who, batch, channels, spatial, &total);
    if (rc) return rc;
    hipStream_t s = as_stream(stream);
    const bool rvec = spatial % 4 == 0 && aligned16(delta) && aligned16(x) && aligned16(pre_activation);
    const ResidentForm form = resident_form(batch, channels, spatial, rvec, activation, true);
    const bool asks = asks_for_workspace(batch, channels, spatial, rvec);
    void* ws = nullptr;
    ClippedRegions region{};
    ClipArgs clip{};
    if (cs.on) {
        rc = resolve_workspace(workspace, workspace_bytes_given, clipped_workspace_bytes(batch, channels, spatial), &ws, s);
        if (rc) return rc;
        region = clipped_regions(ws, batch, channels, spatial);
        clip = ClipArgs{ region.norm_partial, region.plan, cs.threshold, cs.clip, cs.norm_out };
    }
    GroupPlan group{};
    // (a saved pre-activation is a third stream, which no register is left for)
    if (!form.small && !form.odd && !pre_activation)
        group = grouped_backward(batch, channels, spatial, rvec, form.per_thread, activation, s);
    if (group.members) {
        const bool exchanges = group.members > 1;
        if (!cs.on && asks) {
            rc = resolve_workspace(workspace, workspace_bytes_given, workspace_bytes(batch, channels, spatial), &ws, s);
            if (rc) return rc;
        }
        GroupGeom g = group_geom(group, batch, channels, spatial);
        if (exchanges) {
            rc = start_exchange(who, g, static_cast<char*>(ws) + (cs.on ? group_figure_bytes(channels) : 0),
                                cs.on ? kFirstWords : kSumWords, cs.on, s);
            if (rc) return rc;
        }
        if (exchanges && cs.on) {
            // no sums: the members' words hold them
            char* const base = reinterpret_cast<char*>(region.channel_sums);
            region.channel_before = reinterpret_cast<float2*>(base);
            region.channel_done = reinterpret_cast<int*>(base + static_cast<size_t>(channels) * sizeof(float2));
        }
        const ResidentBwdArgs r{ BackwardArgs{ delta, x, nullptr, mean, var, scale, bias }, scale_updates,
                                 bias_updates, mean_delta, var_delta, g.g, region.channel_norm, region.channel_sums,
                                 region.channel_before, region.channel_done, clip };
        return launch_grouped_backward(who, r, g, group.places, cs.on, rvec, activation, s);
    }
    if (form) {
        if (!cs.on && asks) {
            // not used, but still the caller's part of this shape (as in the forward)
            rc = resolve_workspace(workspace, workspace_bytes_given, workspace_bytes(batch, channels, spatial), &ws, s);
            if (rc) return rc;
        }
        const ResidentBwdArgs r{ BackwardArgs{ delta, x, pre_activation, mean, var, scale, bias }, scale_updates,
                                 bias_updates, mean_delta, var_delta, resident_geom(batch, channels, spatial),
                                 region.channel_norm, region.channel_sums, region.channel_before, region.channel_done,
                                 clip };
        return launch_resident_backward(who, r, cs.on, form, activation, s);
    }
    if (!cs.on) {
        rc = resolve_workspace(workspace, workspace_bytes_given, workspace_bytes(batch, channels, spatial), &ws, s);
        if (rc) return rc;
    }
    const ReduceGeom g = make_geom(batch, channels, spatial);
    double2* partial = static_cast<double2*>(ws);
    DxCoef* coef = static_cast<DxCoef*>(coef_region(ws, batch, channels, spatial));

    BackwardArgs b{ delta, x, pre_activation, mean, var, scale, bias };
    const bool vec = rvec;
    const int tensors = pre_activation ? 3 : 2;
    const bool nt = vec && streams_past_cache(total, tensors);
    const dim3 grid(static_cast<unsigned>(channels) * g.blocks);
    const dim3 finish_grid(grid_for(channels, kBlock / kWave));
    const auto sums = [&]<int ACT, int MODE>() {
        if (nt) {
            hipLaunchKernelGGL((bwd_partial_kernel<ACT, true, false, 4, true, MODE>), grid, dim3(kBlock), 0, s, b, g,
                               partial, clip);
        } else if (vec) {
            hipLaunchKernelGGL((bwd_partial_kernel<ACT, true, false, 4, false, MODE>), grid, dim3(kBlock), 0, s, b, g,
                               partial, clip);
        } else if (sums_in_vectors(spatial, activation)) {
            hipLaunchKernelGGL((bwd_partial_kernel<ACT, true, false, 4, false, MODE, true>), grid, dim3(kBlock), 0, s, b, g,
                               partial, clip);
        } else {
            hipLaunchKernelGGL((bwd_partial_kernel<ACT, true, false, 1, false, MODE>), grid, dim3(kBlock), 0, s, b, g,
                               partial, clip);
        }
    };
    const auto finish = [&]<int MODE>() {
        if constexpr (MODE == kFirst)
            hipLaunchKernelGGL((bwd_finish_kernel<true, MODE, kPlanThreads>), dim3(grid_for(channels, kPlanThreads / kWave)),
                               dim3(kPlanThreads), 0, s, partial, channels, g.blocks, batch * spatial, mean, var, scale,
                               bias, scale_updates, bias_updates, mean_delta, var_delta, coef, clip);
        else
            hipLaunchKernelGGL((bwd_finish_kernel<true, MODE>), finish_grid, dim3(kBlock), 0, s, partial, channels,
                               g.blocks, batch * spatial, mean, var, scale, bias, scale_updates, bias_updates,
                               mean_delta, var_delta, coef, clip);
    };
    const bool known = dispatch_activation(activation, [&]<int ACT>() {
        if (!cs.on) {
            sums.template operator()<ACT, kPlain>();
        } else {
            sums.template operator()<ACT, kFirst>();
            finish.template operator()<kFirst>();
            sums.template operator()<ACT, kRedo>();
        }
    });
    if (!known) return fail_invalid("%s: unknown activation %d", who, activation);
    rc = check_launch("bn_backward_partial");
    if (rc) return rc;
    if (!cs.on && finishes_inside(g, total, kFusedBackward)) {
        const BackwardFinish f{ partial, scale_updates, bias_updates, mean_delta, var_delta, batch * spatial };
        dispatch_activation(activation, [&]<int ACT>() {
            if (vec) hipLaunchKernelGGL((bn_finish_dx_kernel<ACT, false>), grid, dim3(kBlock), 0, s, b, g, f);
            else hipLaunchKernelGGL((bn_finish_dx_kernel<ACT, true>), grid, dim3(kBlock), 0, s, b, g, f);
        });
        return check_launch("bn_backward_finish_dx");
    }
    if (cs.on) finish.template operator()<kRedo>();
    else finish.template operator()<kPlain>();
    rc = check_launch("bn_backward_finish");
    if (rc) return rc;

    DxArgs d{};
    d.delta = delta; d.x = x; d.pre = pre_activation; d.coef = coef;
    d.by_spatial = FastDiv(spatial); d.by_channels = FastDiv(channels); d.total = total;
    d.plan = cs.on ? region.plan : nullptr;
    const bool dx_vec = aligned16(delta) && aligned16(x) && aligned16(pre_activation);
    const bool dx_nt = streams_past_cache(total, tensors + 1);
    const auto dx = [&]<int ACT, bool CLIPPED>() {
        if (dx_vec) {
            const dim3 dx_grid(grid_for(total, static_cast<size_t>(kBlock) * 4));
            if (dx_nt) hipLaunchKernelGGL((bn_dx_kernel<ACT, true, CLIPPED>), dx_grid, dim3(kBlock), 0, s, d);
            else hipLaunchKernelGGL((bn_dx_kernel<ACT, false, CLIPPED>), dx_grid, dim3(kBlock), 0, s, d);
        } else {
            hipLaunchKernelGGL((bn_dx_scalar_kernel<ACT, CLIPPED>), dim3(grid_for(total, kBlock)), dim3(kBlock), 0, s, d);
        }
    };
    dispatch_activation(activation, [&]<int ACT>() {
        if (cs.on) dx.template operator()<ACT, true>();
        else dx.template operator()<ACT, false>();
    });
    return check_launch("bn_backward_dx");
}

int pxh_bn_act_backward(float* delta, const float* x, const float* pre_activation, const float* mean,
                        const float* var, const float* scale, const float* bias, float* scale_updates,
                        float* bias_updates, float* mean_delta, float* var_delta, int batch, int channels,
                        int spatial, int activation, void* workspace, size_t workspace_bytes_given, void* stream)
{
    return bn_backward("pxh_bn_act_backward", delta, x, pre_activation, mean, var, scale, bias, scale_updates,
                       bias_updates, mean_delta, var_delta, batch, channels, spatial, activation,
                       ClipSpec{ false, 0.0f, 0.0f, nullptr }, workspace, workspace_bytes_given, stream);
}

size_t pxh_bn_clipped_workspace_bytes(int batch, int channels, int spatial)
{
    if (batch <= 0 || channels <= 0 || spatial <= 0) return 0;
    return clipped_workspace_bytes_with(partial_bytes_up_to(batch, channels, spatial), channels);
}

int pxh_bn_act_backward_clipped(float* delta, const float* x, const float* pre_activation, const float* mean,
                                const float* var, const float* scale, const float* bias, float* scale_updates,
                                float* bias_updates, float* mean_delta, float* var_delta, int batch, int channels,
                                int spatial, int activation, float threshold, float clip, float* norm_out,
                                void* workspace, size_t workspace_bytes_given, void* stream)
{
    return bn_backward("pxh_bn_act_backward_clipped", delta, x, pre_activation, mean, var, scale, bias, scale_updates,
                       bias_updates, mean_delta, var_delta, batch, channels, spatial, activation,
                       ClipSpec{ true, threshold, clip, norm_out }, workspace, workspace_bytes_given, stream);
}

static int bias_backward(const char* who, float* delta, const float* pre_activation, float* bias_updates, int batch,
                         int channels, int spatial, int activation, const ClipSpec& cs, void* workspace,
                         size_t workspace_bytes_given, void* stream)
{
    if (!delta || !bias_updates) return fail_invalid("%s: null pointer", who);
    if (activation != PXH_LINEAR && !pre_activation)
        return fail_invalid("%s: pre_activation is required for a non-linear activation", who);
    uint32_t total;
    int rc = check_shape(who, batch, channels, spatial, &total);
    if (rc) return rc;
    hipStream_t s = as_stream(stream);
    void* ws;
    rc = resolve_workspace(workspace, workspace_bytes_given,
                           cs.on ? clipped_workspace_bytes(batch, channels, spatial)
                                 : workspace_bytes(batch, channels, spatial), &ws, s);
    if (rc) return rc;
    const ReduceGeom g = make_geom(batch, channels, spatial);
    double2* partial = static_cast<double2*>(ws);
    ClipArgs clip{};
    if (cs.on) {
        const ClippedRegions region = clipped_regions(ws, batch, channels, spatial);
        clip = ClipArgs{ region.norm_partial, region.plan, cs.threshold, cs.clip, cs.norm_out };
    }
    BackwardArgs b{ delta, nullptr, pre_activation, nullptr, nullptr, nullptr, nullptr };
    const bool vec = spatial % 4 == 0 && aligned16(delta) && aligned16(pre_activation);
    const dim3 grid(static_cast<unsigned>(channels) * g.blocks);
    const dim3 finish_grid(grid_for(channels, kBlock / kWave));
    const auto sums = [&]<int ACT, bool WRITE, int MODE>() {
        if (vec) {
            hipLaunchKernelGGL((bwd_partial_kernel<ACT, false, WRITE, 4, false, MODE>), grid, dim3(kBlock), 0, s, b, g,
                               partial, clip);
        } else if (sums_in_vectors(spatial, activation)) {
            hipLaunchKernelGGL((bwd_partial_kernel<ACT, false, WRITE, 4, false, MODE, true>), grid, dim3(kBlock), 0, s, b, g,
                               partial, clip);
        } else {
            hipLaunchKernelGGL((bwd_partial_kernel<ACT, false, WRITE, 1, false, MODE>), grid, dim3(kBlock), 0, s, b, g,
                               partial, clip);
        }
    };
    const auto finish = [&]<int MODE>() {
        if constexpr (MODE == kFirst)
            hipLaunchKernelGGL((bwd_finish_kernel<false, MODE, kPlanThreads>), dim3(grid_for(channels, kPlanThreads / kWave)),
                               dim3(kPlanThreads), 0, s, partial, channels, g.blocks, batch * spatial, nullptr, nullptr,
                               nullptr, nullptr, nullptr, bias_updates, nullptr, nullptr, nullptr, clip);
        else
            hipLaunchKernelGGL((bwd_finish_kernel<false, MODE>), finish_grid, dim3(kBlock), 0, s, partial, channels,
                               g.blocks, batch * spatial, nullptr, nullptr, nullptr, nullptr, nullptr, bias_updates,
                               nullptr, nullptr, nullptr, clip);
    };
    const bool known = dispatch_activation(activation, [&]<int ACT>() {
        if (!cs.on) {
            sums.template operator()<ACT, true, kPlain>();
        } else {
            // the sums of the delta as it came (nothing written), the plan, then the pass that writes:
            // it leaves at once when nothing changes and the activation is linear
            sums.template operator()<ACT, false, kFirst>();
            finish.template operator()<kFirst>();
            sums.template operator()<ACT, true, kRedo>();
        }
    });
    if (!known) return fail_invalid("%s: unknown activation %d", who, activation);
    rc = check_launch("bias_backward_partial");
    if (rc) return rc;
    if (cs.on) finish.template operator()<kRedo>();
    else finish.template operator()<kPlain>();
    return check_launch("bias_backward_finish");
}

int pxh_bias_act_backward(float* delta, const float* pre_activation, float* bias_updates, int batch, int channels,
                          int spatial, int activation, void* workspace, size_t workspace_bytes_given, void* stream)
{
    return bias_backward("pxh_bias_act_backward", delta, pre_activation, bias_updates, batch, channels, spatial,
                         activation, ClipSpec{ false, 0.0f, 0.0f, nullptr }, workspace, workspace_bytes_given, stream);
}

int pxh_bias_act_backward_clipped(float* delta, const float* pre_activation, float* bias_updates, int batch,
                                  int channels, int spatial, int activation, float threshold, float clip,
                                  float* norm_out, void* workspace, size_t workspace_bytes_given, void* stream)
{
    return bias_backward("pxh_bias_act_backward_clipped", delta, pre_activation, bias_updates, batch, channels,
                         spatial, activation, ClipSpec{ true, threshold, clip, norm_out }, workspace,
                         workspace_bytes_given, stream);
}

int pxh_backward_bias(float* bias_updates, const float* delta, int batch, int n, int size, void* workspace,
                      size_t workspace_bytes_given, void* stream)
{
    // delta is only read on the linear path
    return pxh_bias_act_backward(const_cast<float*>(delta), nullptr, bias_updates, batch, n, size, PXH_LINEAR,
                                 workspace, workspace_bytes_given, stream);
}

}
