// The one-launch training passes: what their kernels share, which shapes take them, and their launches.
#pragma once

#include "batchnorm.h"

namespace pxh {

// ---------------------------------------------------------------- channel-resident training passes
// For a tensor whose per-channel slice (batch * spatial floats) fits the registers of one
// workgroup, the three launches of epilogue.hip (partial sums, finish, apply) collapse into one: workgroup c
// holds channel c, reduces it, finishes the statistics and applies them.  The tensor is read from
// memory once, and a small layer costs one launch instead of three.
constexpr int kResidentThreads = 1024;
// The scalar forms also come with workgroups of half the size, four to a compute unit instead of two:
// for the layers with a thousand channels of 19 x 19, whose workgroups would otherwise run in two rounds.
constexpr int kResidentNarrowThreads = 512;
constexpr int kResidentVectors = 8;            // per lane of the forms without an LDS part

// Sum of two doubles over the workgroup; every thread returns both totals.
template<int T>
__device__ __forceinline__ void resident_sum2(double& a, double& b, double (*slots)[T / kWave])
{
    a = wave_sum(a);
    b = wave_sum(b);
    const int lane = threadIdx.x & (kWave - 1);
    const int wave = threadIdx.x / kWave;
    __syncthreads();
    if (lane == 0) {
        slots[0][wave] = a;
        slots[1][wave] = b;
    }
    __syncthreads();
    double ta = 0.0, tb = 0.0;
#pragma unroll
    for (int w = 0; w < T / kWave; ++w) {
        ta += slots[0][w];
        tb += slots[1][w];
    }
    a = ta;
    b = tb;
}

// The same for a workgroup of half the size whose thread t stands in for threads t and t + T of a workgroup
// of 2 T threads (sums a of the first, b of the second): the additions of resident_sum2<2 * T>, in its order.
template<int T>
__device__ __forceinline__ void resident_sum2_twin(double& a1, double& a2, double b1, double b2,
                                                   double (*slots)[2 * T / kWave])
{
    a1 = wave_sum(a1);
    a2 = wave_sum(a2);
    b1 = wave_sum(b1);
    b2 = wave_sum(b2);
    const int lane = threadIdx.x & (kWave - 1);
    const int wave = threadIdx.x / kWave;
    __syncthreads();
    if (lane == 0) {
        slots[0][wave] = a1;
        slots[1][wave] = a2;
        slots[0][wave + T / kWave] = b1;
        slots[1][wave + T / kWave] = b2;
    }
    __syncthreads();
    double ta = 0.0, tb = 0.0;
#pragma unroll
    for (int w = 0; w < 2 * T / kWave; ++w) {
        ta += slots[0][w];
        tb += slots[1][w];
    }
    a1 = ta;
    a2 = tb;
}

// The same for three sums and a maximum (the first pass of a clipped backward).
template<int T>
__device__ __forceinline__ void resident_sum3_max(double& a, double& b, double& q, float& top,
                                                  double (*slots)[T / kWave], float* tops)
{
    a = wave_sum(a);
    b = wave_sum(b);
    q = wave_sum(q);
    top = wave_max(top);
    const int lane = threadIdx.x & (kWave - 1);
    const int wave = threadIdx.x / kWave;
    __syncthreads();
    if (lane == 0) {
        slots[0][wave] = a;
        slots[1][wave] = b;
        slots[2][wave] = q;
        tops[wave] = top;
    }
    __syncthreads();
    double ta = 0.0, tb = 0.0, tq = 0.0;
    float tt = 0.0f;
    // four waves' figures at a time: all sixteen at once are 100 registers of LDS loads in flight
#pragma unroll 4
    for (int w = 0; w < T / kWave; ++w) {
        ta += slots[0][w];
        tb += slots[1][w];
        tq += slots[2][w];
        tt = fmaxf(tt, tops[w]);
    }
    a = ta;
    b = tb;
    q = tq;
    top = tt;
}

struct ResidentGeom {
    int channels, spatial;
    uint32_t per_channel;     // batch * spatial
    FastDiv by_spatial;
    // offset of element e of channel c's slice (e counts through the images)
    __device__ __forceinline__ size_t at(uint32_t c, uint32_t e) const
    {
        uint32_t n, r;
        by_spatial.divmod(e, n, r);
        return (static_cast<size_t>(n) * channels + c) * spatial + r;
    }
};

// The sums of a slice: fp32 per lane, except in the scalar forms that hold more than kResidentVectors values per lane.
// Those shapes otherwise take three launches, which add a lane's share of one image in fp32 (three values of a 13 x 13
// plane, one of a plane of up to 64) and carry on in doubles; sixteen or twenty-four values in fp32 lose two to three
// times as much.  Here two values are added in fp32 where the three launches add as many or more, none where they add
// fewer, and everything beyond in doubles.  Against fp32 throughout, forward and backward, us: 64 x 256 x 13^2 8.5 -> 8.7
// and 11.6 -> 11.8, 64 x 1024 x 13^2 27.6 -> 27.7 and 37.3 -> 38.6.  (Every value into a double of its own: 9.1 and 12.1,
// 28.2 and 39.0.)
template<int V, int R, int L, int T>
constexpr bool kWideSlice = V == 1 && (R + L) * T > kResidentVectors * kResidentThreads;
constexpr int kPairSpatial = 2 * kWave;        // from this plane on a lane of the three launches adds two values and more

__device__ __forceinline__ void add_two(double& sum, float v, float w, bool pair)
{
    if (pair) {
        sum += static_cast<double>(v + w);
    } else {
        asm volatile("" : "+v"(v));     // a branch, not both ways and a choice: `pair` is the same for every lane
        sum += static_cast<double>(v);
        sum += static_cast<double>(w);
    }
}

// The small forms (small_slice below): a lane adds the values of a vector in fp32 and its vectors in doubles -- no further
// from 64 bits than a lane of the other forms that holds one vector -- and the backward keeps x beside the delta.
template<int V, int R, int L, int T>
constexpr bool kSmallSlice = L == 0 && T < kResidentThreads && V * R <= (V == 4 ? 32 : 12);

// A thread keeps R vectors in registers and L more in LDS (dynamic, L * kResidentThreads vectors:
// thread-major, so every access is the conflict-free 128-bit one).
template<int V, int R>
__device__ __forceinline__ Pack<V>* resident_lds_slot(float* lds, int r)
{
    return reinterpret_cast<Pack<V>*>(lds) + static_cast<size_t>(r - R) * kResidentThreads + threadIdx.x;
}

struct ResidentFwdArgs {
    const float* x;
    float* y;
    float* pre;        // nullable
    float* x_saved;    // nullable
    float* x_norm;     // nullable
    float* mean;
    float* var;
    float* rolling_mean;
    float* rolling_var;
    const float* scale;
    const float* bias;
    ResidentGeom g;
    // the shortcut that follows the layer (else null), as in EpilogueArgs
    const float* residual;
    float res_alpha, res_beta;
};

struct ResidentBwdArgs {
    BackwardArgs b;
    float* scale_updates;
    float* bias_updates;
    float* mean_delta;   // nullable
    float* var_delta;    // nullable
    ResidentGeom g;
    // the clipped form (else null): per channel the (sum of squares, largest magnitude) of its delta,
    // the two sums it was finished with, its bias and scale updates before that, and whether it was
    // finished at all
    double2* channel_norm;
    double2* channel_sums;
    float2* channel_before;
    int* channel_done;
    ClipArgs clip;
};

// Vectors per thread the resident kernels are built for, and whether a shape takes that path:
// the channel slice must fit, and there must be enough channels to occupy the machine.  (Measured
// with 24 vectors per thread: the registers spill and 128 workgroups of 16x128x76^2 are slower than
// the three launches; with a third of them in LDS they do not.)
// The forms without an LDS part hold kResidentVectors (above);
// the large form (128-bit vectors only) 16 vectors in registers + 8 in LDS (128 KB of the CU's 160)
constexpr int kResidentLargeRegs = 16, kResidentLargeLds = 8;
constexpr size_t kResidentLargeLdsBytes = static_cast<size_t>(kResidentLargeLds) * kResidentThreads * 16;
// The scalar forms (odd planes) with more values per lane: 16 in 64 registers, two workgroups per compute unit; the
// backward also 24 in 128 registers.  Against the three launches, us:
//                       forward        + shortcut     backward
//   64 x 256 x 13^2     15.2 ->  8.7   16.0 -> 11.8   21.8 -> 11.8   leaky
//   64 x 512 x 13^2     22.1 -> 14.4   24.1 -> 17.6   32.0 -> 18.5
//   49 x 1024 x 13^2    31.4 -> 23.5   35.7 -> 30.0   43.2 -> 32.1
//   64 x 1024 x 13^2    36.5 -> 27.7   41.7 -> 38.4   49.1 -> 38.6
//   32 x 1024 x 19^2    29.9 -> 27.4   41.6 -> 35.8   49.7 -> 37.2
//   64 x 512 x 19^2     29.7 -> 28.3   38.9 -> 54.0   49.9 -> 36.6   24 values
//   64 x 256 x 13^2     15.7 -> 12.1   16.4 -> 13.4   28.5 -> 20.8   mish
//   64 x 512 x 13^2     22.7 -> 19.2   25.1 -> 21.4   40.4 -> 35.8
//   32 x 1024 x 19^2    30.8 -> 37.1   39.6 -> 52.4   64.8 -> 66.5
//   64 x 512 x 19^2     30.1 -> 34.7   40.3 -> 64.3   64.5 -> 61.8   24 values
// An activation with an exponential leaves a workgroup that waits for its own channel more to do after the wait, and a
// thousand channels keep the three launches' many small workgroups busy: it takes the one-launch form only up to 512
// channels, and 24 values only where the backward's gradient is a select.  (Forward with 24 values the shortcut would
// lose, and a layer has the same statistics to the bit with and without one: no such form.)
constexpr int kResidentScalarMid = 16, kResidentScalarWide = 24;
constexpr int kResidentScalarFew = 512;
// Beyond this the riding form runs two workgroups to a compute unit (64 x 512 x 13^2, leaky: 17.6 against 20.7 us); up to
// it every channel finds a compute unit of its own, and the form that keeps its addresses is ahead (64 x 256 x 13^2: 11.2
// against 11.8, mish 12.6 against 14.2).
constexpr int kResidentTight = 256;

constexpr bool selects(int activation)
{
    return activation == PXH_LEAKY || activation == PXH_RELU || activation == PXH_LINEAR;
}

constexpr int kResidentChannels = 96;

// The small forms.  A launch over short slices is one chain -- the loads, the sums across the workgroup, the thread that
// finishes the channel, the stores -- and a workgroup of 1024 lanes that holds 50 vectors walks it at the pace of its
// sixteen waves: seven of the eight steps of a lane are loads of nothing, and a thousand such workgroups run in two rounds.
// Few lanes with two to eight steps each shorten every link; what the backward's finish takes from the variance alone is
// formed while the slice is on its way (0.5 us of each backward).  Against workgroups of 1024 lanes (from 96 channels on)
// or three launches, us, leaky: forward, forward + shortcut, backward, backward with rescale + clip
//   2 x 1024 x 10^2    12.8 -> 4.1   12.4 -> 4.2   11.3 -> 4.9   20.0 ->  8.0     64 lanes, 2 vectors
//   2 x 512 x 20^2      7.9 -> 4.0    7.7 -> 4.3    7.1 -> 4.7   13.0 ->  7.8    128 lanes, 2
//   2 x 256 x 40^2      6.1 -> 4.5    6.4 -> 4.7    6.7 -> 5.4   11.2 ->  8.1    256 lanes, 4
//   8 x 512 x 26^2      9.2 -> 6.6    9.6 -> 7.8   10.7 -> 9.0   16.4 -> 12.4    512 lanes, 4
//   2 x 128 x 80^2      6.8 -> 6.0    7.7 -> 6.2    9.0 -> 8.0   13.4 -> 11.1    512 lanes, 8
//   1 x 64 x 104^2      9.6 -> 5.5   10.8 -> 5.6   13.4 -> 7.3   19.1 -> 10.6    (three launches before)
//   1 x 1024 x 13^2     8.4 -> 3.9   11.2 -> 4.0   11.9 -> 4.8   17.7 ->  8.3     64 lanes, 4 values
//   4 x 1024 x 13^2     9.0 -> 5.3   11.8 -> 5.4   12.8 -> 6.1   17.5 ->  9.6    256 lanes, 4
//   8 x 512 x 19^2      7.1 -> 6.0    8.3 -> 6.7   10.1 -> 7.9   14.8 -> 11.2    512 lanes, 8
//   16 x 512 x 19^2     8.3 -> 7.7   10.5 -> 10.3  11.2 -> 10.6  16.3 -> 13.8    512 lanes, 12
//   16 x 1024 x 19^2   14.1 -> 13.8  19.5 -> 19.6  19.1 -> 19.3  23.2 -> 23.3
// With more lanes at the same capacity each is slower (2 x 1024 x 10^2 in 128, 256, 512 lanes: backward 4.7, 6.5, 10.0).
// Eight vectors a lane take a workgroup's 256 registers a lane, one to a compute unit: up to as many channels only
// (4 x 512 x 52^2, leaky: backward 16.5 us against 14.2).  An activation with an exponential is bound by its gradient, and
// there the waves count: beyond 512 vectors a slice its backward keeps the full workgroups where it has them
// (8 x 256 x 38^2, mish: 15.5 us against 13.4; 2 x 256 x 40^2: 8.5 against 8.0; 2 x 512 x 20^2: 6.4 against 7.8).
constexpr uint32_t kSmallVectors = 4096, kSmallScalars = 6144;
constexpr uint32_t kSmallVectorsMany = 2048;      // beyond kSmallChannels channels
constexpr int kSmallChannels = 256;
constexpr uint32_t kSmallVectorsSmooth = 512;

// The vectors (or scalars) of a channel's slice where the shape takes a small form, else 0.
inline uint32_t small_slice(int batch, int channels, int spatial, bool vec, int activation, bool backward)
{
    const size_t per_channel = static_cast<size_t>(batch) * spatial;
    const size_t items = vec ? per_channel / 4 : per_channel;
    size_t most = !vec ? kSmallScalars : channels <= kSmallChannels ? kSmallVectors : kSmallVectorsMany;
    if (vec && backward && !selects(activation) && channels >= kResidentChannels) most = kSmallVectorsSmooth;
    return items <= most ? static_cast<uint32_t>(items) : 0;
}

// Calls launch.operator()<V, R, T>() with the form for `items`: vectors or scalars, steps per lane, lanes.
template<typename F>
void dispatch_small_form(bool vec, uint32_t items, F&& launch)
{
    if (vec) {
        if (items <= 64 * 2) return launch.template operator()<4, 2, 64>();
        if (items <= 128 * 2) return launch.template operator()<4, 2, 128>();
        if (items <= 256 * 4) return launch.template operator()<4, 4, 256>();
        if (items <= 512 * 4) return launch.template operator()<4, 4, 512>();
        return launch.template operator()<4, 8, 512>();
    }
    if (items <= 64 * 4) return launch.template operator()<1, 4, 64>();
    if (items <= 256 * 4) return launch.template operator()<1, 4, 256>();
    if (items <= 256 * 8) return launch.template operator()<1, 8, 256>();
    if (items <= 512 * 8) return launch.template operator()<1, 8, 512>();
    return launch.template operator()<1, 12, 512>();
}

inline int resident_vectors(int batch, int channels, int spatial, bool vec, int activation, bool backward)
{
    if (channels < kResidentChannels) return 0;
    const size_t per_channel = static_cast<size_t>(batch) * spatial;
    const size_t vectors = (per_channel + (vec ? 3 : 0)) / (vec ? 4 : 1);
    const size_t per_thread = (vectors + kResidentThreads - 1) / kResidentThreads;
    if (per_thread <= kResidentVectors) return kResidentVectors;
    if (vec) return per_thread <= kResidentLargeRegs + kResidentLargeLds ? kResidentLargeRegs + kResidentLargeLds : 0;
    const bool light = selects(activation);
    if (per_thread <= kResidentScalarMid && (light || channels <= kResidentScalarFew)) return kResidentScalarMid;
    if (per_thread <= kResidentScalarWide && light && backward) return kResidentScalarWide;
    return 0;
}

// The scalar form with workgroups of kResidentNarrowThreads (twice the values per thread): when the full
// workgroups would outnumber the two places a compute unit has for them.  Measured at 16 x 1024 x 19^2:
// forward 14.6 against 16.3 us, backward 23.1 against 26.5; at 512 channels the forward gains 5 %, the
// backward loses 20 %.
constexpr int kResidentNarrowVectors = 2 * kResidentVectors;
inline bool resident_narrow(const ResidentGeom& g, int per_thread, bool vec, bool backward)
{
    if (vec || per_thread != kResidentVectors || g.channels < (backward ? 1024 : 512)) return false;
    return (g.per_channel + kResidentNarrowThreads - 1) / kResidentNarrowThreads <= kResidentNarrowVectors;
}

inline ResidentGeom resident_geom(int batch, int channels, int spatial)
{
    return ResidentGeom{ channels, spatial, static_cast<uint32_t>(batch) * static_cast<uint32_t>(spatial),
                         FastDiv(static_cast<uint32_t>(spatial)) };
}

// A kernel that asks for more than 64 KB of dynamic LDS has to be allowed to, once.
int allow_large_lds(const void* kernel);

// `per_thread`: resident_vectors() of the shape, `small`: small_slice().
int launch_resident_forward(const char* who, const ResidentFwdArgs& r, bool vec, int per_thread, uint32_t small,
                            int activation, hipStream_t s);
int launch_resident_backward(const char* who, const ResidentBwdArgs& r, bool clipped, bool vec, int per_thread,
                             uint32_t small, int activation, hipStream_t s);

}  // namespace pxh
