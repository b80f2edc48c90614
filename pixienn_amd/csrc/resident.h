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
// Workgroups of half the size: the 128-bit form with a shortcut on top, and odd planes (dispatch_odd_form).
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
    // Odd planes: vectors of a plane, the last one moved back to end with the plane, and of the slice.
    FastDiv by_row;
    uint32_t vectors;
};

// A step of a lane: where its values are, whether the slice has them, and how many of the first ones the vector in front
// holds too.
struct Step {
    size_t at;
    bool valid;
    int held;
};

template<int V, bool RAGGED>
__device__ __forceinline__ Step step_of(const ResidentGeom& g, uint32_t c, uint32_t item)
{
    if constexpr (RAGGED) {
        const bool valid = item < g.vectors;
        uint32_t n, j;
        g.by_row.divmod(valid ? item : 0u, n, j);
        const int beyond = static_cast<int>(j) * 4 + 4 - g.spatial;
        const int held = beyond > 0 ? beyond : 0;
        return Step{ (static_cast<size_t>(n) * g.channels + c) * g.spatial + (static_cast<int>(j) * 4 - held), valid, held };
    } else {
        const uint32_t e = item * V;
        const bool valid = e < g.per_channel;
        return Step{ g.at(c, valid ? e : 0u), valid, 0 };
    }
}

template<int V, bool NT, bool RAGGED>
__device__ __forceinline__ Pack<V> ld_step(const float* p, const Step& s)
{
    if constexpr (RAGGED) return ld_word<NT>(p + s.at);
    else return ld<V, NT>(p, s.at);
}

// OWN: without the values that the vector in front holds too.
template<int V, bool RAGGED, bool OWN = false>
__device__ __forceinline__ void st_step(float* p, const Step& s, const Pack<V>& v)
{
    if constexpr (!RAGGED) {
        st<V, true>(p, s.at, v);
    } else if (OWN) {
        st_own(p + s.at, v, s.held);
    } else {
        st_word(p + s.at, v);
    }
}

// The small forms (small_slice below): a lane adds the values of a vector in fp32 and its vectors in doubles -- no further
// from 64 bits than a lane of the other forms that holds one vector -- and the backward keeps x beside the delta.  (Odd
// planes, and one value a step in whatever form: every value in doubles.)
template<int V, int R, int L, int T>
constexpr bool kSmallSlice = L == 0 && T < kResidentThreads && V * R <= 32;

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
// What a forward takes u = 1 + exp(x) through.
constexpr bool chains_exponential(int activation)
{
    return activation == PXH_MISH || activation == PXH_SOFTPLUS;
}

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
// With more lanes at the same capacity each is slower (2 x 1024 x 10^2 in 128, 256, 512 lanes: backward 4.7, 6.5, 10.0).
// Eight vectors a lane take a workgroup's 256 registers a lane, one to a compute unit: up to as many channels only
// (4 x 512 x 52^2, leaky: backward 16.5 us against 14.2).  An activation with an exponential is bound by its gradient, and
// there the waves count: beyond 512 vectors a slice its backward keeps the full workgroups where it has them
// (8 x 256 x 38^2, mish: 15.5 us against 13.4; 2 x 256 x 40^2: 8.5 against 8.0; 2 x 512 x 20^2: 6.4 against 7.8).
constexpr uint32_t kSmallVectors = 4096;
constexpr uint32_t kSmallVectorsMany = 2048;      // beyond kSmallChannels channels
constexpr int kSmallChannels = 256;
constexpr uint32_t kSmallVectorsSmooth = 512;

// The vectors of a channel's slice where the shape takes a small form, else 0.
inline uint32_t small_slice(int batch, int channels, int spatial, bool vec, int activation, bool backward)
{
    if (!vec) return 0;
    const size_t items = static_cast<size_t>(batch) * spatial / 4;
    size_t most = channels <= kSmallChannels ? kSmallVectors : kSmallVectorsMany;
    if (backward && !selects(activation) && channels >= kResidentChannels) most = kSmallVectorsSmooth;
    return items <= most ? static_cast<uint32_t>(items) : 0;
}

// Calls launch.operator()<R, T>() with the form for `items` vectors: steps per lane, lanes.
template<typename F>
void dispatch_small_form(uint32_t items, F&& launch)
{
    if (items <= 64 * 2) return launch.template operator()<2, 64>();
    if (items <= 128 * 2) return launch.template operator()<2, 128>();
    if (items <= 256 * 4) return launch.template operator()<4, 256>();
    if (items <= 512 * 4) return launch.template operator()<4, 512>();
    return launch.template operator()<8, 512>();
}

inline int resident_vectors(int batch, int channels, int spatial, bool vec)
{
    if (!vec || channels < kResidentChannels) return 0;
    const size_t vectors = static_cast<size_t>(batch) * spatial / 4;
    const size_t per_thread = (vectors + kResidentThreads - 1) / kResidentThreads;
    if (per_thread <= kResidentVectors) return kResidentVectors;
    return per_thread <= kResidentLargeRegs + kResidentLargeLds ? kResidentLargeRegs + kResidentLargeLds : 0;
}

// Odd planes (and tensors off a 16-byte boundary).  A 128-bit access needs the alignment of a word only, so their planes
// are taken in vectors too, the last of a plane moved back to end with it: the values that it shares with the vector in
// front are loaded twice, added once, and written twice with the same result, or once where a lane may read what another
// has written.  One value per access was what bound these layers (a quarter of the bytes on their way per instruction and
// four times the addresses); a lane that keeps both tensors needs no second read of x either.
// One value a step, or three launches (*) -> vectors, us, leaky and mish: forward, + shortcut, backward, backward with rescale + clip
//   64 x 1024 x 13^2  28.4 -> 23.8  39.8 -> 34.3  40.4 -> 35.0  48.0 -> 37.1   6 x 512   38.6*-> 24.0  43.5*-> 33.7  62.6*-> 36.0  72.2*-> 47.6
//   64 x 512 x 13^2   15.2 -> 11.2  19.0 -> 16.3  19.8 -> 16.8  24.8 -> 19.0   6 x 512   18.5 -> 12.4  22.3 -> 16.6  25.0 -> 19.1  34.0 -> 25.5
//   64 x 256 x 13^2    9.3 ->  8.0  12.6 ->  8.9  12.3 -> 10.6  16.7 -> 13.8   6 x 512   11.9 ->  8.8  14.1 -> 10.0  15.3 -> 13.0  21.2 -> 17.1
//   64 x 512 x 19^2   31.9*-> 21.4  38.2*-> 31.9  37.5 -> 35.3  43.5 -> 41.0   6 x 1024  33.2*-> 20.9  41.6*-> 33.5  57.4*-> 40.1  66.0*-> 56.5
//   16 x 1024 x 19^2  13.3 -> 10.6  19.5 -> 15.7  18.8 -> 16.7  22.5 -> 19.1   6 x 256   17.5 -> 12.6  21.7 -> 16.5  21.9 -> 19.2  29.3 -> 25.1
//   16 x 512 x 19^2    7.7 ->  7.5   9.4 ->  8.4  10.6 ->  9.4  13.8 -> 12.7   3 x 512   10.8 ->  8.1  12.0 ->  9.3  13.0 -> 11.3  17.4 -> 15.6
//   8 x 512 x 19^2     5.9 ->  5.7   6.4 ->  6.0   7.7 ->  6.6  10.8 ->  9.8   3 x 256    7.6 ->  6.5   8.0 ->  6.9   9.7 ->  8.0  13.0 -> 11.5
//   8 x 96 x 45^2      9.2 ->  6.8  12.7 ->  9.0  12.5 ->  9.5  17.2 -> 13.3   4 x 1024  14.3 ->  8.7  15.8 -> 10.8  16.0 -> 12.3  20.7 -> 17.1
//   4 x 1024 x 13^2    5.1 ->  4.9   5.3 ->  5.2   5.6 ->  5.5   9.3 ->  8.9   2 x 128    5.8 ->  5.4   5.9 ->  5.7   6.7 ->  6.3  10.2 ->  9.7
//   1 x 1024 x 13^2    4.2 ->  4.0   4.3 ->  4.3   4.4 ->  4.3   7.2 ->  7.1   1 x 64     4.6 ->  4.4   4.9 ->  4.7   4.9 ->  4.3   7.7 ->  7.3
//   1 x 1024 x 19^2    5.1 ->  4.5   5.2 ->  4.6   5.4 ->  4.5   9.0 ->  7.4   1 x 128    5.4 ->  5.0   5.5 ->  5.2   5.9 ->  4.9   9.1 ->  7.8
// (steps x lanes of the form.)  More lanes than the slice needs are slower everywhere (64 x 1024 x 13^2, backward: 4 x 1024
// 41.4, 8 x 512 43.0; 16 x 512 x 19^2: 3 x 1024 14.3); six steps in workgroups of 256 lanes serve a thousand channels, whose
// workgroups then run in one round (16 x 1024 x 19^2 16.7 against 18.2 with 3 x 512), three in 512 lanes up to half as many
// (16 x 512 x 19^2, mish: 11.3 against 12.5).  Up to 128 vectors a step is enough (1 x 256 x 17^2, mish, backward: 1 x 128 3.8,
// 2 x 128 4.3), and a slice of a value per lane needs no vectors, whose addresses and shared values are then the longer part of
// a short launch (1 x 1024 x 7^2, mish: forward 3.8 against 4.2 in vectors, + shortcut 3.8 and 4.5).
// A step that few lanes or none of a workgroup need is computed all the same.  With many channels: 20 x 1024 x 7^2 (260 vectors), leaky and
// mish, backward, 2 x 256 7.4 and 9.1, 3 x 256 8.1 and 10.5; 64 x 1024 x 7^2 (832) 4 x 256 15.1 and 17.1, 6 x 256 15.4 and 19.8.  With few, where
// an exponential is, twice the lanes are ahead: 2 x 512 x 19^2, mish, forward 1 x 256 4.8, 2 x 128 5.2, backward 4.9 and 6.2;
// 6 x 512 x 13^2 1 x 512 6.6, 3 x 256 7.3; 40 x 300 x 9^2 2 x 512 9.2, 3 x 512 10.5.  (Leaky, 6 x 512 x 13^2: 5.5 and 5.2; with a thousand
// channels 4 x 1024 x 13^2, leaky, 1 x 256 5.9, 2 x 128 5.6.)
// Planes below kOddSpatial have no vector: one value a step, in forms that hold as much as those of the others.  Three launches
// give each plane a wave of its own.
// us, leaky and mish, one launch and (*) several: forward, + shortcut, backward
//   2731 x 5 x 2       7.7, 9.7, 9.2      8.1, 10.3, 10.6    12 x 512     12.6*, 12.6*, 13.7*   12.8*, 12.8*, 16.0*
//   2048 x 64 x 3      16.7, 25.8, 24.7   16.9, 25.9, 25.4   12 x 512     34.7*, 34.0*, 37.1*   34.2*, 33.6*, 47.3*
//   4000 x 256 x 3     59, 93, 92         60, 94, 92         16 x 1024    191*, 192*, 209*      191*, 192*, 292*
//   8000 x 256 x 3     127, 192, 185      128, 194, 185      24 x 1024    369*, 374*, 402*      369*, 374*, 605*
// Workgroups of the size that just holds the slice: 64 x 1024 x 1 in 64 lanes 6.7, 7.6, 8.2, in 256 7.2, 8.6, 8.4;
// 513 x 97 x 2 in 256 lanes 7.9, 8.6, 9.2, in 1024 8.7, 11.1, 11.2.
constexpr int kOddSpatial = 4;
constexpr uint32_t kOddVectors = 6144;
constexpr uint32_t kOddVectorsFew = 4096;         // with fewer than kResidentChannels channels (as kSmallVectors)
// ... where an exponential is followed by another chain: workgroups of 1024 lanes, with fewer of them than compute units, are longer
// than several launches, us, mish, forward, backward, clipped with nothing to change, rescaled, clamped throughout: 90 x 16 x 13^2 10.1 -> 8.9,
// 14.6 -> 11.9, 18.7 -> 17.6, 26.0 -> 17.5, 32.0 -> 20.2, 8 x 64 x 45^2 10.8 -> 10.1, 16.4 -> 16.1, 20.7 -> 24.3, 27.8 -> 24.0, 34.8 -> 30.1.  Not
// logistic (8 x 64 x 45^2: 7.8 and 8.4, 11.0 and 11.5, 15.1 and 21.0), nor 60 x 64 x 13^2 (2640 vectors: 8.3 and 10.3, 12.6 and 15.2).
constexpr uint32_t kOddVectorsFewChain = 3072;
constexpr uint32_t kOddValues = 4 * kOddVectors, kOddValuesFew = 6144;
constexpr int kOddChannels = 512;

// The vectors (values in planes below kOddSpatial) of a channel's slice where such a shape takes a one-launch form, else 0.
inline uint32_t odd_slice(int batch, int channels, int spatial, bool vec, int activation, bool backward)
{
    if (vec) return 0;
    const bool few = channels < kResidentChannels;
    const bool values = spatial < kOddSpatial;
    const size_t items = static_cast<size_t>(batch) * (values ? spatial : (spatial + 3) / 4);
    // (the forward of planes of up to a wave's width stays: several launches give each a wave)
    const bool chain = chains_exponential(activation) && (backward || spatial > kWave);
    const uint32_t most = values ? (few ? kOddValuesFew : kOddValues) : few ? (chain ? kOddVectorsFewChain : kOddVectorsFew) : kOddVectors;
    return items <= most ? static_cast<uint32_t>(items) : 0;
}

// Vectors of a slice up to which a lane takes one, with few channels: an exponential is worth more than waves, and its gradient
// twice as much.
template<int ACT, bool BACKWARD>
constexpr int kOddOneStep = selects(ACT) ? 128 : BACKWARD ? 512 : 256;

// Calls launch.operator()<V, R, T>() with the form for `items`: values per step, steps per lane, lanes.  ONE: kOddOneStep.
template<int ONE, typename F>
void dispatch_odd_form(uint32_t items, const ResidentGeom& g, F&& launch)
{
    if (g.per_channel <= 64) return launch.template operator()<1, 1, 64>();
    if (g.spatial < kOddSpatial) {
        if (items <= 64 * 4) return launch.template operator()<1, 4, 64>();
        if (items <= 256 * 4) return launch.template operator()<1, 4, 256>();
        if (items <= 256 * 8) return launch.template operator()<1, 8, 256>();
        if (items <= 512 * 8) return launch.template operator()<1, 8, 512>();
        if (items <= 512 * 12) return launch.template operator()<1, 12, 512>();
        if (items <= 1024 * 8) return launch.template operator()<1, 8, 1024>();
        if (items <= 1024 * 16) return launch.template operator()<1, 16, 1024>();
        return launch.template operator()<1, 24, 1024>();
    }
    const bool many = g.channels > kOddChannels;
    if (items <= 64) return launch.template operator()<4, 1, 64>();
    if (items <= 128) return launch.template operator()<4, 1, 128>();
    if constexpr (ONE >= 256)
        if (items <= 256 && !many) return launch.template operator()<4, 1, 256>();
    if constexpr (ONE >= 512) {
        if (items > 256 && items <= 512 && !many) return launch.template operator()<4, 1, 512>();
        if (items > 256 * 3 && items <= 512 * 2 && !many) return launch.template operator()<4, 2, 512>();
    }
    if (items <= 128 * 2) return launch.template operator()<4, 2, 128>();
    if (items <= 256 * 2 && many) return launch.template operator()<4, 2, 256>();
    if (items <= 256 * 3) return launch.template operator()<4, 3, 256>();
    if (items <= 256 * 4 && many) return launch.template operator()<4, 4, 256>();
    if (items <= 256 * 6 && many) return launch.template operator()<4, 6, 256>();
    if (items <= 512 * 3) return launch.template operator()<4, 3, 512>();
    if (items <= 512 * 4) return launch.template operator()<4, 4, 512>();
    if (items <= 512 * 6) return launch.template operator()<4, 6, 512>();
    if (items <= 1024 * 4) return launch.template operator()<4, 4, 1024>();
    return launch.template operator()<4, 6, 1024>();
}

// Whether the sums over odd planes in several launches, which give each segment of a plane a wave, take them in vectors.  Up to
// a value per lane those only leave lanes idle, each with four times the arithmetic; in the backward of an activation with an
// exponential, up to two, whose arithmetic is worth more than the loads.  There a lane takes a value a step, in no more steps than
// that.  In vectors -> so, us, forward, bias-only backward, backward, clipped with nothing to change:
//   6000 x 64 x 5, mish     113 -> 49     132 -> 55     160 -> 75      205 -> 99
//   3000 x 16 x 3^2, leaky  22.8 -> 12.6  14.3 -> 10.9  22.1 -> 17.6   30.6 -> 25.2
//   3000 x 16 x 7 x 9, mish 27.5 -> 19.3  26.8 -> 16.9  42.9 -> 32.1   53.1 -> 38.6
//   3000 x 16 x 7 x 11, mish              26.7 -> 21.7  43.1 -> 35.2   53.7 -> 42.8
//   1500 x 32 x 11^2, mish                25.5 -> 22.0  44.2 -> 37.7   55.0 -> 45.4
// From 65 to 128 values the others are level, but for the bias-only backward (3000 x 16 x 7 x 11, leaky: 20.4 so, 19.1 in vectors).
constexpr int kValueSteps = 2;
inline bool sums_in_vectors(int spatial, int activation = PXH_LINEAR)
{
    return spatial > (selects(activation) ? 1 : kValueSteps) * kWave;
}

// Whether a plain call of a shape asks for a workspace: unless it takes a one-launch form that never depended on measured
// limits.  Those of the others may move, also between activations, and a workspace that is too small for a shape is refused
// on either side of them (as is growth in a capture).
inline bool asks_for_workspace(int batch, int channels, int spatial, bool vec)
{
    if (vec) return resident_vectors(batch, channels, spatial, true) == 0;
    return channels < kResidentChannels || static_cast<size_t>(batch) * spatial > kResidentVectors * kResidentThreads;
}

inline ResidentGeom resident_geom(int batch, int channels, int spatial)
{
    return ResidentGeom{ channels, spatial, static_cast<uint32_t>(batch) * static_cast<uint32_t>(spatial),
                         FastDiv(static_cast<uint32_t>(spatial)), FastDiv(static_cast<uint32_t>(spatial + 3) / 4),
                         static_cast<uint32_t>(batch) * (static_cast<uint32_t>(spatial + 3) / 4) };
}

// A kernel that asks for more than 64 KB of dynamic LDS has to be allowed to, once.
int allow_large_lds(const void* kernel);

// How a shape takes the one-launch passes: the vectors per lane of the forms of 1024 lanes (resident_vectors), or the vectors of
// a slice in a small form (small_slice) or of odd planes (odd_slice); all 0 where it does not.
struct ResidentForm {
    int per_thread;
    uint32_t small, odd;
    explicit operator bool() const { return per_thread || small || odd; }
};

inline ResidentForm resident_form(int batch, int channels, int spatial, bool vec, int activation, bool backward)
{
    return ResidentForm{ resident_vectors(batch, channels, spatial, vec),
                         small_slice(batch, channels, spatial, vec, activation, backward),
                         odd_slice(batch, channels, spatial, vec, activation, backward) };
}

int launch_resident_forward(const char* who, const ResidentFwdArgs& r, const ResidentForm& form, int activation, hipStream_t s);
int launch_resident_backward(const char* who, const ResidentBwdArgs& r, bool clipped, const ResidentForm& form, int activation,
                             hipStream_t s);

}  // namespace pxh
