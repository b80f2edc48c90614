// Max-pool (values + int32 argmax) and nearest upsample, forward and backward, for gfx950.
// Index and copy work is bit-exact against the CPU layers; accumulation follows their order.
#include "stream.h"

#include <algorithm>
#include <cfloat>

namespace pxh {
namespace {

struct PoolGeom {
    int ih, iw, oh, ow, kernel, stride, origin;   // origin = -padding / 2
};

// ------------------------------------------------------------------ max-pool, any geometry
// One window.  Taps in row-major order; the first in-bounds tap is taken, later taps only when strictly
// greater (include/MaxPoolLayer.h:106-127 of the reference).
__device__ __forceinline__ void scan_window(const float* in, const PoolGeom& g, uint32_t plane, uint32_t oy, uint32_t ox,
                                            float& best, int& best_at)
{
    best = -FLT_MAX;
    best_at = -1;
    for (int ky = 0; ky < g.kernel; ++ky) {
        const int y = g.origin + static_cast<int>(oy) * g.stride + ky;
        if (y < 0 || y >= g.ih) continue;
        for (int kx = 0; kx < g.kernel; ++kx) {
            const int x = g.origin + static_cast<int>(ox) * g.stride + kx;
            if (x < 0 || x >= g.iw) continue;
            const int at = x + g.iw * (y + g.ih * static_cast<int>(plane));
            const float v = in[at];
            if (best_at < 0 || v > best) {
                best_at = at;
                best = v;
            }
        }
    }
}

// One output per lane.
__global__ __launch_bounds__(kBlock) void maxpool_fwd_generic_kernel(const float* in, float* out, int* indexes,
                                                                     uint32_t total, PoolGeom g, FastDiv by_ow,
                                                                     FastDiv by_oh)
{
    const uint32_t o = blockIdx.x * kBlock + threadIdx.x;
    if (o >= total) return;
    uint32_t rows, ox, plane, oy;
    by_ow.divmod(o, rows, ox);
    by_oh.divmod(rows, plane, oy);
    float best;
    int best_at;
    scan_window(in, g, plane, oy, ox, best, best_at);
    out[o] = best;
    indexes[o] = best_at;
}

// Windows of 2 that move by one cell over a tensor of the output's size: four outputs of the flat tensor to a lane, whose cells
// are the five from the first output on and the five a row further, whatever rows they lie in.  One output per lane read
// each of its cells by itself; us: 32768 planes of 13 x 13 22.5 -> 13.4, 512 of 13 x 13 2.9 -> 2.7, of 26 x 26 3.5 -> 3.1.  (A
// launch this short is one trip to memory: the outputs whose row further would end behind the tensor, taken one after the other
// by a scan, made it 4.5.)
__global__ __launch_bounds__(kBlock) void maxpool_fwd_step1_kernel(const float* in, float* out, int* indexes, uint32_t total,
                                                                   FastDiv by_w, FastDiv by_h)
{
    const uint32_t o = (blockIdx.x * kBlock + threadIdx.x) * 4;
    if (o >= total) return;
    uint32_t rows, x, plane, y;
    by_w.divmod(o, rows, x);
    by_h.divmod(rows, plane, y);
    const uint32_t w = by_w.d, h = by_h.d;
    float a[5], b[5];
    if (o + w + 5 <= total) {
        const Pack<4> a4 = ld_word<false>(in + o), b4 = ld_word<false>(in + o + w);
#pragma unroll
        for (int q = 0; q < 4; ++q) {
            a[q] = a4.v[q];
            b[q] = b4.v[q];
        }
        a[4] = in[o + 4];
        b[4] = in[o + w + 4];
    } else {
        // the cells of a row further end with the tensor: those beyond are no output's
#pragma unroll
        for (int q = 0; q < 5; ++q) {
            a[q] = in[min(o + q, total - 1)];
            b[q] = in[min(o + q + w, total - 1)];
        }
    }
    Pack<4> value, index;
#pragma unroll
    for (int q = 0; q < 4; ++q) {
        const bool right = x + 1 < w, below = y + 1 < h;
        float best = a[q];
        uint32_t at = o + q;
        if (right && a[q + 1] > best) { best = a[q + 1]; at = o + q + 1; }
        if (below && b[q] > best) { best = b[q]; at = o + q + w; }
        if (right && below && b[q + 1] > best) { best = b[q + 1]; at = o + q + w + 1; }
        value.v[q] = best;
        index.v[q] = __int_as_float(static_cast<int>(at));
        if (!right) {
            x = 0;
            y = below ? y + 1 : 0;
        } else {
            ++x;
        }
    }
    if (o + 4 <= total) {
        st_word<false>(out + o, value);
        st_word<false>(reinterpret_cast<float*>(indexes) + o, index);
    } else {
#pragma unroll
        for (int q = 0; q < 3; ++q) {
            if (o + q >= total) break;
            out[o + q] = value.v[q];
            indexes[o + q] = __float_as_int(index.v[q]);
        }
    }
}

// ------------------------------------------------------------------ max-pool through LDS
// Overlapping windows read every input k * k times; from the caches, at one lane per output, that is what
// the kernel above costs (8192 planes of 19 x 19: k = 5 44 us, k = 13 191 us, for 36 MB of traffic).  Here a
// workgroup takes a tile -- whole planes while they are small, else a strip of rows of one plane -- into LDS
// and works separably: the first largest tap of every row segment, then the first largest of k segments,
// 2k reads in place of k * k (17 and 24 us).  Row-major first-wins order survives the split: a segment keeps
// its first largest tap, and a later segment only wins when strictly greater.  The tile is framed by -inf,
// so that no tap has to be checked against the border; where that could decide (a window whose largest
// value is -inf) or a NaN is in the tile (as the first tap it is taken, later it is not), the window is
// scanned as above.
struct PoolTile {
    uint32_t planes;        // of the tensor
    uint32_t per_tile;      // planes per tile; more than one only of whole planes
    uint32_t strips;        // tiles per plane
    uint32_t rows;          // output (forward) or input (backward) rows per strip
};

// K: the window, or 0 for any other
template<int K>
__global__ __launch_bounds__(kBlock) void maxpool_fwd_tile_kernel(const float* in, float* out, int* indexes,
                                                                  PoolTile tile, PoolGeom g, FastDiv by_strips,
                                                                  FastDiv by_iw, FastDiv by_ih, FastDiv by_ow,
                                                                  FastDiv by_oh, uint32_t tile_cells, uint32_t segments)
{
    extern __shared__ float lds[];
    float* cells = lds;                                        // [tile_cells]: framed rows
    float* best_of = lds + tile_cells;                         // [segments]
    uint8_t* tap_of = reinterpret_cast<uint8_t*>(best_of + segments);
    const int k = K ? K : g.kernel;
    uint32_t group, strip;
    by_strips.divmod(blockIdx.x, group, strip);
    const uint32_t p0 = group * tile.per_tile;
    const uint32_t planes = min(tile.per_tile, tile.planes - p0);
    const int oy0 = static_cast<int>(strip * tile.rows);
    const int rows_out = min(static_cast<int>(tile.rows), g.oh - oy0);
    // the frame: what the windows of the tile cover, from row y_frame and column g.origin on
    const int y_frame = g.origin + oy0 * g.stride;
    const uint32_t frame_h = (rows_out - 1) * g.stride + k, frame_w = (g.ow - 1) * g.stride + k;
    int y_lo = 0, rows_in = g.ih;
    if (tile.strips > 1) {
        y_lo = min(max(0, y_frame), g.ih);
        rows_in = max(0, min(g.ih, y_frame + static_cast<int>(frame_h)) - y_lo);
    }
    for (uint32_t i = threadIdx.x; i < planes * rows_in * frame_w; i += kBlock) cells[i] = -INFINITY;
    for (uint32_t i = threadIdx.x; i < planes * frame_h * g.ow; i += kBlock) best_of[i] = -INFINITY;
    __syncthreads();
    const uint32_t in0 = (p0 * g.ih + y_lo) * g.iw;
    bool nan = false;
    for (uint32_t i = threadIdx.x; i < planes * rows_in * g.iw; i += kBlock) {
        uint32_t row, x;
        by_iw.divmod(i, row, x);
        const float v = in[in0 + i];
        nan |= v != v;
        const uint32_t column = x - g.origin;
        if (column < frame_w) cells[row * frame_w + column] = v;
    }
    const bool by_scan = __syncthreads_or(nan) != 0;
    for (uint32_t j = threadIdx.x; j < planes * rows_in * g.ow; j += kBlock) {
        uint32_t row, ox, plane = 0;
        by_ow.divmod(j, row, ox);
        const float* line = cells + row * frame_w + ox * g.stride;
        if (tile.strips == 1) by_ih.divmod(row, plane, row);
        const uint32_t frame_row = y_lo + row - y_frame;
        if (frame_row >= frame_h) continue;
        float best = line[0];
        int tap = 0;
#pragma unroll
        for (int kx = 1; kx < k; ++kx) {
            const float v = line[kx];
            tap = v > best ? kx : tap;
            best = v > best ? v : best;         // not fmaxf: of two zeros the first stays
        }
        const uint32_t seg = (plane * frame_h + frame_row) * g.ow + ox;
        best_of[seg] = best;
        tap_of[seg] = static_cast<uint8_t>(tap);
    }
    __syncthreads();
    const uint32_t out0 = (p0 * g.oh + oy0) * g.ow;
    for (uint32_t j = threadIdx.x; j < planes * rows_out * g.ow; j += kBlock) {
        uint32_t row, ox, plane = 0;
        by_ow.divmod(j, row, ox);
        if (tile.strips == 1) by_oh.divmod(row, plane, row);
        const uint32_t seg = (plane * frame_h + row * g.stride) * g.ow + ox;
        float best = best_of[seg];
        int tap = 0;
#pragma unroll
        for (int ky = 1; ky < k; ++ky) {
            const float v = best_of[seg + ky * g.ow];
            tap = v > best ? ky : tap;
            best = v > best ? v : best;         // not fmaxf: of two zeros the first stays
        }
        const int x = g.origin + static_cast<int>(ox) * g.stride + tap_of[seg + tap * g.ow];
        const int y = y_frame + static_cast<int>(row) * g.stride + tap;
        int at = x + g.iw * (y + g.ih * static_cast<int>(p0 + plane));
        if (by_scan || best == -INFINITY) scan_window(in, g, p0 + plane, oy0 + row, ox, best, at);
        out[out0 + j] = best;
        indexes[out0 + j] = at;
    }
}

// The same for windows that move by one cell, the usual case, with the LDS work of several outputs shared: the tile comes in
// by 128-bit loads that are in flight while its frame is laid out; a lane takes four neighbouring outputs of a row from one
// reading of their K + 3 cells (128 bits at a time), then four outputs of a column from one reading of their K + 3 segments.
// Rows beyond the image are left out by their numbers, so that only columns have a frame.  Against the kernel above, us,
// 8192 planes of 19 x 19: k = 5 16.8 -> 12.9, 9 20.9 -> 16.2, 13 23.5 -> 19.2; 64 of 300 x 300, k = 3, 25.5 -> 19.9.
struct SlideTile {
    uint32_t pitch, groups;     // cells of a framed row; fours of outputs of a row
};

constexpr int kSlideRun = 4;

constexpr uint32_t slide_pitch(int k, uint32_t groups)
{
    return 4 * (groups - 1) + (k + kSlideRun - 1 + 3) / 4 * 4;
}

template<int K>
__global__ __launch_bounds__(kBlock) void maxpool_fwd_slide_kernel(const float* in, float* out, int* indexes,
                                                                   PoolTile tile, PoolGeom g, SlideTile st,
                                                                   FastDiv by_strips, FastDiv by_iw, FastDiv by_groups,
                                                                   FastDiv by_ow, FastDiv by_runs)
{
    extern __shared__ __align__(16) float lds[];
    constexpr int kRead = (K + kSlideRun - 1 + 3) / 4 * 4;
    constexpr int kLoads = 2;       // vectors of a lane on their way at once: what a tile of 2048 cells has
    uint32_t group, strip;
    by_strips.divmod(blockIdx.x, group, strip);
    const uint32_t p0 = group * tile.per_tile;
    const uint32_t planes = min(tile.per_tile, tile.planes - p0);
    const int oy0 = static_cast<int>(strip * tile.rows);
    const int rows_out = min(static_cast<int>(tile.rows), g.oh - oy0);
    const int y_frame = g.origin + oy0;
    int y_lo = 0, rows_in = g.ih;
    if (tile.strips > 1) {
        y_lo = min(max(0, y_frame), g.ih);
        rows_in = max(0, min(g.ih, y_frame + rows_out - 1 + K) - y_lo);
    }
    const uint32_t all_rows = planes * rows_in, width = 4 * st.groups;
    float* const cells = lds;                                  // [all_rows][pitch], column 0 at x = g.origin
    float* const best_of = cells + all_rows * st.pitch;        // [all_rows][width]
    uint8_t* const tap_of = reinterpret_cast<uint8_t*>(best_of + all_rows * width);
    const uint32_t in0 = (p0 * g.ih + y_lo) * g.iw;
    const uint32_t values = all_rows * g.iw, vectors = values > kBlock ? values / 4 : 0;      // (a value to a lane where that is all)
    Pack<4> v[kLoads];
    const auto fetch = [&](uint32_t first) {
#pragma unroll
        for (int u = 0; u < kLoads; ++u) {
            const uint32_t i = first + u * kBlock + threadIdx.x;
            if (i < vectors) v[u] = ld_word<false>(in + in0 + 4 * static_cast<size_t>(i));
        }
    };
    fetch(0);
    const Pack<4> outside{ { -INFINITY, -INFINITY, -INFINITY, -INFINITY } };
    for (uint32_t i = threadIdx.x; i < all_rows * (st.pitch / 4); i += kBlock) *reinterpret_cast<Pack<4>*>(cells + 4 * i) = outside;
    __syncthreads();
    bool nan = false;
    const auto put = [&](uint32_t row, uint32_t x, float value) {
        nan |= value != value;
        const uint32_t column = x - g.origin;
        if (column < st.pitch) cells[row * st.pitch + column] = value;
    };
    for (uint32_t first = 0; first < vectors; first += kLoads * kBlock) {
        if (first) fetch(first);
#pragma unroll
        for (int u = 0; u < kLoads; ++u) {
            const uint32_t i = first + u * kBlock + threadIdx.x;
            if (i >= vectors) continue;
            uint32_t row, x;
            by_iw.divmod(4 * i, row, x);
#pragma unroll
            for (int q = 0; q < 4; ++q) {
                put(row, x, v[u].v[q]);
                if (++x == static_cast<uint32_t>(g.iw)) {
                    x = 0;
                    ++row;
                }
            }
        }
    }
    if (threadIdx.x < values - 4 * vectors) {
        uint32_t row, x;
        by_iw.divmod(4 * vectors + threadIdx.x, row, x);
        put(row, x, in[in0 + 4 * vectors + threadIdx.x]);
    }
    const bool by_scan = __syncthreads_or(nan) != 0;
    for (uint32_t j = threadIdx.x; j < all_rows * st.groups; j += kBlock) {
        uint32_t row, four;
        by_groups.divmod(j, row, four);
        const float* const line = cells + row * st.pitch + 4 * four;
        float w[kRead];
#pragma unroll
        for (int q = 0; q < kRead / 4; ++q) {
            const Pack<4> t = *reinterpret_cast<const Pack<4>*>(line + 4 * q);
#pragma unroll
            for (int k = 0; k < 4; ++k) w[4 * q + k] = t.v[k];
        }
        Pack<4> best;
        uint32_t taps = 0;
#pragma unroll
        for (int o = 0; o < 4; ++o) {
            best.v[o] = w[o];
            uint32_t tap = 0;
#pragma unroll
            for (int kx = 1; kx < K; ++kx) {
                tap = w[o + kx] > best.v[o] ? kx : tap;
                best.v[o] = w[o + kx] > best.v[o] ? w[o + kx] : best.v[o];      // not fmaxf: of two zeros the first stays
            }
            taps |= tap << (8 * o);
        }
        *reinterpret_cast<Pack<4>*>(best_of + row * width + 4 * four) = best;
        *reinterpret_cast<uint32_t*>(tap_of + row * width + 4 * four) = taps;
    }
    __syncthreads();
    // runs of kSlideRun rows
    for (uint32_t j = threadIdx.x; j < planes * by_runs.d * g.ow; j += kBlock) {
        uint32_t run, ox, plane;
        by_ow.divmod(j, run, ox);
        by_runs.divmod(run, plane, run);
        const int row0 = static_cast<int>(run) * kSlideRun;
        const int seg0 = y_frame + row0 - y_lo;       // of the tile's rows of this plane; the first may lie before them
        const uint32_t column = plane * rows_in * width + ox;
        float w[K + kSlideRun - 1];
#pragma unroll
        for (int q = 0; q < K + kSlideRun - 1; ++q) {
            const bool inside = static_cast<uint32_t>(seg0 + q) < static_cast<uint32_t>(rows_in);
            const float value = best_of[column + (inside ? seg0 + q : 0) * width];
            w[q] = inside ? value : -INFINITY;
        }
#pragma unroll
        for (int o = 0; o < kSlideRun; ++o) {
            if (row0 + o >= rows_out) break;
            float best = w[o];
            int tap = 0;
#pragma unroll
            for (int ky = 1; ky < K; ++ky) {
                tap = w[o + ky] > best ? ky : tap;
                best = w[o + ky] > best ? w[o + ky] : best;
            }
            int at;
            if (by_scan || best == -INFINITY) {
                scan_window(in, g, p0 + plane, oy0 + row0 + o, ox, best, at);
            } else {
                const int x = g.origin + static_cast<int>(ox) + tap_of[column + (seg0 + o + tap) * width];
                const int y = y_frame + row0 + o + tap;
                at = x + g.iw * (y + g.ih * static_cast<int>(p0 + plane));
            }
            const size_t to = (static_cast<size_t>(p0 + plane) * g.oh + oy0 + row0 + o) * g.ow + ox;
            out[to] = best;
            indexes[to] = at;
        }
    }
}

// 2x2 / stride 2 windows that all lie inside the input: VX outputs per lane from two
// (2*VX)-wide row loads, stored as VX-wide value and index vectors.
template<int VX, bool NT>
__global__ __launch_bounds__(kBlock) void maxpool_fwd_2x2_kernel(const float* in, float* out, int* indexes,
                                                                 uint32_t units, int iw, int ow, FastDiv by_owv,
                                                                 FastDiv by_oh)
{
    const uint32_t t = blockIdx.x * kBlock + threadIdx.x;
    if (t >= units) return;
    uint32_t rows, oxv, plane, oy;
    by_owv.divmod(t, rows, oxv);
    by_oh.divmod(rows, plane, oy);
    const uint32_t ih = by_oh.d * 2;
    const uint32_t ox = oxv * VX;
    const uint32_t in0 = (plane * ih + 2 * oy) * iw + 2 * ox;   // < 2^31 checked by the host
    const Pack<2 * VX> r0 = ld<2 * VX, NT>(in, in0);
    const Pack<2 * VX> r1 = ld<2 * VX, NT>(in, in0 + iw);
    Pack<VX> v;
    IPack<VX> ix;
#pragma unroll
    for (int k = 0; k < VX; ++k) {
        float best = r0.v[2 * k];
        int at = in0 + 2 * k;
        if (r0.v[2 * k + 1] > best) { best = r0.v[2 * k + 1]; at = in0 + 2 * k + 1; }
        if (r1.v[2 * k] > best) { best = r1.v[2 * k]; at = in0 + iw + 2 * k; }
        if (r1.v[2 * k + 1] > best) { best = r1.v[2 * k + 1]; at = in0 + iw + 2 * k + 1; }
        v.v[k] = best;
        ix.v[k] = at;
    }
    const uint32_t o = (plane * by_oh.d + oy) * ow + ox;
    st<VX, NT>(out, o, v);
    sti<VX, NT>(indexes, o, ix);
}

// The same for an even output width (input rows of a multiple of 4 floats) and a multiple of 4
// outputs in all, with one 128-bit access per lane and stream: a lane takes 2 consecutive
// outputs of the flat output tensor (they share a row), i.e. 4 floats of each of two input rows;
// the lanes of a pair then swap halves so that the even lane stores the pair's 4 values and the
// odd lane its 4 indexes.  Every address is 16-byte aligned: rows start at multiples of 4 floats.
template<bool NT>
__global__ __launch_bounds__(kBlock) void maxpool_fwd_2x2_pair_kernel(const float* in, float* out, int* indexes,
                                                                      uint32_t lanes, int iw, int ow, FastDiv by_owh,
                                                                      FastDiv by_oh)
{
    // the grid is a whole number of waves and `lanes` is even: a pair is never split by the guard
    const uint32_t t = blockIdx.x * kBlock + threadIdx.x;
    const bool live = t < lanes;
    const uint32_t u = live ? t : 0;
    const uint32_t half = u & 1;
    uint32_t rows, oxh, plane, oy;
    by_owh.divmod(u, rows, oxh);
    by_oh.divmod(rows, plane, oy);
    const uint32_t ih = by_oh.d * 2;
    const uint32_t ox = oxh * 2;
    const uint32_t in0 = (plane * ih + 2 * oy) * iw + 2 * ox;   // < 2^31 checked by the host
    const Pack<4> r0 = ld<4, NT>(in, in0);
    const Pack<4> r1 = ld<4, NT>(in, in0 + iw);
    float v[2];
    int ix[2];
#pragma unroll
    for (int k = 0; k < 2; ++k) {
        float best = r0.v[2 * k];
        int at = in0 + 2 * k;
        if (r0.v[2 * k + 1] > best) { best = r0.v[2 * k + 1]; at = in0 + 2 * k + 1; }
        if (r1.v[2 * k] > best) { best = r1.v[2 * k]; at = in0 + iw + 2 * k; }
        if (r1.v[2 * k + 1] > best) { best = r1.v[2 * k + 1]; at = in0 + iw + 2 * k + 1; }
        v[k] = best;
        ix[k] = at;
    }
    // even lane: gives its indexes, takes the partner's values; odd lane the other way round
    const float pv0 = __shfl_xor(v[0], 1, kWave), pv1 = __shfl_xor(v[1], 1, kWave);
    const int pi0 = __shfl_xor(ix[0], 1, kWave), pi1 = __shfl_xor(ix[1], 1, kWave);
    if (!live) return;
    const uint32_t o = (u >> 1) * 4;       // the pair's 4 flat outputs
    if (half == 0) {
        const Pack<4> w{ { v[0], v[1], pv0, pv1 } };
        st<4, NT>(out, o, w);
    } else {
        const IPack<4> w{ { pi0, pi1, ix[0], ix[1] } };
        sti<4, NT>(indexes, o, w);
    }
}

// Backward, any geometry: one input cell per lane gathers, in ascending output order, the
// deltas of the windows whose recorded argmax is this cell.  Ascending output order is the
// order in which the sequential CPU loop reaches this cell (include/MaxPoolLayer.h:150-156).
__global__ __launch_bounds__(kBlock) void maxpool_bwd_generic_kernel(const float* delta, const int* indexes,
                                                                     float* grad, uint32_t total, PoolGeom g,
                                                                     FastDiv by_iw, FastDiv by_ih)
{
    const uint32_t cell = blockIdx.x * kBlock + threadIdx.x;
    if (cell >= total) return;
    uint32_t rows, x, plane, y;
    by_iw.divmod(cell, rows, x);
    by_ih.divmod(rows, plane, y);
    // windows with origin + o*stride <= p <= origin + o*stride + kernel - 1
    const int py = static_cast<int>(y) - g.origin, px = static_cast<int>(x) - g.origin;
    int oy0 = py - g.kernel + 1;
    oy0 = oy0 <= 0 ? 0 : (oy0 + g.stride - 1) / g.stride;
    int ox0 = px - g.kernel + 1;
    ox0 = ox0 <= 0 ? 0 : (ox0 + g.stride - 1) / g.stride;
    const int oy1 = min(g.oh - 1, py >= 0 ? py / g.stride : -1);
    const int ox1 = min(g.ow - 1, px >= 0 ? px / g.stride : -1);
    float acc = grad[cell];
    bool touched = false;
    for (int oy = oy0; oy <= oy1; ++oy)
        for (int ox = ox0; ox <= ox1; ++ox) {
            const int o = ox + g.ow * (oy + g.oh * static_cast<int>(plane));
            if (indexes[o] == static_cast<int>(cell)) {
                acc += delta[o];
                touched = true;
            }
        }
    if (touched) grad[cell] = acc;
}

// Backward through LDS.  A lane per cell that looks at all k * k windows of its cell reads k * k indexes to
// find one on average (8192 planes of 19 x 19: k = 5 75 us, k = 13 274 us; here 14 and 44).  Here each output of the tile sets ONE bit, in
// the mask of the cell its index names, at the output's position among the cell's windows in ascending
// order; the cells with a bit (one in nine for k = 5) are then listed, so that lanes are not idle, and each
// adds its deltas in that order.  An index that names no cell of the output's own window is ignored, as it
// is by the kernel above.
struct PoolWindows {
    int along;              // windows over a cell along one axis: ceil(kernel / stride)
    uint32_t words;         // of a cell's mask
    FastDiv by_stride, by_along;
};

// K: the window of a kernel that moves by one cell over rows of at least K, or 0 for any geometry.  There a window's taps are
// told apart by one division of the distance from its first cell.  The outputs come in by 128-bit loads that are in flight
// while the masks are cleared, one at a time where a lane has one or two (four to some of the lanes: 512 planes of 13 x 13, 3 / 2, 3.8 -> 4.5).
// us, 8192 planes of 19 x 19: k = 5 19.3 -> 14.2, 9 34.3 -> 22.8, 13 55.5 -> 44.0; 64 of 300 x 300,
// k = 3, 32.8 -> 24.9; 32768 of 13 x 13, k = 2, 30.1 -> 21.3.  (Any geometry, by the loads alone: 1024 of 151 x 151, 3 / 2,
// 53.2 -> 48.7.)
template<int K>
__global__ __launch_bounds__(kBlock) void maxpool_bwd_tile_kernel(const float* delta, const int* indexes, float* grad,
                                                                  PoolTile tile, PoolGeom g, PoolWindows w,
                                                                  FastDiv by_strips, FastDiv by_ow, FastDiv by_oh,
                                                                  FastDiv by_iw, FastDiv by_ih, uint32_t tile_cells,
                                                                  uint32_t tile_outputs)
{
    extern __shared__ __align__(16) float lds[];
    constexpr int kLoads = 2;
    constexpr uint32_t kSteps = K ? 1 : 2;      // up to as many outputs a lane are taken one at a time
    const int k = K ? K : g.kernel;
    const uint32_t along = K ? K : w.along, words = K ? (K * K + 31) / 32 : w.words;
    const int past = g.ow - static_cast<int>(along);       // from the last of a cell's windows of a row to the first of the next
    const auto by_stride = [&](uint32_t n) { return K ? n : w.by_stride.div(n); };
    uint32_t* masks = reinterpret_cast<uint32_t*>(lds);                      // [word][tile_cells]
    float* deltas = lds + words * tile_cells;                                // [tile_outputs]
    uint16_t* listed = reinterpret_cast<uint16_t*>(deltas + tile_outputs);   // [tile_cells]
    __shared__ uint32_t listed_count;
    uint32_t group, strip;
    by_strips.divmod(blockIdx.x, group, strip);
    const uint32_t p0 = group * tile.per_tile;
    const uint32_t planes = min(tile.per_tile, tile.planes - p0);
    const int y_lo = static_cast<int>(strip * tile.rows);
    const int rows_in = min(static_cast<int>(tile.rows), g.ih - y_lo);
    int oy_lo = 0, rows_out = g.oh;
    if (tile.strips > 1) {
        // windows that reach row y_lo or later and begin no later than the last row
        const int reach = y_lo - g.origin - k + 1;
        oy_lo = min(reach <= 0 ? 0 : static_cast<int>(by_stride(reach + g.stride - 1)), g.oh);
        const int last = static_cast<int>(by_stride(y_lo + rows_in - 1 - g.origin));
        rows_out = max(0, min(g.oh, last + 1) - oy_lo);
    }
    const uint32_t cells = planes * rows_in * g.iw;
    const uint32_t cell0 = (p0 * g.ih + y_lo) * g.iw, out0 = (p0 * g.oh + oy_lo) * g.ow;
    const uint32_t outputs = planes * rows_out * g.ow, vectors = outputs > kSteps * kBlock ? outputs / 4 : 0;
    Pack<4> d[kLoads], at[kLoads];
    const auto fetch = [&](uint32_t first) {
#pragma unroll
        for (int u = 0; u < kLoads; ++u) {
            const uint32_t i = first + u * kBlock + threadIdx.x;
            if (i >= vectors) continue;
            d[u] = ld_word<false>(delta + out0 + 4 * static_cast<size_t>(i));
            at[u] = ld_word<false>(reinterpret_cast<const float*>(indexes) + out0 + 4 * static_cast<size_t>(i));
        }
    };
    fetch(0);
    for (uint32_t i = threadIdx.x; i < words * tile_cells; i += kBlock) masks[i] = 0;
    if (threadIdx.x == 0) listed_count = 0;
    __syncthreads();
    // output (row, ox) of the plane, `j` of the tile
    const auto take = [&](uint32_t j, uint32_t plane, uint32_t row, uint32_t ox, float value, int index) {
        deltas[j] = value;
        const uint32_t cell = static_cast<uint32_t>(index) - cell0;     // negative: beyond any tile
        if (cell >= cells) return;
        uint32_t ty, tx;
        if constexpr (K > 0) {
            const int y0 = oy_lo + static_cast<int>(row) + g.origin - y_lo, x0 = static_cast<int>(ox) + g.origin;
            const int from = (static_cast<int>(plane) * rows_in + y0) * g.iw + x0;
            const int away = static_cast<int>(cell) - from;
            if (away < 0) return;
            by_iw.divmod(away, ty, tx);
            if (ty >= K || tx >= K || static_cast<uint32_t>(x0 + static_cast<int>(tx)) >= static_cast<uint32_t>(g.iw) ||
                static_cast<uint32_t>(y0 + static_cast<int>(ty)) >= static_cast<uint32_t>(rows_in))
                return;
        } else {
            uint32_t y, x, cell_plane = 0;
            by_iw.divmod(cell, y, x);
            if (tile.strips == 1) by_ih.divmod(y, cell_plane, y);
            ty = y_lo + y - g.origin - (oy_lo + row) * g.stride;
            tx = x - g.origin - ox * g.stride;
            if (plane != cell_plane || ty >= static_cast<uint32_t>(k) || tx >= static_cast<uint32_t>(k)) return;
        }
        const uint32_t bit = by_stride(k - 1 - ty) * along + by_stride(k - 1 - tx);
        atomicOr(&masks[(bit >> 5) * tile_cells + cell], 1u << (bit & 31));
    };
    const auto place = [&](uint32_t j, uint32_t& plane, uint32_t& row, uint32_t& ox) {
        by_ow.divmod(j, row, ox);
        plane = 0;
        if (tile.strips == 1) by_oh.divmod(row, plane, row);
    };
    for (uint32_t first = 0; first < vectors; first += kLoads * kBlock) {
        if (first) fetch(first);
#pragma unroll
        for (int u = 0; u < kLoads; ++u) {
            const uint32_t i = first + u * kBlock + threadIdx.x;
            if (i >= vectors) continue;
            uint32_t plane, row, ox;
            place(4 * i, plane, row, ox);
#pragma unroll
            for (int q = 0; q < 4; ++q) {
                take(4 * i + q, plane, row, ox, d[u].v[q], __float_as_int(at[u].v[q]));
                if (++ox == static_cast<uint32_t>(g.ow)) {
                    ox = 0;
                    if (++row == static_cast<uint32_t>(rows_out)) {
                        row = 0;
                        ++plane;
                    }
                }
            }
        }
    }
#pragma unroll
    for (uint32_t step = 0; step < kSteps; ++step) {
        const uint32_t j = 4 * vectors + step * kBlock + threadIdx.x;
        if (j >= outputs) break;
        uint32_t plane, row, ox;
        place(j, plane, row, ox);
        take(j, plane, row, ox, delta[out0 + j], indexes[out0 + j]);
    }
    __syncthreads();
    const uint32_t lane = threadIdx.x & (kWave - 1);
    for (uint32_t i0 = threadIdx.x - lane; i0 < cells; i0 += kBlock) {
        const uint32_t i = i0 + lane;
        uint32_t any = 0;
        if (i < cells)
            for (uint32_t word = 0; word < words; ++word) any |= masks[word * tile_cells + i];
        const uint64_t hit = __ballot(any != 0);
        if (hit == 0) continue;
        uint32_t next = 0;
        if (lane == 0) next = atomicAdd(&listed_count, static_cast<uint32_t>(__popcll(hit)));
        next = __builtin_amdgcn_readfirstlane(next);
        if (any) listed[next + __popcll(hit & ((1ull << lane) - 1))] = static_cast<uint16_t>(i);
    }
    __syncthreads();
    for (uint32_t n = threadIdx.x; n < listed_count; n += kBlock) {
        const uint32_t cell = listed[n];
        float acc = grad[cell0 + cell];
        uint32_t y, x, plane = 0;
        by_iw.divmod(cell, y, x);
        if (tile.strips == 1) by_ih.divmod(y, plane, y);
        // the first window that reaches the cell along each axis (it may lie before the first output)
        const int lift = k * g.stride;
        const int oy = static_cast<int>(by_stride(y_lo + y - g.origin - k + g.stride + lift)) - k;
        const int ox = static_cast<int>(by_stride(x - g.origin - k + g.stride + lift)) - k;
        int first = (static_cast<int>(plane) * rows_out + oy - oy_lo) * g.ow + ox;
        if constexpr (K == 0) asm volatile("" : "+v"(first));      // formed here, not in parts between the additions, which are a chain
        for (uint32_t word = 0; word < words; ++word)
            for (uint32_t bits = masks[word * tile_cells + cell]; bits; bits &= bits - 1) {
                const uint32_t bit = word * 32 + __builtin_ctz(bits);
                if constexpr (K > 0) {
                    const uint32_t wy = bit / K, wx = bit - wy * K;
                    acc += deltas[first + static_cast<int>(wy) * g.ow + static_cast<int>(wx)];
                } else {
                    acc += deltas[first + static_cast<int>(bit) + static_cast<int>(w.by_along.div(bit)) * past];
                }
            }
        grad[cell0 + cell] = acc;
    }
}

// Backward for the 2x2 / stride 2 in-bounds case: one window per output, VX windows per lane,
// the two grad rows are updated as full vectors so the read-modify-write stays coalesced.
template<int VX, bool NT>
__global__ __launch_bounds__(kBlock) void maxpool_bwd_2x2_kernel(const float* delta, const int* indexes, float* grad,
                                                                 uint32_t units, int iw, int ow, FastDiv by_owv,
                                                                 FastDiv by_oh)
{
    const uint32_t t = blockIdx.x * kBlock + threadIdx.x;
    if (t >= units) return;
    uint32_t rows, oxv, plane, oy;
    by_owv.divmod(t, rows, oxv);
    by_oh.divmod(rows, plane, oy);
    const uint32_t ih = by_oh.d * 2;
    const uint32_t ox = oxv * VX;
    const uint32_t in0 = (plane * ih + 2 * oy) * iw + 2 * ox;
    const uint32_t o = (plane * by_oh.d + oy) * ow + ox;
    const Pack<VX> d = ld<VX, NT>(delta, o);
    const IPack<VX> ix = ldi<VX, NT>(indexes, o);
    Pack<2 * VX> g0 = ld<2 * VX, NT>(grad, in0);
    Pack<2 * VX> g1 = ld<2 * VX, NT>(grad, in0 + iw);
#pragma unroll
    for (int k = 0; k < VX; ++k) {
        const int at = ix.v[k];
        const int base = static_cast<int>(in0) + 2 * k;
        if (at == base) g0.v[2 * k] += d.v[k];
        else if (at == base + 1) g0.v[2 * k + 1] += d.v[k];
        else if (at == base + iw) g1.v[2 * k] += d.v[k];
        else if (at == base + iw + 1) g1.v[2 * k + 1] += d.v[k];
    }
    st<2 * VX, NT>(grad, in0, g0);
    st<2 * VX, NT>(grad, in0 + iw, g1);
}

// The pair form of the backward pass: the even lane reads the pair's 4 deltas, the odd lane its
// 4 indexes, they swap halves, and every lane updates 4 floats of each of the two grad rows.
template<bool NT>
__global__ __launch_bounds__(kBlock) void maxpool_bwd_2x2_pair_kernel(const float* delta, const int* indexes,
                                                                      float* grad, uint32_t lanes, int iw, int ow,
                                                                      FastDiv by_owh, FastDiv by_oh)
{
    const uint32_t t = blockIdx.x * kBlock + threadIdx.x;
    const bool live = t < lanes;
    const uint32_t u = live ? t : 0;
    const uint32_t half = u & 1;
    uint32_t rows, oxh, plane, oy;
    by_owh.divmod(u, rows, oxh);
    by_oh.divmod(rows, plane, oy);
    const uint32_t ih = by_oh.d * 2;
    const uint32_t ox = oxh * 2;
    const uint32_t in0 = (plane * ih + 2 * oy) * iw + 2 * ox;
    const uint32_t o = (u >> 1) * 4;
    // one 128-bit load per lane: deltas (even) or indexes (odd), as raw bits
    const Pack<4> mine = half == 0 ? ld<4, NT>(delta, o) : ld<4, NT>(reinterpret_cast<const float*>(indexes), o);
    Pack<4> theirs;
#pragma unroll
    for (int k = 0; k < 4; ++k) theirs.v[k] = __shfl_xor(mine.v[k], 1, kWave);
    // this lane's two windows are outputs 2*half, 2*half + 1 of the pair
    float d[2];
    int ix[2];
    if (half == 0) {
        d[0] = mine.v[0]; d[1] = mine.v[1];
        ix[0] = __float_as_int(theirs.v[0]); ix[1] = __float_as_int(theirs.v[1]);
    } else {
        d[0] = theirs.v[2]; d[1] = theirs.v[3];
        ix[0] = __float_as_int(mine.v[2]); ix[1] = __float_as_int(mine.v[3]);
    }
    if (!live) return;
    Pack<4> g0 = ld<4, NT>(grad, in0);
    Pack<4> g1 = ld<4, NT>(grad, in0 + iw);
#pragma unroll
    for (int k = 0; k < 2; ++k) {
        const int at = ix[k];
        const int base = static_cast<int>(in0) + 2 * k;
        if (at == base) g0.v[2 * k] += d[k];
        else if (at == base + 1) g0.v[2 * k + 1] += d[k];
        else if (at == base + iw) g1.v[2 * k] += d[k];
        else if (at == base + iw + 1) g1.v[2 * k + 1] += d[k];
    }
    st<4, NT>(grad, in0, g0);
    st<4, NT>(grad, in0 + iw, g1);
}

__global__ __launch_bounds__(kBlock) void maxpool_bwd_scatter_kernel(const float* delta, const int* indexes,
                                                                     float* grad, int size)
{
    const int i = blockIdx.x * kBlock + threadIdx.x;
    if (i >= size) return;
    const int at = indexes[i];
    if (at >= 0) atomicAdd(grad + at, delta[i]);
}

// ------------------------------------------------------------------ upsample
// The large tensor may be a channel slice of a wider one (a concatenation buffer): image n then
// starts `extra` elements later than in a dense tensor, for every image before it.
struct ImageGap {
    FastDiv by_channels;
    uint32_t extra;     // image stride of the large tensor minus channels * its plane size
    __device__ uint32_t of_plane(uint32_t plane) const { return extra ? by_channels.div(plane) * extra : 0u; }
};

// stride 2: VX inputs per lane; forward writes the 2 x (2*VX) block, backward folds it into the
// input cell as (((acc + s*o00) + s*o01) + s*o10) + s*o11, the raster order of the CPU loop.
template<int VX, bool FORWARD>
__global__ __launch_bounds__(kBlock) void upsample2_kernel(const float* in, float* acc, float* out, uint32_t units,
                                                           int w, float scale, FastDiv by_wv, FastDiv by_h,
                                                           ImageGap gap)
{
    const uint32_t t = blockIdx.x * kBlock + threadIdx.x;
    if (t >= units) return;
    uint32_t rows, xv, plane, y;
    by_wv.divmod(t, rows, xv);
    by_h.divmod(rows, plane, y);
    const uint32_t x = xv * VX;
    const uint32_t ii = rows * w + x;                                   // rows = plane*h + y
    const uint32_t ow = 2 * w;
    const uint32_t oi = (2 * rows) * ow + 2 * x + gap.of_plane(plane);  // (plane*2h + 2y)*2w + 2x
    if constexpr (FORWARD) {
        const Pack<VX> v = ld<VX>(in, ii);
        Pack<2 * VX> o;
#pragma unroll
        for (int k = 0; k < VX; ++k) {
            const float s = scale * v.v[k];
            o.v[2 * k] = s;
            o.v[2 * k + 1] = s;
        }
        st<2 * VX>(out, oi, o);
        st<2 * VX>(out, oi + ow, o);
    } else {
        Pack<VX> a = ld<VX>(acc, ii);
        const Pack<2 * VX> r0 = ld<2 * VX>(out, oi);
        const Pack<2 * VX> r1 = ld<2 * VX>(out, oi + ow);
#pragma unroll
        for (int k = 0; k < VX; ++k) {
            float g = a.v[k];
            float p = scale * r0.v[2 * k];
            g = g + p;
            p = scale * r0.v[2 * k + 1];
            g = g + p;
            p = scale * r1.v[2 * k];
            g = g + p;
            p = scale * r1.v[2 * k + 1];
            g = g + p;
            a.v[k] = g;
        }
        st<VX>(acc, ii, a);
    }
}

// any stride: one input cell per lane
template<bool FORWARD>
__global__ __launch_bounds__(kBlock) void upsample_generic_kernel(const float* in, float* acc, float* out,
                                                                  uint32_t total, int w, int stride, float scale,
                                                                  FastDiv by_w, FastDiv by_h, ImageGap gap)
{
    const uint32_t cell = blockIdx.x * kBlock + threadIdx.x;
    if (cell >= total) return;
    uint32_t rows, x, plane, y;
    by_w.divmod(cell, rows, x);
    by_h.divmod(rows, plane, y);
    const size_t ow = static_cast<size_t>(w) * stride;
    const size_t o0 = static_cast<size_t>(rows) * stride * ow + static_cast<size_t>(x) * stride + gap.of_plane(plane);
    if constexpr (FORWARD) {
        const float s = scale * in[cell];
        for (int dy = 0; dy < stride; ++dy)
            for (int dx = 0; dx < stride; ++dx) out[o0 + dy * ow + dx] = s;
    } else {
        float g = acc[cell];
        for (int dy = 0; dy < stride; ++dy)
            for (int dx = 0; dx < stride; ++dx) {
                const float p = scale * out[o0 + dy * ow + dx];
                g = g + p;
            }
        acc[cell] = g;
    }
}

int check_pool_args(const char* who, int batch, int channels, int ih, int iw, int oh, int ow, int kernel, int stride,
                    int padding)
{
    if (batch <= 0 || channels <= 0 || ih <= 0 || iw <= 0 || oh <= 0 || ow <= 0)
        return fail_invalid("%s: dimensions must be positive", who);
    if (kernel <= 0) return fail_invalid("%s: MaxPool kernel must be positive", who);
    if (stride <= 0) return fail_invalid("%s: MaxPool stride must be positive", who);
    if (padding < 0) return fail_invalid("%s: MaxPool padding cannot be negative", who);
    const unsigned long long in_total = 1ull * batch * channels * ih * iw;
    const unsigned long long out_total = 1ull * batch * channels * oh * ow;
    if (in_total >= (1ull << 31) || out_total >= (1ull << 31)) {
        // the index tensor is int32: larger inputs cannot be represented by the layer at all
        set_error("%s: tensors of 2^31 elements or more are not supported", who);
        return PXH_ERR_UNSUPPORTED;
    }
    return PXH_OK;
}

// all windows 2x2, stride 2, inside the input
bool is_2x2_inbounds(int ih, int iw, int oh, int ow, int kernel, int stride, int padding)
{
    return kernel == 2 && stride == 2 && padding <= 1 && ih % 2 == 0 && iw % 2 == 0 && oh == ih / 2 && ow == iw / 2;
}

// Tiles of about `target` cells: whole planes while one fits, else strips.  `rows` and `width` are those of the
// tensor that is tiled.
PoolTile pool_tile(uint32_t planes, int rows, int width, uint32_t target)
{
    PoolTile t{ planes, 1, 1, static_cast<uint32_t>(rows) };
    const uint32_t plane = static_cast<uint32_t>(rows) * width;
    if (plane <= target) {
        t.per_tile = target / plane;
        // enough workgroups for the chip before larger ones
        const uint32_t spread = planes / 1024 > 0 ? planes / 1024 : 1;
        if (t.per_tile > spread) t.per_tile = spread;
        return t;
    }
    t.rows = target / width > 0 ? target / width : 1;
    t.strips = (rows + t.rows - 1) / t.rows;
    return t;
}

constexpr size_t kPoolLds = 40u << 10;      // four workgroups per compute unit
constexpr uint32_t kPoolCells = 2048;       // eight per lane; halved until the tile fits

// Launches the tiled forward pass; false when the geometry does not suit it.
bool launch_fwd_tile(const float* in, float* out, int* indexes, uint32_t planes, const PoolGeom& g, hipStream_t s)
{
    // Every input is a tap of (k / stride)^2 windows.  Measured, us one lane per output -> tiled: 3 / 1, 64 planes
    // of 300 x 300, 45 -> 20; 5 / 1, 8192 of 19 x 19, 44 -> 13; 13 / 1 190 -> 19; but 3 / 2, 64 of 300 x 300,
    // 13.3 -> 18.8 (and 2 / 1 in a form of its own, above): with so few taps the detour through LDS costs more.
    if (g.kernel > 64 || g.kernel * g.kernel < 8 * g.stride * g.stride) return false;
    for (uint32_t target = kPoolCells; target >= 256; target /= 2) {
        const PoolTile t = pool_tile(planes, g.oh, g.ow, target);
        // strips of few rows read most of their input for the rows of the next one
        if (t.strips > 1 && t.rows * g.stride < static_cast<uint32_t>(g.kernel)) return false;
        const size_t frame_h = static_cast<size_t>(t.rows - 1) * g.stride + g.kernel;
        const size_t frame_w = static_cast<size_t>(g.ow - 1) * g.stride + g.kernel;
        const size_t rows_in = t.strips == 1 ? g.ih : std::min<size_t>(g.ih, frame_h);
        const size_t cells = t.per_tile * rows_in * frame_w, segments = t.per_tile * frame_h * g.ow;
        const size_t bytes = cells * 4 + segments * 5;
        const dim3 grid((planes + t.per_tile - 1) / t.per_tile * t.strips);
        const uint32_t groups = static_cast<uint32_t>(g.ow + 3) / 4;
        // A lane takes four outputs a step: a tile needs two for each lane before that is shorter than one output per lane.  us,
        // k = 5 and 13, 512 planes of 13 x 13 3.4 -> 4.0 and 3.7 -> 4.6, of 19 x 19 4.1 -> 4.4 and 4.6 -> 5.3, but of 26 x 26 4.9 -> 4.5 and
        // 5.7 -> 5.4.  (Windows: those that have a form of their own, whose runs are unrolled.)
        const SlideTile st{ slide_pitch(g.kernel, groups), groups };
        const bool runs = t.per_tile * t.rows * static_cast<uint32_t>(g.ow) > 2 * kBlock;
        const size_t slide_bytes = t.per_tile * rows_in * (4 * st.pitch + 5 * 4 * groups);
        const auto slide = [&]<int K>() {
            hipLaunchKernelGGL((maxpool_fwd_slide_kernel<K>), grid, dim3(kBlock), slide_bytes, s, in, out, indexes, t, g, st,
                               FastDiv(t.strips), FastDiv(g.iw), FastDiv(groups), FastDiv(g.ow),
                               FastDiv((t.rows + kSlideRun - 1) / kSlideRun));
            return true;
        };
        if (g.stride == 1 && slide_bytes <= kPoolLds && runs) {
            if (g.kernel == 3) return slide.template operator()<3>();
            if (g.kernel == 5) return slide.template operator()<5>();
            if (g.kernel == 9) return slide.template operator()<9>();
            if (g.kernel == 13) return slide.template operator()<13>();
        }
        if (bytes > kPoolLds) continue;
#define PXH_POOL_TILE(K)                                                                                       \
        hipLaunchKernelGGL((maxpool_fwd_tile_kernel<K>), grid, dim3(kBlock), bytes, s, in, out, indexes, t, g, \
                           FastDiv(t.strips), FastDiv(g.iw), FastDiv(g.ih), FastDiv(g.ow), FastDiv(g.oh),      \
                           static_cast<uint32_t>(cells), static_cast<uint32_t>(segments))
        switch (g.kernel) {
        case 3: PXH_POOL_TILE(3); break;
        case 5: PXH_POOL_TILE(5); break;
        case 9: PXH_POOL_TILE(9); break;
        case 13: PXH_POOL_TILE(13); break;
        default: PXH_POOL_TILE(0);
        }
#undef PXH_POOL_TILE
        return true;
    }
    return false;
}

bool launch_bwd_tile(const float* delta, const int* indexes, float* grad, uint32_t planes, const PoolGeom& g,
                     hipStream_t s)
{
    // masks of up to eight words; few windows per cell gain less (2 / 2, 1024 planes of 151 x 151, 86 -> 53 us; 3 / 2,
    // 64 of 300 x 300, 38 -> 19), and launches too small to matter stay level
    if (g.kernel > 16 || g.stride > 16) return false;
    PoolWindows w;
    w.along = (g.kernel + g.stride - 1) / g.stride;
    w.words = static_cast<uint32_t>(w.along * w.along + 31) / 32;
    w.by_stride = FastDiv(g.stride);
    w.by_along = FastDiv(w.along);
    for (uint32_t target = kPoolCells; target >= 256; target /= 2) {
        const PoolTile t = pool_tile(planes, g.ih, g.iw, target);
        if (t.strips > 1 && t.rows < static_cast<uint32_t>(g.kernel)) return false;
        const size_t cells = static_cast<size_t>(t.per_tile) * t.rows * g.iw;
        const size_t rows_out = t.strips == 1 ? g.oh : std::min<size_t>(g.oh, (t.rows + g.kernel - 2) / g.stride + 2);
        const size_t outputs = t.per_tile * rows_out * g.ow;
        const size_t bytes = cells * (4 * w.words + 2) + outputs * 4;
        if (bytes > kPoolLds) continue;
        const dim3 grid((planes + t.per_tile - 1) / t.per_tile * t.strips);
        const auto launch = [&]<int K>() {
            hipLaunchKernelGGL((maxpool_bwd_tile_kernel<K>), grid, dim3(kBlock), bytes, s, delta, indexes, grad, t, g, w,
                               FastDiv(t.strips), FastDiv(g.ow), FastDiv(g.oh), FastDiv(g.iw), FastDiv(g.ih),
                               static_cast<uint32_t>(cells), static_cast<uint32_t>(outputs));
        };
        switch (g.stride == 1 && g.iw >= g.kernel ? g.kernel : 0) {
        case 2: launch.template operator()<2>(); break;
        case 3: launch.template operator()<3>(); break;
        case 5: launch.template operator()<5>(); break;
        case 9: launch.template operator()<9>(); break;
        case 13: launch.template operator()<13>(); break;
        default: launch.template operator()<0>();
        }
        return true;
    }
    return false;
}

}  // namespace
}  // namespace pxh

using namespace pxh;

extern "C" {

int pxh_maxpool_forward(const float* in, float* out, int* indexes, int batch, int channels, int ih, int iw, int oh,
                        int ow, int kernel, int stride, int padding, void* stream)
{
    if (!in || !out || !indexes) return fail_invalid("pxh_maxpool_forward: null pointer");
    int rc = check_pool_args("pxh_maxpool_forward", batch, channels, ih, iw, oh, ow, kernel, stride, padding);
    if (rc) return rc;
    hipStream_t s = as_stream(stream);
    const uint32_t planes = static_cast<uint32_t>(batch) * channels;
    const uint32_t total = planes * oh * ow;
    if (is_2x2_inbounds(ih, iw, oh, ow, kernel, stride, padding) && aligned16(in) && aligned16(out) &&
        aligned16(indexes)) {
        // 4 bytes in, 8 bytes out per input element / 4
        const bool nt = static_cast<size_t>(total) * 24 >= kStreamingBytes;
        // the pair form needs an even output width and whole output quads; it pays for wide rows
        if (iw % 8 == 0 && total % 4 == 0) {
            const uint32_t lanes = total / 2;
            const dim3 grid(grid_for(lanes, kBlock));
            if (nt) hipLaunchKernelGGL((maxpool_fwd_2x2_pair_kernel<true>), grid, dim3(kBlock), 0, s, in, out, indexes,
                                       lanes, iw, ow, FastDiv(ow / 2), FastDiv(oh));
            else hipLaunchKernelGGL((maxpool_fwd_2x2_pair_kernel<false>), grid, dim3(kBlock), 0, s, in, out, indexes,
                                    lanes, iw, ow, FastDiv(ow / 2), FastDiv(oh));
        } else if (iw % 4 == 0) {
            const uint32_t units = total / 2;
            const dim3 grid(grid_for(units, kBlock));
            if (nt) hipLaunchKernelGGL((maxpool_fwd_2x2_kernel<2, true>), grid, dim3(kBlock), 0, s, in, out, indexes,
                                       units, iw, ow, FastDiv(ow / 2), FastDiv(oh));
            else hipLaunchKernelGGL((maxpool_fwd_2x2_kernel<2, false>), grid, dim3(kBlock), 0, s, in, out, indexes,
                                    units, iw, ow, FastDiv(ow / 2), FastDiv(oh));
        } else {
            const dim3 grid(grid_for(total, kBlock));
            if (nt) hipLaunchKernelGGL((maxpool_fwd_2x2_kernel<1, true>), grid, dim3(kBlock), 0, s, in, out, indexes,
                                       total, iw, ow, FastDiv(ow), FastDiv(oh));
            else hipLaunchKernelGGL((maxpool_fwd_2x2_kernel<1, false>), grid, dim3(kBlock), 0, s, in, out, indexes,
                                    total, iw, ow, FastDiv(ow), FastDiv(oh));
        }
        return check_launch("pxh_maxpool_forward");
    }
    const PoolGeom g{ ih, iw, oh, ow, kernel, stride, -padding / 2 };
    if (kernel == 2 && stride == 1 && g.origin == 0 && oh == ih && ow == iw) {
        hipLaunchKernelGGL(maxpool_fwd_step1_kernel, dim3(grid_for(total, static_cast<size_t>(kBlock) * 4)), dim3(kBlock), 0, s,
                           in, out, indexes, total, FastDiv(ow), FastDiv(oh));
        return check_launch("pxh_maxpool_forward");
    }
    if (launch_fwd_tile(in, out, indexes, planes, g, s)) return check_launch("pxh_maxpool_forward");
    hipLaunchKernelGGL(maxpool_fwd_generic_kernel, dim3(grid_for(total, kBlock)), dim3(kBlock), 0, s, in, out, indexes,
                       total, g, FastDiv(ow), FastDiv(oh));
    return check_launch("pxh_maxpool_forward");
}

int pxh_maxpool_backward(const float* delta, const int* indexes, float* grad, int batch, int channels, int ih, int iw,
                         int oh, int ow, int kernel, int stride, int padding, void* stream)
{
    if (!delta || !indexes || !grad) return fail_invalid("pxh_maxpool_backward: null pointer");
    int rc = check_pool_args("pxh_maxpool_backward", batch, channels, ih, iw, oh, ow, kernel, stride, padding);
    if (rc) return rc;
    hipStream_t s = as_stream(stream);
    const uint32_t planes = static_cast<uint32_t>(batch) * channels;
    const uint32_t out_total = planes * oh * ow;
    if (is_2x2_inbounds(ih, iw, oh, ow, kernel, stride, padding) && aligned16(delta) && aligned16(indexes) &&
        aligned16(grad)) {
        // 8 bytes per output, 8 bytes per grad cell
        const bool nt = static_cast<size_t>(out_total) * 40 >= kStreamingBytes;
        if (iw % 8 == 0 && out_total % 4 == 0) {
            const uint32_t lanes = out_total / 2;
            const dim3 grid(grid_for(lanes, kBlock));
            if (nt) hipLaunchKernelGGL((maxpool_bwd_2x2_pair_kernel<true>), grid, dim3(kBlock), 0, s, delta, indexes,
                                       grad, lanes, iw, ow, FastDiv(ow / 2), FastDiv(oh));
            else hipLaunchKernelGGL((maxpool_bwd_2x2_pair_kernel<false>), grid, dim3(kBlock), 0, s, delta, indexes,
                                    grad, lanes, iw, ow, FastDiv(ow / 2), FastDiv(oh));
        } else if (iw % 4 == 0) {
            const uint32_t units = out_total / 2;
            const dim3 grid(grid_for(units, kBlock));
            if (nt) hipLaunchKernelGGL((maxpool_bwd_2x2_kernel<2, true>), grid, dim3(kBlock), 0, s, delta, indexes,
                                       grad, units, iw, ow, FastDiv(ow / 2), FastDiv(oh));
            else hipLaunchKernelGGL((maxpool_bwd_2x2_kernel<2, false>), grid, dim3(kBlock), 0, s, delta, indexes, grad,
                                    units, iw, ow, FastDiv(ow / 2), FastDiv(oh));
        } else {
            const dim3 grid(grid_for(out_total, kBlock));
            if (nt) hipLaunchKernelGGL((maxpool_bwd_2x2_kernel<1, true>), grid, dim3(kBlock), 0, s, delta, indexes,
                                       grad, out_total, iw, ow, FastDiv(ow), FastDiv(oh));
            else hipLaunchKernelGGL((maxpool_bwd_2x2_kernel<1, false>), grid, dim3(kBlock), 0, s, delta, indexes, grad,
                                    out_total, iw, ow, FastDiv(ow), FastDiv(oh));
        }
        return check_launch("pxh_maxpool_backward");
    }
    const PoolGeom g{ ih, iw, oh, ow, kernel, stride, -padding / 2 };
    if (launch_bwd_tile(delta, indexes, grad, planes, g, s)) return check_launch("pxh_maxpool_backward");
    const uint32_t in_total = planes * ih * iw;
    hipLaunchKernelGGL(maxpool_bwd_generic_kernel, dim3(grid_for(in_total, kBlock)), dim3(kBlock), 0, s, delta,
                       indexes, grad, in_total, g, FastDiv(iw), FastDiv(ih));
    return check_launch("pxh_maxpool_backward");
}

int pxh_maxpool_backward_scatter(const float* delta, const int* indexes, float* grad, int size, void* stream)
{
    if (size < 0 || ((!delta || !indexes || !grad) && size)) return fail_invalid("pxh_maxpool_backward_scatter: bad argument");
    if (size == 0) return PXH_OK;
    hipLaunchKernelGGL(maxpool_bwd_scatter_kernel, dim3(grid_for(size, kBlock)), dim3(kBlock), 0, as_stream(stream),
                       delta, indexes, grad, size);
    return check_launch("pxh_maxpool_backward_scatter");
}

int pxh_upsample_strided(const float* in, int w, int h, int c, int batch, int stride, int forward, float scale,
                         float* acc, float* out, long long out_image_stride, void* stream)
{
    if (w <= 0 || h <= 0 || c <= 0 || batch <= 0 || stride <= 0)
        return fail_invalid("pxh_upsample: dimensions and stride must be positive");
    if (!out || (forward && !in) || (!forward && !acc)) return fail_invalid("pxh_upsample: null pointer");
    const unsigned long long image = 1ull * c * h * w * stride * stride;
    if (out_image_stride < 0 || static_cast<unsigned long long>(out_image_stride) < image)
        return fail_invalid("pxh_upsample: image stride %lld is smaller than one upsampled image (%llu)",
                            out_image_stride, image);
    if (1ull * batch * static_cast<unsigned long long>(out_image_stride) >= (1ull << 31)) {
        set_error("pxh_upsample: tensors of 2^31 elements or more are not supported");
        return PXH_ERR_UNSUPPORTED;
    }
    hipStream_t s = as_stream(stream);
    const uint32_t total = static_cast<uint32_t>(batch) * c * h * w;
    const ImageGap gap{ FastDiv(c), static_cast<uint32_t>(static_cast<unsigned long long>(out_image_stride) - image) };
    const float* small = forward ? in : acc;
    if (stride == 2 && aligned16(small) && aligned16(out) && gap.extra % 4 == 0) {
        // VX inputs per lane; the input vector needs 4*VX-byte alignment of every row start
        const int vx = (w % 4 == 0) ? 4 : (w % 2 == 0 ? 2 : 1);
        const uint32_t units = total / vx;
        const dim3 grid(grid_for(units, kBlock));
#define PXH_UPSAMPLE2(VX, FWD)                                                                              \
        hipLaunchKernelGGL((upsample2_kernel<VX, FWD>), grid, dim3(kBlock), 0, s, in, acc, out, units, w, \
                           scale, FastDiv(w / VX), FastDiv(h), gap)
        if (forward) {
            if (vx == 4) PXH_UPSAMPLE2(4, true); else if (vx == 2) PXH_UPSAMPLE2(2, true); else PXH_UPSAMPLE2(1, true);
        } else {
            if (vx == 4) PXH_UPSAMPLE2(4, false); else if (vx == 2) PXH_UPSAMPLE2(2, false); else PXH_UPSAMPLE2(1, false);
        }
#undef PXH_UPSAMPLE2
        return check_launch("pxh_upsample");
    }
    const dim3 grid(grid_for(total, kBlock));
    if (forward) {
        hipLaunchKernelGGL((upsample_generic_kernel<true>), grid, dim3(kBlock), 0, s, in, acc, out, total, w, stride,
                           scale, FastDiv(w), FastDiv(h), gap);
    } else {
        hipLaunchKernelGGL((upsample_generic_kernel<false>), grid, dim3(kBlock), 0, s, in, acc, out, total, w, stride,
                           scale, FastDiv(w), FastDiv(h), gap);
    }
    return check_launch("pxh_upsample");
}

int pxh_upsample(const float* in, int w, int h, int c, int batch, int stride, int forward, float scale, float* acc,
                 float* out, void* stream)
{
    if (w <= 0 || h <= 0 || c <= 0 || batch <= 0 || stride <= 0)
        return fail_invalid("pxh_upsample: dimensions and stride must be positive");
    return pxh_upsample_strided(in, w, h, c, batch, stride, forward, scale, acc, out,
                                1ll * c * h * w * stride * stride, stream);
}

}
