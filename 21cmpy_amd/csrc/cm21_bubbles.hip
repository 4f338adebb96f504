// find_HII_bubbles on the GPU: k-space filter, f_coll with its FP64 box sum,
// threshold / final paint, sphere paint and the radius-loop driver.
//
// Reference: Programs/find_bubbles.cu:12-158 (kernels) and
// Programs/find_HII_bubbles.py:17-193 (loop).  Differences by design:
//  * the forward transform runs once per box (the reference re-uploads and
//    re-transforms the same box every radius, find_HII_bubbles.py:141-144);
//  * the 1/N of the inverse transform and the growth factor of nonlinear
//    input are folded into the filter multiply;
//  * the box mean of f_coll is an FP64 device scalar read by the threshold
//    kernel, so the loop never synchronises with the host.
#include <algorithm>
#include <cmath>
#include <cstring>
#include <mutex>
#include <unordered_map>
#include <vector>

#include "cm21_internal.hpp"
#include "cm21_window.hpp"
#include "cm21_fused_dev.hpp"

using namespace cm21;

namespace {

constexpr int kThreshCells = 4 * kThreads;  // cells per threshold block
constexpr size_t kChunkAlign = kThreshCells;

// W(kR) times the spectrum.  Bound by memory where modes survive (2 x 8 bytes a
// mode); a mode that the cut surely takes (|k|R 0.1 % past it) is written as
// zero without being read and without the FP64 root and the Gaussian of the
// exact test.  The blocks run over the D*H modes of a plane in memory order (64
// modes of a row to a block left 49 % of the lanes idle at H = 65 and 21 % at
// H = 101); (i * row_magic) >> 32 is i / H there.  At 200^3, over the 37 radii of a
// k-space top-hat, 22.5 -> 9.5 us a radius.
__global__ void k_filter(float2* __restrict__ out, const float2* __restrict__ in, int D, WindowParams wp,
                         float scale, float ksq_cut, unsigned row_magic) {
    const unsigned H = D / 2 + 1, i = blockIdx.x * kThreads + threadIdx.x;
    if (i >= D * H) return;
    const int a = blockIdx.y, b = (int)__umulhi(i, row_magic), c = (int)(i - b * H);
    const size_t idx = (size_t)a * D * H + i;
    const float ka = (float)mode_of(a, D) * wp.dk, kb = (float)mode_of(b, D) * wp.dk, kc = (float)c * wp.dk;
    if (ka * ka + kb * kb + kc * kc > ksq_cut) {
        out[idx] = make_float2(0.0f, 0.0f);
        return;
    }
    float w0, w2;
    bool cut;
    window_of(kmag_of(a, b, c, D, wp.dk, wp.korder), wp, w0, cut, w2);
    out[idx] = apply_window(in[idx], w0, cut, w2, scale);
}

__global__ void k_fill(float* __restrict__ p, size_t n, float v) {
    const size_t i = (size_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (i < n) p[i] = v;
}

// Cells per block of the f_coll sum: consecutive cells, so that the maximum a
// block stores lets the threshold and the sphere paint pass its cells over.
inline size_t sum_chunk(size_t N) { return align_up((N + kReduceBlocks - 1) / kReduceBlocks, kChunkAlign); }

// FP64 partial sum of f_coll and maximum of the smoothed field of a chunk.
// Bound by the VALU (erfcf and its divided argument).
__global__ void k_fcoll_partial(const float* __restrict__ sm, size_t N, size_t chunk, float deltac, float denom,
                                double* __restrict__ partial, float* __restrict__ cmax) {
    const size_t p0 = (size_t)blockIdx.x * chunk, p1 = p0 + chunk < N ? p0 + chunk : N;
    double acc = 0.0;
    float most = -INFINITY;
    for (size_t p = p0 + threadIdx.x; p < p1; p += blockDim.x) {
        const float d = sm[p];
        acc += (double)fcoll_of(d, deltac, denom);
        most = fmaxf(most, d);  // a NaN is no hit
    }
    acc = block_sum(acc);
    if (threadIdx.x == 0) partial[blockIdx.x] = acc;
    if (cmax) {
        __shared__ float part[kWaves];
#pragma unroll
        for (int off = 32; off > 0; off >>= 1) most = fmaxf(most, __shfl_xor(most, off, 64));
        if ((threadIdx.x & 63) == 0) part[threadIdx.x >> 6] = most;
        __syncthreads();
        if (threadIdx.x == 0) {
            for (int w = 1; w < kWaves; ++w) most = fmaxf(most, part[w]);
            cmax[blockIdx.x] = most;
        }
    }
}

// The centre-pixel test of a radius on the generic path.
struct CellTest {
    float deltac, denom;
    double zeta, inv_zeta;
    const double* sum;              // nonlinear input: the f_coll sum ...
    float fc_mean;
    double ncells;
    const ScaledThreshold* scaled;  // ... or what follows from it, or NULL
    DensityThreshold th;            // linear input
    const float* cmax;              // chunk maxima of the f_coll sum, or NULL
    size_t chunk;
};

// The density threshold holds for f_coll falling with the argument; other
// denominators leave every cell to the float32 test.
__device__ __host__ inline bool plain_denom(float denom) { return denom > 0.0f && denom < INFINITY; }

__device__ inline ScaledThreshold scaled_of_sum(double sum, double ncells, float fc_mean, float deltac, float denom,
                                                double zeta) {
    ScaledThreshold s;
    s.scale = (float)((double)fc_mean / (sum / ncells));
    s.th.dstar = 0.0f;
    s.th.band = INFINITY;
    if (plain_denom(denom)) s.th = density_threshold(deltac, denom, zeta, s.scale);
    s.neutral = 0;
    return s;
}

// Sums `n` partials in a fixed order into *out (one block); with `scaled` also
// the box-mean scale and the density threshold of the radius, once for every
// cell of the following pass (per cell they were two FP64 divisions).
__global__ void k_sum_partials(const double* __restrict__ partial, int n, double* __restrict__ out, CellTest t,
                               ScaledThreshold* __restrict__ scaled) {
    double acc = 0.0;
    for (int i = threadIdx.x; i < n; i += blockDim.x) acc += partial[i];
    acc = block_sum(acc);
    if (threadIdx.x == 0) {
        *out = acc;
        if (scaled) *scaled = scaled_of_sum(acc, t.ncells, t.fc_mean, t.deltac, t.denom, t.zeta);
    }
}

// Scale and threshold of a block.  Without a prepared one (a call of the
// threshold alone) only the scale: its cells take the float32 test.
__device__ inline ScaledThreshold block_threshold(const CellTest& t) {
    if (t.scaled) return *t.scaled;
    ScaledThreshold s{1.0f, t.th, 0};
    if (t.sum) {
        s.scale = (float)((double)t.fc_mean / (*t.sum / t.ncells));
        s.th.dstar = 0.0f;
        s.th.band = INFINITY;
    }
    return s;
}

__device__ __forceinline__ bool cell_hits(float d, const CellTest& t, const ScaledThreshold& s) {
    return cell_hit(d, s.th, t.deltac, t.denom, t.sum != nullptr, s.scale, t.inv_zeta);
}

// Threshold and final paint.  A block takes kThreshCells consecutive cells;
// kThreshCells divides the chunk of the sum, so one maximum tells whether any of
// them can be ionized.  Bound by memory: 22 us at 200^3 with the exact test
// and two FP64 divisions per cell, 5.5 with the density threshold and the maxima.
__global__ void k_threshold(float* __restrict__ ion, const float* __restrict__ sm, size_t N, CellTest t,
                            int final_step) {
    const size_t p0 = (size_t)blockIdx.x * kThreshCells;
    const ScaledThreshold s = block_threshold(t);
    if (!final_step && t.cmax && t.cmax[p0 / t.chunk] < s.th.dstar - s.th.band) return;
#pragma unroll
    for (int k = 0; k < kThreshCells / kThreads; ++k) {
        const size_t p = p0 + k * kThreads + threadIdx.x;
        if (p >= N) return;
        if (ion[p] == 1.0f) continue;
        const float d = sm[p];
        if (cell_hits(d, t, s)) {
            ion[p] = 1.0f;
        } else if (final_step) {
            float f = fcoll_of(d, t.deltac, t.denom);
            if (t.sum) f = __fmul_rn(f, s.scale);
            ion[p] = (float)((double)f * t.zeta);
        }
    }
}

// ------------------------------------------------------------------ sphere paint
// A cell is painted when its squared distance to an ionizing centre is below
// R^2 (Programs/find_bubbles.cu:97-98), in whole numbers: a separable squared
// distance transform over the offsets with o^2 < R^2.
//   rows:   the centres of a line of axis 2 as bits; the distance g to the
//           nearest one along the line by bit scans (kNoCentre: none in reach);
//   planes: h = min over o of g(b + o)^2 + o^2 along axis 1;
//   paint:  whether h(a + o) + o^2 < R^2 for some o along axis 0.
// The rows flag lines without a centre and the planes flag tiles without a
// distance: nothing of those is written or read, and a tile of cells that are
// all painted already is passed over.  Reaches up to kNarrowReach cells (all
// but boxes of very small cells) hold g^2 and h in 16 bits, where sums saturate at
// kNarrowMax, and take the tiles below.  A reach that the side cuts short can come
// with an R^2 beyond that.  Where no cell is as far as R (R >= D in a periodic box, R
// past the diagonal of a clipped one), one centre paints all of it, saturated or not;
// between, only the 32-bit form can compare (180^3 with R = 256.5: 1.66 ms, the
// tiles 0.19; 128^3 periodic with R = 300: 0.30 to 0.42 ms, the tiles 0.05).  The tiles:
// saturating 16-bit adds and minima, two cells an instruction, against a column
// of the tile in LDS, eight cells along the axis per thread, so that one LDS
// read serves eight offsets and the squares stay in scalar registers.
// Bound by those adds and minima, one instruction per cell and offset, and by
// their launches: 4.9 + 3.5 + 4.3 us a radius at 128^3 (reach 0 to 30), for 8.4
// (centres) + 3 x 29.6 (three 32-bit passes from global memory over all offsets) +
// 5 (paint); the whole box 5.45 -> 2.29 ms.
constexpr uint32_t kNoCentre = 0xFFFFu;
constexpr int kNarrowReach = 190;  // the column of a tile stays below 64 KB of LDS
constexpr float kNarrowMax = 65535.0f;
constexpr int kTile = 64;          // cells along either side of a tile
constexpr int kTileRun = 8;        // cells along the axis per thread
static_assert(kTile / kTileRun * (kTile / 2) == kThreads, "one thread per run and pair of lines");

// Position of the nearest set bit at or before x within `reach`, as a distance
// (periodic: also across the line's start), or kNoCentre.
__device__ __forceinline__ uint32_t reach_back(const unsigned long long* words, int nw, int D, int x, int reach,
                                               int periodic) {
    int w = x >> 6;
    unsigned long long m = words[w] & (~0ull >> (63 - (x & 63)));
    while (!m && --w >= 0 && x - (w * 64 + 63) <= reach) m = words[w];
    if (m) return (uint32_t)(x - (w * 64 + 63 - __clzll((long long)m)));
    if (!periodic) return kNoCentre;
    for (w = nw - 1; w >= 0 && x + D - min(w * 64 + 63, D - 1) <= reach; --w)
        if (words[w]) return (uint32_t)(x + D - (w * 64 + 63 - __clzll((long long)words[w])));
    return kNoCentre;
}

__device__ __forceinline__ uint32_t reach_on(const unsigned long long* words, int nw, int D, int x, int reach,
                                             int periodic) {
    int w = x >> 6;
    unsigned long long m = words[w] & (~0ull << (x & 63));
    while (!m && ++w < nw && w * 64 - x <= reach) m = words[w];
    if (m) return (uint32_t)(w * 64 + __ffsll(m) - 1 - x);
    if (!periodic) return kNoCentre;
    for (w = 0; w < nw && w * 64 + D - x <= reach; ++w)
        if (words[w]) return (uint32_t)(w * 64 + __ffsll(words[w]) - 1 + D - x);
    return kNoCentre;
}

// One wave per line of axis 2 (D^2 lines, a multiple of four).
__global__ __launch_bounds__(kThreads) void k_sphere_rows(uint16_t* __restrict__ g, uint8_t* __restrict__ any_row,
                                                          const float* __restrict__ sm, int D, CellTest t, int reach,
                                                          int periodic) {
    __shared__ unsigned long long bits[kWaves][32];
    const int lane = threadIdx.x & 63, w = threadIdx.x >> 6, nw = (D + 63) >> 6;
    const size_t row = (size_t)blockIdx.x * kWaves + w, p0 = row * D;
    const ScaledThreshold s = block_threshold(t);
    bool quiet = false;
    if (t.cmax) {  // a line lies in one or two chunks, or is longer than they are
        quiet = true;
        for (size_t c = p0 / t.chunk; c <= (p0 + D - 1) / t.chunk; ++c)
            quiet = quiet && t.cmax[c] < s.th.dstar - s.th.band;
    }
    bool any = false;
    for (int c = 0; c < nw && !quiet; ++c) {
        const int x = c * 64 + lane;
        const unsigned long long m = __ballot(x < D && cell_hits(sm[p0 + x], t, s));
        if (lane == 0) bits[w][c] = m;
        any = any || m;
    }
    if (lane == 0) any_row[row] = any;
    __syncthreads();
    if (!any) return;
    for (int x = lane; x < D; x += 64) {
        const uint32_t l = reach_back(bits[w], nw, D, x, reach, periodic);
        const uint32_t r = reach_on(bits[w], nw, D, x, reach, periodic);
        const uint32_t m = min(l, r);
        g[p0 + x] = (uint16_t)(m <= (uint32_t)reach ? m : kNoCentre);
    }
}

typedef unsigned short u16x2 __attribute__((ext_vector_type(2)));

// Minimum over the offsets of the LDS column + o^2 for the thread's run of
// cells.  col: the thread's pair of lines at the run's first cell less `reach`.
// Offsets past the reach (the run's ends) change nothing: they have o^2 >= R^2 or,
// where the side cut the reach short, no cell or one that a nearer offset has too.
__device__ __forceinline__ void run_minimum(const u16x2* col, int reach, u16x2 best[kTileRun]) {
#pragma unroll
    for (int i = 0; i < kTileRun; ++i) best[i] = u16x2{0xFFFF, 0xFFFF};
    u16x2 sq[kTileRun];  // sq[(j - i) % 8] = (j - i)^2 of the eight latest offsets
#pragma unroll
    for (int i = 1; i < kTileRun; ++i) {
        const int o = -reach - i;
        const unsigned short q = (unsigned short)min(o * o, 0xFFFF);
        sq[(kTileRun - i) % kTileRun] = u16x2{q, q};
    }
    for (int j0 = 0; j0 < 2 * reach + kTileRun; j0 += kTileRun) {
#pragma unroll
        for (int u = 0; u < kTileRun; ++u) {
            const int o = j0 + u - reach;
            const unsigned short q = (unsigned short)min(o * o, 0xFFFF);
            sq[u] = u16x2{q, q};
            const u16x2 v = col[(j0 + u) * (kTile / 2)];
#pragma unroll
            for (int i = 0; i < kTileRun; ++i)
                best[i] = __builtin_elementwise_min(
                    best[i], __builtin_elementwise_add_sat(v, sq[(u - i + kTileRun) % kTileRun]));
        }
    }
}

// Rows of a tile's LDS column: the tile, the reach on both sides and the run's
// rounding up.
inline size_t tile_lds(int reach) { return sizeof(u16x2) * (kTile / 2) * (size_t)(kTile + 2 * reach + kTileRun); }

// Position along the axis of column row r of the tile that starts at x0, or -1.
__device__ __forceinline__ int tile_position(int x0, int r, int reach, int D, int periodic) {
    int q = x0 + r - reach;
    if (periodic) {
        q %= D;
        return q < 0 ? q + D : q;
    }
    return q < 0 || q >= D ? -1 : q;
}

// PAINT: axis 0, from h into `ion`; otherwise axis 1, from g into h.  `from`
// flags what was written of the input, `any_tile` what is written of h.
template <bool PAINT>
__global__ __launch_bounds__(kThreads) void k_sphere_tile(const uint16_t* __restrict__ in,
                                                          const uint8_t* __restrict__ from, uint16_t* __restrict__ h,
                                                          uint8_t* __restrict__ any_tile, float* __restrict__ ion,
                                                          int D, int reach, int periodic, float R2) {
    extern __shared__ u16x2 col[];
    const int t = threadIdx.x, pair = t & 31, run = t >> 5;
    const int x = blockIdx.x * kTile + 2 * pair;       // axis 2 (D is even: a pair is inside or outside)
    const int s0 = blockIdx.y * kTile;                 // first cell of the tile along the axis
    const int other = blockIdx.z;                      // the third axis
    const int nt = gridDim.y, nx = gridDim.x;
    const size_t stride = PAINT ? (size_t)D * D : (size_t)D;
    const size_t base = PAINT ? (size_t)other * D : (size_t)other * D * D;
    const int rows = kTile + 2 * reach + kTileRun;
    bool todo = false;
    for (int r = t; r < rows && !todo; r += kThreads) {
        const int q = tile_position(s0, r, reach, D, periodic);
        if (q >= 0) todo = PAINT ? from[((size_t)q * nt + other / kTile) * nx + blockIdx.x]
                                 : from[(size_t)other * D + q];
    }
    todo = __syncthreads_or(todo);
    if (PAINT && todo) {
        bool open = false;
        for (int i = 0; i < kTileRun; ++i) {
            const int q = s0 + run * kTileRun + i;
            if (x < D && q < D) {
                const size_t p = base + (size_t)q * stride + x;
                open = open || ion[p] != 1.0f || ion[p + 1] != 1.0f;
            }
        }
        todo = __syncthreads_or(open);
    }
    if (!PAINT && t == 0) any_tile[((size_t)other * nt + blockIdx.y) * nx + blockIdx.x] = todo;
    if (!todo) return;
    for (int r = run; r < rows; r += kThreads / 32) {
        const int q = tile_position(s0, r, reach, D, periodic);
        u16x2 v{0xFFFF, 0xFFFF};
        if (q >= 0 && x < D &&
            (PAINT ? from[((size_t)q * nt + other / kTile) * nx + blockIdx.x] : from[(size_t)other * D + q])) {
            const size_t p = base + (size_t)q * stride + x;
            v = *reinterpret_cast<const u16x2*>(in + p);
            if (!PAINT) {
                v.x = v.x == kNoCentre ? v.x : (unsigned short)(v.x * v.x);
                v.y = v.y == kNoCentre ? v.y : (unsigned short)(v.y * v.y);
            }
        }
        col[r * (kTile / 2) + pair] = v;
    }
    __syncthreads();
    u16x2 best[kTileRun];
    run_minimum(col + run * kTileRun * (kTile / 2) + pair, reach, best);
    if (x >= D) return;
#pragma unroll
    for (int i = 0; i < kTileRun; ++i) {
        const int q = s0 + run * kTileRun + i;
        if (q >= D) return;
        const size_t p = base + (size_t)q * stride + x;
        if (PAINT) {
            if ((float)best[i].x < R2) ion[p] = 1.0f;
            if ((float)best[i].y < R2) ion[p + 1] = 1.0f;
        } else {
            *reinterpret_cast<u16x2*>(h + p) = best[i];
        }
    }
}

// The planes and the paint for a reach or an R^2 beyond the tiles': 32-bit, a thread
// per cell, from offset 0 outwards until none can be nearer.
constexpr uint32_t kFar = 0x3FFFFFFFu;

template <bool PAINT>
__global__ void k_sphere_far(const uint16_t* __restrict__ g, const uint8_t* __restrict__ any_row,
                             uint32_t* __restrict__ h, float* __restrict__ ion, int D, int reach, int periodic,
                             float R2) {
    const size_t p = (size_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (p >= (size_t)D * D * D) return;
    if (PAINT && ion[p] == 1.0f) return;
    const size_t stride = PAINT ? (size_t)D * D : (size_t)D;
    const int pos = (int)((p / stride) % D);
    const size_t base = p - (size_t)pos * stride;
    uint32_t best = kFar;
    for (int o = 0; o <= reach && (uint32_t)(o * o) < best; ++o) {
        for (int side = 0; side < 2; ++side) {
            int q = side ? pos + o : pos - o;
            if (periodic)
                q = q < 0 ? q + D : (q >= D ? q - D : q);  // (the reach is below D)
            if (q < 0 || q >= D) continue;
            const size_t at = base + (size_t)q * stride;
            uint32_t v = kFar;
            if (PAINT)
                v = h[at];
            else if (any_row[at / D] && g[at] != kNoCentre)
                v = (uint32_t)g[at] * g[at];
            if (v < kFar) best = min(best, v + (uint32_t)(o * o));
        }
        if (PAINT && (float)best < R2) break;
    }
    if (!PAINT)
        h[p] = best;
    else if ((float)best < R2)
        ion[p] = 1.0f;
}

int launch_filter(void* spec_out, const void* spec_in, int D, const WindowParams& wp, float scale,
                  hipStream_t st) {
    // |k|^2 past which the cut of window_of takes every mode
    float ksq_cut = INFINITY;
    if (wp.filter_type == 1 || (wp.filter_type == 0 && wp.ref_fallthrough)) {
        const double k = 1.001 / (0.413566994 * (double)wp.R);
        if (wp.R > 0.0f) ksq_cut = (float)(k * k);
    }
    // ceil(2^32 / H): exact for i < D*H <= 2^21 + 2^11, i * H < 2^32
    const unsigned H = D / 2 + 1, magic = (unsigned)(((1ull << 32) + H - 1) / H);
    k_filter<<<dim3(grid_for((size_t)D * H), D), kThreads, 0, st>>>((float2*)spec_out, (const float2*)spec_in, D, wp,
                                                                    scale, ksq_cut, magic);
    CM21_LAUNCH_CHECK("k_filter");
    return CM21_OK;
}

// The f_coll sum; with t and scaled also the radius' scale and threshold, and
// the chunk maxima.
int launch_fcoll_sum(const float* sm, int D, float deltac, float denom, double* dev_sum, void* work,
                     hipStream_t st, const CellTest* t = nullptr, float* cmax = nullptr,
                     ScaledThreshold* scaled = nullptr) {
    const size_t N = (size_t)D * D * D;
    double* partial = (double*)work;
    k_fcoll_partial<<<kReduceBlocks, kThreads, 0, st>>>(sm, N, sum_chunk(N), deltac, denom, partial, cmax);
    CM21_LAUNCH_CHECK("k_fcoll_partial");
    k_sum_partials<<<1, kThreads, 0, st>>>(partial, kReduceBlocks, dev_sum, t ? *t : CellTest{}, scaled);
    CM21_LAUNCH_CHECK("k_sum_partials");
    return CM21_OK;
}

CellTest cell_test(int D, float deltac, float denom, double zeta, const double* sum, float fc_mean) {
    CellTest t{};
    t.deltac = deltac;
    t.denom = denom;
    t.zeta = zeta;
    t.inv_zeta = 1.0 / zeta;
    t.sum = sum;
    t.fc_mean = fc_mean;
    t.ncells = (double)((size_t)D * D * D);
    t.th.dstar = 0.0f;
    t.th.band = INFINITY;
    if (!sum && plain_denom(denom)) t.th = density_threshold_host(deltac, denom, zeta, 1.0f);
    return t;
}

int launch_threshold(float* ion, const float* sm, int D, const CellTest& t, int final_step, hipStream_t st) {
    const size_t N = (size_t)D * D * D;
    k_threshold<<<grid_for(N, kThreshCells), kThreads, 0, st>>>(ion, sm, N, t, final_step);
    CM21_LAUNCH_CHECK("k_threshold");
    return CM21_OK;
}

int launch_sphere(float* ion, const float* sm, int D, const CellTest& test, float R_cells, int periodic, void* work,
                  hipStream_t st) {
    const size_t N = (size_t)D * D * D;
    if (!(R_cells > 0.0f)) return CM21_OK;  // (a negative sphere scale) no offset is inside
    const float R2 = R_cells * R_cells;     // float32(R*R), find_bubbles.cu:98
    int reach = (int)std::ceil((double)R_cells);
    while (reach > 0 && (float)(reach * reach) >= R2) --reach;  // largest o with o^2 < R^2
    if (reach >= D) reach = periodic ? D / 2 : D - 1;
    // of the 8 N bytes: h (4 N, or 2 N in 16 bits), g (2 N), the flags (2 N)
    uint16_t* g = (uint16_t*)((char*)work + 4 * N);
    uint8_t* any_row = (uint8_t*)work + 6 * N;
    uint8_t* any_tile = any_row + (size_t)D * D;
    k_sphere_rows<<<(unsigned)((size_t)D * D / kWaves), kThreads, 0, st>>>(g, any_row, sm, D, test, reach, periodic);
    CM21_LAUNCH_CHECK("k_sphere_rows");
    const float diagonal = 3.0f * (float)(D - 1) * (float)(D - 1);  // its square; exact for the tiles' sides
    if (reach <= kNarrowReach && (R2 <= kNarrowMax || periodic || R2 > diagonal)) {
        const unsigned n = (unsigned)((D + kTile - 1) / kTile);
        uint16_t* h = (uint16_t*)work;
        k_sphere_tile<false><<<dim3(n, n, D), kThreads, tile_lds(reach), st>>>(g, any_row, h, any_tile, nullptr, D,
                                                                              reach, periodic, R2);
        CM21_LAUNCH_CHECK("k_sphere_tile");
        k_sphere_tile<true><<<dim3(n, n, D), kThreads, tile_lds(reach), st>>>(h, any_tile, nullptr, nullptr, ion, D,
                                                                             reach, periodic, R2);
        CM21_LAUNCH_CHECK("k_sphere_tile");
        return CM21_OK;
    }
    uint32_t* h = (uint32_t*)work;
    k_sphere_far<false><<<grid_for(N), kThreads, 0, st>>>(g, any_row, h, nullptr, D, reach, periodic, R2);
    CM21_LAUNCH_CHECK("k_sphere_far");
    k_sphere_far<true><<<grid_for(N), kThreads, 0, st>>>(nullptr, nullptr, h, ion, D, reach, periodic, R2);
    CM21_LAUNCH_CHECK("k_sphere_far");
    return CM21_OK;
}

bool valid_dim(int D) { return D >= 2 && D <= 2048 && D % 2 == 0; }

}  // namespace

extern "C" int cm21_hii_filter(void* spec_out, const void* spec_in, int D, float delta_k, int filter_type,
                               int ref_fallthrough, int korder, float R, float scale, void* stream) {
    CM21_REQUIRE(spec_out && spec_in, "cm21_hii_filter: NULL spectrum");
    CM21_REQUIRE(valid_dim(D), "cm21_hii_filter: D=%d must be even in [2,2048]", D);
    CM21_REQUIRE(filter_type >= 0 && filter_type <= 2, "cm21_hii_filter: filter_type=%d not in {0,1,2}", filter_type);
    CM21_REQUIRE(korder == 0 || korder == 1, "cm21_hii_filter: korder=%d not in {0,1}", korder);
    WindowParams wp{delta_k, R, filter_type, ref_fallthrough ? 1 : 0, korder};
    return launch_filter(spec_out, spec_in, D, wp, scale, (hipStream_t)stream);
}

extern "C" size_t cm21_reduce_workspace_bytes(void) { return align_up(sizeof(double) * kReduceBlocks, 256); }

extern "C" int cm21_fcoll_sum(const float* smoothed, int D, float deltac, float denom, double* dev_sum,
                              void* work, void* stream) {
    CM21_REQUIRE(smoothed && dev_sum && work, "cm21_fcoll_sum: NULL argument");
    CM21_REQUIRE(valid_dim(D), "cm21_fcoll_sum: D=%d must be even in [2,2048]", D);
    return launch_fcoll_sum(smoothed, D, deltac, denom, dev_sum, work, (hipStream_t)stream);
}

extern "C" int cm21_fcoll_threshold(float* ionized, const float* smoothed, int D, float deltac, float denom,
                                    double zeta, const double* dev_sum, float fc_mean, int final_step,
                                    void* stream) {
    CM21_REQUIRE(ionized && smoothed, "cm21_fcoll_threshold: NULL argument");
    CM21_REQUIRE(valid_dim(D), "cm21_fcoll_threshold: D=%d must be even in [2,2048]", D);
    CM21_REQUIRE(zeta > 0.0, "cm21_fcoll_threshold: zeta must be positive");
    return launch_threshold(ionized, smoothed, D, cell_test(D, deltac, denom, zeta, dev_sum, fc_mean), final_step,
                            (hipStream_t)stream);
}

extern "C" size_t cm21_sphere_workspace_bytes(int D) {
    return align_up(sizeof(uint32_t) * 2 * (size_t)D * D * D, 256);
}

extern "C" int cm21_update_sphere(float* ionized, const float* smoothed, int D, float deltac, float denom,
                                  double zeta, const double* dev_sum, float fc_mean, float R_cells, int periodic,
                                  void* work, void* stream) {
    CM21_REQUIRE(ionized && smoothed && work, "cm21_update_sphere: NULL argument");
    CM21_REQUIRE(valid_dim(D), "cm21_update_sphere: D=%d must be even in [2,2048]", D);
    CM21_REQUIRE(zeta > 0.0, "cm21_update_sphere: zeta must be positive");
    CM21_REQUIRE(R_cells >= 0.0f && R_cells <= 1024.0f, "cm21_update_sphere: R_cells=%g not in [0,1024]",
                 (double)R_cells);
    return launch_sphere(ionized, smoothed, D, cell_test(D, deltac, denom, zeta, dev_sum, fc_mean), R_cells,
                         periodic ? 1 : 0, work, (hipStream_t)stream);
}

// Workspace carve-up of the loop driver.
namespace {
// Pipelined fused loop: a radius uses one of loop_inter(D) intermediates in
// turn and the small per-radius buffers r % kSlots; a launch touches radii
// r-2 .. r+3.
// From side 256 on the columns and rows of the first radii (neutral_radii: where
// the bound of the rows pass may tell that the box stays neutral) run one launch
// further ahead, so that the launch between the rows and the box sums of a
// radius can decide it: one more intermediate, only then used.  Deciding
// it in every box-sum block instead cost 5 us of each 31 us launch at 256^3;
// running every radius ahead cost 3 to 8 % there, its intermediates outliving
// the caches.  (Smaller sides take this loop only with the least workspace.)
constexpr int kInterMax = 6, kSlots = 3;
constexpr int kRowBounds = 4;  // bounds per plane (kBoundGroups of the rows pass)
constexpr int loop_inter(int D) { return D >= 256 ? 6 : 5; }

struct LoopWork {
    float2* spec;
    float2* filt;             // generic path: filtered spectrum
    float* smoothed;          // generic path: smoothed box
    float2* inter[kInterMax]; // fused path: intermediates (inter[0] is filt,
                              // inter[1] shares smoothed's region)
    double* partial;
    float* cmax;              // generic path: chunk maxima of the f_coll sum
    double* sums;
    void* sphere;
    unsigned long long* mask;
    double* lpart[kSlots];    // box-sum partials
    float* bmax[kSlots];      // per line group maxima
    int* active[kSlots];      // line groups the threshold pass visits, and their number
    int* nactive[kSlots];
    float* bound[kSlots];     // bounds of the rows pass
    ScaledThreshold* scaled;  // per radius
    size_t bytes;
};

LoopWork carve(void* base, int D, int n_radii, int update) {
    const size_t N = (size_t)D * D * D;
    const size_t Nc = (size_t)D * D * (D / 2 + 1);
    const size_t Nt = (size_t)D * D * padded_row(D / 2 + 1);  // an intermediate (padded rows)
    char* p = (char*)base;
    LoopWork w{};
    size_t off = 0;
    // the spectrum: the r2c layout (stride D/2+1) for the paint path, the
    // fused transform's b-major layout with padded rows otherwise
    w.spec = (float2*)(p + off);
    off = align_up(off + sizeof(float2) * (update ? Nc : Nt), 256);
    w.filt = w.inter[0] = (float2*)(p + off);
    off = align_up(off + sizeof(float2) * Nt, 256);
    // 8Nt >= 4N bytes
    w.smoothed = (float*)(p + off);
    w.inter[1] = (float2*)(p + off);
    off = align_up(off + std::max(sizeof(float) * N, sizeof(float2) * Nt), 256);
    // the fused path (update == 0 only) needs three or four more intermediates
    for (int k = 2; k < loop_inter(D) && !update; ++k) {
        w.inter[k] = (float2*)(p + off);
        off = align_up(off + sizeof(float2) * Nt, 256);
    }
    w.partial = (double*)(p + off);
    off = align_up(off + cm21_reduce_workspace_bytes(), 256);
    w.cmax = (float*)(p + off);
    off = align_up(off + sizeof(float) * kReduceBlocks, 256);
    w.sums = (double*)(p + off);
    off = align_up(off + sizeof(double) * (size_t)(n_radii > 0 ? n_radii : 1), 256);
    w.sphere = update ? (void*)(p + off) : nullptr;
    if (update) off = align_up(off + cm21_sphere_workspace_bytes(D), 256);
    w.mask = (unsigned long long*)(p + off);
    off = align_up(off + sizeof(unsigned long long) * ((N + 63) / 64), 256);
    for (int k = 0; k < kSlots; ++k) {
        w.lpart[k] = (double*)(p + off);
        off = align_up(off + sizeof(double) * (fused_partials(D) + 1), 256);
        w.bmax[k] = (float*)(p + off);
        off = align_up(off + sizeof(float) * (fused_partials(D) + 1), 256);
        w.active[k] = (int*)(p + off);
        off = align_up(off + sizeof(int) * (fused_partials(D) + 1), 256);
        w.nactive[k] = (int*)(p + off);
        off = align_up(off + sizeof(int), 256);
        w.bound[k] = (float*)(p + off);
        off = align_up(off + sizeof(float) * kRowBounds * D, 256);
    }
    w.scaled = (ScaledThreshold*)(p + off);
    off = align_up(off + sizeof(ScaledThreshold) * (size_t)(n_radii > 0 ? n_radii : 1), 256);
    w.bytes = off;
    return w;
}

// The all-radii form (sides up to 160): its buffers behind the standard
// carve-up's spectrum, or bytes = 0 when the form does not apply.
struct AllWork {
    AllRadii a;
    size_t bytes;
};

bool loop_is_fused(const FusedShape* sh, const cm21_bubble_params* prm) {
    return prm->fused && sh && prm->update == 0 && (prm->filter_type == 1 || prm->filter_type == 2);
}

float loop_scale(int D, const cm21_bubble_params* prm) {
    const double n = (double)((size_t)D * D * D);
    return prm->linear_input ? (float)(1.0 / n) : (float)((double)prm->growth_inv / n);
}

float loop_delta_k(const cm21_bubble_params* prm) { return (float)(2.0 * M_PI / (double)prm->box_len); }

// Whether the launch per radius is the faster form for a side that has both: with the
// Gaussian window at 160^3 the intermediates of every radius (0.8 GB) are past the caches,
// and on a box that is expected to be all ionized at the largest radius (zeta <f_coll>)
// its threshold launches end at once, where the all-radii form transforms every line
// of every radius.  All radii at once, 160^3, BOX_LEN 250, by zeta <f_coll> = 1.0 / 1.1 / 1.2 / 3:
// linear 838 831 817 809 us against 884 797 662 662, nonlinear 1069 1051 1030 1018 against
// 1236 1162 889 884.  At 128^3 (463 against 528 at 3) and with the k-space top-hat (326
// against 318 at 3, 353 against 467 at 1.2) all at once is as fast or faster throughout.
bool per_radius_is_faster(int D, const cm21_bubble_params* prm) {
    return D > 128 && prm->filter_type == 2 && prm->zeta * (double)prm->fc_mean > 1.2;
}

AllWork carve_all(void* base, int D, const float* radii, const float* denoms, int n_radii,
                  const cm21_bubble_params* prm) {
    AllWork w{};
    const FusedShape* sh = fused_shape(D);
    if (!loop_is_fused(sh, prm) || per_radius_is_faster(D, prm)) return w;
    const size_t nt = all_radii_table(*sh, loop_delta_k(prm), radii, denoms, n_radii, prm->filter_type,
                                      prm->ref_fallthrough, loop_scale(D, prm), &w.a);
    if (nt == 0) return w;
    const size_t N = (size_t)D * D * D, row = (size_t)D * D * padded_row(D / 2 + 1);
    const size_t cells = (size_t)n_radii * w.a.nblk;
    char* p = (char*)base;
    size_t off = 0;
    auto take = [&](size_t bytes) {
        void* q = p + off;
        off = align_up(off + bytes, 256);
        return q;
    };
    AllRadii& a = w.a;
    a.S = (float2*)take(sizeof(float2) * row);
    // the forward transform passes through the intermediates' region
    a.T = (float2*)take(sizeof(float2) * std::max(nt, row));
    a.sums = (double*)take(sizeof(double) * n_radii);
    a.bound = (float*)take(sizeof(float) * kRowBounds * D * n_radii);
    a.scaled = (ScaledThreshold*)take(sizeof(ScaledThreshold) * n_radii);
    a.hits = (unsigned*)take(sizeof(unsigned) * cells);
    a.planes = (unsigned long long*)take(sizeof(unsigned long long) * n_radii * (N / 64));
    if (!prm->linear_input) {
        a.partial = (double*)take(sizeof(double) * cells);
        a.bmax = (float*)take(sizeof(float) * cells);
    }
    w.bytes = off;
    return w;
}
}  // namespace

namespace {
int run_loop(cm21_plan* plan, const float* delta, float* ionized, const float* radii, const float* denoms,
             int n_radii, const cm21_bubble_params* prm, void* work, size_t work_bytes, hipStream_t st);
int graph_loop(cm21_plan* plan, const float* delta, float* ionized, const float* radii, const float* denoms,
               int n_radii, const cm21_bubble_params* prm, void* work, size_t work_bytes, hipStream_t st);
}  // namespace

extern "C" size_t cm21_find_bubbles_workspace_bytes(int D, int n_radii, int update) {
    if (!valid_dim(D)) return 0;
    return carve(nullptr, D, n_radii, update).bytes;
}

extern "C" size_t cm21_find_bubbles_full_workspace_bytes(int D, const float* radii, int n_radii,
                                                         const cm21_bubble_params* prm) {
    if (!valid_dim(D) || !radii || n_radii < 1 || !prm || !(prm->box_len > 0.0f)) return 0;
    return std::max(carve(nullptr, D, n_radii, prm->update).bytes,
                    carve_all(nullptr, D, radii, nullptr, n_radii, prm).bytes);
}

namespace {
// Argument checks shared by cm21_find_bubbles and cm21_find_bubbles_noalloc.
int check_loop_args(const char* fn, cm21_plan* plan, const float* delta, float* ionized, const float* radii,
                    const float* denoms, int n_radii, const cm21_bubble_params* prm) {
    CM21_REQUIRE(plan && delta && ionized && radii && denoms && prm, "%s: NULL argument", fn);
    CM21_REQUIRE(plan_batch(plan) == 1, "%s: plan must have batch 1", fn);
    CM21_REQUIRE(n_radii >= 1 && n_radii <= 4096, "%s: n_radii=%d out of range", fn, n_radii);
    CM21_REQUIRE(prm->filter_type >= 0 && prm->filter_type <= 2, "%s: filter_type=%d", fn, prm->filter_type);
    CM21_REQUIRE(prm->zeta > 0.0, "%s: zeta must be positive", fn);
    CM21_REQUIRE(prm->box_len > 0.0f, "%s: box_len must be positive", fn);
    for (int r = 0; r < n_radii; ++r) {
        if (!(denoms[r] > 0.0f) || !std::isfinite(denoms[r]))
            return cm21::fail(CM21_ERR_DOMAIN,
                              "%s: denominator %g at R=%g is not positive and finite (sigma_min^2 <= S(R))", fn,
                              (double)denoms[r], (double)radii[r]);
        if (prm->update && !(radii[r] * prm->sphere_r_scale <= 1024.0f))
            return cm21::fail(CM21_ERR_INVALID, "%s: sphere radius %g cells exceeds 1024", fn,
                              (double)(radii[r] * prm->sphere_r_scale));
    }
    return CM21_OK;
}
}  // namespace

extern "C" int cm21_find_bubbles(cm21_plan* plan, const float* delta, float* ionized, const float* radii,
                                 const float* denoms, int n_radii, const cm21_bubble_params* prm, void* work,
                                 size_t work_bytes, void* stream) {
    CM21_TRY(check_loop_args("cm21_find_bubbles", plan, delta, ionized, radii, denoms, n_radii, prm));
    CM21_REQUIRE(work, "cm21_find_bubbles: NULL argument");
    const size_t need = carve(nullptr, plan_dim(plan), n_radii, prm->update).bytes;
    if (work_bytes < need)
        return cm21::fail(CM21_ERR_NOMEM, "cm21_find_bubbles: workspace %zu bytes < required %zu", work_bytes, need);
    hipStream_t st = (hipStream_t)stream;
    if (prm->graph && st != nullptr && !prof_any())
        return graph_loop(plan, delta, ionized, radii, denoms, n_radii, prm, work, work_bytes, st);
    return run_loop(plan, delta, ionized, radii, denoms, n_radii, prm, work, work_bytes, st);
}

namespace {
int run_loop(cm21_plan* plan, const float* delta, float* ionized, const float* radii, const float* denoms,
             int n_radii, const cm21_bubble_params* prm, void* work, size_t work_bytes, hipStream_t st) {
    void* stream = (void*)st;
    const int D = plan_dim(plan);
    const size_t N = (size_t)D * D * D;
    const LoopWork w = carve(work, D, n_radii, prm->update);

    const float dk = loop_delta_k(prm);
    const float scale = loop_scale(D, prm);
    const FusedShape* sh = fused_shape(D);
    if (loop_is_fused(sh, prm)) {
        const float2* tw = plan_twiddles(plan);
        // the forward transform forms only the modes the widest window keeps
        FusedParams widest = fused_params(D, dk, radii[0], prm->filter_type, prm->ref_fallthrough, scale);
        for (int r = 1; r < n_radii; ++r) {
            const FusedParams f = fused_params(D, dk, radii[r], prm->filter_type, prm->ref_fallthrough, scale);
            if (f.m2max > widest.m2max) widest = f;
        }
        // every radius at once where the workspace holds their intermediates
        AllWork all = carve_all(work, D, radii, denoms, n_radii, prm);
        if (all.bytes && work_bytes >= all.bytes) {
            AllRadii& a = all.a;
            a.linear = prm->linear_input ? 1 : 0;
            a.deltac = prm->deltac;
            a.fc_mean = prm->fc_mean;
            a.zeta = prm->zeta;
            a.ncells = (double)N;
            a.out = ionized;
            CM21_TRY(fused_forward(*sh, delta, a.T, a.S, tw, widest, st));
            return fused_all_radii(*sh, a, tw, st);
        }
        // through the intermediate of the last radius, which the box before left in
        // the caches (256^3 forward 89 us; 97 to 102 through any other), and ahead of what
        // the host works out for the schedule
        CM21_TRY(fused_forward(*sh, delta, w.inter[0], w.spec, tw, widest, st));
        CM21_TRY(fused_mask_clear(w.mask, (N + 63) / 64, st));
        // One launch per radius on the caller's stream, each with up to six
        // independent roles over neighbouring radii (k_fused_radius): launch
        // j holds the columns pass of radius j+2, the rows pass of radius j+1,
        // the box-sum pass of radius j, the box-sum reduction of radius j-1
        // and the threshold pass of radius j-2 (nonlinear input), or the
        // threshold pass of radius j (linear input, threshold from the host).
        // In-order launches carry every dependency (rows after columns, sum
        // after rows, reduction after sum, threshold after reduction), so the
        // loop needs no events, and the pruned transforms of later radii
        // share the chip with the box sums instead of waiting for them.
        // The threshold pass recomputes the last-axis transform in the line
        // groups whose maximum can reach the threshold rather than storing and
        // re-reading the smoothed field; the final paint is one more launch.
        const int nblk = D * D / sh->L;
        const bool nl = !prm->linear_input;
        auto params = [&](int r) {
            return fused_params(D, dk, radii[r], prm->filter_type, prm->ref_fallthrough, scale);
        };
        std::vector<DensityThreshold> linear_th(nl ? 0 : n_radii);
        for (size_t r = 0; r < linear_th.size(); ++r)
            linear_th[r] = density_threshold_host(prm->deltac, denoms[r], prm->zeta, 1.0f);
        const int last = n_radii - 1;
        // radii 0 .. ahead-1 run their columns and rows one launch further
        // ahead and get a verdict (never the last radius, which is painted)
        int ahead = 0;
        if (D >= 256) {
            std::vector<int> cmax(n_radii);
            for (int r = 0; r < n_radii; ++r) cmax[r] = params(r).cmax;
            ahead = neutral_radii(*prm, denoms, n_radii, cmax.data());
        }
        // the intermediate of each radius: a ring of six while radii run
        // ahead, of five afterwards (the fewer, the more of them stay cached)
        std::vector<int> inter_of(n_radii);
        for (int r = 0; r < n_radii; ++r)
            inter_of[r] = ahead > 0 && r <= ahead ? r % kInterMax : (r >= 5 ? inter_of[r - 5] : r);
        const int q_last = inter_of[last];  // takes the place of number 0
        auto inter = [&](int r) {
            const int q = inter_of[r];
            return w.inter[q == q_last ? 0 : (q == 0 ? q_last : q)];
        };
        auto col_launch = [&](int r) { return r - (r < ahead ? 3 : 2); };
        auto row_launch = [&](int r) { return r - (r < ahead ? 2 : 1); };
        // the radius whose pass falls into launch j, or -1
        auto radius_in = [&](auto&& launch_of, int j, int d) {
            for (int r = j + d; r <= j + d + 1; ++r)
                if (r >= 0 && r <= last && launch_of(r) == j) return r;
            return -1;
        };
        // launches j = -2 .. j_end-1: the last one holds the reduction of the
        // last radius and the threshold pass of the one before (nonlinear), or
        // the threshold pass of the radius before the last (linear)
        const int j_end = nl ? n_radii + 1 : n_radii - 1;
        for (int j = ahead > 0 ? -3 : -2; j < j_end; ++j) {
            RadiusRoles a{};
            AskRoles q{};
            a.deltac = prm->deltac;
            a.zeta = prm->zeta;
            if (const int r = radius_in(col_launch, j, 2); r >= 0) {
                a.S = w.spec;
                a.Tcols = inter(r);
                a.fp_cols = params(r);
                int nb = 0;
                column_groups(*sh, a.fp_cols, &a.ncg_cols, &nb);
                a.n_cols = a.ncg_cols * nb;
            }
            a.n_mem = a.n_cols;
            if (const int r = radius_in(row_launch, j, 1); r >= 0) {
                a.Trows = inter(r);
                const FusedParams fp = params(r);
                a.m2max_rows = fp.m2max;
                a.cmax_rows = fp.cmax;
                int nb = 0;
                column_groups(*sh, fp, &a.ncg_rows, &nb);
                a.n_mem += a.ncg_rows * D;
                q.bound_rows = r < ahead && a.ncg_rows <= kRowBounds ? w.bound[r % kSlots] : nullptr;
            }
            if (j + 1 >= 0 && j + 1 < ahead) {
                const int r = j + 1;
                const FusedParams fp = params(r);
                int ncg = 0, nb = 0;
                column_groups(*sh, fp, &ncg, &nb);
                q.n_ver = 1;
                q.skip.bound = ncg <= kRowBounds ? w.bound[r % kSlots] : nullptr;
                q.skip.S0 = w.spec;
                q.skip.groups = ncg;
                q.skip.linear = nl ? 0 : 1;
                q.skip.deltac = prm->deltac;
                q.skip.zeta_fc_mean = (float)(prm->zeta * (double)prm->fc_mean);
                if (!nl) q.skip.th = linear_th[r];
                q.skip_scale = fp.scale;
                q.skip_denom = denoms[r];
                q.verdict = w.scaled + r;
            }
            if (nl && j - 1 >= 0 && j - 1 <= last) {
                const int r = j - 1, s = r % kSlots;
                a.partial = w.lpart[s];
                a.total = w.sums + r;
                a.scaled_red = w.scaled + r;
                a.fc_mean = prm->fc_mean;
                a.denom_red = denoms[r];
                a.bmax_red = w.bmax[s];
                a.active_red = r < last ? w.active[s] : nullptr;
                a.nactive_red = r < last ? w.nactive[s] : nullptr;
                if (r < ahead) q.state_red = w.scaled + r;
                a.n_red = 1;
            }
            const int rt = nl ? j - 2 : j;  // the threshold pass (the last radius is painted below)
            if (rt >= 0 && rt < last) {
                a.Uthr = inter(rt);
                a.cmax_thr = params(rt).cmax;
                a.denom_thr = denoms[rt];
                a.mask = w.mask;
                if (nl) {
                    a.scaled_thr = w.scaled + rt;
                    a.bmax_thr = w.bmax[rt % kSlots];
                    a.active_thr = w.active[rt % kSlots];
                    a.nactive_thr = w.nactive[rt % kSlots];
                } else {
                    a.th = linear_th[rt];
                }
                a.n_thr = nblk;
                if (!nl && rt < ahead) q.state_thr = w.scaled + rt;
            }
            if (nl && j >= 0 && j <= last) {
                const int r = j, s = r % kSlots;
                a.Usum = inter(r);
                a.cmax_sum = params(r).cmax;
                a.denom_sum = denoms[r];
                a.partial_sum = w.lpart[s];
                a.bmax_sum = w.bmax[s];
                if (r < ahead) q.state_sum = w.scaled + r;
                a.n_sum = nblk;
            }
            q.any = q.n_ver || q.bound_rows || q.state_thr || q.state_sum || q.state_red;
            CM21_TRY(fused_radius_launch(*sh, a, q, tw, st));
        }
        // mode 2: the final paint of the last radius
        LineEpilogue e = line_epilogue(prm->deltac, denoms[last], prm->zeta, w.mask, ionized);
        if (nl)
            e.scaled = w.scaled + last;
        else
            e.th = linear_th[last];
        CM21_TRY(fused_lines(*sh, inter(last), tw, params(last), e, st, CM21_STAGE_FUSED_LINES_THRESHOLD));
        return CM21_OK;
    }
    {
        ProfToken t = prof_begin(CM21_STAGE_R2C, st);
        CM21_TRY(cm21_r2c(plan, delta, w.spec, stream));
        prof_end(t, st);
    }
    k_fill<<<grid_for(N), kThreads, 0, st>>>(ionized, N, 0.0f);
    CM21_LAUNCH_CHECK("k_fill");
    for (int r = 0; r < n_radii; ++r) {
        const bool final_step = r == n_radii - 1;
        WindowParams wp{dk, radii[r], prm->filter_type, prm->ref_fallthrough ? 1 : 0, 0};
        ProfToken t = prof_begin(CM21_STAGE_FILTER, st);
        CM21_TRY(launch_filter(w.filt, w.spec, D, wp, scale, st));
        prof_end(t, st);
        t = prof_begin(CM21_STAGE_C2R, st);
        CM21_TRY(cm21_c2r(plan, w.filt, w.smoothed, stream));
        prof_end(t, st);
        CellTest test = cell_test(D, prm->deltac, denoms[r], prm->zeta, prm->linear_input ? nullptr : w.sums + r,
                                  prm->fc_mean);
        if (!prm->linear_input) {
            t = prof_begin(CM21_STAGE_FCOLL_SUM, st);
            CM21_TRY(launch_fcoll_sum(w.smoothed, D, prm->deltac, denoms[r], w.sums + r, w.partial, st, &test, w.cmax,
                                      w.scaled + r));
            prof_end(t, st);
            test.scaled = w.scaled + r;
            test.cmax = w.cmax;
            test.chunk = sum_chunk(N);
        }
        if (prm->update && !final_step) {
            t = prof_begin(CM21_STAGE_SPHERE, st);
            CM21_TRY(launch_sphere(ionized, w.smoothed, D, test, radii[r] * prm->sphere_r_scale,
                                   prm->sphere_periodic, w.sphere, st));
            prof_end(t, st);
        } else {
            t = prof_begin(CM21_STAGE_THRESHOLD, st);
            CM21_TRY(launch_threshold(ionized, w.smoothed, D, test, final_step ? 1 : 0, st));
            prof_end(t, st);
        }
    }
    return CM21_OK;
}

// Graph replay of the whole loop.  The first call with a given set of
// arguments (pointers, parameters, radii, denominators, stream) captures the
// launches into a HIP graph; identical later calls replay it, which removes
// the host launch cost of the ~5 kernels per radius.  One graph is kept per
// plan.  A capture that fails falls back to eager launches.
struct GraphKey {
    const void* delta;
    const void* ionized;
    const void* work;
    size_t work_bytes;
    hipStream_t stream;
    cm21_bubble_params prm;
    std::vector<float> radii, denoms;
    bool operator==(const GraphKey& o) const {
        return delta == o.delta && ionized == o.ionized && work == o.work &&
               work_bytes == o.work_bytes && stream == o.stream &&
               std::memcmp(&prm, &o.prm, sizeof(prm)) == 0 && radii == o.radii && denoms == o.denoms;
    }
};
struct GraphEntry {
    GraphKey key;
    hipGraphExec_t exec = nullptr;
};
std::mutex g_graph_mu;
std::unordered_map<const cm21_plan*, GraphEntry> g_graphs;

int graph_loop(cm21_plan* plan, const float* delta, float* ionized, const float* radii, const float* denoms,
               int n_radii, const cm21_bubble_params* prm, void* work, size_t work_bytes, hipStream_t st) {
    GraphKey key{delta, ionized, work, work_bytes, st, *prm, std::vector<float>(radii, radii + n_radii),
                 std::vector<float>(denoms, denoms + n_radii)};
    std::lock_guard<std::mutex> lk(g_graph_mu);
    auto it = g_graphs.find(plan);
    if (it != g_graphs.end() && it->second.exec && it->second.key == key) {
        CM21_HIP_CHECK(hipGraphLaunch(it->second.exec, st));
        return CM21_OK;
    }
    if (it != g_graphs.end() && it->second.exec) {
        (void)hipGraphExecDestroy(it->second.exec);
        it->second.exec = nullptr;
    }
    if (hipStreamBeginCapture(st, hipStreamCaptureModeThreadLocal) != hipSuccess) {
        (void)hipGetLastError();
        return run_loop(plan, delta, ionized, radii, denoms, n_radii, prm, work, work_bytes, st);
    }
    const int rc = run_loop(plan, delta, ionized, radii, denoms, n_radii, prm, work, work_bytes, st);
    hipGraph_t graph = nullptr;
    const hipError_t ec = hipStreamEndCapture(st, &graph);
    hipGraphExec_t exec = nullptr;
    bool ok = rc == CM21_OK && ec == hipSuccess && graph;
    if (ok) ok = hipGraphInstantiate(&exec, graph, nullptr, nullptr, 0) == hipSuccess;
    if (graph) (void)hipGraphDestroy(graph);
    if (!ok) {
        (void)hipGetLastError();
        if (rc != CM21_OK) return rc;
        return run_loop(plan, delta, ionized, radii, denoms, n_radii, prm, work, work_bytes, st);
    }
    g_graphs[plan] = GraphEntry{std::move(key), exec};
    CM21_HIP_CHECK(hipGraphLaunch(exec, st));
    return CM21_OK;
}
}  // namespace

// ------------------------------------------------------------------ no-alloc loop
// cm21_find_bubbles_noalloc runs the loop of cm21_find_bubbles with its
// workspace in a file-scope device array instead of a caller's buffer.  Each
// GPU holds its own copy of the array (CM21_NOALLOC_SCRATCH_BYTES) from the
// library's load until the process ends; host code reaches it only through
// the address hipGetSymbolAddress returns on that device, taken once per
// device at the first call.  Calls on one GPU share the array.
namespace {
constexpr size_t kScratchBytes = (size_t)CM21_NOALLOC_SCRATCH_BYTES;
static __device__ __align__(256) unsigned char scratch[kScratchBytes];

constexpr int kMaxDevices = 64;
std::mutex g_scratch_mu;
void* g_scratch[kMaxDevices] = {};

int scratch_on_current_device(void** out) {
    int dev = 0;
    CM21_HIP_CHECK(hipGetDevice(&dev));
    CM21_REQUIRE(dev >= 0 && dev < kMaxDevices, "cm21_find_bubbles_noalloc: device %d out of range", dev);
    std::lock_guard<std::mutex> lk(g_scratch_mu);
    if (!g_scratch[dev]) {
        void* p = nullptr;
        const hipError_t e = hipGetSymbolAddress(&p, HIP_SYMBOL(scratch));
        if (e != hipSuccess || p == nullptr)
            return cm21::fail(CM21_ERR_HIP, "cm21_find_bubbles_noalloc: hipGetSymbolAddress(scratch) on device %d: %s",
                              dev, hipGetErrorString(e));
        g_scratch[dev] = p;
    }
    *out = g_scratch[dev];
    return CM21_OK;
}
}  // namespace

extern "C" int cm21_find_bubbles_noalloc(cm21_plan* plan, const float* delta, float* ionized, const float* radii,
                                         const float* denoms, int n_radii, const cm21_bubble_params* prm,
                                         void* stream) {
    CM21_TRY(check_loop_args("cm21_find_bubbles_noalloc", plan, delta, ionized, radii, denoms, n_radii, prm));
    const int D = plan_dim(plan);
    const size_t need = carve(nullptr, D, n_radii, prm->update).bytes;
    if (need > kScratchBytes)
        return cm21::fail(CM21_ERR_NOMEM,
                          "cm21_find_bubbles_noalloc: D=%d with %d radii (update %d) needs %zu bytes of workspace, "
                          "more than the %zu-byte static scratch; use cm21_find_bubbles with a caller workspace",
                          D, n_radii, prm->update, need, kScratchBytes);
    void* base = nullptr;
    CM21_TRY(scratch_on_current_device(&base));
    // the launches go straight to the stream (params->graph is ignored), so a
    // caller that captures the stream records them into its own graph
    return run_loop(plan, delta, ionized, radii, denoms, n_radii, prm, base, kScratchBytes, (hipStream_t)stream);
}

namespace cm21 {
void forget_plan_graphs(const cm21_plan* plan) {
    std::lock_guard<std::mutex> lk(g_graph_mu);
    auto it = g_graphs.find(plan);
    if (it != g_graphs.end()) {
        if (it->second.exec) (void)hipGraphExecDestroy(it->second.exec);
        g_graphs.erase(it);
    }
}
}  // namespace cm21
