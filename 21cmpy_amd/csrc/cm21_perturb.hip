// Zel'dovich mass move on the GPU (perturb_field stage).
//
// Reference: Programs/perturb_field.cu:90-133 (move_mass) and
// Programs/perturb_field.py:93-105, in the reference's float32 position
// arithmetic.  NGP deposits the whole mass in the truncated cell (bit-exact
// indices); CIC shares it over the 8 nearest cell centres.  Deposits are float
// atomics: the summation order varies from run to run at the 1e-7 relative level,
// the target cells never do.
//
// The particles of one HII cell share their displacement and deposit
// together (k_move_cells, k_move_waves), through an LDS tile around their block's patch.
#include <algorithm>
#include <cmath>

#include "cm21_internal.hpp"

using namespace cm21;

namespace {

struct MoveParams {
    int DIM, sw, q;     // q = DIM / sw
    float disp_scale;   // (D(z) - D_init)/BOX_LEN
    float growth_init;  // D_init
};

// Start of particle index i on one axis, in box units.
__device__ inline float particle_start(int i, int DIM) { return (float)(((double)i + 0.5) / (double)DIM); }

// Position on one axis from the start, after the wrap loops of
// perturb_field.cu:102-118.  Returns false for a non-finite position.
__device__ __forceinline__ bool particle_coord(float start, float v, const MoveParams& mp, float& f) {
    const float swf = (float)mp.sw;
    f = __fadd_rn(start, __fmul_rn(v, mp.disp_scale));
    f = __fmul_rn(f, swf);
    if (!isfinite(f)) return false;
    if (f >= 0.0f && f < swf) return true;
    // The reference loops until in range; bound the loop and finish with an
    // exact floor-based wrap for displacements of many box lengths.
    int it = 0;
    while (f >= swf && it < 64) { f = __fsub_rn(f, swf); ++it; }
    while (f < 0.0f && it < 128) { f = __fadd_rn(f, swf); ++it; }
    if (f >= swf || f < 0.0f) {
        f = f - swf * floorf(f / swf);
        if (f >= swf) f = 0.0f;
    }
    return true;
}

__device__ inline float particle_mass(float delta, float growth_init) {
    return (float)(1.0 + (double)__fmul_rn(growth_init, delta));
}

// Deposit by displacement cells.  The q^3 particles of one HII cell share
// their displacement (q = DIM/sw), so they move as a rigid lattice less than
// one HII cell wide: along each axis their target cells are base + {0, 1}
// (NGP) or base + {0, 1, 2} (CIC; one less at q = 1), and the CIC weight of a particle in a cell
// is the product of its three axis weights.  A thread therefore takes one HII
// cell, forms the C weights of each of its q planes per axis (C = 1, 2 or 3) and
// contracts the q^3 masses with them, along z, then y, then x, into C^3 sums:
// 27 deposits for q^3 particles instead of 8 q^3 (q > 1).
//
// A block of 512 threads takes kNY x kNZ columns of HII cells, each column
// shared by two threads that walk half of its PX cells in x; it accumulates
// into an LDS tile around where the middle of its patch goes: the patch and kHalo cells
// on its sides, room for displacements that differ from the middle's by 3 cells
// (displacements are smooth; with the tile around the patch itself, 256^3 cells moved by
// 40 took 859 us for 223, CIC at q = 1, and a smooth field of 8 cells rms 2723 for 517).  Cells
// whose lattice leaves the tile deposit straight into global memory, and cells with a non-finite mass
// or position go particle by particle, so that one bad particle reaches only
// the cells that it touches.
//
// The tile is FP64 because the float32 LDS atomic is slow on this hardware:
// ds_add_f32 takes 195 cycles of a CU's LDS per wavefront, ds_add_f64 9 (and
// ds_add_u32 5), all on distinct addresses.  The float atomics were the bound
// of every earlier form (2.1 to 2.3 ms at 512 -> 256, per particle or per
// cell alike: 27 a cell are 7 M of them, 2.2 ms).
//
// Then each non-zero tile cell is one global atomic.  Storing the tiles and
// adding those that cover a cell in a second kernel, without atomics, was
// slower at every size (512 -> 256: 432 against 305 us, 128 -> 64: 35 against
// 24).  In all, with the clearing and the renormalisation, 512 -> 256 takes
// 305 us (CIC; 2.14 ms before), of which reading delta and the displacements
// is 0.16 ms at the rate of a copy.
constexpr int kHalo = 4, kReach = 2 * kHalo;  // tile side: patch side + kReach
constexpr int kNY = 16, kNZ = 16, kWalk = 8, kMoveThreads = 512;

__device__ __forceinline__ int wrapped(int x, int sw) {
    x %= sw;
    return x < 0 ? x + sw : x;
}
__device__ __forceinline__ void add_global(float* acc, int sw, int x, int y, int z, float w) {
    atomicAdd(&acc[((size_t)wrapped(x, sw) * sw + wrapped(y, sw)) * sw + wrapped(z, sw)], w);
}

struct Tile {
    int ox, oy, oz, Tx, Ty, Tz, sw;
    bool use;

    __device__ __forceinline__ int local(int x, int o) const {  // (x - o) mod sw, x in [-1, sw), o in [0, sw)
        const int l = x - o;
        return l < 0 ? l + sw : l;
    }
};

// Target of one plane of a cell's lattice on one axis: its offset from the
// base cell and its C weights.
template <int SCHEME, int Q>
struct AxisWeights {
    static constexpr int C = (SCHEME == 0 ? 2 : 3) - (Q == 1 ? 1 : 0);
    float w[C];
    int cell;  // NGP: the target; CIC: the lower target
    float t;   // CIC: share of the upper target

    // f: position in [0, sw)
    __device__ __forceinline__ void place(float f) {
        if (SCHEME == 0) {
            cell = (int)f;
            t = 0.0f;
        } else {
            const float c = __fsub_rn(f, 0.5f), fl = floorf(c);
            cell = (int)fl;
            t = __fsub_rn(c, fl);
        }
    }
    // weights relative to `base`; false when the offset is not 0 or 1
    __device__ __forceinline__ bool weigh(int base, int sw) {
        int o = cell - base;
        o += o < 0 ? sw : 0;
        const float lo = SCHEME == 0 ? 1.0f : __fsub_rn(1.0f, t);
        if constexpr (Q == 1) {  // one plane: its own cell is the base
            w[0] = lo;
            if constexpr (C == 2) w[1] = t;
            return true;
        } else {
            w[0] = o ? 0.0f : lo;
            w[1] = o ? lo : t;
            if constexpr (C == 3) w[2] = o ? t : 0.0f;
            return o == 0 || o == 1;
        }
    }
};

// Deposits of one particle.
template <int SCHEME>
__device__ __forceinline__ void move_particle(float* __restrict__ acc, float delta, int i, int j, int k,
                                              const float (&pv)[3], const MoveParams& mp) {
    const int at[3] = {i, j, k};
    AxisWeights<SCHEME, 0> o[3];
#pragma unroll
    for (int ax = 0; ax < 3; ++ax) {
        float f;
        if (!particle_coord(particle_start(at[ax], mp.DIM), pv[ax], mp, f)) return;
        o[ax].place(f);
    }
    const float mass = particle_mass(delta, mp.growth_init);
    for (int c = 0; c < (SCHEME == 0 ? 1 : 8); ++c) {
        const int a = c >> 2, b = (c >> 1) & 1, e = c & 1;
        float wt = mass;
        if (SCHEME == 1) {
            wt = __fmul_rn(wt, a ? o[0].t : __fsub_rn(1.0f, o[0].t));
            wt = __fmul_rn(wt, b ? o[1].t : __fsub_rn(1.0f, o[1].t));
            wt = __fmul_rn(wt, e ? o[2].t : __fsub_rn(1.0f, o[2].t));
        }
        if (wt != 0.0f) add_global(acc, mp.sw, o[0].cell + a, o[1].cell + b, o[2].cell + e, wt);
    }
}

// Q: DIM/sw when it is 1 to 4 (the weights of every plane stay in registers),
// or 0 (formed again per row) for a larger ratio, few of them (by_waves), and
// for masses that are not aligned.
template <int SCHEME, int Q>
__global__ __launch_bounds__(kMoveThreads) void k_move_cells(float* __restrict__ acc, const float* __restrict__ delta,
                                                    const float* __restrict__ vx, const float* __restrict__ vy,
                                                    const float* __restrict__ vz, MoveParams mp, int PX, int Tx, int Ty,
                                                    int Tz) {
    using W = AxisWeights<SCHEME, Q>;
    constexpr int C = W::C, NQ = Q > 0 ? Q : 1;
    extern __shared__ double tile[];
    __shared__ float startx[kWalk * NQ];  // particle_start of the walk's planes
    const int DIM = mp.DIM, sw = mp.sw, q = Q > 0 ? Q : mp.q;
    const int nz = (sw + kNZ - 1) / kNZ, ny = (sw + kNY - 1) / kNY;
    const int z0 = (blockIdx.x % nz) * kNZ, y0 = (blockIdx.x / nz % ny) * kNY, x0 = (int)(blockIdx.x / (nz * ny)) * PX;
    const int t = threadIdx.x;
    const int hy = y0 + t / kNZ % kNY, hz = z0 + t % kNZ;
    const int half = t / (kNY * kNZ), xa = x0 + half * (PX / 2);  // this thread's part of the walk
    // displacement of the patch's middle, in flight while the tile is cleared
    const size_t hm = ((size_t)min(x0 + PX / 2, sw - 1) * sw + min(y0 + kNY / 2, sw - 1)) * sw + min(z0 + kNZ / 2, sw - 1);
    const float mid[3] = {vx[hm], vy[hm], vz[hm]};
    const bool use_tile = sw >= Tx && sw >= Ty && sw >= Tz;
    if (use_tile)
        for (int c = t; c < Tx * Ty * Tz; c += kMoveThreads) tile[c] = 0.0;
    if (t < kWalk * NQ) startx[t] = particle_start(x0 * NQ + t, DIM);
    __syncthreads();
    auto origin = [&](int p0, float v) {
        const float d = rintf(v * mp.disp_scale * (float)sw);
        int o = p0 - kHalo + (fabsf(d) < 1e6f ? (int)d : 0);
        if (o < 0) o += sw;
        return (unsigned)o < (unsigned)sw ? o : wrapped(o, sw);
    };
    const Tile tl{origin(x0, mid[0]), origin(y0, mid[1]), origin(z0, mid[2]), Tx, Ty, Tz, sw, use_tile};
    const int xb = hy < sw && hz < sw ? min(sw, xa + PX / 2) : xa;
    for (int hx = xa; hx < xb; ++hx) {
        const size_t h = ((size_t)hx * sw + hy) * sw + hz;  // C_INDEX(HII_k, HII_j, HII_i, sw)
        const float pv[3] = {vx[h], vy[h], vz[h]};
        const int i0 = hx * q, j0 = hy * q, k0 = hz * q;  // the cell's first particle
        const float* dp = delta + ((size_t)i0 * DIM + j0) * DIM + k0;
        float m[NQ][NQ][NQ];
        if (Q > 0) {
#pragma unroll
            for (int i = 0; i < NQ; ++i)
#pragma unroll
                for (int j = 0; j < NQ; ++j) {
                    const float* row = dp + ((size_t)i * DIM + j) * DIM;
                    // rows start at multiples of q floats from `delta`, which the launch
                    // found aligned to q of them, and DIM is a multiple of 8
                    if constexpr (Q == 2) {
                        const float2 d = *(const float2*)row;
                        m[i][j][0] = d.x, m[i][j][1] = d.y;
                    } else if constexpr (Q == 4) {
                        const float4 d = *(const float4*)row;
                        m[i][j][0] = d.x, m[i][j][1] = d.y, m[i][j][2] = d.z, m[i][j][3] = d.w;
                    } else {
#pragma unroll
                        for (int k = 0; k < NQ; ++k) m[i][j][k] = row[k];
                    }
                }
        }
        W w[3][NQ];
        int base[3];
        bool ok = true;
        const int first[3] = {i0, j0, k0};
#pragma unroll
        for (int ax = 0; ax < 3; ++ax) {
            float f;
            auto start = [&](int p) {
                return Q > 0 && ax == 0 ? startx[(hx - x0) * NQ + p] : particle_start(first[ax] + p, DIM);
            };
            ok = particle_coord(start(0), pv[ax], mp, f) && ok;
            w[ax][0].place(f);
            base[ax] = w[ax][0].cell;
            w[ax][0].weigh(base[ax], sw);
#pragma unroll
            for (int p = 1; p < NQ; ++p) {
                ok = particle_coord(start(p), pv[ax], mp, f) && ok;
                w[ax][p].place(f);
                ok = w[ax][p].weigh(base[ax], sw) && ok;
            }
        }
        float s[C][C][C];
#pragma unroll
        for (int a = 0; a < C; ++a)
#pragma unroll
            for (int b = 0; b < C; ++b)
#pragma unroll
                for (int c = 0; c < C; ++c) s[a][b][c] = 0.0f;
        float total = 0.0f;
        auto weight = [&](int ax, int p, W& o) {
            float f;
            ok = particle_coord(particle_start(first[ax] + p, DIM), pv[ax], mp, f) && ok;
            o.place(f);
            ok = o.weigh(base[ax], sw) && ok;
        };
        if (Q > 0) {
#pragma unroll
            for (int i = 0; i < NQ; ++i) {
                float p2[C][C];
#pragma unroll
                for (int j = 0; j < NQ; ++j) {
                    float p1[C];
#pragma unroll
                    for (int k = 0; k < NQ; ++k) {
                        const float mass = particle_mass(m[i][j][k], mp.growth_init);
                        total += mass;
#pragma unroll
                        for (int c = 0; c < C; ++c) p1[c] = k ? fmaf(w[2][k].w[c], mass, p1[c]) : w[2][k].w[c] * mass;
                    }
#pragma unroll
                    for (int b = 0; b < C; ++b)
#pragma unroll
                        for (int c = 0; c < C; ++c)
                            p2[b][c] = j ? fmaf(w[1][j].w[b], p1[c], p2[b][c]) : w[1][j].w[b] * p1[c];
                }
#pragma unroll
                for (int a = 0; a < C; ++a)
#pragma unroll
                    for (int b = 0; b < C; ++b)
#pragma unroll
                        for (int c = 0; c < C; ++c) s[a][b][c] = fmaf(w[0][i].w[a], p2[b][c], s[a][b][c]);
            }
        } else {
            for (int i = 0; i < q; ++i) {
                float p2[C][C];
#pragma unroll
                for (int b = 0; b < C; ++b)
#pragma unroll
                    for (int c = 0; c < C; ++c) p2[b][c] = 0.0f;
                for (int j = 0; j < q; ++j) {
                    float p1[C];
#pragma unroll
                    for (int c = 0; c < C; ++c) p1[c] = 0.0f;
                    const float* row = dp + ((size_t)i * DIM + j) * DIM;
                    for (int k = 0; k < q; ++k) {
                        W wk;
                        weight(2, k, wk);
                        const float mass = particle_mass(row[k], mp.growth_init);
                        total += mass;
#pragma unroll
                        for (int c = 0; c < C; ++c) p1[c] = fmaf(wk.w[c], mass, p1[c]);
                    }
                    W wj;
                    weight(1, j, wj);
#pragma unroll
                    for (int b = 0; b < C; ++b)
#pragma unroll
                        for (int c = 0; c < C; ++c) p2[b][c] = fmaf(wj.w[b], p1[c], p2[b][c]);
                }
                W wi;
                weight(0, i, wi);
#pragma unroll
                for (int a = 0; a < C; ++a)
#pragma unroll
                    for (int b = 0; b < C; ++b)
#pragma unroll
                        for (int c = 0; c < C; ++c) s[a][b][c] = fmaf(wi.w[a], p2[b][c], s[a][b][c]);
            }
        }
        if (!(ok && isfinite(total))) {
            for (int p = 0; p < q * q * q; ++p) {
                const int i = p / (q * q), j = p / q % q, k = p % q;
                move_particle<SCHEME>(acc, dp[((size_t)i * DIM + j) * DIM + k], i0 + i, j0 + j, k0 + k, pv, mp);
            }
            continue;
        }
        const int lx = tl.local(base[0], tl.ox), ly = tl.local(base[1], tl.oy), lz = tl.local(base[2], tl.oz);
        if (tl.use && lx <= Tx - C && ly <= Ty - C && lz <= Tz - C) {
            double* p = tile + (lx * Ty + ly) * Tz + lz;
#pragma unroll
            for (int a = 0; a < C; ++a)
#pragma unroll
                for (int b = 0; b < C; ++b)
#pragma unroll
                    for (int c = 0; c < C; ++c) atomicAdd(p + (a * Ty + b) * Tz + c, (double)s[a][b][c]);
        } else {
#pragma unroll
            for (int a = 0; a < C; ++a)
#pragma unroll
                for (int b = 0; b < C; ++b)
#pragma unroll
                    for (int c = 0; c < C; ++c)
                        if (s[a][b][c] != 0.0f) add_global(acc, sw, base[0] + a, base[1] + b, base[2] + c, s[a][b][c]);
        }
    }
    if (!tl.use) return;
    __syncthreads();
    for (int c = t; c < Ty * Tz; c += kMoveThreads) {
        const int ly = c / Tz, lz = c - ly * Tz;
        int gx = tl.ox, gy = tl.oy + ly, gz = tl.oz + lz;
        gy = gy >= sw ? gy - sw : gy;
        gz = gz >= sw ? gz - sw : gz;
        float* col = acc + (size_t)gy * sw + gz;
        for (int lx = 0; lx < Tx; ++lx) {
            const float v = (float)tile[lx * Ty * Tz + c];
            if (v != 0.0f) atomicAdd(col + (size_t)gx * sw * sw, v);
            gx = gx + 1 == sw ? 0 : gx + 1;
        }
    }
}

// Larger ratios: a wavefront per displacement cell, or per share of one, where a
// thread per cell leaves the chip idle (8 blocks at 512 -> 16).  A share is `len` of the
// cell's planes along x and one of `parts` shares of a plane's q^2 columns.  A lane
// sums its columns along x against the C weights of the planes, which the lanes
// hold one plane each, then with the column's own weights into C^3 sums; these
// are added over the lanes, half of them handed over at each step, after which lane l
// has one sum.  A block takes a patch of P^3 cells (P = 1: up to eight shares of one)
// and adds the sums up in an FP64 LDS tile around where its first cell goes, because
// a global atomic per sum is 0.2 ns each and was the bound (512 -> 64: 1.7 ms).
// CIC, against a thread per cell and a thread per 16 particles of a 16^3 patch:
// 512 -> 16 108 us (9700, 943; 5 TB/s), 512 -> 32 138 (1282, 985), 512 -> 8 116 (66700,
// 129600), 256 -> 32 57 (172, 168), 128 -> 16 22 (146, 42).  Bound by memory from q = 16
// on, below by the sums' 31 exchanges a cell, and by the three launches up to 128^3.
constexpr int kShareLen = 32;     // planes of a share (a lane each, up to 64 - kAhead)
constexpr int kAhead = 8;         // planes whose loads are in flight together
constexpr int kFillWaves = 8192;  // wavefronts wanted, eight per SIMD
constexpr int kTileEdge = 10;     // P = 4, two cells on both sides and the CIC neighbours

struct WaveSplit {
    int P, halo;             // cells along a patch, tile cells on its sides
    int len, chunks, parts;  // planes of a share, shares along x and of a plane
    int shares;              // shares of a cell in a block
};

template <int SCHEME>
__global__ __launch_bounds__(kMoveThreads, 6) void k_move_waves(float* __restrict__ acc, const float* __restrict__ delta,
                                                             const float* __restrict__ vx, const float* __restrict__ vy,
                                                             const float* __restrict__ vz, MoveParams mp, WaveSplit ws) {
    using W = AxisWeights<SCHEME, 0>;
    constexpr int C = W::C, C3 = C * C * C, CP = SCHEME == 0 ? 8 : 32;
    __shared__ double tile[kTileEdge * kTileEdge * kTileEdge];
    const int DIM = mp.DIM, sw = mp.sw, q = mp.q, lane = threadIdx.x & 63;
    const int P = ws.P, T = P + C - 1 + 2 * ws.halo, np = (sw + P - 1) / P;
    for (int c = threadIdx.x; c < T * T * T; c += kMoveThreads) tile[c] = 0.0;
    const int x0 = (int)(blockIdx.x / (np * np)) * P, y0 = (int)(blockIdx.x / np % np) * P, z0 = (int)(blockIdx.x % np) * P;
    int org[3];  // the tile's first cell
    {
        const size_t h = ((size_t)x0 * sw + y0) * sw + z0;
        const float pv[3] = {vx[h], vy[h], vz[h]};
        const int first[3] = {x0 * q, y0 * q, z0 * q};
#pragma unroll
        for (int ax = 0; ax < 3; ++ax) {
            float f;
            W o;
            o.place(particle_coord(particle_start(first[ax], DIM), pv[ax], mp, f) ? f : 0.0f);
            org[ax] = o.cell - ws.halo;
        }
    }
    __syncthreads();
    const int cells = P * P * P;
    for (int u = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6); u < cells * ws.shares; u += kMoveThreads / 64) {
        const int pc = u % cells, share = blockIdx.y * ws.shares + u / cells;
        const int hx = x0 + pc / (P * P), hy = y0 + pc / P % P, hz = z0 + pc % P;
        if (hx >= sw || hy >= sw || hz >= sw || share >= ws.chunks * ws.parts) continue;
        const int chunk = share / ws.parts, part = share % ws.parts, len = ws.len, parts = ws.parts;
        const size_t h = ((size_t)hx * sw + hy) * sw + hz;
        const float pv[3] = {vx[h], vy[h], vz[h]};
        const int first[3] = {hx * q, hy * q, hz * q};
        const int i0 = first[0] + chunk * len, ni = min(len, q - chunk * len);
        const float* dp = delta + ((size_t)i0 * DIM + first[1]) * DIM + first[2];
        int base[3];
        bool ok = true;
        auto weigh = [&](int ax, int p, W& o) {
            float f;
            ok = particle_coord(particle_start(p, DIM), pv[ax], mp, f) && ok;
            o.place(f);
            ok = o.weigh(base[ax], sw) && ok;
        };
#pragma unroll
        for (int ax = 0; ax < 3; ++ax) {
            float f;
            W o;
            ok = particle_coord(particle_start(first[ax], DIM), pv[ax], mp, f) && ok;
            o.place(f);
            base[ax] = o.cell;
        }
        W wx;  // of plane `lane` of the share, nothing past its end
        weigh(0, i0 + min(lane, ni - 1), wx);
#pragma unroll
        for (int a = 0; a < C; ++a)
            if (lane >= ni) wx.w[a] = 0.0f;
        float s[CP];
#pragma unroll
        for (int c = 0; c < CP; ++c) s[c] = 0.0f;
        float total = 0.0f;
        const int cols = q * q, dj = parts * 64 / q, dk = parts * 64 - dj * q;
        int col = part * 64 + lane, j = col / q, k = col - j * q;
        for (int c0 = part * 64; c0 < cols; c0 += parts * 64) {
            const bool in = col < cols;  // the last lanes of a plane read its first column
            const float* p = in ? dp + (size_t)j * DIM + k : dp;
            float m[C];
#pragma unroll
            for (int a = 0; a < C; ++a) m[a] = 0.0f;
            for (int i = 0; i < ni; i += kAhead) {
                float d[kAhead];
#pragma unroll
                for (int u = 0; u < kAhead; ++u) d[u] = p[(size_t)min(i + u, ni - 1) * DIM * DIM];
#pragma unroll
                for (int u = 0; u < kAhead; ++u) {
                    const float mass = particle_mass(d[u], mp.growth_init);
                    total += mass;
#pragma unroll
                    for (int a = 0; a < C; ++a)
                        m[a] = fmaf(__int_as_float(__builtin_amdgcn_readlane(__float_as_int(wx.w[a]), i + u)), mass, m[a]);
                }
            }
            W wy, wz;
            weigh(1, first[1] + (in ? j : 0), wy);
            weigh(2, first[2] + (in ? k : 0), wz);
#pragma unroll
            for (int a = 0; a < C; ++a)
#pragma unroll
                for (int b = 0; b < C; ++b) {
                    const float w = in ? m[a] * wy.w[b] : 0.0f;
#pragma unroll
                    for (int c = 0; c < C; ++c) s[(a * C + b) * C + c] = fmaf(w, wz.w[c], s[(a * C + b) * C + c]);
                }
            col += parts * 64;
            j += dj;
            k += dk;
            if (k >= q) {
                k -= q;
                ++j;
            }
        }
        if (!__all(ok && isfinite(total))) {
            for (int p = part * 64 + lane; p < ni * cols; p += parts * 64) {
                const int i = p / cols, y = p / q % q, z = p % q;
                move_particle<SCHEME>(acc, dp[((size_t)i * DIM + y) * DIM + z], i0 + i, first[1] + y, first[2] + z, pv, mp);
            }
            continue;
        }
        // lane l ends with sum number (bits of l reversed)
#pragma unroll
        for (int n = CP / 2, bit = 1; n > 0; n >>= 1, bit <<= 1) {
            const bool up = lane & bit;
#pragma unroll
            for (int c = 0; c < n; ++c) {
                const float give = up ? s[c] : s[c + n];
                s[c] = (up ? s[c + n] : s[c]) + __shfl_xor(give, bit, 64);
            }
        }
#pragma unroll
        for (int bit = CP; bit < 64; bit <<= 1) s[0] += __shfl_xor(s[0], bit, 64);
        const int n = (int)(__brev((unsigned)lane) >> (SCHEME == 0 ? 29 : 27));
        if (lane < CP && n < C3 && s[0] != 0.0f) {
            const int lx = wrapped(base[0] - org[0], sw), ly = wrapped(base[1] - org[1], sw);
            const int lz = wrapped(base[2] - org[2], sw);
            const int a = n / (C * C), b = n / C % C, c = n % C;
            if (lx <= T - C && ly <= T - C && lz <= T - C)
                atomicAdd(&tile[((lx + a) * T + ly + b) * T + lz + c], (double)s[0]);
            else
                add_global(acc, sw, base[0] + a, base[1] + b, base[2] + c, s[0]);
        }
    }
    __syncthreads();
    for (int c = threadIdx.x; c < T * T * T; c += kMoveThreads) {
        const float v = (float)tile[c];
        if (v != 0.0f) add_global(acc, sw, org[0] + c / (T * T), org[1] + c / T % T, org[2] + c % T, v);
    }
}

// Whether the cells go to a wavefront each.  Time of a thread per cell over that,
// CIC: q = 5 2.0 at sw = 16, 0.9 at 32, 0.3 at 64 and 80; q = 6 2.9 at 16, 1.5 at 32,
// 0.97 at 40, 0.6 at 48 and 56; q = 8 3.0 at 32, 1.3 at 48, 1.5 at 56, 1.1 at 64 and 128;
// q = 9 0.9 at 64, 80 and 128; q = 10 1.6 at 48, 1.2 at 64, 1.1 at 80; q = 12 1.5 at 64;
// q = 16 3.2 at 64.  Up to q = 4 the thread has its weights in registers and is never
// slower by more than the launches.
bool by_waves(const MoveParams& mp) { return mp.q >= 10 || (mp.q >= 5 && mp.sw < (mp.q < 8 ? 40 : 64)); }

int patches(int sw, int P) {
    const int n = (sw + P - 1) / P;
    return n * n * n;
}

// The largest patch with two blocks to a CU, and shares that fill the chip.
WaveSplit wave_split(const MoveParams& mp) {
    WaveSplit ws;
    ws.P = patches(mp.sw, 4) >= 512 ? 4 : (patches(mp.sw, 2) >= 512 ? 2 : 1);
    ws.halo = ws.P > 1 ? 2 : 0;
    ws.len = std::min(mp.q, kShareLen);
    ws.chunks = (mp.q + ws.len - 1) / ws.len;
    const long waves = (long)mp.sw * mp.sw * mp.sw * ws.chunks, most = ((long)mp.q * mp.q + 63) / 64;
    ws.parts = (int)std::min((kFillWaves + waves - 1) / waves, most);
    ws.shares = ws.P > 1 ? ws.chunks * ws.parts : std::min(ws.chunks * ws.parts, kMoveThreads / 64);
    return ws;
}

template <int SCHEME>
int launch_move(float* acc, const float* delta, const float* vx, const float* vy, const float* vz, const MoveParams& mp,
                hipStream_t st) {
    if (by_waves(mp)) {
        const WaveSplit ws = wave_split(mp);
        const int all = ws.chunks * ws.parts;
        k_move_waves<SCHEME><<<dim3(patches(mp.sw, ws.P), (all + ws.shares - 1) / ws.shares), kMoveThreads, 0, st>>>(
            acc, delta, vx, vy, vz, mp, ws);
        CM21_LAUNCH_CHECK("k_move_waves");
        return CM21_OK;
    }
    auto blocks = [&](int n) { return (unsigned)((mp.sw + n - 1) / n); };
    // a walk of kWalk cells, or of 2 where that would leave CUs without a block
    const int PX = blocks(kWalk) * blocks(kNY) * blocks(kNZ) >= 512 ? kWalk : 2;
    const int Tx = PX + kReach, Ty = kNY + kReach, Tz = kNZ + kReach;
    const unsigned grid = blocks(PX) * blocks(kNY) * blocks(kNZ);
    const size_t lds = sizeof(double) * Tx * Ty * Tz;  // 72 KB, two blocks a CU (45 KB for the short walk)
    // two and four masses of a row are one load; a view that does not start at a
    // multiple of them takes the kernel that loads them one by one
    const bool aligned = (uintptr_t)delta % (sizeof(float) * mp.q) == 0;
    auto* k = mp.q == 1              ? k_move_cells<SCHEME, 1>
              : mp.q == 2 && aligned ? k_move_cells<SCHEME, 2>
              : mp.q == 3            ? k_move_cells<SCHEME, 3>
              : mp.q == 4 && aligned ? k_move_cells<SCHEME, 4>
                                     : k_move_cells<SCHEME, 0>;
    k<<<grid, kMoveThreads, lds, st>>>(acc, delta, vx, vy, vz, mp, PX, Tx, Ty, Tz);
    CM21_LAUNCH_CHECK("k_move_cells");
    return CM21_OK;
}

__global__ void k_zero(float* __restrict__ p, size_t n) {
    const size_t i = (size_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (i < n) p[i] = 0.0f;
}

__global__ void k_renorm(float* __restrict__ p, size_t n, float mass_factor) {
    const size_t i = (size_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (i < n) p[i] = __fsub_rn(__fdiv_rn(p[i], mass_factor), 1.0f);
}

}  // namespace

extern "C" int cm21_move_mass(float* updated, const float* deltax, const float* vx, const float* vy,
                              const float* vz, int DIM, int sw, float disp_scale, float growth_init, int scheme,
                              void* stream) {
    CM21_REQUIRE(updated && deltax && vx && vy && vz, "cm21_move_mass: NULL argument");
    CM21_REQUIRE(DIM >= 8 && DIM <= 2048 && DIM % 8 == 0, "cm21_move_mass: DIM=%d must be a multiple of 8 in [8,2048]",
                 DIM);
    CM21_REQUIRE(sw >= 1 && sw <= DIM && DIM % sw == 0, "cm21_move_mass: sw=%d must divide DIM=%d", sw, DIM);
    CM21_REQUIRE(scheme == 0 || scheme == 1, "cm21_move_mass: scheme=%d not in {0 (NGP), 1 (CIC)}", scheme);
    if (scheme == 1 && DIM % 16 != 0)
        return cm21::fail(CM21_ERR_INVALID, "cm21_move_mass: CIC needs DIM %% 16 == 0");
    hipStream_t st = (hipStream_t)stream;
    const size_t n_small = (size_t)sw * sw * sw;
    const float pff = (float)DIM / (float)sw;  // PIXEL_FACTOR (INIT_PARAMS.py:7)
    const MoveParams mp{DIM, sw, DIM / sw, disp_scale, growth_init};
    k_zero<<<grid_for(n_small), kThreads, 0, st>>>(updated, n_small);
    CM21_LAUNCH_CHECK("k_zero");
    CM21_TRY((scheme ? launch_move<1> : launch_move<0>)(updated, deltax, vx, vy, vz, mp, st));
    const float mass_factor = (float)std::pow((double)pff, 3.0);  // MASS_FACTOR (INIT_PARAMS.py:8)
    k_renorm<<<grid_for(n_small), kThreads, 0, st>>>(updated, n_small, mass_factor);
    CM21_LAUNCH_CHECK("k_renorm");
    return CM21_OK;
}
