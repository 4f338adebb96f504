// Fused, pruned inverse transforms of the find_HII_bubbles radius loop.
//
// For each radius the filtered spectrum W(kR) S(k) is transformed back to real
// space in three passes over the half spectrum S[a][b][c] (a, b full axes, c the
// halved axis, c fastest):
//   columns: window multiply + inverse DFT along a, written to T[p][b][c];
//   rows:    inverse DFT along b, in place, T[p][q][c];
//   lines:   c2r along c (as a length-D/2 complex DFT) fused with the f_coll
//            epilogue (FP64 box sum, threshold into an ionization bitmask, or
//            the final paint into the float output).
// With the k-space top-hat (HII_FILTER 0 and 1 cut modes with kR > 2.418 in
// the reference's fall-through chain, Programs/find_bubbles.cu:33-37) every
// mode with |n|^2 > m2max is zero, so the columns pass reads and writes only
// columns inside the disc b^2 + c^2 <= m2max, the rows pass only c <= cmax and
// the lines pass only c <= cmax of each line.  Large radii keep a few modes;
// the work per radius follows the number of surviving modes.
//
// Each DFT of length D = D1*D2 is a four-step transform: D2-point DFTs in
// registers (one per thread), a twiddle by w_D^(n1 k2), an LDS transpose, then
// D1-point DFTs in registers.  The window is evaluated per mode from its
// integer |n|^2: the Gaussian factor as exp2(m2 * gcoef) and the cut by an
// integer bound, except in a thin shell around the cut where the reference's
// float32 test (find_bubbles.cu:26-35) decides, so cut decisions are
// bit-identical to the reference arithmetic.
#include <algorithm>

#include "cm21_fused_dev.hpp"

#pragma clang fp contract(fast)

namespace cm21 {

// Box-sum reduction of one radius by the NT threads of one block: strided
// per-thread FP64 sums, the wavefront tree, then the waves in order (the order
// is fixed, so the total is bitwise reproducible).  With `scaled` thread 0
// also derives the box-mean scale float32(fc_mean / (sum / ncells)) and its
// density threshold, once for every block of the threshold pass; with
// `active` the block lists the line groups whose maximum is not below
// d* - band (the order of the list does not matter: each group writes only
// its own mask words).
// A radius at which no cell can be ionized has no box sums: its list is empty.
template <int NT>
__device__ void finish_box_sum(const double* partial, int n, int nblk, double* out, const SumScaleArgs& sa,
                               const ScaledThreshold* state = nullptr) {
    if (state && state->neutral) {
        if (threadIdx.x == 0 && sa.active) *sa.nactive = 0;
        return;
    }
    __shared__ double part[NT / 64];
    __shared__ DensityThreshold sth;
    __shared__ int count;
    double acc = 0.0;
    for (int i = threadIdx.x; i < n; i += NT) acc += partial[i];
    acc = wave_sum(acc);
    if ((threadIdx.x & 63) == 0) part[threadIdx.x >> 6] = acc;
    __syncthreads();
    if (threadIdx.x == 0) {
        double r = 0.0;
        for (int w = 0; w < NT / 64; ++w) r += part[w];
        *out = r;
        if (sa.scaled) {
            const float scale = (float)((double)sa.fc_mean / (r / sa.ncells));
            ScaledThreshold s;
            s.scale = scale;
            s.th = density_threshold(sa.deltac, sa.denom, sa.zeta, scale);
            s.neutral = 0;
            *sa.scaled = s;
            sth = s.th;
        }
        count = 0;
    }
    if (!sa.scaled || !sa.active) return;
    __syncthreads();
    const float lim = sth.dstar - sth.band;
    for (int i = threadIdx.x; i < nblk; i += NT)
        if (!(sa.bmax[i] < lim)) sa.active[atomicAdd(&count, 1)] = i;
    __syncthreads();
    if (threadIdx.x == 0) *sa.nactive = count;
}

// Pass 3: c2r along axis 2 for L consecutive lines, then the f_coll epilogue:
// FP64 block partial of the box sum and the block's maximum of the smoothed
// field (MODE kLineSum), threshold into the ionization bitmask
// (kLineThreshold) or the final paint (kLineFinal).  In sum mode a one-block
// kernel adds the partials in a fixed order (deterministic), and the kernel
// boundary makes them visible across the chip's L2 slices.
//
// Before any transform work a threshold block returns when it cannot change
// the mask: every one of its cells is already ionized, or the box-sum pass
// found its maximum below d* - band (no cell can reach the threshold; cells
// inside the band take the exact test, so the skip never drops a hit).  A
// final-paint block whose cells are all ionized writes 1 without transforming.
// `blk` is the index of the L-line group the block works on.
// `hs` is the line stride of U.  kLinePaint is kLineFinal with the block's mask
// words in `word` (thread t holds word t) instead of ep.mask.
template <int N1, int N2, int L, int MODE_>
__device__ __forceinline__ void lines_block(const float2* __restrict__ U, int hs, const float2* __restrict__ tw,
                                            int cmax, const LineEpilogue& ep, int blk, float2* buf,
                                            float2* stw, unsigned long long* smask, unsigned long long word = 0ull) {
    using C = LinesCore<N1, N2, L>;
    constexpr int D = C::D, NT = C::NT, WORDS = C::WORDS;
    constexpr int MODE = MODE_ == kLinePaint ? (int)kLineFinal : MODE_;
    // the lines and threads of a box-sum partial
    constexpr int SL = sum_lines(D, L), SNT = NT / (L / SL);
    const int t = threadIdx.x;
    const size_t line0 = (size_t)blk * L;
    const size_t word0 = line0 * D / 64;
    const size_t cell0 = line0 * D;
    const bool use_scale = ep.scaled != nullptr;
    float scale = 1.0f;
    DensityThreshold th = ep.th;
    unsigned long long mword = 0ull;
    if (MODE != kLineSum) {
        if (use_scale) {
            const ScaledThreshold s = *ep.scaled;
            scale = s.scale;
            th = s.th;
        }
        mword = t < WORDS ? (MODE_ == kLinePaint ? word : ep.mask[word0 + t]) : ~0ull;
        const bool all_ionized = __syncthreads_and(mword == ~0ull);
        if (all_ionized) {
            if (MODE == kLineFinal)
                for (int q = t; q < L * D; q += NT) ep.out[cell0 + q] = 1.0f;
            return;
        }
        if (MODE == kLineThreshold && ep.bmax != nullptr && ep.bmax[blk] < th.dstar - th.band) return;
    }
    // all global loads in flight before the first LDS store
    float2 tmp[C::LOADS];
    C::load(U + line0 * hs, hs, cmax + 1, tmp);
    for (int q = t; q < D; q += NT) stw[q] = tw[q];
    C::store(tmp, buf);
    if (MODE != kLineSum && t < WORDS) smask[t] = mword;
    __syncthreads();
    C::transform(buf, stw, cmax + 1);
    double acc = 0.0;
    float vmax = -INFINITY;
    const int lane = t & 63;
    const float* xrf = reinterpret_cast<const float*>(buf);
    const float inv_denom = 1.0f / ep.denom;
    // box sum: four float32 partials per thread (a quarter of its cells each,
    // a few roundings of values in [0, 2]), added in FP64 after the loop
    static_assert((L * D) % (4 * NT) == 0, "whole sets of four cells per thread");
    float part[4] = {0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll 4
    for (int q = 0; q < L * D / NT; ++q) {
        const int f = MODE == kLineSum && SNT != NT ? t / SNT * SL * D + t % SNT + q * SNT : t + q * NT;
        const int i = f / D, r = f - i * D;
        const float delta = xrf[i * 2 * C::HP + r];
        if (MODE == kLineSum) {
            part[q & 3] += fcoll_for_sum(delta, ep.deltac, ep.denom, inv_denom);
            vmax = fmaxf(vmax, delta);
        } else {
            const bool hit = cell_hit(delta, th, ep.deltac, ep.denom, use_scale, scale, ep.inv_zeta);
            const unsigned long long old = smask[f >> 6];
            if (MODE == kLineThreshold) {
                const unsigned long long bits = __ballot(hit);
                if (lane == 0) smask[f >> 6] = old | bits;
            } else {
                const bool was = (old >> (f & 63)) & 1ull;
                float val = 1.0f;
                if (!was && !hit) val = final_value(delta, ep.deltac, ep.denom, use_scale, scale, ep.zeta, ep.inv_zeta);
                ep.out[cell0 + f] = val;
            }
        }
    }
    if (MODE == kLineSum) {
        acc = ((double)part[0] + (double)part[1]) + ((double)part[2] + (double)part[3]);
        if (ep.bmax != nullptr) {
            __shared__ float wmax[NT / 64];
#pragma unroll
            for (int off = 32; off > 0; off >>= 1) vmax = fmaxf(vmax, __shfl_xor(vmax, off, 64));
            if (lane == 0) wmax[t >> 6] = vmax;
            __syncthreads();
            if (t == 0) {
                float m = wmax[0];
                for (int w = 1; w < NT / 64; ++w) m = fmaxf(m, wmax[w]);
                ep.bmax[blk] = m;
            }
        }
        if (SNT == NT) {
            acc = block_sum(acc);
            if (t == 0) ep.partial[blk] = acc;
        } else {
            __shared__ double wsum[NT / 64];
            acc = wave_sum(acc);
            if (lane == 0) wsum[t >> 6] = acc;
            __syncthreads();
            if (t % SNT == 0) {
                double sum = 0.0;
                for (int w = 0; w < SNT / 64; ++w) sum += wsum[(t >> 6) + w];
                ep.partial[blk * (L / SL) + t / SNT] = sum;
            }
        }
    }
    if (MODE == kLineThreshold) {
        __syncthreads();
        if (t < WORDS && smask[t] != mword) ep.mask[word0 + t] = smask[t];
    }
}

// The final paint of the loop with a launch per radius.
template <int N1, int N2, int L>
__global__ __launch_bounds__(L* N1) void k_fused_lines(const float2* __restrict__ U, const float2* __restrict__ tw,
                                                      int cmax, LineEpilogue ep) {
    using C = LinesCore<N1, N2, L>;
    __shared__ float2 buf[L * C::HP];
    __shared__ float2 stw[C::D];
    __shared__ unsigned long long smask[C::WORDS];
    lines_block<N1, N2, L, kLineFinal>(U, C::HO, tw, cmax, ep, blockIdx.x, buf, stw, smask);
}

// One launch of the pipelined radius loop.  Its blocks take one of six
// roles: the columns pass of radius r+2 and the rows pass of radius r+1 (into
// intermediates no other role of the launch touches; r+3 and r+2 for the
// first radii), the one-block box-sum reduction of radius r-1 (scale,
// threshold and active list), the one-block verdict whether the box stays
// neutral at radius r+1 (the first radii), the threshold pass of radius r-2
// and the box-sum pass of radius r.  A radius without a cell to ionize costs 10
// us at 256^3 instead of 31 (box sums, nonlinear) and 25 us at 512^3 instead of
// 220 (thresholds, linear).  Every role reads only what earlier launches wrote
// and writes buffers no other role of the launch reads or writes, so the roles
// need no ordering among themselves; in-order launches on one stream order the
// radii.
// Block order: the reduction, then for nonlinear input the box-sum blocks,
// the columns/rows blocks and the threshold blocks (block i of these takes
// the i-th listed line group; those past the end of the list return at
// once), for linear input the threshold blocks and then the columns/rows
// blocks.  The VALU-bound box sums fill every CU first and the
// memory-bound transposes take the slots they free; against the columns/rows
// blocks interleaved one for one with the box sums after the threshold
// blocks, 578 -> 603 boxes/s (literal) and 450 -> 457 (partly ionized) at
// 256^3; thresholds first stay better for linear input (128^3: 2530
// against 2399 boxes/s with thresholds last).
// The kernel asks for eight waves per SIMD, the box-sum role's full
// occupancy (about 52 VGPRs, 19.5 KB of LDS at D = 256); the columns/rows
// roles fit it without spilling through the re/im-staged transpose.
// ASK: the launch has a verdict, bounds or states to look at (launches of the
// first radii); without it the kernel carries none of that.
template <int D1, int D2, int W, int N1, int N2, int L, bool ASK>
__device__ __forceinline__ void radius_roles(const RadiusRoles& a, const AskRoles& q, const float2* __restrict__ tw) {
    using C = LinesCore<N1, N2, L>;
    constexpr int D = D1 * D2, NT = W * D1;
    static_assert(C::D == D && C::NT == NT, "columns/rows and lines tiles must share D and the block size");
    // the columns/rows transposes stage real and imaginary parts in turn
    // (a float tile) when their one-round float2 tile would need more LDS
    // than the lines pass, and so lower the occupancy of the box sums
    constexpr int kLdsLines = L * C::HP + D + C::WORDS;
    constexpr int kRounds = W * (D + 1) > kLdsLines + kLdsLines / 4 ? 0 : 1;
    constexpr int kLdsCR = kRounds == 0 ? (W * (D + 1) + 1) / 2 : W * (D + 1);
    __shared__ float2 lds[kLdsCR > kLdsLines ? kLdsCR : kLdsLines];
    float2* buf = lds;
    float2* stw = lds + L * C::HP;
    unsigned long long* smask = reinterpret_cast<unsigned long long*>(lds + L * C::HP + D);
    int b = blockIdx.x;
    if (b < a.n_red) {
        const SumScaleArgs sa{a.scaled_red,   a.fc_mean,    a.deltac,     a.denom_red,    (double)D * D * D,
                              a.zeta,         a.bmax_red,   a.active_red, a.nactive_red};
        finish_box_sum<NT>(a.partial, D * D / sum_lines(D, L), D * D / L, a.total, sa, ASK ? q.state_red : nullptr);
        return;
    }
    b -= a.n_red;
    if (ASK && b < q.n_ver) {
        const bool neutral = box_stays_neutral<NT, D>(q.skip, q.skip_scale, q.skip_denom);
        if (threadIdx.x == 0) q.verdict->neutral = neutral ? 1 : 0;
        return;
    }
    if (ASK) b -= q.n_ver;
    // nonlinear input: box sums, transposes, thresholds; linear input (no
    // box sums): thresholds, transposes
    const int thr0 = a.n_sum > 0 ? a.n_sum + a.n_mem : 0;
    if (b >= thr0 && b < thr0 + a.n_thr) {
        b -= thr0;
        if (a.active_thr != nullptr) {
            if (b >= *a.nactive_thr) return;
            b = a.active_thr[b];
        }
        if (ASK && q.state_thr && q.state_thr->neutral) return;
        LineEpilogue ep{};
        ep.deltac = a.deltac;
        ep.denom = a.denom_thr;
        ep.inv_zeta = 1.0 / a.zeta;
        ep.mask = a.mask;
        ep.bmax = const_cast<float*>(a.bmax_thr);
        ep.th = a.th;
        ep.scaled = a.scaled_thr;
        lines_block<N1, N2, L, kLineThreshold>(a.Uthr, C::HO, tw, a.cmax_thr, ep, b, buf, stw, smask);
        return;
    }
    if (b >= thr0 + a.n_thr) b -= a.n_thr;
    const bool mem = b >= a.n_sum;
    int i = mem ? b - a.n_sum : b;
    if (!mem) {
        if (ASK && q.state_sum && q.state_sum->neutral) return;
        LineEpilogue ep{};
        ep.deltac = a.deltac;
        ep.denom = a.denom_sum;
        ep.partial = a.partial_sum;
        ep.bmax = a.bmax_sum;
        lines_block<N1, N2, L, kLineSum>(a.Usum, C::HO, tw, a.cmax_sum, ep, i, buf, stw, smask);
    } else if (i < a.n_cols) {
        columns_body<D1, D2, W, kRounds, true>(a.S, a.Tcols, C::HO, tw, a.fp_cols, a.fp_cols.scale, i / a.ncg_cols,
                                i % a.ncg_cols, lds);
    } else {
        i -= a.n_cols;
        FusedParams fp{};
        fp.m2max = a.m2max_rows;
        fp.cmax = a.cmax_rows;
        rows_body<D1, D2, W, kRounds>(a.Trows, C::HO, tw, fp, i / a.ncg_rows, i % a.ncg_rows, lds,
                                      ASK ? q.bound_rows : nullptr);
    }
}

template <int D1, int D2, int W, int N1, int N2, int L>
__global__ __launch_bounds__(W* D1, 8) void k_fused_radius(RadiusRoles a, const float2* __restrict__ tw) {
    radius_roles<D1, D2, W, N1, N2, L, false>(a, AskRoles{}, tw);
}
template <int D1, int D2, int W, int N1, int N2, int L>
__global__ __launch_bounds__(W* D1, 8) void k_fused_radius_ask(RadiusRoles a, AskRoles q,
                                                              const float2* __restrict__ tw) {
    radius_roles<D1, D2, W, N1, N2, L, true>(a, q, tw);
}

// ------------------------------------------------------------------ all radii at once
// For sides up to 160 a launch per radius leaves most of the chip idle (64 to
// 800 line groups on 2048 block slots) and the ~45 launches of a box cost more
// than their work.  Here each role runs once, over every (radius, group): the
// columns, the rows, the box sums, the reductions (nonlinear input), the
// thresholds and the paint, with the same device bodies on the same tiles, so
// the results are those of the launch per radius bit for bit.  What the loop
// orders, the ionization mask, becomes one bit plane per radius: a group's
// threshold block writes its hits where it has any, and the paint ORs the
// flagged planes.  The thresholds of linear input are found on the device with
// the verdicts on whole radii (box_stays_neutral).
// A call of conv_bubbles takes 65 us at 64^3 (linear, 37 radii; 279 with a
// launch per radius) and 210 us at 128^3 (nonlinear, 40 radii; 463), 90 of them
// the box sums (VALU-bound; 130 without the verdicts).
__device__ __forceinline__ int radius_of_block(const int* blk, int nr, int x) {
    int lo = 0, hi = nr - 1;  // last r with blk[r] <= x
    while (lo < hi) {
        const int mid = (lo + hi + 1) >> 1;
        if (blk[mid] <= x)
            lo = mid;
        else
            hi = mid - 1;
    }
    return lo;
}

// LDS rounds and tile of the columns and rows bodies, as in k_fused_radius.
template <int D1, int D2, int W, int N1, int N2, int L>
struct ColumnTile {
    using C = LinesCore<N1, N2, L>;
    static constexpr int D = D1 * D2;
    static constexpr int kLdsLines = L * C::HP + D + C::WORDS;
    static constexpr int kRounds = W * (D + 1) > kLdsLines + kLdsLines / 4 ? 0 : 1;
    static constexpr int kLdsCR = kRounds == 0 ? (W * (D + 1) + 1) / 2 : W * (D + 1);
};

template <int D1, int D2, int W, int N1, int N2, int L>
__global__ __launch_bounds__(W* D1) void k_all_columns(AllRadii a, const float2* __restrict__ tw) {
    using CT = ColumnTile<D1, D2, W, N1, N2, L>;
    __shared__ float2 lds[CT::kLdsCR];
    const int x = blockIdx.x;
    const int r = radius_of_block(a.cblk, a.nr, x), i = x - a.cblk[r];
    const AllRadius& R = a.r[r];
    columns_body<D1, D2, W, CT::kRounds, true>(a.S, a.T + R.toff, R.ho, tw, R.fp, R.fp.scale, i / R.ncg, i % R.ncg, lds);
}

__device__ __forceinline__ bool bounded(const AllRadius& R) {
    return R.fp.cmax < kBoundModes && R.ncg <= kBoundGroups;
}

template <int D1, int D2, int W, int N1, int N2, int L>
__global__ __launch_bounds__(W* D1) void k_all_rows(AllRadii a, const float2* __restrict__ tw) {
    using CT = ColumnTile<D1, D2, W, N1, N2, L>;
    __shared__ float2 lds[CT::kLdsCR];
    const int x = blockIdx.x;
    const int r = radius_of_block(a.rblk, a.nr, x), i = x - a.rblk[r];
    const AllRadius& R = a.r[r];
    rows_body<D1, D2, W, CT::kRounds>(a.T + R.toff, R.ho, tw, R.fp, i / R.ncg, i % R.ncg, lds,
                                      bounded(R) ? a.bound + (size_t)r * CT::D * kBoundGroups : nullptr);
}

// One block per radius: the threshold of linear input, and whether the box
// stays neutral there (never asked of the last radius, which is painted).
template <int NT, int D>
__global__ __launch_bounds__(NT) void k_all_verdicts(AllRadii a) {
    const int r = blockIdx.x;
    const AllRadius& R = a.r[r];
    SkipArgs sk{};
    ScaledThreshold s{};
    s.scale = 1.0f;
    if (a.linear) s.th = density_threshold(a.deltac, R.denom, a.zeta, 1.0f);
    if (r < a.nr - 1 && bounded(R)) {
        sk.bound = a.bound + (size_t)r * D * kBoundGroups;
        sk.S0 = a.S;
        sk.groups = R.ncg;
        sk.linear = a.linear;
        sk.deltac = a.deltac;
        sk.zeta_fc_mean = (float)(a.zeta * (double)a.fc_mean);
        sk.th = s.th;
    }
    s.neutral = box_stays_neutral<NT, D>(sk, R.fp.scale, R.denom) ? 1 : 0;
    if (threadIdx.x == 0) a.scaled[r] = s;
}

template <int N1, int N2, int L>
__global__ __launch_bounds__(L* N1) void k_all_sums(AllRadii a, const float2* __restrict__ tw) {
    using C = LinesCore<N1, N2, L>;
    __shared__ float2 buf[L * C::HP];
    __shared__ float2 stw[C::D];
    __shared__ unsigned long long smask[C::WORDS];
    const int r = blockIdx.y;
    const AllRadius& R = a.r[r];
    if (a.scaled[r].neutral) return;
    LineEpilogue ep{};
    ep.deltac = a.deltac;
    ep.denom = R.denom;
    ep.partial = a.partial + (size_t)r * a.nblk;
    ep.bmax = a.bmax + (size_t)r * a.nblk;
    lines_block<N1, N2, L, kLineSum>(a.T + R.toff, R.ho, tw, R.fp.cmax, ep, blockIdx.x, buf, stw, smask);
}

template <int NT>
__global__ __launch_bounds__(NT) void k_all_reduce(AllRadii a) {
    const int r = blockIdx.x;
    const SumScaleArgs sa{a.scaled + r, a.fc_mean, a.deltac, a.r[r].denom, a.ncells, a.zeta,
                          nullptr,      nullptr,   nullptr};
    finish_box_sum<NT>(a.partial + (size_t)r * a.nblk, a.nblk, a.nblk, a.sums + r, sa, a.scaled + r);
}

template <int N1, int N2, int L>
__global__ __launch_bounds__(L* N1) void k_all_thresholds(AllRadii a, const float2* __restrict__ tw) {
    using C = LinesCore<N1, N2, L>;
    constexpr int D = C::D, NT = C::NT, WORDS = C::WORDS;
    __shared__ float2 buf[L * C::HP];
    __shared__ float2 stw[D];
    __shared__ unsigned long long smask[WORDS];
    const int t = threadIdx.x, r = blockIdx.y, blk = blockIdx.x;
    const AllRadius& R = a.r[r];
    const ScaledThreshold sc = a.scaled[r];
    unsigned* hit_flag = a.hits + (size_t)r * a.nblk + blk;
    const size_t line0 = (size_t)blk * L;
    // no cell of the group can reach the threshold (cells inside the band
    // take the exact test, so the skip never drops a hit)
    const bool none =
        sc.neutral || (!a.linear && a.bmax[(size_t)r * a.nblk + blk] < sc.th.dstar - sc.th.band);
    if (none) {
        if (t == 0) *hit_flag = 0u;
        return;
    }
    float2 tmp[C::LOADS];
    C::load(a.T + R.toff + line0 * R.ho, R.ho, R.fp.cmax + 1, tmp);
    for (int q = t; q < D; q += NT) stw[q] = tw[q];
    C::store(tmp, buf);
    __syncthreads();
    C::transform(buf, stw, R.fp.cmax + 1);
    const float* xrf = reinterpret_cast<const float*>(buf);
    const double inv_zeta = 1.0 / a.zeta;
    unsigned long long any = 0ull;
#pragma unroll 4
    for (int q = 0; q < L * D / NT; ++q) {
        const int f = t + q * NT;
        const int i = f / D, c = f - i * D;
        const unsigned long long bits = __ballot(
            cell_hit(xrf[i * 2 * C::HP + c], sc.th, a.deltac, R.denom, !a.linear, sc.scale, inv_zeta));
        if ((t & 63) == 0) smask[f >> 6] = bits;
        any |= bits;
    }
    const bool hit = __syncthreads_or(any != 0ull);
    if (t == 0) *hit_flag = hit ? 1u : 0u;
    if (hit && t < WORDS) a.planes[((size_t)r * a.nblk + blk) * WORDS + t] = smask[t];
}

template <int N1, int N2, int L>
__global__ __launch_bounds__(L* N1) void k_all_paint(AllRadii a, const float2* __restrict__ tw) {
    using C = LinesCore<N1, N2, L>;
    __shared__ float2 buf[L * C::HP];
    __shared__ float2 stw[C::D];
    __shared__ unsigned long long smask[C::WORDS];
    const int t = threadIdx.x, blk = blockIdx.x, last = a.nr - 1;
    const AllRadius& R = a.r[last];
    // every wave reads the group's flags at once (last < 64) and ORs the flagged planes
    const int lane = t & 63;
    unsigned long long word = 0ull, flags = __ballot(lane < last && a.hits[(size_t)lane * a.nblk + blk]);
    for (; flags; flags &= flags - 1) {
        const int r = __ffsll((long long)flags) - 1;
        if (t < C::WORDS) word |= a.planes[((size_t)r * a.nblk + blk) * C::WORDS + t];
    }
    LineEpilogue ep{};
    ep.deltac = a.deltac;
    ep.denom = R.denom;
    ep.zeta = a.zeta;
    ep.inv_zeta = 1.0 / a.zeta;
    ep.out = a.out;
    ep.th = a.scaled[last].th;
    ep.scaled = a.linear ? nullptr : a.scaled + last;
    lines_block<N1, N2, L, kLinePaint>(a.T + R.toff, R.ho, tw, R.fp.cmax, ep, blk, buf, stw, smask, word);
}

// Pruned r2c of the fused loop (three launches): only the modes that the
// smallest radius keeps (|n|^2 <= m2max, c <= cmax) are formed.
// Lines: the r2c along c of L lines per block, from the real box into T0
// (stride HO, c <= cmax).  Bound by memory: 170 us at 512^3 with 160 of 257 modes
// kept (5.1 TB/s), 320 with each load waiting for the store of the one before and
// a division per mode of the second loop.
template <int N1, int N2, int L>
__global__ __launch_bounds__(L* N1) void k_fwd_lines(const float* __restrict__ delta, float2* __restrict__ T0,
                                                    const float2* __restrict__ tw, int cmax) {
    using C = LinesCore<N1, N2, L>;
    constexpr int N = C::N, D = C::D, NT = C::NT, HP = C::HP;
    __shared__ float2 buf[L * HP];
    __shared__ float2 stw[D];
    const int t = threadIdx.x;
    const size_t line0 = (size_t)blockIdx.x * L;
    const float2* src = reinterpret_cast<const float2*>(delta + line0 * D);
    // all global loads in flight before the first LDS store
    static_assert(L * N % NT == 0, "whole loads");
    float2 tmp[L * N / NT];
#pragma unroll
    for (int q = 0; q < L * N / NT; ++q) tmp[q] = src[t + q * NT];
    for (int q = t; q < D; q += NT) stw[q] = tw[q];
#pragma unroll
    for (int q = 0; q < L * N / NT; ++q) {
        const int f = t + q * NT, i = f / N;
        buf[i * HP + f - i * N] = tmp[q];
    }
    __syncthreads();
    forward_pairs<N1, N2, L>(buf, stw);
    // N1 lanes to a line
    const int i = t / N1;
    for (int k = t % N1; k <= cmax; k += N1) {
        const float2 Wk = buf[i * HP + (k == N ? 0 : k)];
        const float2 Wmk = buf[i * HP + (k == 0 ? 0 : N - k)];
        T0[(line0 + i) * C::HO + k] = line_spectrum(Wk, Wmk, stw[k]);
    }
}

// Rows and columns of the forward transform: the re/im-staged transpose (a
// float tile of W*(D+1)) keeps the LDS of a block at half the
// one-round tile; at six waves per SIMD they need no scratch (at eight they
// spill a few registers at D = 256 and run slower).
template <int D1, int D2, int W>
__global__ __launch_bounds__(W* D1, 6) void k_fwd_rows(float2* __restrict__ T0, const float2* __restrict__ tw,
                                                      int cmax, int m2max) {
    constexpr int D = D1 * D2;
    __shared__ float lds[W * (D + 1)];
    fwd_rows_body<D1, D2, W, 0>(T0, padded_row(D / 2 + 1), tw, cmax, m2max, blockIdx.y, blockIdx.x,
                                reinterpret_cast<float2*>(lds));
}

template <int D1, int D2, int W>
__global__ __launch_bounds__(W* D1, 6) void k_fwd_columns(const float2* __restrict__ T0, float2* __restrict__ S,
                                                         const float2* __restrict__ tw, int bm, int cmax, int m2max) {
    constexpr int D = D1 * D2;
    __shared__ float lds[W * (D + 1)];
    fwd_columns_body<D1, D2, W, 0>(T0, padded_row(D / 2 + 1), S, tw, bm, cmax, m2max, blockIdx.y, blockIdx.x,
                                   reinterpret_cast<float2*>(lds));
}

// Whole c2r of a half spectrum S[a][b][c] (no window): columns along a into the
// padded rows T[p][b][c], rows along b in place, lines along c into the box.
// Bound by memory, three passes over the half box: 261 + 231 + 278 us at 512^3, at
// 4.1 to 4.9 TB/s, where a large copy runs at 4.7 (the library's transform, which
// overwrites its input, 1460 us and 200 for a copy of it); 79 us at 256^3 (152 and
// 22).  A block has 16 columns or more, 128 bytes of a line.
template <int D1, int D2, int W>
struct InverseTile {
    static constexpr int D = D1 * D2, H = D / 2 + 1, HO = padded_row(H), NCG = (H + W - 1) / W;
    static_assert(D % 8 == 0, "whole lines per XCD");
    // The column groups of a line follow each other on one XCD, so that a 128-byte
    // line of S that two groups share is fetched into one L2: blocks go to
    // the eight XCDs in turn.
    __device__ static __forceinline__ void of_block(int x, int* line, int* group) {
        const int i = x >> 3;
        *line = (x & 7) + 8 * (i / NCG);
        *group = i % NCG;
    }
};

template <int D1, int D2, int W>
__global__ __launch_bounds__(W* D1) void k_inv_columns(const float2* __restrict__ S, float2* __restrict__ T,
                                                      const float2* __restrict__ tw) {
    using I = InverseTile<D1, D2, W>;
    constexpr int D = I::D, H = I::H;
    __shared__ float lds[W * (D + 1)];
    int b, group;
    I::of_block(blockIdx.x, &b, &group);
    const int t = threadIdx.x, n1 = t / W, c0 = group * W, c = c0 + t % W;
    float2 v[D2];
#pragma unroll
    for (int n2 = 0; n2 < D2; ++n2)
        v[n2] = c < H ? S[((size_t)(n1 + D1 * n2) * D + b) * H + c] : make_float2(0.0f, 0.0f);
    dft<D2>(v);
    transpose_finish<D1, D2, W, 0>(v, tw, reinterpret_cast<float2*>(lds), [&](int jj, int k2, int k1, float2 u) {
        if (c0 + jj < H) T[((size_t)(k2 + D2 * k1) * D + b) * I::HO + c0 + jj] = u;
    });
}

template <int D1, int D2, int W>
__global__ __launch_bounds__(W* D1) void k_inv_rows(float2* __restrict__ T, const float2* __restrict__ tw) {
    using I = InverseTile<D1, D2, W>;
    constexpr int D = I::D, H = I::H;
    __shared__ float lds[W * (D + 1)];
    int p, group;
    I::of_block(blockIdx.x, &p, &group);
    const int t = threadIdx.x, n1 = t / W, c0 = group * W, c = c0 + t % W;
    float2 v[D2];
#pragma unroll
    for (int n2 = 0; n2 < D2; ++n2)
        v[n2] = c < H ? T[((size_t)p * D + n1 + D1 * n2) * I::HO + c] : make_float2(0.0f, 0.0f);
    dft<D2>(v);
    transpose_finish<D1, D2, W, 0>(v, tw, reinterpret_cast<float2*>(lds), [&](int jj, int k2, int k1, float2 u) {
        if (c0 + jj < H) T[((size_t)p * D + k2 + D2 * k1) * I::HO + c0 + jj] = u;
    });
}

template <int N1, int N2, int L>
__global__ __launch_bounds__(L* N1) void k_inv_lines(const float2* __restrict__ T, float2* __restrict__ out,
                                                    const float2* __restrict__ tw) {
    using C = LinesCore<N1, N2, L>;
    __shared__ float2 buf[L * C::HP];
    __shared__ float2 stw[C::D];
    const int t = threadIdx.x;
    const size_t line0 = (size_t)blockIdx.x * L;
    float2 tmp[C::LOADS];
    C::load(T + line0 * C::HO, C::HO, C::H, tmp);
    for (int q = t; q < C::D; q += C::NT) stw[q] = tw[q];
    C::store(tmp, buf);
    __syncthreads();
    C::transform(buf, stw);
    for (int f = t; f < L * C::N; f += C::NT) {
        const int i = f / C::N, m = f - i * C::N;
        out[line0 * C::N + f] = buf[i * C::HP + m];
    }
}

__global__ void k_fill_u64(unsigned long long* __restrict__ p, size_t n) {
    const size_t i = (size_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (i < n) p[i] = 0ull;
}


// ------------------------------------------------------------------ host side

template <int N1, int N2, int L>
int launch_lines(const float2* U, const float2* tw, int cmax, const LineEpilogue& ep, hipStream_t st) {
    constexpr int D = 2 * N1 * N2;
    k_fused_lines<N1, N2, L><<<(unsigned)((size_t)D * D / L), L * N1, 0, st>>>(U, tw, cmax, ep);
    CM21_LAUNCH_CHECK("k_fused_lines");
    return CM21_OK;
}

template <int D1, int D2, int W, int N1, int N2, int L>
int launch_radius(const RadiusRoles& a, const AskRoles& q, const float2* tw, hipStream_t st) {
    const int blocks = a.n_red + q.n_ver + a.n_thr + a.n_mem + a.n_sum;
    if (blocks <= 0) return CM21_OK;
    if (q.any)
        k_fused_radius_ask<D1, D2, W, N1, N2, L><<<blocks, W * D1, 0, st>>>(a, q, tw);
    else
        k_fused_radius<D1, D2, W, N1, N2, L><<<blocks, W * D1, 0, st>>>(a, tw);
    CM21_LAUNCH_CHECK("k_fused_radius");
    return CM21_OK;
}

template <int D1, int D2, int W, int N1, int N2, int L>
int launch_forward(const float* delta, float2* T0, float2* S, const float2* tw, const FusedParams& fp,
                   hipStream_t st) {
    constexpr int D = D1 * D2, H = D / 2 + 1;
    const int cmax = fp.cmax < H - 1 ? fp.cmax : H - 1;
    k_fwd_lines<N1, N2, L><<<D * D / L, L * N1, 0, st>>>(delta, T0, tw, cmax);
    CM21_LAUNCH_CHECK("k_fwd_lines");
    const int ncg = cmax / W + 1;
    k_fwd_rows<D1, D2, W><<<dim3(ncg, D), W * D1, 0, st>>>(T0, tw, cmax, fp.m2max);
    CM21_LAUNCH_CHECK("k_fwd_rows");
    const int bpos = fp.bm < D / 2 ? fp.bm : D / 2;
    const int bneg = fp.bm < D / 2 - 1 ? fp.bm : D / 2 - 1;
    k_fwd_columns<D1, D2, W><<<dim3(ncg, bpos + 1 + bneg), W * D1, 0, st>>>(T0, S, tw, fp.bm, cmax, fp.m2max);
    CM21_LAUNCH_CHECK("k_fwd_columns");
    return CM21_OK;
}

template <int D1, int D2, int W, int N1, int N2, int L>
int launch_inverse(const float2* S, float2* T, float* out, const float2* tw, hipStream_t st) {
    using I = InverseTile<D1, D2, W>;
    k_inv_columns<D1, D2, W><<<I::D * I::NCG, W * D1, 0, st>>>(S, T, tw);
    CM21_LAUNCH_CHECK("k_inv_columns");
    k_inv_rows<D1, D2, W><<<I::D * I::NCG, W * D1, 0, st>>>(T, tw);
    CM21_LAUNCH_CHECK("k_inv_rows");
    k_inv_lines<N1, N2, L><<<I::D * I::D / L, L * N1, 0, st>>>(T, reinterpret_cast<float2*>(out), tw);
    CM21_LAUNCH_CHECK("k_inv_lines");
    return CM21_OK;
}

template <int D1, int D2, int W, int N1, int N2, int L>
int launch_all(const AllRadii& a, const float2* tw, hipStream_t st) {
    constexpr int NT = W * D1;
    auto timed = [&](int stage, auto&& launch, const char* name) {
        const ProfToken t = prof_begin(stage, st);
        launch();
        CM21_LAUNCH_CHECK(name);
        prof_end(t, st);
        return (int)CM21_OK;
    };
    const dim3 groups(a.nblk, a.nr);
    CM21_TRY(timed(CM21_STAGE_FUSED_COLUMNS, [&] {
        k_all_columns<D1, D2, W, N1, N2, L><<<a.cblk[a.nr], NT, 0, st>>>(a, tw);
    }, "k_all_columns"));
    CM21_TRY(timed(CM21_STAGE_FUSED_ROWS, [&] {
        k_all_rows<D1, D2, W, N1, N2, L><<<a.rblk[a.nr], NT, 0, st>>>(a, tw);
    }, "k_all_rows"));
    k_all_verdicts<NT, D1 * D2><<<a.nr, NT, 0, st>>>(a);
    CM21_LAUNCH_CHECK("k_all_verdicts");
    if (!a.linear) {
        CM21_TRY(timed(CM21_STAGE_FCOLL_SUM, [&] { k_all_sums<N1, N2, L><<<groups, NT, 0, st>>>(a, tw); }, "k_all_sums"));
        k_all_reduce<NT><<<a.nr, NT, 0, st>>>(a);
        CM21_LAUNCH_CHECK("k_all_reduce");
    }
    if (a.nr > 1)
        CM21_TRY(timed(CM21_STAGE_FUSED_LINES_THRESHOLD, [&] {
            k_all_thresholds<N1, N2, L><<<dim3(a.nblk, a.nr - 1), NT, 0, st>>>(a, tw);
        }, "k_all_thresholds"));
    return timed(CM21_STAGE_FUSED_LINES, [&] { k_all_paint<N1, N2, L><<<a.nblk, NT, 0, st>>>(a, tw); }, "k_all_paint");
}

// At 512^3 blocks of 256 threads on 16 columns (128 bytes) and 16 lines: 11.0 ms a box
// with linear input and 14.3 with nonlinear, against 14.1 and 17.4 with blocks of 128 on
// eight, whose 64-byte pieces fetched a line's halves into two L2s.
// D, all radii, lines (N1, N2, L), radius (columns/rows D1, D2, W; lines N1, N2, L), forward, inverse
const FusedShape kShapes[] = {
    {64, launch_all<8, 8, 32, 4, 8, 64>, launch_lines<4, 8, 64>,
     launch_radius<8, 8, 32, 4, 8, 64>, launch_forward<8, 8, 32, 4, 8, 64>, launch_inverse<8, 8, 32, 4, 8, 64>,
     32, 64},
    {96, launch_all<8, 12, 32, 4, 12, 64>, launch_lines<4, 12, 64>,
     launch_radius<8, 12, 32, 4, 12, 64>, launch_forward<8, 12, 32, 4, 12, 64>, launch_inverse<8, 12, 32, 4, 12, 64>,
     32, 64},
    {128, launch_all<8, 16, 32, 8, 8, 32>, launch_lines<8, 8, 32>,
     launch_radius<8, 16, 32, 8, 8, 32>, launch_forward<8, 16, 32, 8, 8, 32>, launch_inverse<8, 16, 32, 8, 8, 32>,
     32, 32},
    {160, launch_all<16, 10, 16, 8, 10, 32>, launch_lines<8, 10, 32>,
     launch_radius<16, 10, 16, 8, 10, 32>, launch_forward<16, 10, 16, 8, 10, 32>, launch_inverse<16, 10, 16, 8, 10, 32>,
     16, 32},
    {256, nullptr, launch_lines<16, 8, 16>,
     launch_radius<16, 16, 16, 16, 8, 16>, launch_forward<16, 16, 16, 16, 8, 16>, launch_inverse<16, 16, 16, 16, 8, 16>,
     16, 16},
    {512, nullptr, launch_lines<16, 16, 16>,
     launch_radius<16, 32, 16, 16, 16, 16>, launch_forward<16, 32, 16, 16, 16, 8>, launch_inverse<16, 32, 16, 16, 16, 8>,
     16, 16},
};

const FusedShape* fused_shape(int D) {
    for (const auto& s : kShapes)
        if (s.D == D) return &s;
    return nullptr;
}

size_t fused_partials(int D) {
    const FusedShape* s = fused_shape(D);
    return s ? (size_t)D * D / sum_lines(D, s->L) : 0;
}

// Per-radius bounds of the pruned transforms.
FusedParams fused_params(int D, float dk, float R, int filter_type, int ref_fallthrough, float scale) {
    FusedParams fp{};
    const int h = D / 2;
    const int all = 3 * h * h;
    fp.dk = dk;
    fp.R = R;
    fp.scale = scale;
    const double ln2 = 0.69314718055994530942;
    const bool cut = filter_type == 1;  // type 0 stays on the generic path
    if (cut) {
        const double kcut = 1.0 / (0.413566994 * (double)dk * (double)R);  // in units of dk
        const double m2c = kcut * kcut;
        const double hi = std::floor(m2c * (1.0 + 1e-5)), lo = std::ceil(m2c * (1.0 - 1e-5));
        fp.m2max = hi >= (double)all ? all : (int)hi;
        fp.m2lo = lo >= (double)all ? all + 1 : (int)lo;
        fp.exact_cut = 1;
    } else {
        fp.m2max = all;
        fp.m2lo = all + 1;
        fp.exact_cut = 0;
    }
    double kappa = 0.0;
    if (ref_fallthrough)
        kappa = filter_type == 1 ? 0.413566994 * 0.643 : 0.643;
    else
        kappa = filter_type == 2 ? 0.643 : 0.0;
    const double g = kappa * (double)dk * (double)R;
    fp.gcoef = (float)(-(g * g) / 2.0 / ln2);
    int bm = (int)std::floor(std::sqrt((double)fp.m2max));
    while ((long)(bm + 1) * (bm + 1) <= fp.m2max) ++bm;
    while ((long)bm * bm > fp.m2max) --bm;
    fp.bm = bm < h ? bm : h;
    fp.cmax = fp.bm;
    return fp;
}

void column_groups(const FusedShape& sh, const FusedParams& fp, int* ncg, int* nb) {
    const int D = sh.D, H = D / 2 + 1;
    const int bpos = fp.bm < D / 2 ? fp.bm : D / 2;
    const int bneg = fp.bm < D / 2 - 1 ? fp.bm : D / 2 - 1;
    *nb = bpos + 1 + bneg;
    const int ncg_all = (H + sh.W - 1) / sh.W;
    *ncg = std::min(fp.cmax / sh.W + 1, ncg_all);
}

int fused_lines(const FusedShape& sh, const float2* U, const float2* tw, const FusedParams& fp,
                const LineEpilogue& ep, hipStream_t st, int stage) {
    ProfToken t = prof_begin(stage, st);
    CM21_TRY(sh.lines(U, tw, fp.cmax, ep, st));
    prof_end(t, st);
    return CM21_OK;
}

int fused_forward(const FusedShape& sh, const float* delta, float2* T0, float2* S, const float2* tw,
                  const FusedParams& fp, hipStream_t st) {
    ProfToken t = prof_begin(CM21_STAGE_R2C, st);
    CM21_TRY(sh.forward(delta, T0, S, tw, fp, st));
    prof_end(t, st);
    return CM21_OK;
}

int fused_radius_launch(const FusedShape& sh, const RadiusRoles& a, const AskRoles& q, const float2* tw,
                        hipStream_t st) {
    ProfToken t = prof_begin(CM21_STAGE_FUSED_RADIUS, st);
    CM21_TRY(sh.radius(a, q, tw, st));
    prof_end(t, st);
    return CM21_OK;
}

size_t all_radii_table(const FusedShape& sh, float dk, const float* radii, const float* denoms, int n_radii,
                       int filter_type, int ref_fallthrough, float scale, AllRadii* a) {
    if (!sh.all || n_radii > kAllRadii) return 0;
    const int D = sh.D;
    size_t off = 0;
    int nc = 0, nrow = 0;
    a->nr = n_radii;
    a->nblk = (int)fused_partials(D);
    for (int r = 0; r < n_radii; ++r) {
        AllRadius& R = a->r[r];
        R.fp = fused_params(D, dk, radii[r], filter_type, ref_fallthrough, scale);
        R.denom = denoms ? denoms[r] : 0.0f;
        R.ho = padded_row(std::min(R.fp.cmax, D / 2) + 1);
        R.toff = off;
        off += (size_t)D * D * R.ho;
        int nb = 0;
        column_groups(sh, R.fp, &R.ncg, &nb);
        a->cblk[r] = nc;
        a->rblk[r] = nrow;
        nc += R.ncg * nb;
        nrow += R.ncg * D;
    }
    a->cblk[n_radii] = nc;
    a->rblk[n_radii] = nrow;
    return off;
}

int fused_all_radii(const FusedShape& sh, const AllRadii& a, const float2* tw, hipStream_t st) {
    return sh.all(a, tw, st);
}

int fused_mask_clear(unsigned long long* mask, size_t words, hipStream_t st) {
    k_fill_u64<<<grid_for(words), kThreads, 0, st>>>(mask, words);
    CM21_LAUNCH_CHECK("k_fill_u64");
    return CM21_OK;
}

// erfc^-1 on the host: bisection on std::erfc (monotone decreasing) to the
// last bit, for y in (0, 2).
static double erfcinv_host(double y) {
    double lo = -6.0, hi = 27.3;  // erfc(-6) = 2 - 2e-17, erfc(27.3) < 1e-300
    for (int i = 0; i < 200 && hi - lo > 0.0; ++i) {
        const double mid = 0.5 * (lo + hi);
        if (mid == lo || mid == hi) break;
        if (std::erfc(mid) > y)
            lo = mid;
        else
            hi = mid;
    }
    return 0.5 * (lo + hi);
}

// The bound of the rows pass is the largest sum of moduli of a line's modes: on
// Gaussian and lognormal boxes of this path's spectra 1.5 to 2.5 (mostly 1.7 to 2)
// times sqrt(cmax + 1) standard deviations.  So a verdict can only come out neutral
// where the threshold (of linear input, or with the box mean at its value for
// mean density) is that many standard deviations away; sigma^2 = S(R) follows
// from the denominators and sigma_min^2 from fc_mean, where it is given.  This
// only decides whether to ask: boxes that would never pass keep the shorter
// schedule (asking in vain costs 2 % at 256^3).  With it a 256^3 box takes 1664
// us for 1822 (nonlinear, half ionized) and a 512^3 one (blocks of eight columns) 14.1 ms for 15.8 (linear).
int neutral_radii(const cm21_bubble_params& prm, const float* denoms, int n_radii, const int* cmax) {
    const double dc = prm.deltac, fc = prm.fc_mean;
    double smin = 0.5 * (double)denoms[0] * denoms[0];  // S at the largest radius counted as 0
    if (fc > 1e-30 && fc < 1.0) {
        const double x = dc / erfcinv_host(fc);
        if (0.5 * x * x > smin) smin = 0.5 * x * x;
    }
    int n = 0;
    for (; n < n_radii - 1 && cmax[n] < kBoundModes; ++n) {
        const double dn = denoms[n], s = smin - 0.5 * dn * dn;
        double y = 1.0 / prm.zeta;
        if (!prm.linear_input) y *= std::erfc(dc / dn) / fc;
        if (!(y > 1e-30 && y < 1.999)) break;
        if (dc - dn * erfcinv_host(y) < 1.7 * std::sqrt((cmax[n] + 1.0) * (s > 0.0 ? s : 0.0))) break;
    }
    return n < 4 ? 0 : n;  // the schedule's one launch more has to pay
}

DensityThreshold density_threshold_host(float deltac, float denom, double zeta, float scale) {
    const double y = 1.0 / (zeta * (double)scale);
    DensityThreshold t;
    if (!(y > 1e-30 && y < 1.999)) {
        t.dstar = 0.0f;
        t.band = INFINITY;
        return t;
    }
    const double ds = (double)deltac - (double)denom * erfcinv_host(y);
    t.dstar = (float)ds;
    t.band = (float)(1e-4 * (1.0 + std::fabs((double)deltac) + (double)denom + std::fabs(ds)));
    return t;
}

LineEpilogue line_epilogue(float deltac, float denom, double zeta, unsigned long long* mask, float* out) {
    LineEpilogue ep{};
    ep.deltac = deltac;
    ep.denom = denom;
    ep.zeta = zeta;
    ep.inv_zeta = 1.0 / zeta;
    ep.mask = mask;
    ep.out = out;
    return ep;
}

}  // namespace cm21
