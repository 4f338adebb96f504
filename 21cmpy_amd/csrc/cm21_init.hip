// Initial conditions on the GPU: the Gaussian random field written directly
// as a Hermitian r2c half spectrum, the nearest-pick subsample and the
// Zel'dovich displacement ("velocity") spectra.
//
// Reference: Programs/initialize.cu:58-95 (init_kernel), :133-146 (subsample),
// :148-190 (set_velocity); Programs/initialize.py:33-111 (driver).
#include <algorithm>
#include <cmath>

#include "cm21_internal.hpp"
#include "cm21_window.hpp"
#include "cm21_fused_api.hpp"

using namespace cm21;

namespace {

// Philox4x32-10 (Salmon et al., SC'11): ten rounds of two 32x32->64-bit
// multiplies; the key is bumped by the Weyl constants before rounds 2..10.
__device__ inline uint4 philox4x32_10(uint4 c, uint2 k) {
#pragma unroll
    for (int r = 0; r < 10; ++r) {
        if (r) {
            k.x += 0x9E3779B9u;
            k.y += 0xBB67AE85u;
        }
        // one 64-bit product instruction for both halves (they run at a quarter of
        // the rate of an add: with the ten rounds' halves apart, most of k_grf)
        const uint64_t p0 = (uint64_t)0xD2511F53u * c.x, p1 = (uint64_t)0xCD9E8D57u * c.z;
        c = make_uint4((uint32_t)(p1 >> 32) ^ c.y ^ k.x, (uint32_t)p1, (uint32_t)(p0 >> 32) ^ c.w ^ k.y, (uint32_t)p0);
    }
    return c;
}

// Box-Muller in float32, r = sqrt(-2 ln a), theta = 2 pi b, with the
// uniforms a = ((u0 >> 8) + 0.5) 2^-24 and b likewise, handled so that no
// argument is rounded: a = m 2^-25 with m = 2 (u0 >> 8) + 1 is its nearest float f
// and an exact remainder d, ln a = ln f + d/f (the next term is below 2^-26 of it);
// 2b = m' 2^-24 is exact below 1, and 2b - 1 is exact above (sin and cos change
// sign), so sincospi sees an exact argument.  Each result is within a few
// float32 ulp of the FP64 values.
__device__ inline void box_muller(uint32_t u0, uint32_t u1, float& g1, float& g2) {
    const uint32_t m0 = 2u * (u0 >> 8) + 1u;
    const float f = (float)m0, d = (float)(int)(m0 - (uint32_t)f);
    const float lna = fmaf(d, __builtin_amdgcn_rcpf(f), logf(f * 0x1p-25f));
    const float r = sqrtf(-2.0f * lna);
    const uint32_t m1 = 2u * (u1 >> 8) + 1u;
    const uint32_t half = m1 & (1u << 24);
    float s, c;
    sincospif((float)(m1 ^ half) * 0x1p-24f, &s, &c);
    g1 = r * (half ? -c : c);
    g2 = r * (half ? -s : s);
}

struct GrfParams {
    float dkf;          // 2 pi / box_len
    float norm;         // power law: sqrt(P(k) normalisation / box_len^3 * dk^n), and the
    float quarter_n;    // exponents of the amplitude norm * exp2(quarter_n log2 |n|^2
    float half_cut;     //   - half_cut |n|^2)
    float inv_volume;   // 1 / box_len^3
    uint32_t seed, box_id;
    const float* ktab;  // tabulated P(k): increasing K (NULL = power law)
    const float* ptab;
    int ntab;
};

constexpr int kMaxTable = 2048;

// Where to start looking for k in a table: the index of k if the table were
// spaced uniformly in log k between its end points (the P(k) tables are),
// from log2 K[0] and (n-1) / log2(K[n-1]/K[0]); any table works, the search
// then only walks further.
struct TableGuess {
    float l0, inv;
};

__device__ inline TableGuess table_guess(const float* K, int n) {
    TableGuess g{0.0f, 0.0f};
    if (K[0] > 0.0f && K[n - 1] > K[0]) {
        g.l0 = __log2f(K[0]);
        g.inv = (float)(n - 1) / (__log2f(K[n - 1]) - g.l0);
    }
    return g;
}

// P(k) from the table by the rule of initialize.cu:87-90: i is the first
// index with K[i] >= k and P is interpolated linearly between i-1 and i in
// float32, as init_kernel does; modes outside [K[0], K[n-1]] get 0.  The
// index is found from the log-uniform guess by stepping down while K[i-1] >= k
// and up while K[i] < k: the same first index as a bisection, in one or two
// steps on a log-spaced table.
__device__ inline float table_pk(float k, const float* K, const float* Pt, int n, const TableGuess& tg) {
    if (!(k >= K[0]) || k > K[n - 1]) return 0.0f;
    const float x = (__log2f(k) - tg.l0) * tg.inv + 1.0f;
    int hi = (int)fminf(fmaxf(x, 1.0f), (float)(n - 1));  // in [1, n-1]
    while (hi > 1 && K[hi - 1] >= k) --hi;
    while (K[hi] < k) ++hi;  // stops at n-1 at the latest: K[n-1] >= k
    const int lo = hi - 1;
    if (K[lo] >= k) return Pt[lo];  // k == K[0]
    return Pt[lo] + (Pt[hi] - Pt[lo]) * ((k - K[lo]) / (K[hi] - K[lo]));
}

// One mode: its Philox draw, amplitude and Hermitian placement.
template <bool TABLE>
__device__ __forceinline__ void grf_mode(float2* __restrict__ spec, int D, int a, int b, int c, const GrfParams& gp,
                                         const float* sK, const float* sP, const TableGuess& tg) {
    const int H = D / 2 + 1;
    const size_t idx = ((size_t)a * D + b) * H + c;
    if (a == 0 && b == 0 && c == 0) {
        spec[idx] = make_float2(0.0f, 0.0f);
        return;
    }
    // Modes on the c = 0 and c = D/2 planes pair with (-a, -b) in the same
    // plane; the pair shares the random numbers of its lower linear index.
    const bool edge = (c == 0) || (c == D / 2);
    const int ma = a ? D - a : 0, mb = b ? D - b : 0;
    const int lin_self = a * D + b, lin_mirror = ma * D + mb;  // below 2^22
    const bool use_mirror = edge && lin_mirror < lin_self;
    const bool selfconj = edge && lin_mirror == lin_self;
    const uint64_t rep = (uint64_t)(uint32_t)(use_mirror ? lin_mirror : lin_self) * (uint32_t)H + (uint32_t)c;
    const uint4 u = philox4x32_10(make_uint4((uint32_t)rep, (uint32_t)(rep >> 32), 0u, 0u), make_uint2(gp.seed, gp.box_id));
    float g1, g2;
    box_muller(u.x, u.y, g1, g2);

    // |n|^2 is an exact integer (and an exact float); the amplitude in float32
    const int na = mode_of(a, D), nb = mode_of(b, D);
    const float m2 = (float)(na * na + nb * nb + c * c);
    float amp;
    if (TABLE) {
        amp = sqrtf(table_pk(gp.dkf * sqrtf(m2), sK, sP, gp.ntab, tg) * gp.inv_volume);
    } else {
        // sqrt(k^n exp(-(k/k_cut)^2)) by one log2 and one exp2 of the hardware (1 ulp
        // each).  With |n|^2 = f 2^e, f in [1, 2), the power of 2^e goes into the result's
        // exponent and the logarithm stays below 1: 9e-8 rms of the mode (1.5e-7
        // with exp2f(n log2f(k)), expf and sqrtf, twice the instructions)
        const int e = __builtin_amdgcn_frexp_expf(m2) - 1;
        const float f = 2.0f * __builtin_amdgcn_frexp_mantf(m2);
        const float whole = rintf(gp.quarter_n * (float)e);
        const float x = fmaf(gp.quarter_n, (float)e, -whole) +
                        fmaf(gp.quarter_n, __builtin_amdgcn_logf(f), -gp.half_cut * m2);
        amp = ldexpf(gp.norm * __builtin_amdgcn_exp2f(x), (int)whole);
    }
    if (selfconj) {
        spec[idx] = make_float2(amp * g1, 0.0f);
    } else {
        const float h = amp * 0.70710678118654752f;
        spec[idx] = make_float2(h * g1, use_mirror ? -(h * g2) : h * g2);
    }
}

// Block (0, y, z) covers a = z and the kGrfRows rows b from y * kGrfRows, its 256
// threads walking the rows' modes as one run (no lane idles at the end of each
// row of D/2+1 modes), so the P(k) table is loaded into LDS once per
// kGrfRows * H modes.  Bound by the VALU (the integer products of the ten rounds
// first): 335 us at 512^3, 630 with the halves of the products apart, logarithm
// and sincos twice over and a modulo in each mode; its writes alone take 115.
constexpr int kGrfRows = 16;

template <bool TABLE>
__global__ __launch_bounds__(kThreads) void k_grf(float2* __restrict__ spec, int D, GrfParams gp) {
    __shared__ float sK[TABLE ? kMaxTable : 1], sP[TABLE ? kMaxTable : 1];
    if (TABLE) {
        for (int i = threadIdx.x; i < gp.ntab; i += kThreads) {
            sK[i] = gp.ktab[i];
            sP[i] = gp.ptab[i];
        }
        __syncthreads();
    }
    const TableGuess tg = TABLE ? table_guess(sK, gp.ntab) : TableGuess{0.0f, 0.0f};
    const int H = D / 2 + 1;
    const int a = blockIdx.z;
    const int b0 = blockIdx.y * kGrfRows;
    const int rows = min(D, b0 + kGrfRows) - b0;
    const int dr = kThreads / H, dc = kThreads - dr * H;
    int row = threadIdx.x / H, c = threadIdx.x - row * H;
    while (row < rows) {
        grf_mode<TABLE>(spec, D, a, b0 + row, c, gp, sK, sP, tg);
        row += dr;
        c += dc;
        if (c >= H) {
            c -= H;
            ++row;
        }
    }
}

__global__ void k_subsample(float* __restrict__ small, const float* __restrict__ large, int D, int sw, float pf) {
    const int k = blockIdx.x * kModeBlockX + threadIdx.x, j = blockIdx.y * kModeBlockY + threadIdx.y;
    const int i = blockIdx.z;
    if (k >= sw || j >= sw) return;
    const size_t p = ((size_t)i * sw + j) * sw + k;
    // floor(k*pixel_factor + 0.5): product in float, + 0.5 in double.
    const int lk = (int)floor((double)__fmul_rn((float)k, pf) + 0.5);
    const int lj = (int)floor((double)__fmul_rn((float)j, pf) + 0.5);
    const int li = (int)floor((double)__fmul_rn((float)i, pf) + 0.5);
    if (li >= D || lj >= D || lk >= D) return;  // never taken for pf = D/sw
    small[p] = large[((size_t)li * D + lj) * D + lk];
}

__global__ void k_velocity(float2* __restrict__ out, const float2* __restrict__ in, int D, float dk, int comp,
                           int filter_type, float R) {
    const int H = D / 2 + 1;
    const int c = blockIdx.x * kModeBlockX + threadIdx.x, b = blockIdx.y * kModeBlockY + threadIdx.y;
    const int a = blockIdx.z;
    if (c >= H || b >= D) return;
    const size_t idx = ((size_t)a * D + b) * H + c;
    const float k0 = __fmul_rn((float)mode_of(a, D), dk);
    const float k1 = __fmul_rn((float)mode_of(b, D), dk);
    const float k2 = __fmul_rn((float)c, dk);
    // initialize.cu:162: k_sq = k_x^2 + k_y^2 + k_z^2 with x the slowest axis.
    const float ksq = __fadd_rn(__fadd_rn(__fmul_rn(k0, k0), __fmul_rn(k1, k1)), __fmul_rn(k2, k2));
    const int idx_c = comp == 0 ? a : (comp == 1 ? b : c);
    const float kc = comp == 0 ? k0 : (comp == 1 ? k1 : k2);
    if (ksq == 0.0f || idx_c == D / 2) {
        out[idx] = make_float2(0.0f, 0.0f);
        return;
    }
    const float f = __fdiv_rn(kc, ksq);
    const float2 v = in[idx];
    float2 r = make_float2(-__fmul_rn(f, v.y), __fmul_rn(f, v.x));  // (i f) * v
    if (filter_type >= 0) {
        WindowParams wp{dk, R, filter_type, 1, 1};
        float w0, w2;
        bool cut;
        window_of(sqrt_rn(ksq), wp, w0, cut, w2);
        r = apply_window(r, w0, cut, w2, 1.0f);
    }
    out[idx] = r;
}

// window_of's type-0 fall-through window inside its cut (kR <= 2.4181) with the
// sine and cosine from their Taylor series in FP64 (the next terms are below 3e-15;
// both are rounded to float32 as there) and the Gaussian from the hardware's exp2:
// gauss = -(0.413566994 0.643)^2 log2(e) / 2.
__device__ __forceinline__ float window_inside(float kR, float gauss) {
    const double x = (double)kR, u = x * x;
    float w0 = 1.0f;
    double s = -3.86817017063068413e-23, c = -8.89679139245057408e-22;
    s = fma(s, u, 1.95729410633912626e-20);
    c = fma(c, u, 4.11031762331216484e-19);
    s = fma(s, u, -8.22063524662432950e-18);
    c = fma(c, u, -1.56192069685862253e-16);
    s = fma(s, u, 2.81145725434552060e-15);
    c = fma(c, u, 4.77947733238738525e-14);
    s = fma(s, u, -7.64716373181981641e-13);
    c = fma(c, u, -1.14707455977297245e-11);
    s = fma(s, u, 1.60590438368216133e-10);
    c = fma(c, u, 2.08767569878681002e-09);
    s = fma(s, u, -2.50521083854417202e-08);
    c = fma(c, u, -2.75573192239858883e-07);
    s = fma(s, u, 2.75573192239858925e-06);
    c = fma(c, u, 2.48015873015873016e-05);
    s = fma(s, u, -1.98412698412698413e-04);
    c = fma(c, u, -1.38888888888888894e-03);
    s = fma(s, u, 8.33333333333333322e-03);
    c = fma(c, u, 4.16666666666666644e-02);
    s = fma(s, u, -1.66666666666666657e-01);
    c = fma(c, u, -5.00000000000000000e-01);
    s = fma(s, u, 1.0);
    c = fma(c, u, 1.0);
    const float p3 = (float)(u * x), p2 = (float)u;
    const float inner = __fsub_rn(__fdiv_rn((float)(s * x), p3), __fdiv_rn((float)c, p2));
    if (x > 1e-4) w0 = (float)(3.0 * (double)inner);
    return w0 * __builtin_amdgcn_exp2f(gauss * p2);
}

// Spectra of boxes that are only read on every q-th cell (q = D/d): a field
// of the D^3 grid picked at multiples of q is the inverse transform on the
// d^3 grid of its spectrum folded modulo d, Y[m] = sum of W(n) X[n] over n = m
// (mod d).  One thread per mode m of the small half spectrum adds the one to
// eight modes n inside the window's cut (|n|^2 <= m2max; negative n_c through
// the conjugate of -n), in a fixed order, and forms the smoothed spectrum and
// the three displacement spectra i k/k^2 W X from one read of X.  The threads
// take a plane's modes in memory order.
//
// What bounds it: the writes of the small spectra (four of 68 MB at d = 256) and
// the FP64 window, of 8.4 M modes instead of the 67 M of the 512^3 spectrum.  At
// 512 -> 256 it takes 110 us (216 with window_of and its library functions, 185
// with those in memory order) and the four 256^3 inverse transforms 316 us, for a
// filter (585 us), three displacement passes (3 x 500), four 512^3 transforms
// (4 x 1450) and four picks (4 x 50): initial conditions 10.2 -> 1.52 ms with the
// transform of the whole box at 775 and the field at 335, perturbed density and
// velocity boxes 9.6 -> 1.11 ms with the pruned forward transform.  The strides are
// those of the spectrum's first two axes.
__global__ void k_fold_fields(float2* __restrict__ out, const float2* __restrict__ in, int D, int d, WindowParams wp,
                              float scale, int bm, int m2max, int smoothed, int velocity, size_t stride_a,
                              size_t stride_b, float gauss) {
    const int h = d / 2 + 1;
    const int i = blockIdx.x * kThreads + threadIdx.x, ma = blockIdx.y;  // a plane's modes in memory order
    if (i >= d * h) return;
    const int mb = i / h, mc = i - mb * h;
    const int lo = -min(bm, D / 2 - 1), hi = min(bm, D / 2);  // index D/2 is the mode +D/2
    float2 y[4];
#pragma unroll
    for (int q = 0; q < 4; ++q) y[q] = make_float2(0.0f, 0.0f);
    // the largest n <= hi with n = m (mod d), then down to lo
    auto first = [&](int m) { return m + (hi - m >= 0 ? (hi - m) / d : -((m - hi + d - 1) / d)) * d; };
    const int fa = first(ma), fb = first(mb), fc = first(mc);
    for (int na = fa; na >= lo; na -= d) {
        for (int nb = fb; nb >= lo; nb -= d) {
            const int left = m2max - na * na - nb * nb;
            if (left < 0) continue;
            for (int nc = fc; nc >= lo; nc -= d) {
                if (nc * nc > left) continue;
                // the stored mode: n, or -n for negative n_c
                const bool neg = nc < 0;
                int a = neg ? -na : na, b = neg ? -nb : nb;
                const int c = neg ? -nc : nc;
                if (a < 0) a += D;
                if (b < 0) b += D;
                const float k0 = __fmul_rn((float)mode_of(a, D), wp.dk);
                const float k1 = __fmul_rn((float)mode_of(b, D), wp.dk);
                const float k2 = __fmul_rn((float)c, wp.dk);
                const float ksq = __fadd_rn(__fadd_rn(__fmul_rn(k0, k0), __fmul_rn(k1, k1)), __fmul_rn(k2, k2));
                const float kR = __fmul_rn(sqrt_rn(ksq), wp.R);
                if ((float)((double)kR * 0.413566994) > 1.0f) continue;  // cut
                float2 v = in[a * stride_a + b * stride_b + c];
                const float w = window_inside(kR, gauss) * scale;
                v.x *= w;
                v.y *= neg ? -w : w;
                y[0].x += v.x;
                y[0].y += v.y;
                if (velocity && ksq != 0.0f) {
                    // i k/k^2 times the stored mode; of -n the conjugate, where k changes sign
                    const float f = (neg ? -1.0f : 1.0f) / ksq;
                    const float kk[3] = {k0, k1, k2};
                    const int idx[3] = {a, b, c};
#pragma unroll
                    for (int q = 0; q < 3; ++q) {
                        if (idx[q] == D / 2) continue;
                        const float g = f * kk[q];
                        y[q + 1].x -= g * v.y;
                        y[q + 1].y += g * v.x;
                    }
                }
            }
        }
    }
    const size_t nc = (size_t)d * d * h;
    float2* o = out + (size_t)ma * d * h + i;
    if (smoothed) {
        *o = y[0];
        o += nc;
    }
    if (velocity) {
#pragma unroll
        for (int q = 1; q < 4; ++q, o += nc) *o = y[q];
    }
}

bool valid_dim(int D) { return D >= 2 && D <= 2048 && D % 2 == 0; }

dim3 grf_grid(int D) { return dim3(1u, (unsigned)((D + kGrfRows - 1) / kGrfRows), (unsigned)D); }

}  // namespace

extern "C" int cm21_grf_init(void* spec_out, int D, double box_len, double amp, double n_index, double k_cut,
                             uint32_t seed, uint32_t box_id, void* stream) {
    CM21_REQUIRE(spec_out, "cm21_grf_init: NULL spectrum");
    CM21_REQUIRE(valid_dim(D), "cm21_grf_init: D=%d must be even in [2,2048]", D);
    CM21_REQUIRE(box_len > 0.0 && k_cut > 0.0 && amp >= 0.0, "cm21_grf_init: box_len, k_cut must be > 0, amp >= 0");
    const double vol = box_len * box_len * box_len, dk = 2.0 * M_PI / box_len, log2e = 1.4426950408889634;
    GrfParams gp{(float)dk, (float)std::sqrt(amp / vol * std::pow(dk, n_index)), (float)(0.25 * n_index),
                 (float)(0.5 * log2e * dk * dk / (k_cut * k_cut)), (float)(1.0 / vol), seed, box_id, nullptr, nullptr,
                 0};
    k_grf<false><<<grf_grid(D), kThreads, 0, (hipStream_t)stream>>>((float2*)spec_out, D, gp);
    CM21_LAUNCH_CHECK("k_grf");
    return CM21_OK;
}

extern "C" int cm21_grf_init_table(void* spec_out, int D, double box_len, const float* k_table,
                                   const float* p_table, int n_table, uint32_t seed, uint32_t box_id,
                                   void* stream) {
    CM21_REQUIRE(spec_out && k_table && p_table, "cm21_grf_init_table: NULL argument");
    CM21_REQUIRE(valid_dim(D), "cm21_grf_init_table: D=%d must be even in [2,2048]", D);
    CM21_REQUIRE(box_len > 0.0, "cm21_grf_init_table: box_len must be > 0");
    CM21_REQUIRE(n_table >= 2 && n_table <= kMaxTable, "cm21_grf_init_table: n_table=%d not in [2,%d]", n_table,
                 kMaxTable);
    GrfParams gp{(float)(2.0 * M_PI / box_len), 0.0f, 0.0f, 0.0f, (float)(1.0 / (box_len * box_len * box_len)),
                 seed, box_id, k_table, p_table, n_table};
    k_grf<true><<<grf_grid(D), kThreads, 0, (hipStream_t)stream>>>((float2*)spec_out, D, gp);
    CM21_LAUNCH_CHECK("k_grf");
    return CM21_OK;
}

extern "C" int cm21_subsample(float* small, const float* large, int D, int sw, float pixel_factor, void* stream) {
    CM21_REQUIRE(small && large, "cm21_subsample: NULL argument");
    CM21_REQUIRE(D >= 1 && sw >= 1 && sw <= D && D <= 4096, "cm21_subsample: D=%d sw=%d", D, sw);
    // The largest pick is floor((sw-1)*pf + 0.5); it must stay inside the large box.
    const double last = std::floor((double)((float)(sw - 1) * pixel_factor) + 0.5);
    CM21_REQUIRE(pixel_factor > 0.0f && last < (double)D, "cm21_subsample: pixel_factor=%g reads past D=%d",
                 (double)pixel_factor, D);
    k_subsample<<<mode_grid(sw, sw), mode_block(), 0, (hipStream_t)stream>>>(small, large, D, sw, pixel_factor);
    CM21_LAUNCH_CHECK("k_subsample");
    return CM21_OK;
}

extern "C" int cm21_velocity(void* spec_out, const void* spec_in, int D, float delta_k, int comp, int filter_type,
                             float R, void* stream) {
    CM21_REQUIRE(spec_out && spec_in, "cm21_velocity: NULL spectrum");
    CM21_REQUIRE(valid_dim(D), "cm21_velocity: D=%d must be even in [2,2048]", D);
    CM21_REQUIRE(comp >= 0 && comp <= 2, "cm21_velocity: comp=%d not in {0,1,2}", comp);
    CM21_REQUIRE(filter_type <= 2, "cm21_velocity: filter_type=%d", filter_type);
    k_velocity<<<mode_grid(D, D / 2 + 1), mode_block(), 0, (hipStream_t)stream>>>(
        (float2*)spec_out, (const float2*)spec_in, D, delta_k, comp, filter_type, R);
    CM21_LAUNCH_CHECK("k_velocity");
    return CM21_OK;
}

namespace {
// The type-0 window cuts kR > 1/0.413566994 (the kernel's float32 test decides
// inside a shell of 1e-5): the largest |n|^2 and |n| it can keep.
void fold_reach(int D, float delta_k, float R, long* m2max, int* bm) {
    const int hd = D / 2;
    const double all = 3.0 * hd * hd, kcut = 1.0 / (0.413566994 * (double)delta_k * (double)R);
    const double m2 = std::floor(kcut * kcut * (1.0 + 1e-5));
    *m2max = (R > 0.0f && m2 < all) ? (long)m2 : (long)all;
    *bm = (int)std::min<double>(std::sqrt((double)*m2max) + 1.0, (double)hd);
}

int fold(float2* out, const float2* in, int D, int sw, float delta_k, float R, float scale, int smoothed, int velocity,
         size_t stride_a, size_t stride_b, hipStream_t st) {
    long m2max;
    int bm;
    fold_reach(D, delta_k, R, &m2max, &bm);
    WindowParams wp{delta_k, R, 0, 1, 1};
    const double g = 0.413566994 * 0.643;
    const float gauss = (float)(-0.5 * g * g * std::log((double)kE) / std::log(2.0));
    k_fold_fields<<<dim3(grid_for((size_t)sw * (sw / 2 + 1)), sw), kThreads, 0, st>>>(out, in, D, sw, wp, scale, bm, (int)m2max,
                                                                     smoothed ? 1 : 0, velocity ? 1 : 0, stride_a,
                                                                     stride_b, gauss);
    CM21_LAUNCH_CHECK("k_fold_fields");
    return CM21_OK;
}

int check_fold(const char* fn, const void* out, const void* in, int D, int sw, float delta_k, int smoothed,
               int velocity) {
    CM21_REQUIRE(out && in, "%s: NULL argument", fn);
    CM21_REQUIRE(valid_dim(D), "%s: D=%d must be even in [2,2048]", fn, D);
    CM21_REQUIRE(valid_dim(sw) && sw <= D && D % sw == 0, "%s: sw=%d must be even and divide D=%d", fn, sw, D);
    CM21_REQUIRE(smoothed || velocity, "%s: no field asked for", fn);
    CM21_REQUIRE(delta_k > 0.0f, "%s: delta_k must be positive", fn);
    return CM21_OK;
}

size_t padded_spectrum_bytes(int D) { return align_up(sizeof(float2) * D * D * padded_row(D / 2 + 1), 256); }
}  // namespace

extern "C" int cm21_fold_fields(void* spec_out, const void* spec_in, int D, int sw, float delta_k, float R,
                                float scale, int smoothed, int velocity, void* stream) {
    CM21_TRY(check_fold("cm21_fold_fields", spec_out, spec_in, D, sw, delta_k, smoothed, velocity));
    const size_t H = D / 2 + 1;
    return fold((float2*)spec_out, (const float2*)spec_in, D, sw, delta_k, R, scale, smoothed, velocity, D * H, H,
                (hipStream_t)stream);
}

extern "C" size_t cm21_fold_box_workspace_bytes(int D) { return fused_shape(D) ? 2 * padded_spectrum_bytes(D) : 0; }

extern "C" int cm21_fold_box(cm21_plan* plan, void* spec_out, const float* box, int D, int sw, float delta_k, float R,
                             float scale, int smoothed, int velocity, void* work, size_t work_bytes, void* stream) {
    CM21_TRY(check_fold("cm21_fold_box", spec_out, box, D, sw, delta_k, smoothed, velocity));
    const FusedShape* sh = fused_shape(D);
    CM21_REQUIRE(plan && plan_dim(plan) == D && sh, "cm21_fold_box: no transform of D=%d", D);
    CM21_REQUIRE(work && work_bytes >= cm21_fold_box_workspace_bytes(D) && ((uintptr_t)box & 7) == 0,
                 "cm21_fold_box: workspace %zu bytes < required %zu, or a box not aligned to 8 bytes", work_bytes,
                 cm21_fold_box_workspace_bytes(D));
    float2* T = (float2*)work;
    float2* S = (float2*)((char*)work + padded_spectrum_bytes(D));
    long m2max;
    FusedParams fp{};
    fold_reach(D, delta_k, R, &m2max, &fp.bm);
    fp.m2max = (int)m2max;
    fp.cmax = fp.bm;
    CM21_TRY(fused_forward(*sh, box, T, S, plan_twiddles(plan), fp, (hipStream_t)stream));
    const size_t row = padded_row(D / 2 + 1);  // S is b-major
    return fold((float2*)spec_out, S, D, sw, delta_k, R, scale, smoothed, velocity, row, D * row, (hipStream_t)stream);
}

extern "C" size_t cm21_inverse_workspace_bytes(int D) { return fused_shape(D) ? padded_spectrum_bytes(D) : 0; }

extern "C" int cm21_inverse(cm21_plan* plan, const void* spec, float* out, void* work, size_t work_bytes,
                            void* stream) {
    CM21_REQUIRE(plan && spec && out && work, "cm21_inverse: NULL argument");
    const int D = plan_dim(plan);
    const FusedShape* sh = fused_shape(D);
    CM21_REQUIRE(sh, "cm21_inverse: no transform of D=%d", D);
    CM21_REQUIRE(work_bytes >= cm21_inverse_workspace_bytes(D) && (((uintptr_t)out | (uintptr_t)spec) & 7) == 0,
                 "cm21_inverse: workspace %zu bytes < required %zu, or an operand not aligned to 8 bytes", work_bytes,
                 cm21_inverse_workspace_bytes(D));
    return sh->inverse((const float2*)spec, (float2*)work, out, plan_twiddles(plan), (hipStream_t)stream);
}
