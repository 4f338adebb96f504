// 21-cm brightness temperature and its spherically binned power spectrum.
//
// Reference: Programs/delta_T.py:73-98 (host NumPy dT, transform, binning
// driver) and Programs/delta_T.cu:5-29 (pbox_kernel).  Bin sums are FP64 and
// counts are exact integers; the reduction order is fixed, so results are
// bitwise reproducible (the reference kernel races on `+=`, delta_T.cu:27-29).
#include <algorithm>
#include <cmath>

#include "cm21_internal.hpp"

using namespace cm21;

namespace {

__global__ void k_delta_T(float* __restrict__ dT, const float* __restrict__ xH, const float* __restrict__ delta,
                          size_t N, float c, double* __restrict__ partial) {
    double acc = 0.0;
    for (size_t p = (size_t)blockIdx.x * blockDim.x + threadIdx.x; p < N; p += (size_t)gridDim.x * blockDim.x) {
        const float v = __fmul_rn(__fmul_rn(c, xH[p]), __fadd_rn(1.0f, delta[p]));
        dT[p] = v;
        acc += (double)v;
    }
    acc = block_sum(acc);
    if (threadIdx.x == 0) partial[blockIdx.x] = acc;
}

__global__ void k_sum_partials_pk(const double* __restrict__ partial, int n, double* __restrict__ out) {
    double acc = 0.0;
    for (int i = threadIdx.x; i < n; i += blockDim.x) acc += partial[i];
    acc = block_sum(acc);
    if (threadIdx.x == 0) *out = acc;
}

// (field/mean - 1) * V/N [* mean], the array transformed at delta_T.py:80-86.
__global__ void k_pk_prep(float* __restrict__ out, const float* __restrict__ f, size_t N,
                          const double* __restrict__ sum, float vol_over_n, int dimensional) {
    const size_t p = (size_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (p >= N) return;
    const float ave = (float)(*sum / (double)N);
    float v = __fmul_rn(__fsub_rn(__fdiv_rn(f[p], ave), 1.0f), vol_over_n);
    if (dimensional) v = __fmul_rn(v, ave);
    out[p] = v;
}

// lut[m2]: the first bin whose upper edge is not below dk sqrt(m2) (edges
// ascending), -1 for the mean.  A host table of the 49 153 shells of a 256^3 box
// and its upload took longer than the spectrum's kernels.
__global__ void k_bin_lut(const double* __restrict__ edges, int nbins, int n, double dk, int32_t* __restrict__ lut) {
    const int m = blockIdx.x * blockDim.x + threadIdx.x;
    if (m >= n) return;
    const double k = __dmul_rn(dk, __dsqrt_rn((double)m));
    int lo = 0, hi = nbins;
    while (lo < hi) {
        const int mid = (lo + hi) >> 1;
        if (edges[mid] < k)
            lo = mid + 1;
        else
            hi = mid;
    }
    lut[m] = m == 0 ? -1 : lo;
}

// Bins the half spectrum.  The modes (+-a, +-b, c) share |n|^2, so a lane takes
// the up to four of them together: one table look-up and one k for four loads.
// Lanes run over the (b, c) columns of one octant, and a lane walks a segment of
// a = 0 .. D/2, along which its bin only rises: it adds up in registers and
// hands its sums over where the bin changes.  There the wavefront adds to its
// private LDS slots bin by bin, lane 0 with a fixed-order wavefront sum: the
// result does not depend on scheduling.  Blocks then write per-block partials.
// Bound by the loads' latency and the sums at bin changes.  256^3, 40 bins:
// 56 us (194 with a sum per bin present in each 64 modes).
constexpr int kPkBlocks = 1024;

__global__ __launch_bounds__(kThreads) void k_pk_bin(const float2* __restrict__ F, int D,
                                                     const int32_t* __restrict__ lut, int nbins, int segs, int len,
                                                     double dk, double norm, double* __restrict__ part_ps,
                                                     double* __restrict__ part_k,
                                                     unsigned long long* __restrict__ part_n) {
    extern __shared__ unsigned char smem[];
    double* s_ps = (double*)smem;
    double* s_k = s_ps + kWaves * nbins;
    unsigned long long* s_n = (unsigned long long*)(s_k + kWaves * nbins);
    for (int q = threadIdx.x; q < kWaves * nbins; q += blockDim.x) {
        s_ps[q] = 0.0;
        s_k[q] = 0.0;
        s_n[q] = 0ull;
    }
    __syncthreads();
    const int lane = threadIdx.x & 63, wv = threadIdx.x >> 6;
    const int H = D / 2 + 1, cols = H * H, colw = (cols + 63) / 64;
    const size_t plane = (size_t)D * H;
    for (int item = blockIdx.x * kWaves + wv; item < colw * segs; item += gridDim.x * kWaves) {
        const int col = item % colw * 64 + lane, a0 = item / colw * len;
        const int a1 = min(a0 + len, H);
        const bool in = col < cols;
        const int b = in ? col / H : 0, c = in ? col % H : 0;
        const bool two_b = b != 0 && b != D / 2;
        const float2* F0 = F + (size_t)b * H + c;
        const float2* F1 = F + (size_t)(two_b ? D - b : b) * H + c;
        const double wb = (c == 0 || c == D / 2 ? 1.0 : 2.0) * (two_b ? 2.0 : 1.0);
        int bin = -1;
        double ps = 0.0, ks = 0.0, n = 0.0;
        // adds the sums of the lanes with `out` to their bins
        auto hand_over = [&](bool out) {
            unsigned long long mask;
            while ((mask = __ballot(out)) != 0ull) {
                const int b0 = __shfl(bin, __ffsll((long long)mask) - 1, 64);
                const bool mine = out && bin == b0;
                const double sp = wave_sum(mine ? ps : 0.0);
                const double sk = wave_sum(mine ? ks : 0.0);
                const double sn = wave_sum(mine ? n : 0.0);  // whole numbers
                if (lane == 0) {
                    s_ps[wv * nbins + b0] += sp;
                    s_k[wv * nbins + b0] += sk;
                    s_n[wv * nbins + b0] += (unsigned long long)sn;
                }
                out = out && !mine;
            }
        };
        for (int a = a0; a < a1; ++a) {
            const bool two_a = a != 0 && a != D / 2;
            const int m2 = a * a + b * b + c * c;
            const int now = in ? lut[m2] : -1;
            const size_t pa = (size_t)a * plane, pm = (size_t)(two_a ? D - a : a) * plane;
            const float2 v0 = F0[pa], v1 = F1[pa], v2 = F0[pm], v3 = F1[pm];
            const bool live = now >= 0 && now < nbins;
            const bool out = bin >= 0 && now != bin;
            if (__any(out)) {
                hand_over(out);
                if (out) ps = ks = n = 0.0;
            }
            bin = live ? now : -1;
            if (live) {
                double p2 = (double)v0.x * (double)v0.x + (double)v0.y * (double)v0.y;
                if (two_b) p2 += (double)v1.x * (double)v1.x + (double)v1.y * (double)v1.y;
                if (two_a) p2 += (double)v2.x * (double)v2.x + (double)v2.y * (double)v2.y;
                if (two_a && two_b) p2 += (double)v3.x * (double)v3.x + (double)v3.y * (double)v3.y;
                const double kk = dk * sqrt((double)m2), w = two_a ? 2.0 * wb : wb;
                // p2 holds the mirrored modes; of the weights it lacks that of c
                ps += (c == 0 || c == D / 2 ? 1.0 : 2.0) * (kk * kk * kk * p2 * norm);
                ks += w * kk;
                n += w;
            }
        }
        hand_over(bin >= 0);
    }
    __syncthreads();
    for (int q = threadIdx.x; q < nbins; q += blockDim.x) {
        double ps = 0.0, ks = 0.0;
        unsigned long long n = 0;
        for (int v = 0; v < kWaves; ++v) {
            ps += s_ps[v * nbins + q];
            ks += s_k[v * nbins + q];
            n += s_n[v * nbins + q];
        }
        part_ps[(size_t)q * kPkBlocks + blockIdx.x] = ps;
        part_k[(size_t)q * kPkBlocks + blockIdx.x] = ks;
        part_n[(size_t)q * kPkBlocks + blockIdx.x] = n;
    }
}

// One block per bin: each thread adds a strided subset of the per-block
// partials in a fixed order, then a fixed tree over lanes and waves
// (deterministic).
__global__ __launch_bounds__(kThreads) void k_pk_final(const double* __restrict__ part_ps,
                                                       const double* __restrict__ part_k,
                                                       const unsigned long long* __restrict__ part_n, int nblocks,
                                                       double* __restrict__ ps, double* __restrict__ ks,
                                                       unsigned long long* __restrict__ n) {
    __shared__ double wa[kWaves], wb[kWaves];
    __shared__ unsigned long long wc[kWaves];
    const int q = blockIdx.x;
    double a = 0.0, b = 0.0;
    unsigned long long c = 0;
    for (int i = threadIdx.x; i < nblocks; i += kThreads) {
        a += part_ps[(size_t)q * kPkBlocks + i];
        b += part_k[(size_t)q * kPkBlocks + i];
        c += part_n[(size_t)q * kPkBlocks + i];
    }
    a = wave_sum(a);
    b = wave_sum(b);
    c = wave_sum_u64(c);
    const int lane = threadIdx.x & 63, w = threadIdx.x >> 6;
    if (lane == 0) {
        wa[w] = a;
        wb[w] = b;
        wc[w] = c;
    }
    __syncthreads();
    if (threadIdx.x == 0) {
        double ta = 0.0, tb = 0.0;
        unsigned long long tc = 0;
        for (int v = 0; v < kWaves; ++v) {
            ta += wa[v];
            tb += wb[v];
            tc += wc[v];
        }
        ps[q] = ta;
        ks[q] = tb;
        n[q] = tc;
    }
}

struct PkWork {
    float* field;
    float2* spec;
    double* part_ps;
    double* part_k;
    unsigned long long* part_n;
    size_t bytes;
};

PkWork carve_pk(void* base, int D, int nbins) {
    const size_t N = (size_t)D * D * D, Nc = (size_t)D * D * (D / 2 + 1);
    char* p = (char*)base;
    PkWork w{};
    size_t off = 0;
    w.field = (float*)(p + off);
    off = align_up(off + sizeof(float) * N, 256);
    w.spec = (float2*)(p + off);
    off = align_up(off + sizeof(float2) * Nc, 256);
    w.part_ps = (double*)(p + off);
    off = align_up(off + sizeof(double) * kPkBlocks * (size_t)nbins, 256);
    w.part_k = (double*)(p + off);
    off = align_up(off + sizeof(double) * kPkBlocks * (size_t)nbins, 256);
    w.part_n = (unsigned long long*)(p + off);
    off = align_up(off + sizeof(unsigned long long) * kPkBlocks * (size_t)nbins, 256);
    w.bytes = off;
    return w;
}

}  // namespace

namespace cm21 {
int plan_dim(const cm21_plan* p);
int plan_batch(const cm21_plan* p);
}

extern "C" int cm21_delta_T(float* dT, const float* xH, const float* delta, int D, float tb_const, double* dev_sum,
                            void* work, void* stream) {
    CM21_REQUIRE(dT && xH && delta && dev_sum && work, "cm21_delta_T: NULL argument");
    CM21_REQUIRE(D >= 1 && D <= 2048, "cm21_delta_T: D=%d out of range", D);
    hipStream_t st = (hipStream_t)stream;
    const size_t N = (size_t)D * D * D;
    double* partial = (double*)work;
    k_delta_T<<<kReduceBlocks, kThreads, 0, st>>>(dT, xH, delta, N, tb_const, partial);
    CM21_LAUNCH_CHECK("k_delta_T");
    k_sum_partials_pk<<<1, kThreads, 0, st>>>(partial, kReduceBlocks, dev_sum);
    CM21_LAUNCH_CHECK("k_sum_partials_pk");
    return CM21_OK;
}

extern "C" size_t cm21_pk_workspace_bytes(int D, int nbins) {
    if (D < 2 || D > 2048 || D % 2 || nbins < 1) return 0;
    return carve_pk(nullptr, D, nbins).bytes;
}

extern "C" int cm21_bin_lut(const double* edges, int nbins, int D, double dk, int32_t* lut, void* stream) {
    CM21_REQUIRE(edges && lut, "cm21_bin_lut: NULL argument");
    CM21_REQUIRE(D >= 2 && D <= 2048 && D % 2 == 0, "cm21_bin_lut: D=%d must be even in [2,2048]", D);
    CM21_REQUIRE(nbins >= 1 && nbins <= 512, "cm21_bin_lut: nbins=%d not in [1,512]", nbins);
    const int n = 3 * (D / 2) * (D / 2) + 1;
    k_bin_lut<<<grid_for(n), kThreads, 0, (hipStream_t)stream>>>(edges, nbins, n, dk, lut);
    CM21_LAUNCH_CHECK("k_bin_lut");
    return CM21_OK;
}

extern "C" int cm21_power_spectrum(cm21_plan* plan, const float* field, const double* field_sum, int D,
                                   double box_len, const int32_t* bin_lut, int nbins, int dimensional, double* ps_sum,
                                   double* k_sum, uint64_t* counts, void* work, size_t work_bytes, void* stream) {
    CM21_REQUIRE(plan && field && field_sum && bin_lut && ps_sum && k_sum && counts && work,
                 "cm21_power_spectrum: NULL argument");
    CM21_REQUIRE(plan_dim(plan) == D && plan_batch(plan) == 1, "cm21_power_spectrum: plan is not a batch-1 D=%d plan",
                 D);
    CM21_REQUIRE(nbins >= 1 && nbins <= 512, "cm21_power_spectrum: nbins=%d not in [1,512]", nbins);
    CM21_REQUIRE(box_len > 0.0, "cm21_power_spectrum: box_len must be positive");
    PkWork w = carve_pk(work, D, nbins);
    if (work_bytes < w.bytes)
        return cm21::fail(CM21_ERR_NOMEM, "cm21_power_spectrum: workspace %zu bytes < required %zu", work_bytes,
                          w.bytes);
    hipStream_t st = (hipStream_t)stream;
    const size_t N = (size_t)D * D * D;
    const double V = box_len * box_len * box_len;
    k_pk_prep<<<grid_for(N), kThreads, 0, st>>>(w.field, field, N, field_sum, (float)(V / (double)N),
                                                dimensional ? 1 : 0);
    CM21_LAUNCH_CHECK("k_pk_prep");
    CM21_TRY(cm21_r2c(plan, w.field, w.spec, stream));
    const size_t lds = (sizeof(double) * 2 + sizeof(unsigned long long)) * kWaves * (size_t)nbins;
    // segments of a: as many as fill the waves of kPkBlocks blocks
    const int H = D / 2 + 1, colw = (H * H + 63) / 64, want = std::max(kPkBlocks * kWaves / colw, 1);
    const int len = (H + want - 1) / want, segs = (H + len - 1) / len;
    const int blocks = std::min((colw * segs + kWaves - 1) / kWaves, kPkBlocks);
    k_pk_bin<<<blocks, kThreads, lds, st>>>(w.spec, D, bin_lut, nbins, segs, len, 2.0 * M_PI / box_len,
                                            1.0 / (2.0 * M_PI * M_PI * V), w.part_ps, w.part_k, w.part_n);
    CM21_LAUNCH_CHECK("k_pk_bin");
    k_pk_final<<<nbins, kThreads, 0, st>>>(w.part_ps, w.part_k, w.part_n, blocks, ps_sum, k_sum,
                                           (unsigned long long*)counts);
    CM21_LAUNCH_CHECK("k_pk_final");
    return CM21_OK;
}
