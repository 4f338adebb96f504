// Internal interface of the fused, pruned transform passes (cm21_fused.hip)
// used by the radius-loop driver.
#pragma once

#include "cm21_internal.hpp"

namespace cm21 {

struct FusedParams {
    int m2max;      // modes with |n|^2 > m2max are zero
    int m2lo;       // modes with |n|^2 >= m2lo take the exact float32 cut test
    int bm;         // largest |b| with b^2 <= m2max (capped at D/2)
    int cmax;       // largest c with c^2 <= m2max (capped at D/2)
    int exact_cut;  // 1 when the k-space cut applies
    float dk, R;    // for the exact test
    float gcoef;    // Gaussian factor exp2(m2 * gcoef); 0 for none
    float scale;    // 1/N times the growth factor of nonlinear input
};

// Density-space form of the centre-pixel threshold: f = erfcf((deltac -
// d)/denom) * scale >= 1/zeta holds exactly when d >= dstar, up to the float32
// rounding of the left side; cells within `band` of dstar take the exact
// float32 test, the others are decided by comparing d with dstar.
struct DensityThreshold {
    float dstar;  // decided by d > dstar outside the band
    float band;   // +inf: every cell takes the exact test
};

// Box-mean scale of nonlinear input and the threshold it implies, written
// once per radius by the reduction of the box sum.
struct ScaledThreshold {
    float scale;
    DensityThreshold th;
    int neutral;  // no cell of the box can be ionized at this radius (scale and th are then not set)
};

// Radii that keep at least this many modes a line get no bound: the sum of so
// many moduli stays far above any threshold (simulated on Gaussian and
// lognormal boxes, half and a fifth ionized: the last radius that it rules out
// keeps 9 to 23).
constexpr int kBoundModes = 32;

// What box_stays_neutral decides from.
struct SkipArgs {
    const float* bound;  // [D][4] bounds of the rows pass, or NULL: not decided (no)
    const float2* S0;    // the spectrum's k = 0 mode
    int groups;          // column groups that the bounds have
    int linear;
    float deltac, zeta_fc_mean;  // nonlinear input
    DensityThreshold th;  // linear input
};

// The threshold for linear input (scale 1), computed on the host.
DensityThreshold density_threshold_host(float deltac, float denom, double zeta, float scale);

struct LineEpilogue {
    float deltac, denom;
    double zeta, inv_zeta;
    unsigned long long* mask;  // ionization state, one bit per cell
    float* out;                // final float box
    double* partial;           // per-block FP64 partial sums
    float* bmax;               // per-block maximum of the smoothed field: written by
                               // the box-sum pass, read by the threshold pass to skip
                               // blocks no cell of which can reach the threshold; or NULL
    DensityThreshold th;       // threshold when `scaled` is NULL (linear input)
    const ScaledThreshold* scaled;  // nonlinear input: scale and threshold of the radius
};

// Arguments of the box-sum reduction of one radius: the FP64 total, and for
// nonlinear input the box-mean scale float32(fc_mean / (sum / ncells)), its
// density threshold and the list of line groups whose maximum can reach it.
struct SumScaleArgs {
    ScaledThreshold* scaled;
    float fc_mean, deltac, denom;
    double ncells, zeta;
    const float* bmax;
    int* active;
    int* nactive;
};

// The roles of one launch of the pipelined radius loop (k_fused_radius) and
// their block counts; a count of 0 is a role the launch does not have.  Only
// what the roles read: kernel arguments are fetched anew for every launch, and
// 130 bytes more of them (those of AskRoles) made the 33 launches of a linear
// 256^3 box 0.5 us longer each.
struct RadiusRoles {
    int n_red;               // box-sum reduction: 0 or 1 block
    int n_thr;               // threshold blocks (one line group each)
    int n_cols, n_mem;       // columns blocks; columns + rows blocks
    int n_sum;               // box-sum blocks (one line group each)
    int ncg_cols, ncg_rows;  // column groups of the columns and rows roles
    float deltac;
    double zeta;
    const float2* S;         // columns: pristine spectrum -> Tcols
    float2* Tcols;
    FusedParams fp_cols;
    int m2max_rows, cmax_rows;
    float2* Trows;           // rows: in place
    const double* partial;   // reduction: one partial per line group -> total
    double* total;
    ScaledThreshold* scaled_red;
    float fc_mean, denom_red;
    const float* bmax_red;
    int* active_red;         // or NULL (the last radius has no list)
    int* nactive_red;
    const float2* Uthr;      // threshold pass
    int cmax_thr;
    float denom_thr;
    DensityThreshold th;     // linear input
    unsigned long long* mask;
    const ScaledThreshold* scaled_thr;  // nonlinear input
    const float* bmax_thr;
    const int* active_thr;
    const int* nactive_thr;
    const float2* Usum;      // box-sum pass
    int cmax_sum;
    float denom_sum;
    double* partial_sum;
    float* bmax_sum;
};

// What a launch of the first radii has beside its roles.
struct AskRoles {
    int any;
    int n_ver;               // verdict: 0 or 1 block, whether the box stays neutral at a radius
    SkipArgs skip;
    float skip_scale, skip_denom;
    ScaledThreshold* verdict;
    float* bound_rows;                 // rows: bounds of the radius, or NULL
    const ScaledThreshold* state_thr;  // verdicts of the threshold blocks' (linear input), of
    const ScaledThreshold* state_sum;  // the box sums' and of the reduction's radius, or NULL
    const ScaledThreshold* state_red;
};

// The all-radii form of the loop: every role of every radius in one launch
// each (columns, rows, box sums, reductions, thresholds, paint) instead of one
// launch per radius.  One entry per radius; up to kAllRadii of them travel as
// kernel arguments.
constexpr int kAllRadii = 48;  // (at most 64: the paint reads a group's flags with one ballot)
struct AllRadius {
    FusedParams fp;
    int ho;                   // row stride of the radius' intermediate (padded to 16 modes)
    unsigned long long toff;  // its offset (float2) in the intermediates
    float denom;
    int ncg;                  // column groups of its columns and rows blocks
};
struct AllRadii {
    AllRadius r[kAllRadii];
    int cblk[kAllRadii + 1];  // first columns / rows block of each radius
    int rblk[kAllRadii + 1];
    int nr, nblk;             // radii; line groups of the box
    int linear;
    float deltac, fc_mean;
    double zeta, ncells;
    float2* S;                   // spectrum, b-major
    float2* T;                   // intermediates of every radius
    double* partial;             // [nr][nblk] box-sum partials (nonlinear input)
    float* bmax;                 // [nr][nblk] line group maxima
    double* sums;                // [nr]
    float* bound;                // [nr][D][4] bounds of the rows pass
    ScaledThreshold* scaled;     // [nr] box-mean scale (1 for linear input) and density threshold
    unsigned* hits;              // [nr][nblk] whether a line group has a hit at a radius ...
    unsigned long long* planes;  // [nr][N/64] ... and then its hit bits
    float* out;
};

// Lines of a box-sum partial: those of a line group, but eight at side 512, where
// a group has 16 (the float32 sums of a thread cover the cells of eight lines).
__host__ __device__ constexpr int sum_lines(int D, int L) { return D == 512 && L > 8 ? 8 : L; }

struct FusedShape {
    int D;
    int (*all)(const AllRadii&, const float2* tw, hipStream_t);
    int (*lines)(const float2* U, const float2* tw, int cmax, const LineEpilogue&, hipStream_t);
    int (*radius)(const RadiusRoles&, const AskRoles&, const float2* tw, hipStream_t);
    int (*forward)(const float* delta, float2* T0, float2* S, const float2* tw, const FusedParams& fp, hipStream_t);
    int (*inverse)(const float2* S, float2* T, float* out, const float2* tw, hipStream_t);
    int W, L;  // columns per column group, lines per line group
};

// Fills the radius table of the all-radii form (T offsets, blocks) and returns
// the intermediates' size in float2, or 0 when it does not apply: more than
// kAllRadii radii, or a side beyond 160, whose intermediates outgrow the caches
// while one launch per radius already fills the chip.
size_t all_radii_table(const FusedShape& sh, float dk, const float* radii, const float* denoms, int n_radii,
                       int filter_type, int ref_fallthrough, float scale, AllRadii* a);
int fused_all_radii(const FusedShape& sh, const AllRadii& a, const float2* tw, hipStream_t st);

const FusedShape* fused_shape(int D);
size_t fused_partials(int D);
FusedParams fused_params(int D, float dk, float R, int filter_type, int ref_fallthrough, float scale);
LineEpilogue line_epilogue(float deltac, float denom, double zeta, unsigned long long* mask, float* out);
// Column groups and surviving b rows of the columns role at one radius
// (the rows role uses the same column groups over all D rows p).
void column_groups(const FusedShape& sh, const FusedParams& fp, int* ncg, int* nb);
// Leading radii at which asking for a verdict (box_stays_neutral) can pay.
int neutral_radii(const cm21_bubble_params& prm, const float* denoms, int n_radii, const int* cmax);
int fused_radius_launch(const FusedShape& sh, const RadiusRoles& a, const AskRoles& q, const float2* tw,
                        hipStream_t st);
// The r2c of delta into the half spectrum S for the fused loop, stored
// b-major (S[b][a][c]), formed only for the modes the widest window fp keeps
// (|n|^2 <= fp.m2max), through the intermediate T0 (rows padded to 16
// modes).  S entries outside that sphere are left untouched: no radius reads
// them.
int fused_forward(const FusedShape& sh, const float* delta, float2* T0, float2* S, const float2* tw,
                  const FusedParams& fp, hipStream_t st);
// The final paint of the last radius from its intermediate U.
int fused_lines(const FusedShape& sh, const float2* U, const float2* tw, const FusedParams& fp,
                const LineEpilogue& ep, hipStream_t st, int stage = CM21_STAGE_FUSED_LINES);
int fused_mask_clear(unsigned long long* mask, size_t words, hipStream_t st);

}  // namespace cm21
