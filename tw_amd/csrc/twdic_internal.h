// twdic_internal.h -- shared declarations of the HIP implementation of the
// paDIC hot path (context, kernel parameter blocks, launch wrappers).
#pragma once

#include <hip/hip_runtime.h>

#include <atomic>
#include <cstddef>
#include <cstdint>
#include <string>

#include "twdic.h"

namespace twdic {

constexpr int kWave = 64;             // CDNA wavefront width
constexpr int kMaxFftN = 64;          // largest FFT-CC window edge held in LDS
constexpr int kRefStateStride = 48;   // doubles of per-reference state per POI (384 B)

// Per-reference, per-POI state (doubles, kRefStateStride per POI):
//   [0..20]  FP64 Cholesky factor L of the 6x6 Hessian, packed lower, row-major
//   [21..26] A_k = sum SD_k               (steepest-descent sums)
//   [27..32] B_k = sum SD_k (R - mean R)  (BR_k - mean R A_k with BR_k = sum SD_k R, one FMA)
//   [33]     |R - mean R|_2               (R_s)
//   [34]     reference flag: 0 ok, TWDIC_ICGN_DARK_SUBSET, TWDIC_ICGN_SINGULAR_HESSIAN,
//            TWDIC_ICGN_OUT_OF_ROI (subset leaves the ROI)
//   [35]     mean R
//   [36..41] 1 / L_ii (reciprocal pivots of the factor)
enum { RS_L = 0, RS_A = 21, RS_B = 27, RS_NORM = 33, RS_FLAG = 34, RS_MEAN = 35, RS_RDIAG = 36 };
constexpr int kRefStateUsed = 42;     // the doubles above that the iteration kernels read

// IC-GN runs one POI per group of L lanes of a wavefront, 256 / L POIs per
// 256-thread workgroup: L = 32 (a half-wavefront) for sets of at least
// kIcgnHalfWaveMin POIs, where the two POIs of a wavefront share the per-pass
// work between the pixel loops; L = 64 for smaller sets, which leave the GPU
// partly idle and run faster with half the pixel rounds per pass.  The
// choice follows the whole set's POI count (also for a chunk of it, and per
// pair in a batch), so a POI's result does not depend on the path that ran it.
constexpr int kIcgnHalfWaveMin = 32768;
inline int icgn_lanes_for(int n) { return n >= kIcgnHalfWaveMin ? 32 : 64; }

// The reference state: two POIs per wavefront from 4,096 POIs on (its own
// crossover: the sums are exact integers, so the width need not follow the
// iterations'), smaller sets one per wavefront, half the rounds for a GPU left
// partly idle.  A lane sums at most kRefRows rows at a time in 32 bits.
__host__ __device__ inline int ref_lanes_for(int n) { return n >= 4096 ? 32 : 64; }
constexpr int kRefRows = 56;

// How the L lanes of a POI's group walk its subset: strips of `ncol` columns
// from column `col`, each column cut into `segs` row ranges of equal length
// (the first ones a row longer where they do not divide), one lane per column
// and range, ncol segs <= L.
struct Strip {
    int16_t col, ncol, segs;
};
template <int MAX>
struct StripPlan {
    static constexpr int kMax = MAX;
    int count;
    Strip s[MAX];
};
typedef StripPlan<6> IcgnPlan;        // ranges of any length: at most ceil(121 / 32) strips are needed
typedef StripPlan<13> RefPlan;        // ranges of at most kRefRows rows: ceil(121 / 10)

// The strips of a W x H subset (1 <= W, H <= 121; L = 32 or 64) with the
// fewest rounds, a strip costing one round besides its longest row range, and
// no row range longer than max_rows.
template <class Plan>
inline Plan strip_plan(int W, int H, int L, int max_rows)
{
    constexpr int kMaxW = 128;
    int rounds[kMaxW], cost[kMaxW], take[kMaxW];
    auto segs = [&](int c) { return L / c < H ? L / c : H; };
    int widest = 0;
    for (int c = 1; c <= L && c <= W; ++c) {
        rounds[c] = (H + segs(c) - 1) / segs(c);
        if (rounds[c] <= max_rows) widest = c;
    }
    cost[0] = 0;
    for (int w = 1; w <= W; ++w) {
        cost[w] = 1 << 30;
        for (int c = w < widest ? w : widest; c >= 1; --c) {
            const int v = cost[w - c] + rounds[c] + 1;
            if (v < cost[w]) {
                cost[w] = v;
                take[w] = c;
            }
        }
    }
    Plan p{};
    int col = 0, w = W;
    for (; w > 0 && p.count < Plan::kMax; w -= take[w]) {
        p.s[p.count++] = {(int16_t)col, (int16_t)take[w], (int16_t)segs(take[w])};
        col += take[w];
    }
    if (w > 0) {                       // more strips than the table holds: the widest ones instead
        p.count = 0;
        for (col = 0; col < W; col += widest) {
            const int c = W - col < widest ? W - col : widest;
            p.s[p.count++] = {(int16_t)col, (int16_t)c, (int16_t)segs(c)};
        }
    }
    return p;
}

// The walks of one subset size, by the lanes per POI (32, 64).
struct SubsetWalks {
    IcgnPlan icgn[2];
    RefPlan ref[2];
};

inline SubsetWalks subset_walks(int W, int H)
{
    return {{strip_plan<IcgnPlan>(W, H, 32, H), strip_plan<IcgnPlan>(W, H, 64, H)},
            {strip_plan<RefPlan>(W, H, 32, kRefRows), strip_plan<RefPlan>(W, H, 64, kRefRows)}};
}

// Mean and L2 spread of n samples from their exact-or-FP64 sums s1 = sum x,
// s2 = sum x^2.  Shared by the reference-state and iteration kernels so that
// identical subsets give bit-identical statistics.
__device__ __forceinline__ void mean_spread(double s1, double s2, double n, double& mean, double& spread)
{
    mean = s1 / n;
    double var = __fma_rn(-s1, mean, s2);
    spread = sqrt(var > 0.0 ? var : 0.0);
}

// sum SD_k (x - mean) from sum SD_k x and sum SD_k.
__device__ __forceinline__ double centred(double sdx, double mean, double a)
{
    return __fma_rn(-mean, a, sdx);
}

// LDS written by lanes of a wavefront and then read by other lanes of it: its
// LDS accesses complete in issue order; keep the compiler from moving them
// across this point.
__device__ __forceinline__ void wave_lds_sync()
{
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
    __builtin_amdgcn_wave_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
}

struct FftccParams {
    const uint8_t* ref;
    const uint8_t* tar;
    int stride;
    int img_w, img_h;
    const int32_t* poi;
    int n;
    int N;
    const float2* tw;     // N twiddles exp(-2 pi i e / N)
    float tol;            // near-tie tolerance in ZNCC units
    float* u;
    float* v;
    float* zncc;
    uint8_t* status;
};

struct IcgnParams {
    const uint8_t* ref;
    const uint8_t* tar;
    int stride;
    int sx0, sy0, rw, rh;     // ROI
    int Sx, Sy, Wsub, Hsub, s;
    int max_iter;
    int lanes;                // lanes per POI: 32 or 64 (icgn_lanes_for of the set's POI count)
    IcgnPlan strips;          // how those lanes walk the subset
    double delta_p;           // the caller's float, widened: the loop test compares in FP64
    const uint32_t* g2;       // reference gradients (2Rx, 2Ry) as int16 pairs, ROI-relative
    const float* lut;         // target LUT [rh][rw][16]
    const float4* rp;         // target row polynomials [rh + 1][rw] (fused, LUT modes) or B-spline planes
                              // [4][rh][rw]; null: from the image bytes or the LUT
    double* refstate;         // kRefStateStride doubles per POI
    const int32_t* poi;
    int n;
    float* u;
    float* v;
    float* p6;
    int32_t* iters;
    uint8_t* flags;
    float* dpnorm;
};

// One image pair of a batch: the same parameter blocks the single-context
// kernels take, so the persistent kernels reuse the per-POI device code.
struct PairDesc {
    IcgnParams icgn;
    FftccParams fftcc;
    RefPlan ref;              // how ref_lanes_for lanes walk the subset
};

// The lanes per POI of a set of n POIs, and their walks of its subset.
inline void set_icgn_layout(IcgnParams& p, int n, const SubsetWalks& w)
{
    p.lanes = icgn_lanes_for(n);
    p.strips = w.icgn[p.lanes == 64];
}
inline const RefPlan& ref_plan(int n, const SubsetWalks& w) { return w.ref[ref_lanes_for(n) == 64]; }

// A lane's share of a strip (StripPlan): the exact float offsets of its first
// pixel from the POI, that pixel's byte offset in the gradient plane from the
// subset's corner, and, a byte each, its row count (0: the lane has no share),
// the rows that every share of the strip has at least, and the strip's row
// shares per column.  Every POI of a launch has the same subset and ROI width,
// so one table in LDS serves a workgroup.
//
// The shares of a column are ranges of rows where the lane keeps a cell's rows
// (row polynomials), which needs consecutive ones; otherwise the rows are dealt out in
// turn, so that a wavefront reads neighbouring rows of the LUT or the image.
struct StripLane {
    float dx, dy;
    uint32_t go;
    uint32_t rows;
};

template <int L, class Plan>
__device__ __forceinline__ void fill_strips(StripLane* tab, const Plan& plan, const IcgnParams& P, bool ranges,
                                            int t0, int tstride)
{
    // constant strip indices: a run-time index would move the plan to scratch
#pragma unroll
    for (int k = 0; k < Plan::kMax; ++k) {
        if (k >= plan.count) break;
        const Strip s = plan.s[k];
        const int base = P.Hsub / s.segs, rem = P.Hsub - base * s.segs;
        for (int l = t0; l < L; l += tstride) {
            const int seg = l / s.ncol, m = s.col + l - seg * s.ncol;
            const int y = ranges ? seg * base + min(seg, rem) : seg;
            const int rows = seg < s.segs ? base + (seg < rem ? 1 : 0) : 0;
            tab[k * L + l] = {(float)(m - P.Sx), (float)(y - P.Sy), 4u * (uint32_t)(y * P.rw + m),
                              (uint32_t)(rows | (base << 8) | (s.segs << 16))};
        }
    }
}

// Descriptors are never written while a batch kernel runs: reading them
// through the constant address space lets the compiler use scalar loads and
// keep each wave's descriptor in SGPRs.
#if defined(__HIP_DEVICE_COMPILE__)
#define TW_CONST_AS __attribute__((address_space(4)))
#else
#define TW_CONST_AS
#endif
typedef const TW_CONST_AS PairDesc* ConstPairDescPtr;
__device__ __forceinline__ ConstPairDescPtr const_pairs(const PairDesc* p)
{
    return (ConstPairDescPtr)p;
}

// The bytes that IC-GN's target loads may reach, from the pixel (-1, -1) on: the
// rows of the ROI and what its last cells' neighbourhoods add, at most the
// image's 2^31 bytes and three rows of 65,535 more, which an int need not hold.
__host__ __device__ inline uint32_t target_records(int sy0, int rh, int stride)
{
    return (uint32_t)(sy0 + rh + 3) * (uint32_t)stride;
}

// A byte offset past every such range, also with a row of a scalar offset added:
// a load there returns zero.
constexpr uint32_t kNoOffset = 0xC0000000u;

// Kernel launch wrappers (return hipError_t of the launch).
// `bytes` (at most kDownBytes) from device memory to the pinned buffer `out`,
// then seq into *flag.
constexpr size_t kDownBytes = 16384;
hipError_t launch_to_host(const void* src, void* out, size_t bytes, uint32_t* flag, uint32_t seq, hipStream_t st);
hipError_t launch_gradients(const uint8_t* img, int stride, int sx0, int sy0, int rw, int rh,
                            float* gx, float* gy, float* gxy, uint32_t* g2, hipStream_t st);
hipError_t launch_bspline_lut(const uint8_t* tar, int stride, int sx0, int sy0, int rw, int rh, float* lut,
                              hipStream_t st);
// the LUT as its own kernels write it, from the row polynomials, or from the
// B-spline planes, bit for bit; nothing once *done is set, which it then is
hipError_t launch_lut_of_rows(const float4* rp, int rw, int rh, float* lut, int* done, hipStream_t st);
hipError_t launch_lut_of_planes(const float4* planes, int rw, int rh, float* lut, int* done, hipStream_t st);
// the same coefficients as planes, float4[4][rh][rw]
hipError_t launch_bspline_planes(const uint8_t* tar, int stride, int sx0, int sy0, int rw, int rh, float4* planes,
                                 hipStream_t st);
// Catmull-Rom row polynomials of the target, (rh + 1) x rw entries of 16 bytes
hipError_t launch_row_poly(const uint8_t* tar, int stride, int sx0, int sy0, int rw, int rh, float4* rp,
                           hipStream_t st);
// the same for every pair of a batch with a plane (descriptor icgn.rp set);
// max_rh: the largest ROI height among them
hipError_t launch_batch_row_poly(const PairDesc* pairs, int npairs, int max_rh, hipStream_t st);
hipError_t launch_bicubic_lut(const uint8_t* tar, int stride, int sx0, int sy0, int rw, int rh,
                              float* lut, hipStream_t st);
hipError_t launch_poi_grid(int32_t* poi, int start_x, int start_y, int nx, int ny, int mx, int my,
                           int sx, int sy, int gx, int gy, hipStream_t st);
// variant kFftccMma: exact integer correlation on the matrix cores (any even
// N <= 64); 2, 3, 4: the FFT register engine's occupancy target (N = 32, 64,
// else the direct-DFT engine)
constexpr int kFftccMma = 8;
// kFftccDftMfma: N = 64 and most sets with 32 < N <= 60 on fp16 matrix-core DFTs
// with exact re-evaluation of the near-maximal shifts (the others: the integer
// engine); needs dft_tables_init on the device first
constexpr int kFftccDftMfma = 9;
hipError_t dft_tables_init(int device);
hipError_t launch_fftcc(const FftccParams& p, int variant, hipStream_t st);
// The POI sets the matrix-core DFT engine takes in place of the integer one (both
// give the same results): N = 64,
// the even 48 < N <= 60, and 32 < N <= 48 from the count on at which it is the
// faster one: it starts with its tables, 3 us more than the integer engine for
// one POI.  (N = 62 leaves the spectrum no free row, fftcc_dft_mfma_poi.)
// Against the integer engine, 2048^2 speckle, ms:
//   N       34         40         48         50         56         60
//   25      .013/.011  .014/.012  .015/.013  .015/.016  .015/.017  .015/.018
//   800     .016/.012  .016/.013  .016/.015  .016/.018  .016/.020  .016/.021
//   1,200   .016/.014  .016/.016  .016/.019  .016/.024  .017/.026  .016/.027
//   5,000   .025/.034  .023/.038  .025/.044  .03 /.065  .031/.072  .03 /.076
//   155k    .47 /.69   .48 /.82   .51 /1.00  .69 /1.61  .71 /1.86  .72 /1.96
inline bool dft_takes(int N, int n)
{
    return N == 64 || (N > 48 && N <= 60) || (N > 32 && N <= 48 && n >= 1280);
}

// In a flat batch the window edges of one integer kernel (mma_form) share its
// launch, while the DFT engine needs a launch per edge, 14 us before its first
// POIs are through.  Beside other edges it is therefore taken from higher counts
// on.  Batches of one pair per edge with their IC-GN, us, launches of their own /
// one together:
//   POIs per pair   900       1,296     1,764     3,721     7,056
//   50 .. 60        194/173   219/224   231/272   372/483   600/859
//   34 .. 48                            298/257   433/447   707/783
inline bool dft_takes_beside(int N, int n) { return dft_takes(N, n) && (N == 64 || n >= (N > 48 ? 1200 : 3200)); }
// the integer kernel of a window edge, by the largest edge it serves
inline int mma_form(int N) { return N <= 32 ? 32 : N <= 48 ? 48 : 64; }

// batched form: the matrix-core kernels over items (pair, POI): of pairs that
// share the window edge N, by the DFT engine (dft), or whose edges have the
// integer kernel of N
hipError_t launch_batch_fftcc_mma(const PairDesc* pairs, const int2* items, int count, int N, bool dft, hipStream_t st);
// batched form: IC-GN (fused interpolation) over workgroup items (pair, first
// POI), 256 / lanes POIs of one pair per workgroup, every listed pair with
// that many lanes per POI.
// The row-polynomial plane of an ROI is addressed with 32-bit byte offsets
// 16 (iy rw + ix) from entry -(sy0 rw + sx0); true when they all fit.
inline bool row_poly_fits(int sx0, int sy0, int rw, int rh)
{
    return 16ull * ((unsigned long long)(sy0 + rh + 2) * (unsigned long long)rw + (unsigned long long)sx0) <
           (1ull << 32);
}
inline size_t row_poly_bytes(int rw, int rh)
{
    return 16ull * (size_t)rw * (size_t)(rh + 1);
}
// waves: occupancy target 5 or 6; xcd_ranges: contiguous per-XCD item ranges;
// all_rp: every pair's descriptor has its row-polynomial plane
hipError_t launch_batch_icgn_wg(const PairDesc* pairs, const int2* wg, int count, int lanes, int waves,
                                bool xcd_ranges, bool all_rp, hipStream_t st);
hipError_t launch_ref_state(const IcgnParams& p, const RefPlan& plan, hipStream_t st);
hipError_t launch_icgn(const IcgnParams& p, int interp, int variant, hipStream_t st);
// persistent batch kernels: `blocks` workgroups drain a device work counter
hipError_t launch_batch_icgn(const PairDesc* pairs, const int2* items, int total, int* counter, int chunk,
                             int blocks, hipStream_t st);
hipError_t launch_batch_ref_state(const PairDesc* pairs, const int2* items, int total, int* counter, int blocks,
                                  hipStream_t st);
hipError_t launch_batch_fftcc(const PairDesc* pairs, const int2* items, int total, int* counter, int N,
                              int variant, int blocks, hipStream_t st);
hipError_t launch_fill_zero(int* p, int n, hipStream_t st);
hipError_t launch_strain_ls(const float* f, int nx, int ny, int grid, int M, double* dfdx, double* dfdy,
                            hipStream_t st);
// POI tracking across reference resets
hipError_t launch_track_update_poi(int32_t* poi, int n, const float* u, const float* v, hipStream_t st);
hipError_t launch_track_current_poi(const int32_t* poi, int n, const float* u, const float* v, int32_t* out,
                                    hipStream_t st);
hipError_t launch_track_current_poi_acc(const int32_t* poi, int n, const float* u, const float* v, const float* acc_u,
                                        const float* acc_v, int32_t* out, hipStream_t st);
hipError_t launch_track_accumulate_uv(int n, const float* u, const float* v, float* acc_u, float* acc_v,
                                      hipStream_t st);
// occupancy-derived persistent grid sizes
int persistent_blocks_icgn(int device);
int persistent_blocks_state(int device);
int persistent_blocks_fftcc(int device, int N, int variant);

}  // namespace twdic

struct twdic_ctx {
    twdic_config cfg{};
    int device = 0;
    hipStream_t stream = nullptr;
    int nx = 0, ny = 0;
    twdic::SubsetWalks walks{};       // of the configured subset
    int dstride = 0;                  // device image row stride (bytes)
    uint8_t* d_ref = nullptr;
    uint8_t* d_tar = nullptr;
    float* d_rx = nullptr;
    float* d_ry = nullptr;
    float* d_tx = nullptr;
    float* d_ty = nullptr;
    float* d_txy = nullptr;
    float* d_lut = nullptr;
    float4* d_rp = nullptr;           // target row polynomials or B-spline planes (null: not kept)
    uint32_t* d_g2 = nullptr;         // packed (2Rx, 2Ry) int16 pairs
    float2* d_fft_tw = nullptr;
    bool ref_loaded = false, tar_loaded = false;
    bool ref_grads_valid = false;     // Rx/Ry match d_ref
    bool tar_pre_valid = false;       // Tx/Ty/Txy/LUT match d_tar
    bool tar_rp_valid = false;        // d_rp matches d_tar
    bool rp_built = false;            // d_rp was built at some time
    bool tar_exposed = false;         // d_tar was handed out: it may change without twdic_set_target
    bool lut_exposed = false;         // the LUT modes keep d_lut up and read it: it was handed out, or the
                                      // caller captured a call into a graph of its own
    bool lut_behind = false;          // d_rp holds the table of a later build than d_lut's
    bool lut_pending = false;         // d_lut is still to be made from d_rp, unless *d_lut_done
    int* d_lut_done = nullptr;
    uint64_t ref_version = 0;
    // per-reference POI state cache key
    double* d_refstate = nullptr;
    size_t refstate_cap = 0;          // POIs
    uint64_t refstate_version = ~0ull;
    const int32_t* refstate_poi = nullptr;
    int refstate_n = -1;
    // FFT-CC engine (TWDIC_FFTCC_VARIANT): 9 fp16 matrix-core DFTs for N = 64 and
    // most sets with 32 < N <= 60 (else 8), 8 exact integer correlation on the matrix cores, 2-4 FFT registers
    int fftcc_variant = twdic::kFftccDftMfma;
    int icgn_variant = 5;             // occupancy target of the IC-GN kernel (0: compiler's choice)
    uint8_t* h_stage = nullptr;       // pinned staging for host images
    size_t h_stage_bytes = 0;
    // small downloads (twdic_memcpy): a pinned buffer, its device address, and
    // the sequence number that follows its kDownBytes bytes
    uint8_t* h_down = nullptr;
    uint8_t* d_down = nullptr;
    uint32_t down_seq = 0;
    std::atomic_flag down_busy = ATOMIC_FLAG_INIT;
    hipEvent_t ev[16] = {};
    // frame pipeline: FFT-CC of POI chunk i + 1 (on `stream`) overlaps IC-GN of
    // chunk i (on `stream2`)
    static constexpr int kMaxFrameChunks = 16;
    hipStream_t stream2 = nullptr;
    hipEvent_t pev[kMaxFrameChunks + 1] = {};
    int frame_chunks = 1;             // TWDIC_FRAME_CHUNKS; 1 runs the two stages back to back
    // captured frame step (twdic_frame_capture): its graph, the IC-GN
    // parameters it was recorded with, and the per-POI state buffer they name
    hipGraph_t graph = nullptr;
    hipGraphExec_t graph_exec = nullptr;
    twdic::IcgnParams graph_ip{};
    std::string err;
};
