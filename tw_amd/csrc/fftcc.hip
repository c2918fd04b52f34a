// fftcc.hip -- FFT-CC integer-pixel search for gfx950.
//
// Semantics follow Fftcc2D_CPU::ComputeFFTCC (TW_paDIC_FFTCC2D_CPU.cpp:
// 222-326) with the window edge N as a parameter (N = 2S is the reference):
//   window rows POIy - N/2 .. POIy + N/2 - 1, same for columns;
//   C[k] = sum_x R~(x) T~(x+k) (circular), peak = argmax C, lowest row-major
//   index on ties; u = k % N, v = k / N, wrapped by -N when > N/2;
//   ZNCC = C[peak] / sqrt(sum R~^2 sum T~^2).
//
// Exactness: the zero-mean correlation differs from the integer correlation
// I[k] = sum_x R(x) T(x+k) by a constant, so the true peak is an integer
// argmax, and every engine here returns that exact peak.  The reported ZNCC
// is evaluated in FP64 from the exact integer sums at the chosen peak, so
// every output is a function of the two windows alone: results do not depend
// on the engine, batching or pairing.
//
// Engines:
//   * k_fftcc_dft_mfma<CH, FULL> (default for N = 64 and most sets with 32 < N
//     <= 60, dft_takes): the surface from fp16 DFTs on the matrix cores, within
//     a proven error, then the exact integer correlation at the shifts it
//     leaves in question.
//   * k_fftcc_mma<NT, N64, TILE> (the other sets; any even N <= 64): the whole
//     integer correlation surface on the int8 matrix cores, one wavefront per
//     POI (32 x 32 x 32 tiles; 16 x 16 x 64 tiles for 32 < N <= 48).
//   * k_fftcc_fft<P> (N = 4P = 32 or 64): FP32 FFTs.  One workgroup of 4N
//     threads owns a POI pair.  Each window pair is packed into
//     Z = R^ + i T^ (R^, T^ zero-mean, unit norm), so one forward 2-D FFT
//     yields both spectra; the cross-power spectra X_A, X_B are Hermitian, so
//     a single inverse FFT of X_A + i X_B returns both correlation surfaces
//     (real and imaginary parts): 3 complex transforms per 2 POIs.  A 4N-point
//     line transform runs as a P-point radix-4 DFT in registers and a 4-point
//     DFT across a lane quad with DPP quad permutes; transposes go through
//     LDS.  When another shift lies within `tol` (ZNCC units) of the FP32
//     maximum, all such shifts are re-evaluated exactly in integers (lowest
//     index wins ties); with a single candidate the FP32 argmax is provably
//     the exact one.
//   * k_fftcc_dft: FP32 direct DFT along rows/columns for any other even
//     N <= 64, with the same exact re-evaluation.
#include "twdic_internal.h"

#include <algorithm>
#include <cfloat>
#include <climits>
#include <cmath>
#include <mutex>

namespace twdic {

namespace {

constexpr float kTwoPi = 6.283185307179586f;

struct Top2 {
    float best;
    int idx;
    float second;
};

__device__ __forceinline__ Top2 top2_merge(Top2 a, Top2 b)
{
    Top2 r;
    if (a.best > b.best || (a.best == b.best && a.idx < b.idx)) {
        r.best = a.best; r.idx = a.idx; r.second = fmaxf(a.second, b.best);
    } else {
        r.best = b.best; r.idx = b.idx; r.second = fmaxf(b.second, a.best);
    }
    return r;
}

__device__ __forceinline__ Top2 wave_top2(Top2 t)
{
#pragma unroll
    for (int o = 32; o > 0; o >>= 1) {
        Top2 u;
        u.best = __shfl_xor(t.best, o);
        u.idx = __shfl_xor(t.idx, o);
        u.second = __shfl_xor(t.second, o);
        t = top2_merge(t, u);
    }
    return t;
}

__device__ __forceinline__ int wave_sum_i(int v)
{
#pragma unroll
    for (int o = 32; o > 0; o >>= 1) v += __shfl_xor(v, o);
    return v;
}

__device__ __forceinline__ int wave_min_i(int v)
{
#pragma unroll
    for (int o = 32; o > 0; o >>= 1) v = min(v, __shfl_xor(v, o));
    return v;
}

__device__ __forceinline__ float2 cmul(float2 a, float2 b)
{
    return make_float2(a.x * b.x - a.y * b.y, a.x * b.y + a.y * b.x);
}

__device__ __forceinline__ float2 cadd(float2 a, float2 b) { return make_float2(a.x + b.x, a.y + b.y); }
__device__ __forceinline__ float2 csub(float2 a, float2 b) { return make_float2(a.x - b.x, a.y - b.y); }

// i*SGN*d
template <int SGN>
__device__ __forceinline__ float2 rot90(float2 d)
{
    return SGN > 0 ? make_float2(-d.y, d.x) : make_float2(d.y, -d.x);
}

// Add one value to a running top-2 whose indices arrive in increasing order
// (equal values keep the earlier, lower index).  Branch-free.
__device__ __forceinline__ void top2_push(Top2& t, float c, int idx)
{
    t.second = fmaxf(t.second, fminf(t.best, c));
    t.idx = c > t.best ? idx : t.idx;
    t.best = fmaxf(t.best, c);
}

// Wrap a row-major peak index to the reference's (u, v) (:316-322).
__device__ __forceinline__ void wrap_peak(int k, int N, int& u, int& v)
{
    u = k % N;
    v = k / N;
    if (u > N / 2) u -= N;
    if (v > N / 2) v -= N;
}

// ----------------------------------------------------------- register DFTs
// 4-point DFT, natural order, X[k] = sum a[n] exp(i SGN 2 pi n k / 4).
template <int SGN>
__device__ __forceinline__ void dft4(float2& a0, float2& a1, float2& a2, float2& a3)
{
    float2 t0 = cadd(a0, a2), t1 = csub(a0, a2), t2 = cadd(a1, a3), t3 = rot90<SGN>(csub(a1, a3));
    a0 = cadd(t0, t2);
    a2 = csub(t0, t2);
    a1 = cadd(t1, t3);
    a3 = csub(t1, t3);
}

template <int SGN>
__device__ __forceinline__ float2 twc(float2 a, int e, int n)   // a * exp(i SGN 2 pi e / n), e,n constant
{
    const float c = __builtin_cosf(kTwoPi * (float)e / (float)n);
    const float s = (float)SGN * __builtin_sinf(kTwoPi * (float)e / (float)n);
    return make_float2(a.x * c - a.y * s, a.x * s + a.y * c);
}

// P-point DFT in registers, natural order in and out (P = 16: 4 x 4; P = 8: 4 x 2).
template <int P, int SGN>
__device__ __forceinline__ void dft_reg(float2 (&x)[P])
{
    if constexpr (P == 16) {
#pragma unroll
        for (int n2 = 0; n2 < 4; ++n2) dft4<SGN>(x[n2], x[4 + n2], x[8 + n2], x[12 + n2]);
        // x[4*k1 + n2] now holds Y[n2][k1]; twiddle by W16^(n2 k1)
#pragma unroll
        for (int n2 = 1; n2 < 4; ++n2)
#pragma unroll
            for (int k1 = 1; k1 < 4; ++k1) x[4 * k1 + n2] = twc<SGN>(x[4 * k1 + n2], n2 * k1, 16);
        float2 y[16];
#pragma unroll
        for (int k1 = 0; k1 < 4; ++k1) {
            float2 a0 = x[4 * k1], a1 = x[4 * k1 + 1], a2 = x[4 * k1 + 2], a3 = x[4 * k1 + 3];
            dft4<SGN>(a0, a1, a2, a3);
            y[k1] = a0; y[k1 + 4] = a1; y[k1 + 8] = a2; y[k1 + 12] = a3;
        }
#pragma unroll
        for (int i = 0; i < 16; ++i) x[i] = y[i];
    } else {
        static_assert(P == 8, "P must be 8 or 16");
        // n = 2 n1 + n2: 4-point DFTs over n1 for n2 = 0, 1
        dft4<SGN>(x[0], x[2], x[4], x[6]);
        dft4<SGN>(x[1], x[3], x[5], x[7]);
        float2 y[8];
#pragma unroll
        for (int k1 = 0; k1 < 4; ++k1) {
            float2 a = x[2 * k1], b = twc<SGN>(x[2 * k1 + 1], k1, 8);
            y[k1] = cadd(a, b);
            y[k1 + 4] = csub(a, b);
        }
#pragma unroll
        for (int i = 0; i < 8; ++i) x[i] = y[i];
    }
}

// ------------------------------------------------- 4-point DFT across a quad
// DPP quad permutes: xor 1 = quad_perm [1,0,3,2] (0xB1), xor 2 = [2,3,0,1] (0x4E).
__device__ __forceinline__ float dpp_xor1(float v)
{
    return __int_as_float(__builtin_amdgcn_mov_dpp(__float_as_int(v), 0xB1, 0xF, 0xF, true));
}
__device__ __forceinline__ float dpp_xor2(float v)
{
    return __int_as_float(__builtin_amdgcn_mov_dpp(__float_as_int(v), 0x4E, 0xF, 0xF, true));
}

// DIT form: lane q holds index q; returns index brev2(q).
template <int SGN>
__device__ __forceinline__ float2 quad_dit(float2 v, int q)
{
    const float s2 = (q < 2) ? 1.f : -1.f, s1 = (q & 1) ? -1.f : 1.f;
    float2 a = make_float2(fmaf(s2, v.x, dpp_xor2(v.x)), fmaf(s2, v.y, dpp_xor2(v.y)));
    if (q == 3) a = rot90<SGN>(a);
    return make_float2(fmaf(s1, a.x, dpp_xor1(a.x)), fmaf(s1, a.y, dpp_xor1(a.y)));
}

// DIF form: lane q holds index brev2(q); returns index q.
template <int SGN>
__device__ __forceinline__ float2 quad_dif(float2 v, int q)
{
    const float s2 = (q < 2) ? 1.f : -1.f, s1 = (q & 1) ? -1.f : 1.f;
    float2 a = make_float2(fmaf(s1, v.x, dpp_xor1(v.x)), fmaf(s1, v.y, dpp_xor1(v.y)));
    if (q == 3) a = rot90<SGN>(a);
    return make_float2(fmaf(s2, a.x, dpp_xor2(a.x)), fmaf(s2, a.y, dpp_xor2(a.y)));
}

// 4P-point line transforms over a lane quad (tw: LDS table exp(-2 pi i e / 4P)).
//   dif: lane q holds x[j + P*brev2(q)]  ->  X[4k + q]
//   dit: lane q holds x[4j + q]          ->  X[k + P*brev2(q)]
template <int P, int SGN>
__device__ __forceinline__ void line_dif(float2 (&x)[P], int q, const float2* tw)
{
#pragma unroll
    for (int j = 0; j < P; ++j) x[j] = quad_dif<SGN>(x[j], q);
#pragma unroll
    for (int j = 1; j < P; ++j) {
        float2 w = tw[(q * j) & (4 * P - 1)];
        if (SGN > 0) w.y = -w.y;
        x[j] = cmul(x[j], w);
    }
    dft_reg<P, SGN>(x);
}

template <int P, int SGN>
__device__ __forceinline__ void line_dit(float2 (&x)[P], int q, const float2* tw)
{
    dft_reg<P, SGN>(x);
#pragma unroll
    for (int k = 1; k < P; ++k) {
        float2 w = tw[(q * k) & (4 * P - 1)];
        if (SGN > 0) w.y = -w.y;
        x[k] = cmul(x[k], w);
    }
#pragma unroll
    for (int k = 0; k < P; ++k) x[k] = quad_dit<SGN>(x[k], q);
}

}  // namespace

// ===========================================================================
// Fast engine: N = 4P in {32, 64}; 4N threads per workgroup, one POI pair.
// Thread t: line = t / 4 (row or column being transformed), q = t % 4.
// ===========================================================================
template <int P>
struct FftSmem {
    static constexpr int N = 4 * P;
    // complex plane, element (r, c) at r*(N+1) + c + r/P (row skew spreads
    // the four P-row blocks of a column read over distinct banks)
    float2 z[N * (N + 1) + 4];
    float2 tw[N];
    int red[N / 16][8];
    Top2 top[N / 16][2];
    int imin[N / 16];
};

template <int P>
__device__ __forceinline__ int zidx(int r, int c)
{
    return r * (4 * P + 1) + c + r / P;
}

// Exact integer correlation of the thread's R pixels with the LDS T window
// (bytes, row-major N x N) at shift (ku, kv), reduced over the workgroup.
template <int P>
__device__ __forceinline__ int exact_corr(const uint32_t (&rw)[P / 4], const uint8_t* tb, int line, int bq, int ku,
                                          int kv, FftSmem<P>& sm, int slot)
{
    constexpr int N = 4 * P;
    const int row = ((line + kv) & (N - 1)) * N;
    int acc = 0;
#pragma unroll
    for (int j = 0; j < P; ++j) {
        const int r = (rw[j >> 2] >> (8 * (j & 3))) & 255;
        acc += r * (int)tb[row + ((bq * P + j + ku) & (N - 1))];
    }
    acc = wave_sum_i(acc);
    const int wave = threadIdx.x >> 6, lane = threadIdx.x & 63;
    if (lane == 0) sm.red[wave][slot] = acc;
    __syncthreads();
    int s = 0;
#pragma unroll
    for (int w = 0; w < N / 16; ++w) s += sm.red[w][slot];
    __syncthreads();
    return s;
}

// One workgroup's work: the POIs (pa, ia) and (pb, ib); ib < 0 leaves the
// second slot empty.  Both descriptors must share the window edge N = 4P.
template <int P>
__device__ __forceinline__ void fftcc_pair(FftSmem<P>& sm, const FftccParams& pa, int ia, const FftccParams& pb,
                                           int ib)
{
    constexpr int N = 4 * P, NN = N * N, NW = N / 16;   // waves per workgroup
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    const int line = tid >> 2, q = tid & 3, bq = ((q & 1) << 1) | (q >> 1);
    const FftccParams* ps[2] = {&pa, &pb};
    const int idx[2] = {ia, ib};

    if (tid < N) sm.tw[tid] = pa.tw[tid];

    // -- 1. load both window pairs straight into registers (DIF layout: row
    //       `line`, columns bq*P .. bq*P+P-1), exact integer sums ---------------
    uint32_t rw[2][P / 4], tw8[2][P / 4];
    int valid[2], sums[2][4];
    int py[2], px[2];
#pragma unroll
    for (int s = 0; s < 2; ++s) {
        const FftccParams& p = *ps[s];
        const int poi = idx[s];
        valid[s] = 0;
        py[s] = px[s] = 0;
        if (poi >= 0) {
            py[s] = p.poi[2 * poi];
            px[s] = p.poi[2 * poi + 1];
            const int y0 = py[s] - N / 2, x0 = px[s] - N / 2;
            valid[s] = (y0 >= 0 && x0 >= 0 && y0 + N <= p.img_h && x0 + N <= p.img_w) ? 1 : 2;
        }
#pragma unroll
        for (int k = 0; k < P / 4; ++k) { rw[s][k] = 0u; tw8[s][k] = 0u; }
        if (valid[s] == 1) {
            const size_t o = (size_t)(py[s] - N / 2 + line) * p.stride + (px[s] - N / 2 + bq * P);
            __builtin_memcpy(rw[s], p.ref + o, P);
            __builtin_memcpy(tw8[s], p.tar + o, P);
        }
        int a = 0, b = 0, aa = 0, bb = 0;
#pragma unroll
        for (int k = 0; k < P; ++k) {
            const int r = (rw[s][k >> 2] >> (8 * (k & 3))) & 255, t = (tw8[s][k >> 2] >> (8 * (k & 3))) & 255;
            a += r; b += t; aa += r * r; bb += t * t;
        }
        sums[s][0] = wave_sum_i(a); sums[s][1] = wave_sum_i(b);
        sums[s][2] = wave_sum_i(aa); sums[s][3] = wave_sum_i(bb);
        if (lane == 0) {
#pragma unroll
            for (int k = 0; k < 4; ++k) sm.red[wave][4 * s + k] = sums[s][k];
        }
    }
    __syncthreads();
    double nr[2], nt[2];
    float mr[2], mt[2], gr[2], gt[2];
#pragma unroll
    for (int s = 0; s < 2; ++s) {
#pragma unroll
        for (int k = 0; k < 4; ++k) {
            int acc = 0;
#pragma unroll
            for (int w = 0; w < NW; ++w) acc += sm.red[w][4 * s + k];
            sums[s][k] = acc;
        }
        const long long sr = sums[s][0], st = sums[s][1], srr = sums[s][2], stt = sums[s][3];
        // flat window (TW_paDIC_FFTCC2D_CPU.cpp:271-275): exact integer test
        if (valid[s] == 1 && (srr * NN == sr * sr || stt * NN == st * st)) valid[s] = 3;
        nr[s] = (double)srr - (double)sr * (double)sr / (double)NN;
        nt[s] = (double)stt - (double)st * (double)st / (double)NN;
        mr[s] = (float)sr / (float)NN;          // (:253-254)
        mt[s] = (float)st / (float)NN;
        gr[s] = valid[s] == 1 ? (float)(1.0 / sqrt(nr[s])) : 0.f;
        gt[s] = valid[s] == 1 ? (float)(1.0 / sqrt(nt[s])) : 0.f;
    }
    __syncthreads();

    // -- 2. forward transforms and cross-power spectra ---------------------------
    float2 X[2][P];
#pragma unroll
    for (int s = 0; s < 2; ++s) {
        float2 x[P];
#pragma unroll
        for (int j = 0; j < P; ++j) {
            const int r = (rw[s][j >> 2] >> (8 * (j & 3))) & 255, t = (tw8[s][j >> 2] >> (8 * (j & 3))) & 255;
            x[j] = make_float2(((float)r - mr[s]) * gr[s], ((float)t - mt[s]) * gt[s]);
        }
        line_dif<P, -1>(x, q, sm.tw);                       // rows: lane holds kx = 4j + q
#pragma unroll
        for (int j = 0; j < P; ++j) sm.z[zidx<P>(line, 4 * j + q)] = x[j];
        __syncthreads();
#pragma unroll
        for (int j = 0; j < P; ++j) x[j] = sm.z[zidx<P>(bq * P + j, line)];
        __syncthreads();
        line_dif<P, -1>(x, q, sm.tw);                       // columns: lane holds ky = 4j + q, kx = line
#pragma unroll
        for (int j = 0; j < P; ++j) sm.z[zidx<P>(4 * j + q, line)] = x[j];
        __syncthreads();
        // conj(F_R) F_T = Im(Z[k] Z[-k]) / 2 - i (|Z[k]|^2 - |Z[-k]|^2) / 4
        const int mkx = (N - line) & (N - 1);
#pragma unroll
        for (int j = 0; j < P; ++j) {
            const int mky = (N - (4 * j + q)) & (N - 1);
            const float2 a = x[j], b = sm.z[zidx<P>(mky, mkx)];
            const float im_ab = a.x * b.y + a.y * b.x;
            const float d = (a.x * a.x + a.y * a.y) - (b.x * b.x + b.y * b.y);
            X[s][j] = make_float2(0.5f * im_ab, -0.25f * d);
        }
        __syncthreads();
    }

    // -- 3. one inverse transform for both: IFFT(X_A + i X_B) = c_A + i c_B -------
    float2 x[P];
#pragma unroll
    for (int j = 0; j < P; ++j) x[j] = make_float2(X[0][j].x - X[1][j].y, X[0][j].y + X[1][j].x);
    line_dit<P, 1>(x, q, sm.tw);                            // columns: lane holds y = j + P*bq
#pragma unroll
    for (int j = 0; j < P; ++j) sm.z[zidx<P>(j + P * bq, line)] = x[j];
    __syncthreads();
#pragma unroll
    for (int j = 0; j < P; ++j) x[j] = sm.z[zidx<P>(line, 4 * j + q)];
    __syncthreads();
    line_dit<P, 1>(x, q, sm.tw);                            // rows: lane holds x = j + P*bq of row `line`

    // -- 4. peaks: top-2 per POI with lowest-index tie-break (:300-311) ----------
    Top2 t[2];
#pragma unroll
    for (int s = 0; s < 2; ++s) {
        t[s] = Top2{-FLT_MAX, 0x7fffffff, -FLT_MAX};
#pragma unroll
        for (int j = 0; j < P; ++j) top2_push(t[s], s == 0 ? x[j].x : x[j].y, line * N + j + P * bq);
        t[s] = wave_top2(t[s]);
        if (lane == 0) sm.top[wave][s] = t[s];
    }
    // T windows to LDS (bytes, row-major) for the exact integer sums; the
    // complex plane is free once every thread holds its outputs.  The window
    // words are re-read (L2-resident) rather than kept live in registers.
    uint8_t* tb = reinterpret_cast<uint8_t*>(sm.z);
#pragma unroll
    for (int s = 0; s < 2; ++s) {
        if (valid[s] == 1) {
            const FftccParams& p = *ps[s];
            const size_t o = (size_t)(py[s] - N / 2 + line) * p.stride + (px[s] - N / 2 + bq * P);
            __builtin_memcpy(rw[s], p.ref + o, P);
            __builtin_memcpy(tw8[s], p.tar + o, P);
        }
#pragma unroll
        for (int k = 0; k < P / 4; ++k)
            reinterpret_cast<uint32_t*>(tb + s * NN + line * N + bq * P)[k] = tw8[s][k];
    }
    __syncthreads();
#pragma unroll
    for (int s = 0; s < 2; ++s) {
        Top2 r = sm.top[0][s];
#pragma unroll
        for (int w = 1; w < NW; ++w) r = top2_merge(r, sm.top[w][s]);
        t[s] = r;
    }

    // -- 5. exact peak and ZNCC from integers -------------------------------------
#pragma unroll
    for (int s = 0; s < 2; ++s) {
        if (valid[s] != 1) continue;                         // uniform per workgroup
        const float thr = t[s].best - pa.tol * (float)NN;
        int peak = t[s].idx, bestI = 0;
        if (t[s].second < thr) {
            bestI = exact_corr<P>(rw[s], tb + s * NN, line, bq, peak % N, peak / N, sm, 0);
        } else {
            // several shifts within tol of the maximum: evaluate them all exactly,
            // in increasing index order, keeping the first strict maximum
            bestI = -1;
            peak = -1;
            int last = -1;
            for (;;) {
                int cand = 0x7fffffff;
#pragma unroll
                for (int j = 0; j < P; ++j) {
                    const int idx = line * N + j + P * bq;
                    const float c = s == 0 ? x[j].x : x[j].y;
                    if (idx > last && c >= thr) cand = min(cand, idx);
                }
                cand = wave_min_i(cand);
                if (lane == 0) sm.imin[wave] = cand;
                __syncthreads();
                int m = sm.imin[0];
#pragma unroll
                for (int w = 1; w < NW; ++w) m = min(m, sm.imin[w]);
                __syncthreads();
                if (m == 0x7fffffff) break;
                const int I = exact_corr<P>(rw[s], tb + s * NN, line, bq, m % N, m / N, sm, 0);
                if (I > bestI) { bestI = I; peak = m; }
                last = m;
            }
        }
        if (tid == 0) {
            const FftccParams& p = *ps[s];
            int iu, iv;
            wrap_peak(peak, N, iu, iv);
            const double sr = sums[s][0], st = sums[s][1];
            p.u[idx[s]] = (float)iu;
            p.v[idx[s]] = (float)iv;
            p.zncc[idx[s]] = (float)(((double)bestI - sr * st / (double)NN) / sqrt(nr[s] * nt[s]));
        }
    }
    if (tid == 0) {
#pragma unroll
        for (int s = 0; s < 2; ++s)
            if (valid[s] && ps[s]->status)
                ps[s]->status[idx[s]] = valid[s] == 1 ? TWDIC_FFTCC_OK : valid[s] == 2 ? TWDIC_FFTCC_OUT
                                                                                       : TWDIC_FFTCC_FLAT;
    }
}

template <int P, int MINW>
__global__ __launch_bounds__(16 * P, MINW) void k_fftcc_fft(FftccParams p)
{
    __shared__ FftSmem<P> sm;
    const int ia = 2 * blockIdx.x, ib = ia + 1 < p.n ? ia + 1 : -1;
    fftcc_pair<P>(sm, p, ia, p, ib);
}

// Persistent form: each workgroup takes the next pair of (image pair, POI)
// items of one window class from a device counter until the list is
// exhausted.  Consecutive items may belong to different images.
template <int P, int MINW>
__global__ __launch_bounds__(16 * P, MINW) void k_batch_fftcc(const PairDesc* __restrict__ pairs,
                                                              const int2* __restrict__ items, int total, int* counter)
{
    __shared__ FftSmem<P> sm;
    __shared__ int next;
    for (;;) {
        if (threadIdx.x == 0) next = atomicAdd(counter, 1);
        __syncthreads();
        const int k = next;
        __syncthreads();
        if (2 * k >= total) break;
        const int2 a = items[2 * k];
        const int2 b = 2 * k + 1 < total ? items[2 * k + 1] : make_int2(a.x, -1);
        const FftccParams pa = const_pairs(pairs)[__builtin_amdgcn_readfirstlane(a.x)].fftcc;
        const FftccParams pb = const_pairs(pairs)[__builtin_amdgcn_readfirstlane(b.x)].fftcc;
        fftcc_pair<P>(sm, pa, __builtin_amdgcn_readfirstlane(a.y), pb, __builtin_amdgcn_readfirstlane(b.y));
    }
}

// ===========================================================================
// Direct-DFT engine: any even N <= 64, one POI per 256-thread workgroup.
// ===========================================================================
namespace {

constexpr int kDftThreads = 256;
constexpr int kPitch = kMaxFftN + 1;

struct DftSmem {
    float2 z[kMaxFftN * kPitch];
    uint8_t wr[kMaxFftN * kMaxFftN];
    uint8_t wt[kMaxFftN * kMaxFftN];
    float2 tw[kMaxFftN];
    int red[4][4];
    Top2 top[4];
    int imin[4];
};

// In-place DFT of every row (dir 0) or column (dir 1); each wavefront owns
// whole lines and lane k produces output k.  All LDS reads of a line complete
// before its writes within the wavefront.
__device__ void dft_lines(DftSmem& sm, int N, int dir, bool inverse)
{
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    for (int line = wave; line < N; line += 4) {
        float2 acc = make_float2(0.f, 0.f);
        if (lane < N) {
            int e = 0;
            for (int j = 0; j < N; ++j) {
                float2 z = dir == 0 ? sm.z[line * kPitch + j] : sm.z[j * kPitch + line];
                float2 w = sm.tw[e];
                if (inverse) w.y = -w.y;
                acc.x += z.x * w.x - z.y * w.y;
                acc.y += z.x * w.y + z.y * w.x;
                e += lane;
                if (e >= N) e -= N;   // lane < N: one subtraction suffices
            }
        }
        __builtin_amdgcn_wave_barrier();
        if (lane < N) {
            if (dir == 0) sm.z[line * kPitch + lane] = acc;
            else sm.z[lane * kPitch + line] = acc;
        }
    }
}

__device__ int block_sum_i(DftSmem& sm, int v)
{
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    v = wave_sum_i(v);
    __syncthreads();
    if (lane == 0) sm.red[wave][0] = v;
    __syncthreads();
    return sm.red[0][0] + sm.red[1][0] + sm.red[2][0] + sm.red[3][0];
}

__device__ int exact_corr_dft(DftSmem& sm, int N, int ku, int kv)
{
    int acc = 0;
    for (int i = threadIdx.x; i < N * N; i += kDftThreads) {
        int y = i / N, x = i - y * N;
        int yy = y + kv; if (yy >= N) yy -= N;
        int xx = x + ku; if (xx >= N) xx -= N;
        acc += (int)sm.wr[i] * (int)sm.wt[yy * N + xx];
    }
    return block_sum_i(sm, acc);
}

}  // namespace

__device__ void fftcc_dft_poi(DftSmem& sm, const FftccParams& p, int poi)
{
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    const int N = p.N, NN = N * N, half = N >> 1;
    const int py = p.poi[2 * poi], px = p.poi[2 * poi + 1];
    const int y0 = py - half, x0 = px - half;
    if (y0 < 0 || x0 < 0 || y0 + N > p.img_h || x0 + N > p.img_w) {
        if (tid == 0 && p.status) p.status[poi] = TWDIC_FFTCC_OUT;
        return;
    }
    int sr = 0, st = 0, srr = 0, stt = 0;
    for (int i = tid; i < NN; i += kDftThreads) {
        int y = i / N, x = i - y * N;
        size_t o = (size_t)(y0 + y) * p.stride + (x0 + x);
        int a = p.ref[o], b = p.tar[o];
        sm.wr[i] = (uint8_t)a;
        sm.wt[i] = (uint8_t)b;
        sr += a; st += b; srr += a * a; stt += b * b;
    }
    if (tid < N) sm.tw[tid] = p.tw[tid];
    sr = wave_sum_i(sr); st = wave_sum_i(st); srr = wave_sum_i(srr); stt = wave_sum_i(stt);
    if (lane == 0) { sm.red[wave][0] = sr; sm.red[wave][1] = st; sm.red[wave][2] = srr; sm.red[wave][3] = stt; }
    __syncthreads();
    const long long Sr = sm.red[0][0] + sm.red[1][0] + sm.red[2][0] + sm.red[3][0];
    const long long St = sm.red[0][1] + sm.red[1][1] + sm.red[2][1] + sm.red[3][1];
    const long long Srr = sm.red[0][2] + sm.red[1][2] + sm.red[2][2] + sm.red[3][2];
    const long long Stt = sm.red[0][3] + sm.red[1][3] + sm.red[2][3] + sm.red[3][3];
    if (Srr * NN == Sr * Sr || Stt * NN == St * St) {         // (:271-275)
        if (tid == 0 && p.status) p.status[poi] = TWDIC_FFTCC_FLAT;
        return;
    }
    const double nr = (double)Srr - (double)Sr * (double)Sr / (double)NN;
    const double nt = (double)Stt - (double)St * (double)St / (double)NN;
    const float mr = (float)Sr / (float)NN, mt = (float)St / (float)NN;
    const float gr = (float)(1.0 / sqrt(nr)), gt = (float)(1.0 / sqrt(nt));
    for (int i = tid; i < NN; i += kDftThreads) {
        int y = i / N, x = i - y * N;
        sm.z[y * kPitch + x] = make_float2(((float)sm.wr[i] - mr) * gr, ((float)sm.wt[i] - mt) * gt);
    }
    __syncthreads();
    dft_lines(sm, N, 0, false);
    __syncthreads();
    dft_lines(sm, N, 1, false);
    __syncthreads();
    for (int i = tid; i < NN; i += kDftThreads) {
        int ky = i / N, kx = i - ky * N;
        int my = ky ? N - ky : 0, mx = kx ? N - kx : 0;
        int j = my * N + mx;
        if (i <= j) {          // each Hermitian pair is formed by one thread
            float2 a = sm.z[ky * kPitch + kx], b = sm.z[my * kPitch + mx];
            float im_ab = a.x * b.y + a.y * b.x;
            float d = (a.x * a.x + a.y * a.y) - (b.x * b.x + b.y * b.y);
            float2 xk = make_float2(0.5f * im_ab, -0.25f * d);
            sm.z[ky * kPitch + kx] = xk;
            if (j != i) sm.z[my * kPitch + mx] = make_float2(xk.x, -xk.y);
        }
    }
    __syncthreads();
    dft_lines(sm, N, 1, true);
    __syncthreads();
    dft_lines(sm, N, 0, true);
    __syncthreads();

    Top2 t{-FLT_MAX, 0x7fffffff, -FLT_MAX};
    for (int i = tid; i < NN; i += kDftThreads) {
        int y = i / N, x = i - y * N;
        t = top2_merge(t, Top2{sm.z[y * kPitch + x].x, i, -FLT_MAX});
    }
    t = wave_top2(t);
    if (lane == 0) sm.top[wave] = t;
    __syncthreads();
    t = top2_merge(top2_merge(sm.top[0], sm.top[1]), top2_merge(sm.top[2], sm.top[3]));
    const float thr = t.best - p.tol * (float)NN;
    int peak = t.idx, bestI;
    if (t.second < thr) {
        bestI = exact_corr_dft(sm, N, peak % N, peak / N);
    } else {
        bestI = -1;
        peak = -1;
        int last = -1;
        for (;;) {
            int cand = 0x7fffffff;
            for (int i = tid; i < NN; i += kDftThreads) {
                int y = i / N, x = i - y * N;
                if (i > last && sm.z[y * kPitch + x].x >= thr) { cand = i; break; }
            }
            cand = wave_min_i(cand);
            __syncthreads();
            if (lane == 0) sm.imin[wave] = cand;
            __syncthreads();
            cand = min(min(sm.imin[0], sm.imin[1]), min(sm.imin[2], sm.imin[3]));
            if (cand == 0x7fffffff) break;
            const int I = exact_corr_dft(sm, N, cand % N, cand / N);
            if (I > bestI) { bestI = I; peak = cand; }
            last = cand;
        }
    }
    if (tid == 0) {
        int iu, iv;
        wrap_peak(peak, N, iu, iv);
        p.u[poi] = (float)iu;
        p.v[poi] = (float)iv;
        p.zncc[poi] = (float)(((double)bestI - (double)Sr * (double)St / (double)NN) / sqrt(nr * nt));
        if (p.status) p.status[poi] = TWDIC_FFTCC_OK;
    }
}

__global__ __launch_bounds__(kDftThreads) void k_fftcc_dft(FftccParams p)
{
    __shared__ DftSmem sm;
    if ((int)blockIdx.x >= p.n) return;
    fftcc_dft_poi(sm, p, blockIdx.x);
}

__global__ __launch_bounds__(kDftThreads) void k_batch_fftcc_dft(const PairDesc* __restrict__ pairs,
                                                                 const int2* __restrict__ items, int total,
                                                                 int* counter)
{
    __shared__ DftSmem sm;
    __shared__ int next;
    for (;;) {
        if (threadIdx.x == 0) next = atomicAdd(counter, 1);
        __syncthreads();
        const int k = next;
        __syncthreads();
        if (k >= total) break;
        const int2 it = items[k];
        const FftccParams p = const_pairs(pairs)[__builtin_amdgcn_readfirstlane(it.x)].fftcc;
        fftcc_dft_poi(sm, p, __builtin_amdgcn_readfirstlane(it.y));
        __syncthreads();
    }
}

// ===========================================================================
// Matrix-core engine: any even N <= 64, one wavefront per POI.
//
// The inverse transform of the cross-power spectrum (:285-297) is the
// circular cross-correlation C[kv][ku] = sum_{y,x} R[y][x] T[(y+kv)%N][(x+ku)%N],
// up to the zero-mean constant and rounding.  This engine computes it
// directly, exactly, in integers on the int8 matrix cores
// (v_mfma_i32_32x32x32_i8, or v_mfma_i32_16x16x64_i8 for 32 < N <= 48).
// Stored as signed bytes R' = R - 128 and
// T' = T - 128, C'[k] = C[k] - 128 (sum R + sum T) + 128^2 N^2 differs from
// C[k] by a constant, so the argmax (lowest row-major index on ties) is the
// exact integer peak, and |C'| <= 2^14 N^2 <= 2^26 fits int32.
//
// GEMM form, K = (y', x) over target rows y' and columns x:
//   C'[kv][ku] = sum_{y'} sum_x R'[(y' - kv) mod N][x] * T'[y'][(x + ku) mod N]
// A[kv][(y', x)] gathers reference rows (the row index turns with y');
// B[(y', x)][ku] is the circulant of target row y', read from a doubled copy
// of the row, T2[c] = T'[c mod N], at byte offset x + ku.  Outputs are
// NT x NT (NT = 32 for N <= 32, else 64) in 32 x 32 tiles, or 48 x 48 in
// 16 x 16 tiles; rows and columns of K or of the output beyond N are zero
// padding or ignored.
//
// Lane layout (one wavefront, lane l, m = l % 32, h = l / 32): an A operand
// holds row m, bytes 16h .. 16h+15 of a 32-byte K chunk; a B operand holds
// column m, the same 16 K bytes; accumulator register r of lane l is output
// (row 8 (r / 4) + 4 h + r % 4, column m) of the tile.
// ===========================================================================
namespace {

typedef int v4i __attribute__((ext_vector_type(4)));
typedef int v16i __attribute__((ext_vector_type(16)));

// Row strides are multiples of 16 bytes whose dword counts put 8 consecutive
// rows in distinct 4-bank groups, so the row-per-lane 16-byte stores and the
// reference-row reads are conflict-free.
template <int NT, bool N64>
struct MmaSmem {
    static constexpr int RS = NT == 64 ? 80 : 48;     // reference row stride
    static constexpr int TW = N64 ? 96 : 2 * NT;      // bytes of the doubled target row that are read
    static constexpr int TS = N64 ? 112 : NT == 64 ? 144 : 80;   // target row stride
    alignas(16) uint8_t r[NT * RS];
    alignas(16) uint8_t t[NT * TS];
};

// 32 < N <= 48 on 16 x 16 output tiles: 48 rows; the target row is read up
// to byte 111 (offset 16 g + 16 t' + n <= 95, plus 16 bytes)
struct MmaSmem16 {
    static constexpr int RS = 80;
    static constexpr int TW = 112;
    static constexpr int TS = 112;                    // 28 dwords: 8 consecutive rows in distinct bank groups
    alignas(16) uint8_t r[48 * RS];
    alignas(16) uint8_t t[48 * TS];
};

template <int NT, bool N64, int TILE>
struct MmaSel {
    using type = MmaSmem<NT, N64>;
};
template <>
struct MmaSel<64, false, 16> {
    using type = MmaSmem16;
};

// 16 bytes of a doubled target row starting at byte offset o (any alignment)
__device__ __forceinline__ v4i b_operand(const uint32_t* row, int d, int sh)
{
    const uint32_t w0 = row[d], w1 = row[d + 1], w2 = row[d + 2], w3 = row[d + 3], w4 = row[d + 4];
    v4i b;
    b.x = (int)__builtin_amdgcn_alignbyte(w1, w0, sh);
    b.y = (int)__builtin_amdgcn_alignbyte(w2, w1, sh);
    b.z = (int)__builtin_amdgcn_alignbyte(w3, w2, sh);
    b.w = (int)__builtin_amdgcn_alignbyte(w4, w3, sh);
    return b;
}

// The n bytes (2 <= n <= 4 WORDS) at src, any alignment, into w
// (bytes from n on are unspecified).  Only the 16-byte-aligned chunks that
// hold at least one of the n bytes are read; an aligned chunk never crosses a
// page, so nothing beyond the pages of the row itself is touched.  The
// misalignment sh (0..15) is taken out as whole dwords in two select steps,
// then as bytes with v_alignbyte.
template <int WORDS>
__device__ __forceinline__ void load_row(const uint8_t* src, int n, uint32_t (&w)[WORDS])
{
    constexpr int CH = WORDS / 4 + 1;                  // raw words 0 .. WORDS + 3 are used
    const uintptr_t a = reinterpret_cast<uintptr_t>(src);
    const uint4* c = reinterpret_cast<const uint4*>(a & ~(uintptr_t)15);
    const int sh = (int)(a & 15);
    uint32_t raw[4 * CH];
#pragma unroll
    for (int k = 0; k < CH; ++k) {
        uint4 v = make_uint4(0u, 0u, 0u, 0u);
        if (16 * k < sh + n) v = c[k];
        raw[4 * k] = v.x;
        raw[4 * k + 1] = v.y;
        raw[4 * k + 2] = v.z;
        raw[4 * k + 3] = v.w;
    }
    // bitwise selects on opaque masks (v_bfi_b32): a `q ? raw[i + 2] : raw[i]`
    // is folded into a dynamically indexed load, which moves raw to scratch
    uint32_t m2 = (sh & 8) ? ~0u : 0u, m1 = (sh & 4) ? ~0u : 0u;
    asm volatile("" : "+v"(m2), "+v"(m1));
    const int b = sh & 3;
    uint32_t s2[WORDS + 2], s1[WORDS + 1];
#pragma unroll
    for (int i = 0; i < WORDS + 2; ++i) s2[i] = (raw[i + 2] & m2) | (raw[i] & ~m2);
#pragma unroll
    for (int i = 0; i < WORDS + 1; ++i) s1[i] = (s2[i + 1] & m1) | (s2[i] & ~m1);
#pragma unroll
    for (int k = 0; k < WORDS; ++k) w[k] = __builtin_amdgcn_alignbyte(s1[k + 1], s1[k], b);
}

// N64: N == 64 (NT = 64); otherwise N <= NT is a run-time value.  TILE 32:
// v_mfma_i32_32x32x32_i8 on 32 x 32 tiles (N <= 32 in one tile, 32 < N <= 64
// in 2 x 2); TILE 16: v_mfma_i32_16x16x64_i8 on 3 x 3 tiles of 16 x 16 with
// the whole 64-byte row as one K chunk, for 32 < N <= 48, where it issues
// 9 16-cycle MFMAs per row instead of 8 32-cycle ones.
template <int NT, bool N64, int TILE>
__device__ __forceinline__ void fftcc_mma_poi(typename MmaSel<NT, N64, TILE>::type& sm, const FftccParams& p,
                                              int poi)
{
    constexpr int TT = NT / 32;          // output tiles per edge and K chunks per row (TILE 32)
    using Sm = typename MmaSel<NT, N64, TILE>::type;
    const int lane = threadIdx.x, m = lane & 31, h = lane >> 5;
    const int N = N64 ? 64 : p.N, NN = N * N;
    const int py = p.poi[2 * poi], px = p.poi[2 * poi + 1];
    if (py - N / 2 < 0 || px - N / 2 < 0 || py + N / 2 > p.img_h || px + N / 2 > p.img_w) {
        if (lane == 0 && p.status) p.status[poi] = TWDIC_FFTCC_OUT;
        return;
    }

    // -- window rows to LDS (lane = row), exact integer sums -------------------
    int sr = 0, st = 0, srr = 0, stt = 0;
    if (lane < N) {
        const size_t o = (size_t)(py - N / 2 + lane) * p.stride + (px - N / 2);
        uint8_t* rrow = sm.r + lane * Sm::RS;
        uint8_t* trow = sm.t + lane * Sm::TS;
        if (N == NT) {
            uint32_t r[NT / 4], t[NT / 4];
            __builtin_memcpy(r, p.ref + o, NT);
            __builtin_memcpy(t, p.tar + o, NT);
#pragma unroll
            for (int k = 0; k < NT / 4; ++k) {
                sr = (int)__builtin_amdgcn_udot4(r[k], 0x01010101u, (uint32_t)sr, false);
                st = (int)__builtin_amdgcn_udot4(t[k], 0x01010101u, (uint32_t)st, false);
                srr = (int)__builtin_amdgcn_udot4(r[k], r[k], (uint32_t)srr, false);
                stt = (int)__builtin_amdgcn_udot4(t[k], t[k], (uint32_t)stt, false);
            }
            uint4* r4 = reinterpret_cast<uint4*>(rrow);
            uint4* t4 = reinterpret_cast<uint4*>(trow);
#pragma unroll
            for (int k = 0; k < NT / 16; ++k)         // signed bytes
                r4[k] = make_uint4(r[4 * k] ^ 0x80808080u, r[4 * k + 1] ^ 0x80808080u, r[4 * k + 2] ^ 0x80808080u,
                                   r[4 * k + 3] ^ 0x80808080u);
#pragma unroll
            for (int k = 0; k < Sm::TW / 16; ++k) {   // the target row, repeated
                const int q = k % (NT / 16);
                t4[k] = make_uint4(t[4 * q] ^ 0x80808080u, t[4 * q + 1] ^ 0x80808080u, t[4 * q + 2] ^ 0x80808080u,
                                   t[4 * q + 3] ^ 0x80808080u);
            }
        } else {
            // any even N < NT: the rows as words (load_row), signed, reference
            // bytes x >= N zeroed, then the sums from the signed words with
            // explicit dot products.  (A guarded byte sum `if (x < N) s += a * a`
            // was folded by the compiler into a v_dot4 with a wrong accumulator,
            // adding 1 per row.)
            constexpr int WORDS = NT == 32 ? 8 : TILE == 16 ? 12 : 16;   // N <= 30, 48, 62
            uint32_t r[WORDS], t[WORDS];
            load_row<WORDS>(p.ref + o, N, r);
            load_row<WORDS>(p.tar + o, N, t);
            int s1r = 0, s2r = 0, s1t = 0, s2t = 0;
#pragma unroll
            for (int k = 0; k < WORDS; ++k) {
                const int x = 4 * k;
                const uint32_t keep = x + 4 <= N ? ~0u : x >= N ? 0u : 0xffffu;   // N is even
                r[k] = (r[k] ^ 0x80808080u) & keep;
                t[k] ^= 0x80808080u;
                const int wr = (int)r[k], wt = (int)(t[k] & keep);
                s1r = __builtin_amdgcn_sdot4(wr, 0x01010101, s1r, false);
                s2r = __builtin_amdgcn_sdot4(wr, wr, s2r, false);
                s1t = __builtin_amdgcn_sdot4(wt, 0x01010101, s1t, false);
                s2t = __builtin_amdgcn_sdot4(wt, wt, s2t, false);
            }
            uint4* r4 = reinterpret_cast<uint4*>(rrow);
#pragma unroll
            for (int k = 0; k < NT / 16; ++k)
                r4[k] = 4 * k < WORDS ? make_uint4(r[4 * k], r[4 * k + 1], r[4 * k + 2], r[4 * k + 3])
                                      : make_uint4(0u, 0u, 0u, 0u);
            // the target row at byte 0 and again at byte N.  Products that count
            // read bytes x + ku <= 2N - 2 (x, ku < N); later bytes meet zero
            // reference bytes (x >= N) or output columns ku >= N, which are ignored.
            uint4* t4 = reinterpret_cast<uint4*>(trow);
#pragma unroll
            for (int k = 0; k < WORDS / 4; ++k) t4[k] = make_uint4(t[4 * k], t[4 * k + 1], t[4 * k + 2], t[4 * k + 3]);
            uint32_t* t32 = reinterpret_cast<uint32_t*>(trow) + (N >> 2);
            if ((N & 2) == 0) {
#pragma unroll
                for (int e = 0; e < WORDS; ++e) t32[e] = t[e];
            } else {                                       // N = 4 m + 2: bytes 0, 1 at N, then shifted words
                *reinterpret_cast<uint16_t*>(trow + N) = (uint16_t)t[0];
#pragma unroll
                for (int e = 0; e + 1 < WORDS; ++e) t32[1 + e] = __builtin_amdgcn_alignbyte(t[e + 1], t[e], 2);
            }
            // bytes are v - 128: sum v = s1 + 128 N, sum v^2 = s2 + 256 s1 + 16384 N
            sr = s1r + 128 * N;
            srr = s2r + 256 * s1r + 16384 * N;
            st = s1t + 128 * N;
            stt = s2t + 256 * s1t + 16384 * N;
        }
    }
    sr = wave_sum_i(sr); st = wave_sum_i(st); srr = wave_sum_i(srr); stt = wave_sum_i(stt);
    const long long Sr = sr, St = st, Srr = srr, Stt = stt;
    if (Srr * NN == Sr * Sr || Stt * NN == St * St) {          // flat window (:271-275)
        if (lane == 0 && p.status) p.status[poi] = TWDIC_FFTCC_FLAT;
        return;
    }
    __syncthreads();

    int best = INT_MIN, bk = INT_MAX;
    if constexpr (TILE == 32) {
        // -- C' = A B over K = N rows x TT chunks of 32 bytes ------------------------
        int ra[TT];                                        // A row byte offsets, (y' - kv) mod N
#pragma unroll
        for (int t = 0; t < TT; ++t) {
            const int kv = 32 * t + m;
            ra[t] = (kv < N ? (kv == 0 ? 0 : N - kv) : 0) * Sm::RS + 16 * h;
        }
        // B operand j (j = K chunk + output tile) starts at byte 32 j + 16 h + m
        constexpr int NB = TT == 1 ? 1 : N64 ? 2 : 3;      // distinct B operands per row
        int bd[NB], bs[NB];
#pragma unroll
        for (int j = 0; j < NB; ++j) {
            const int o = 32 * j + 16 * h + m;
            bd[j] = o >> 2;
            bs[j] = o & 3;
        }
        const int rwrap = N * Sm::RS;
        v16i acc[TT][TT];
#pragma unroll
        for (int a = 0; a < TT; ++a)
#pragma unroll
            for (int b = 0; b < TT; ++b) acc[a][b] = v16i{};

        // A operands of row y': lane (m, h) holds reference row (y' - kv) mod N,
        // read from LDS for the next row while the MFMAs of this one run.  (Passing
        // them down one lane per row instead, with a DPP shift and two LDS reads,
        // measured 0.8 % slower: the kernel is power-limited, not LDS-bound.)
        v4i A[TT][TT];                                     // [K chunk][output row tile]
#pragma unroll
        for (int xc = 0; xc < TT; ++xc)
#pragma unroll
            for (int t = 0; t < TT; ++t) A[xc][t] = *reinterpret_cast<const v4i*>(sm.r + ra[t] + 32 * xc);

#pragma unroll 2
        for (int y = 0; y < N; ++y) {
            const uint32_t* trow = reinterpret_cast<const uint32_t*>(sm.t + y * Sm::TS);
            v4i B[NB];
#pragma unroll
            for (int j = 0; j < NB; ++j) B[j] = b_operand(trow, bd[j], bs[j]);
#pragma unroll
            for (int xc = 0; xc < TT; ++xc)
#pragma unroll
                for (int t = 0; t < TT; ++t)
#pragma unroll
                    for (int t2 = 0; t2 < TT; ++t2)     // offset 64 is offset 0 when N = 64
                        acc[t][t2] = __builtin_amdgcn_mfma_i32_32x32x32_i8(A[xc][t], B[(xc + t2) % NB], acc[t][t2], 0, 0, 0);
#pragma unroll
            for (int t = 0; t < TT; ++t) {
                ra[t] += Sm::RS;
                if (ra[t] >= rwrap) ra[t] -= rwrap;
            }
#pragma unroll
            for (int xc = 0; xc < TT; ++xc)
#pragma unroll
                for (int t = 0; t < TT; ++t) A[xc][t] = *reinterpret_cast<const v4i*>(sm.r + ra[t] + 32 * xc);
        }

        // -- exact peak: largest C', lowest row-major index on ties (:300-311) -------
        // a lane's values are visited in increasing index order (kv, then ku), so
        // a strict comparison keeps the lowest index among equal values
#pragma unroll
        for (int t = 0; t < TT; ++t)
#pragma unroll
            for (int r = 0; r < 16; ++r)
#pragma unroll
                for (int t2 = 0; t2 < TT; ++t2) {
                    const int kv = 32 * t + 8 * (r >> 2) + 4 * h + (r & 3), ku = 32 * t2 + m;
                    const int v = acc[t][t2][r];
                    const bool take = kv < N && ku < N && v > best;
                    best = take ? v : best;
                    bk = take ? kv * N + ku : bk;
                }
    } else {
        // -- 16 x 16 tiles: lane (n, g), n = lane % 16, g = lane / 16 ----------
        // A tile t: row (y' - kv) mod N, kv = 16 t + n, bytes 16 g .. 16 g + 15
        // of the 64-byte row (zero beyond N); B tile t': the target row at
        // byte offset 16 g + 16 t' + n; accumulator register r of lane l is
        // output (row 4 g + r, column n) of its tile.
        const int n16 = lane & 15, g = lane >> 4;
        int ra[3], bd[3], bs[3];
#pragma unroll
        for (int t = 0; t < 3; ++t) {
            const int kv = 16 * t + n16;
            ra[t] = (kv < N ? (kv == 0 ? 0 : N - kv) : 0) * Sm::RS + 16 * g;
            const int o = 16 * g + 16 * t + n16;
            bd[t] = o >> 2;
            bs[t] = o & 3;
        }
        const int rwrap = N * Sm::RS;
        v4i acc[3][3];
#pragma unroll
        for (int a = 0; a < 3; ++a)
#pragma unroll
            for (int c = 0; c < 3; ++c) acc[a][c] = v4i{};
        v4i A[3];
#pragma unroll
        for (int t = 0; t < 3; ++t) A[t] = *reinterpret_cast<const v4i*>(sm.r + ra[t]);
        for (int y = 0; y < N; ++y) {
            const uint32_t* trow = reinterpret_cast<const uint32_t*>(sm.t + y * Sm::TS);
            v4i B[3];
#pragma unroll
            for (int t = 0; t < 3; ++t) B[t] = b_operand(trow, bd[t], bs[t]);
#pragma unroll
            for (int t = 0; t < 3; ++t)
#pragma unroll
                for (int t2 = 0; t2 < 3; ++t2)
                    acc[t][t2] = __builtin_amdgcn_mfma_i32_16x16x64_i8(A[t], B[t2], acc[t][t2], 0, 0, 0);
#pragma unroll
            for (int t = 0; t < 3; ++t) {
                ra[t] += Sm::RS;
                if (ra[t] >= rwrap) ra[t] -= rwrap;
                A[t] = *reinterpret_cast<const v4i*>(sm.r + ra[t]);
            }
        }
        // increasing index order within the lane: kv = 16 t + 4 g + r, then ku
#pragma unroll
        for (int t = 0; t < 3; ++t)
#pragma unroll
            for (int r = 0; r < 4; ++r)
#pragma unroll
                for (int t2 = 0; t2 < 3; ++t2) {
                    const int kv = 16 * t + 4 * g + r, ku = 16 * t2 + n16;
                    const int v = acc[t][t2][r];
                    const bool take = kv < N && ku < N && v > best;
                    best = take ? v : best;
                    bk = take ? kv * N + ku : bk;
                }
    }
#pragma unroll
    for (int o = 32; o > 0; o >>= 1) {
        const int ov = __shfl_xor(best, o), ok = __shfl_xor(bk, o);
        const bool take = ov > best || (ov == best && ok < bk);
        best = take ? ov : best;
        bk = take ? ok : bk;
    }
    if (lane == 0) {
        const long long I = (long long)best + 128LL * (Sr + St) - 16384LL * NN;   // sum R T at the peak
        const double nr = (double)Srr - (double)Sr * (double)Sr / (double)NN;
        const double nt = (double)Stt - (double)St * (double)St / (double)NN;
        int iu, iv;
        wrap_peak(bk, N, iu, iv);
        p.u[poi] = (float)iu;
        p.v[poi] = (float)iv;
        p.zncc[poi] = (float)(((double)I - (double)Sr * (double)St / (double)NN) / sqrt(nr * nt));
        if (p.status) p.status[poi] = TWDIC_FFTCC_OK;
    }
}

template <int NT, bool N64, int TILE>
__global__ __launch_bounds__(64) void k_fftcc_mma(FftccParams p)
{
    __shared__ typename MmaSel<NT, N64, TILE>::type sm;
    fftcc_mma_poi<NT, N64, TILE>(sm, p, blockIdx.x);
}

// Batched form, one launch over the POIs of many image pairs that share a
// kernel form: block b takes item b, (pair, POI), and that pair's descriptor.
template <int NT, bool N64, int TILE>
__global__ __launch_bounds__(64) void k_batch_fftcc_mma(const PairDesc* __restrict__ pairs,
                                                        const int2* __restrict__ items)
{
    __shared__ typename MmaSel<NT, N64, TILE>::type sm;
    const int2 it = items[blockIdx.x];
    const FftccParams p = const_pairs(pairs)[__builtin_amdgcn_readfirstlane(it.x)].fftcc;
    fftcc_mma_poi<NT, N64, TILE>(sm, p, __builtin_amdgcn_readfirstlane(it.y));
}

// ===========================================================================
// Matrix-core DFT engine, N = 64 and 32 < N <= 60: the correlation surface from
// fp16 2-D DFTs on v_mfma_f32_32x32x16_f16, then the exact integer correlation
// at every shift the surface leaves within its proven error of the maximum.
//
// For N = 64:
//   r = R - a, t = T - b with a, b the rounded window means: integers in
//   [-255, 255], exact in fp16; the correlation of r and t differs from I[k]
//   = sum R T(k) by a constant, so it has the same argmax.
//   Forward: R^ = F r F, T^ = F t F (F[j][y] = w^(j y), w = exp(-2 pi i / 64),
//   rounded to fp16), two passes of fp16 MFMAs with fp32 accumulation, the
//   intermediate rounded to fp16.  r and t are real, so only the columns k =
//   0 .. 32 are needed (column 64 - k is the conjugate of column k, rows
//   negated): the first pass computes k = 0 .. 31 with column 0 carrying Y[.][0]
//   + i Y[.][32] (its table column is 1 + i (-1)^x, exact), and after the
//   second pass W[j] = R^[j][0] + i R^[j][32] is unpacked with its partner
//   row -j: R^[j][0] = (W[j] + conj W[-j]) / 2, R^[j][32] = (W[j] - conj
//   W[-j]) / 2i.  P = conj(R^) T^ s in fp32 (s a power of two putting |P|
//   below 2^14), rounded to fp16, column 0 repacked as P[.][0] + i P[.][32].
//   Inverse: Q = P^T F* for k = 0 .. 31 (scaled by 2^-8, rows k >= 1 doubled
//   for their conjugates), row 0 giving Q[0][a] + i Q[32][a]; then C^T =
//   Re(F* Q) + (-1)^b Q[32][a], the last term through the imaginary table
//   part of k = 0 (zero in F, (-1)^b here): 144 MFMAs per POI against the
//   integer engine's 512 of the same length.
//   Layouts: a 32 x 32 x 16 accumulator holds column n in lane n (+32 h)
//   and rows 8 (r / 4) + 4 h + r % 4 in register r, so registers 8 c' .. 8 c'
//   + 7 of a tile are a ready B (or, for a transposed product, A) operand
//   whose 16 K values are those rows in that order; the other operand, the
//   fp16 DFT matrix, is stored with its K index in the same order (table 1),
//   so no pass transposes through LDS.
//   Error: |C^ - C| <= kDftBound ||r|| ||t|| / N^2 everywhere.  The bound
//   follows from ||fp16(F) - F||_2 = 1.29e-3, the largest entry error of
//   fp16(F) (1.73e-4), the fp16 and fp32 unit roundoffs, the worst-case error
//   of an fp32 sum of n terms (gamma_{n-1} sum |terms|) for each pass and
//   Cauchy-Schwarz; completing the half spectrum by conjugation turns the
//   computation into the full-spectrum one with one set of errors.  It is
//   15.1 with fp16 sub-normals kept and 21.7 if they were flushed to zero;
//   kDftBound covers both, about sixteen times the largest error of a
//   matrix-level model of this arithmetic on stress windows.  Every shift
//   whose approximate value is within twice that (x 1.25) of the approximate
//   maximum is evaluated exactly in integers, in increasing index order,
//   keeping the first strict maximum: the exact argmax with the CPU path's
//   lowest-index tie-break.  (Speckle windows leave about two such shifts; a
//   window of pure noise a handful; at N = 64 the count is not capped.)
//   A workgroup of eight wavefronts, one POI each, shares the fp16 tables in
//   LDS; the window bytes stay in LDS for the exact stage.
//
// For 32 < N <= 60 the same passes run on N x N tables padded with zeros, which
// also silence the window rows and columns beyond N.  The half spectrum k = 0 ..
// N / 2 fits the 32 columns, so no column is packed; columns 0 and N / 2, their
// own conjugates, count once.  Row k = 31 is empty: it carries the mask that
// keeps rows b >= N from being candidates.  N <= 48 needs three K chunks instead
// of four (112 MFMAs instead of 144) and fits 168 registers, so twelve wavefronts,
// three per SIMD, hide each other's chains of dependent MFMAs and conversions,
// which bound the engine: .48 ms for 157k POIs at N = 40, .71 ms at N = 56 and .73 ms
// at N = 64 (two wavefronts per SIMD; on a slower card up to 8 % more).
// ===========================================================================
typedef _Float16 h8 __attribute__((ext_vector_type(8)));
typedef _Float16 h2v __attribute__((ext_vector_type(2)));
typedef float f16x __attribute__((ext_vector_type(16)));

constexpr double kDftBound = 22.0;        // N^2 |C^ - C| / (||r|| ||t||) at N = 64, see above
// the same over N^2 / 4096 for every even 32 < N <= 60 (largest at N = 54: 25.9)
constexpr double kDftBoundN = 26.0;

// F in fp16 as MFMA operands, [table][part][tile][K chunk][lane], lane = 32 h + m,
// parts re, im, -im:
//   table 0: F[16 c + 8 h + q][32 t + m]                 (B operand, K in natural order);
//            in tile 0 the imaginary part of column 0 holds (-1)^x instead of 0
//   table 1: 2^-8 F[32 t + m][16 c + 8 (q / 4) + 4 h + q % 4]   (A operand, K in accumulator
//            row order; the 2^-8, exact, keeps the first inverse pass's output in fp16 range)
__device__ h8 g_dft_tab[2][3][2][4][64];
// the last pass's imaginary table part for K chunk 0 with the k = 0 entry
// (zero in F) set to 2^-8 (-1)^b: the Nyquist row Q[32][a], carried in the
// imaginary part of row 0, then enters C^T[b][a] with its sign (-1)^b
__device__ h8 g_dft_nyq[2][64];
int g_dft_cus[64] = {};                        // compute units per device, set by dft_tables_init

// One workgroup: the tables (read by all its wavefronts) and, per wavefront,
// its POI's R rows and doubled T rows as bytes and, at N = 64, the second
// pass's spectrum column 0 (for the j <-> -j unpacking).  CH: K chunks of 16
// that hold a window edge, 3 for 32 < N <= 48, else 4.  FULL: N = 64.
// Row pitches of R (16 CH bytes) and T (32 CH): 14 and 26, or 18 and 34,
// dwords put the 8-byte operand reads of 16 consecutive rows on distinct banks.
template <int CH, bool FULL>
struct DftWgSmem {
    static constexpr int WAVES = CH == 3 ? 12 : 8;       // POIs in flight, one per wavefront
    static constexpr int ROWS = 16 * CH, RP = CH == 3 ? 56 : 72, TP = CH == 3 ? 104 : 136;
    h8 ta[2][CH][64];
    h8 tb[3][2][CH][64];
    h8 tn[2][64];
    uint8_t ex[WAVES][ROWS * (RP + TP)];
    float col0[FULL ? WAVES : 1][4][64];                // Re R^, Im R^, Re T^, Im T^ of column 0, by row j
    uint32_t xcol[FULL ? WAVES : 1][64];
    static constexpr int KEPT = 32;                     // POIs whose outputs are formed together
    int kept[WAVES][7][KEPT];                           // item, sums of R, T, R^2, T^2, sum R T at the peak, peak
};

// Where a window pair is (no padding bytes: those kept copies in memory).
struct DftItem {
    const uint8_t *ref, *tar;
    int stride, py, px, inside;                         // inside: the windows lie in the image
    __device__ __forceinline__ size_t row(int lane, int N) const
    {
        return (size_t)(py - N / 2 + lane) * stride + (px - N / 2);
    }
};

__device__ __forceinline__ DftItem dft_item(const FftccParams& p, int poi)
{
    const int py = p.poi[2 * poi], px = p.poi[2 * poi + 1], h = p.N / 2;
    return {p.ref, p.tar, p.stride, py, px, py >= h && px >= h && py + h <= p.img_h && px + h <= p.img_w};
}

// A window pair's rows in flight, CH lanes to a row, 16 bytes each, so that a
// load instruction touches the lines of 64 / CH rows (with a lane per row the
// lines of 64, four times over: the loads of eight wavefronts queued up in the
// address unit, 0.81 ms for 157k POIs at N = 64 against 0.73 ms).  Lane l
// holds piece l % CH of the rows k (64 / CH) + l / CH.  A row's last piece ends
// with the row, so nothing outside it is read; words() moves it to its place.
template <int CH, bool FULL>
struct DftRows {
    static constexpr int RL = 64 / CH, LOADS = (16 * CH + RL - 1) / RL;
    uint32_t r[LOADS][4], t[LOADS][4];
    __device__ __forceinline__ static int row(int k, int lane) { return RL * k + lane / CH; }
    __device__ __forceinline__ static bool active(int k, int lane, int N)
    {
        return FULL || (row(k, lane) < N && lane < RL * CH);
    }
    // Any values, or zeros where load() may leave them: nothing has to be kept
    // in these registers until then.
    __device__ __forceinline__ void drop()
    {
#pragma unroll
        for (int k = 0; k < LOADS; ++k)
#pragma unroll
            for (int w = 0; w < 4; ++w) {
                if constexpr (FULL) {
                    asm("" : "=v"(r[k][w]));
                    asm("" : "=v"(t[k][w]));
                } else {
                    r[k][w] = t[k][w] = 0u;
                }
            }
    }
    __device__ __forceinline__ void load(const DftItem& it, int N, int lane)
    {
        const int x = min(16 * (lane % CH), N - 16);
#pragma unroll
        for (int k = 0; k < LOADS; ++k)
            if (active(k, lane, N)) {
                const size_t o = it.row(row(k, lane), N) + x;
                __builtin_memcpy(r[k], it.ref + o, 16);
                __builtin_memcpy(t[k], it.tar + o, 16);
            }
    }
    // The words of bytes 16 (lane % CH) .. + 15 of a row, zero beyond N: the last
    // piece less the 16 CH - N bytes that belong to the one before.
    __device__ __forceinline__ static void words(const uint32_t (&raw)[4], int N, int lane, uint32_t (&w)[4])
    {
        if constexpr (FULL) {
#pragma unroll
            for (int i = 0; i < 4; ++i) w[i] = raw[i];
        } else {
            const int sh = lane % CH == CH - 1 ? 16 * CH - N : 0;
            uint32_t m2 = (sh & 8) ? ~0u : 0u, m1 = (sh & 4) ? ~0u : 0u;
            asm volatile("" : "+v"(m2), "+v"(m1));      // bitwise selects, as in load_row
            uint32_t a[5], b[5];
#pragma unroll
            for (int i = 0; i < 4; ++i) a[i] = ((i < 2 ? raw[(i + 2) & 3] : 0u) & m2) | (raw[i] & ~m2);
            a[4] = 0u;
#pragma unroll
            for (int i = 0; i < 4; ++i) b[i] = (a[i + 1] & m1) | (a[i] & ~m1);
            b[4] = 0u;
#pragma unroll
            for (int i = 0; i < 4; ++i) w[i] = __builtin_amdgcn_alignbyte(b[i + 1], b[i], sh & 3);
        }
    }
};

// Sums over the wavefront of four values at once (as swap_add in icgn.hip:
// pairs folded by permlane swaps, then row rotations), in scalars.
__device__ __forceinline__ void dpp_sum4(int v[4])
{
    int w[2];
#pragma unroll
    for (int i = 0; i < 2; ++i) {
        const auto s = __builtin_amdgcn_permlane32_swap((uint32_t)v[i], (uint32_t)v[i + 2], false, false);
        w[i] = (int)(s[0] + s[1]);                      // lanes 0-31: v[i], 32-63: v[i + 2]
    }
    const auto s = __builtin_amdgcn_permlane16_swap((uint32_t)w[0], (uint32_t)w[1], false, false);
    int x = (int)(s[0] + s[1]);                         // rows 0 .. 3: v[0], v[1], v[2], v[3]
    x += __builtin_amdgcn_update_dpp(0, x, 0x128, 0xF, 0xF, true);
    x += __builtin_amdgcn_update_dpp(0, x, 0x124, 0xF, 0xF, true);
    x += __builtin_amdgcn_update_dpp(0, x, 0x122, 0xF, 0xF, true);
    x += __builtin_amdgcn_update_dpp(0, x, 0x121, 0xF, 0xF, true);
#pragma unroll
    for (int i = 0; i < 4; ++i) v[i] = __builtin_amdgcn_readlane(x, 16 * i);
}

__device__ __forceinline__ f16x mfma16(h8 a, h8 b, f16x c)
{
    return __builtin_amdgcn_mfma_f32_32x32x16_f16(a, b, c, 0, 0, 0);
}

// accumulator registers 8 half .. 8 half + 7, times scale, rounded to fp16
__device__ __forceinline__ h8 to_h8(const f16x& acc, int half, float scale)
{
    h8 r;
#pragma unroll
    for (int q = 0; q < 8; ++q) r[q] = (_Float16)(acc[8 * half + q] * scale);
    return r;
}

// Wave-uniform reductions for the DFT engine: butterflies inside each row of
// 16 lanes by DPP (xor 1, xor 2, half-row mirror, row mirror), then the four
// row results by readlane.  Every lane must be active.
template <class Op>
__device__ __forceinline__ int wave_reduce_dpp(int v, Op op)
{
    v = op(v, __builtin_amdgcn_update_dpp(v, v, 0xB1, 0xF, 0xF, false));
    v = op(v, __builtin_amdgcn_update_dpp(v, v, 0x4E, 0xF, 0xF, false));
    v = op(v, __builtin_amdgcn_update_dpp(v, v, 0x141, 0xF, 0xF, false));
    v = op(v, __builtin_amdgcn_update_dpp(v, v, 0x140, 0xF, 0xF, false));
    const int a = __builtin_amdgcn_readlane(v, 0), b = __builtin_amdgcn_readlane(v, 16);
    const int c = __builtin_amdgcn_readlane(v, 32), d = __builtin_amdgcn_readlane(v, 48);
    return op(op(a, b), op(c, d));
}
__device__ __forceinline__ int dpp_sum(int v)
{
    return wave_reduce_dpp(v, [](int x, int y) { return x + y; });
}
__device__ __forceinline__ float dpp_max(float v)
{
    return __int_as_float(wave_reduce_dpp(__float_as_int(v), [](int x, int y) {
        return __float_as_int(fmaxf(__int_as_float(x), __int_as_float(y)));
    }));
}

// 2 mask + (x >= thr): the compare's lane mask is the carry-in of an add,
// two instructions per bit
__device__ __forceinline__ uint32_t shift_in_ge(uint32_t mask, float x, float thr)
{
    uint32_t r;
    asm("v_cmp_ge_f32_e32 vcc, %1, %2\n\tv_addc_co_u32_e32 %0, vcc, %3, %3, vcc"
        : "=v"(r)
        : "v"(x), "v"(thr), "v"(mask)
        : "vcc");
    return r;
}

// Eight window bytes as the fp16 values byte - off: the byte v becomes the
// half 1024 + v (bits 0x6400 | v), minus off = 1024 + mean, exactly.  The
// byte shuffle is one v_perm_b32 per two values (selector bytes 0-3 take the
// bytes of the second source, 4-7 those of the first: 0x64).
__device__ __forceinline__ h8 centred_h8(uint2 w, h2v off)
{
    const uint32_t q[4] = {__builtin_amdgcn_perm(0x64646464u, w.x, 0x04010400u),
                           __builtin_amdgcn_perm(0x64646464u, w.x, 0x04030402u),
                           __builtin_amdgcn_perm(0x64646464u, w.y, 0x04010400u),
                           __builtin_amdgcn_perm(0x64646464u, w.y, 0x04030402u)};
    h8 r;
#pragma unroll
    for (int k = 0; k < 4; ++k) {
        const h2v v = __builtin_bit_cast(h2v, q[k]) - off;
        r[2 * k] = v[0];
        r[2 * k + 1] = v[1];
    }
    return r;
}

// One window pair's rows (DftRows) to the wavefront's LDS: R row y at y RP, zero
// beyond N, T row y at y TP and again N bytes on; and the exact integer sums of
// R, T, R^2, T^2.
template <int CH, bool FULL>
__device__ __forceinline__ void dft_window(DftWgSmem<CH, FULL>& sm, int wave, int lane, int N,
                                           const DftRows<CH, FULL>& rows, int (&sums)[4])
{
    using Sm = DftWgSmem<CH, FULL>;
    uint8_t* ex = sm.ex[wave];
#pragma unroll
    for (int i = 0; i < 4; ++i) sums[i] = 0;
    using Rows = DftRows<CH, FULL>;
    uint32_t rw[Rows::LOADS][4], tw[Rows::LOADS][4];
#pragma unroll
    for (int k = 0; k < Rows::LOADS; ++k) {
        Rows::words(rows.r[k], N, lane, rw[k]);
        Rows::words(rows.t[k], N, lane, tw[k]);
#pragma unroll
        for (int w = 0; w < 4; ++w) {
            sums[0] = (int)__builtin_amdgcn_udot4(rw[k][w], 0x01010101u, (uint32_t)sums[0], false);
            sums[1] = (int)__builtin_amdgcn_udot4(tw[k][w], 0x01010101u, (uint32_t)sums[1], false);
            sums[2] = (int)__builtin_amdgcn_udot4(rw[k][w], rw[k][w], (uint32_t)sums[2], false);
            sums[3] = (int)__builtin_amdgcn_udot4(tw[k][w], tw[k][w], (uint32_t)sums[3], false);
        }
    }
    wave_lds_sync();                           // the previous POI's reads of this region are done
    uint8_t* er = ex + (lane / CH) * Sm::RP + 16 * (lane % CH);
    uint8_t* et = ex + Sm::ROWS * Sm::RP + (lane / CH) * Sm::TP + 16 * (lane % CH);
#pragma unroll
    for (int k = 0; k < Rows::LOADS; ++k)
        if (Rows::active(k, lane, N)) {
            uint2* e2 = reinterpret_cast<uint2*>(er + k * Rows::RL * Sm::RP);
            uint2* t2 = reinterpret_cast<uint2*>(et + k * Rows::RL * Sm::TP);
#pragma unroll
            for (int e = 0; e < 2; ++e) {
                e2[e] = make_uint2(rw[k][2 * e], rw[k][2 * e + 1]);
                t2[e] = make_uint2(tw[k][2 * e], tw[k][2 * e + 1]);
            }
        }
    // the T rows again from byte N on (up to byte 2 N - 1 they are read),
    // over the zeros of the last piece, which another lane has stored
    if constexpr (!FULL) wave_lds_sync();
#pragma unroll
    for (int k = 0; k < Rows::LOADS; ++k)
        if (Rows::active(k, lane, N)) {
            uint8_t* again = et + k * Rows::RL * Sm::TP + N;
            if constexpr (FULL) {
                reinterpret_cast<uint2*>(again)[0] = make_uint2(tw[k][0], tw[k][1]);
                reinterpret_cast<uint2*>(again)[1] = make_uint2(tw[k][2], tw[k][3]);
            } else {
                __builtin_memcpy(again, tw[k], 16);
            }
        }
    dpp_sum4(sums);
}

// The rounded means a, b of R and T and ||R - a||^2, ||T - b||^2, exact below 2^31:
// zero for a uniform window, whose rounded mean is its value, and for no other.
struct DftNorms {
    int a, b, r2, t2;
    __device__ __forceinline__ DftNorms(const int (&sums)[4], int NN)
        : a((int)((uint32_t)(sums[0] + NN / 2) / (uint32_t)NN)),
          b((int)((uint32_t)(sums[1] + NN / 2) / (uint32_t)NN)),
          r2(sums[2] - 2 * a * sums[0] + a * a * NN), t2(sums[3] - 2 * b * sums[1] + b * b * NN)
    {
    }
    __device__ __forceinline__ bool flat() const { return r2 == 0 || t2 == 0; }       // (:271-275)
};

// Below N = 64 a window pair that leaves more than N shifts in question (it is
// periodic, or nearly so) has its whole integer surface formed instead, in a time
// that does not depend on the image, and so have the wavefront's next
// kDftDirectRun pairs, its neighbours.  After one with more than N / 2 (a texture
// that varies in one direction only gives N) the next pair goes there at once, and
// when the DFTs then find another such, the next 3, 7, ... kDftDirectRun.  Of 32,761 POIs at N = 40 the DFTs take 0.114 ms,
// each candidate 0.0057 and the integer surface 0.25, i.e. 24 candidates more than
// the DFTs and 44 alone; at N = 56 0.165, 0.0081, 0.45: 35 and 55.
constexpr int kDftDirectRun = 31;

// The exact peak of the window pair in the wavefront's LDS rows from the integer
// surface, as k_fftcc_mma forms it (48 x 48 in 16 x 16 tiles for CH = 3, 64 x 64 in
// 32 x 32 ones): lane (m, g) holds bytes 16 g .. 16 g + 15 of a K chunk.  The rows
// are turned signed in place first (reference bytes from N on stay zero).  With
// two or three wavefronts per SIMD the waits for LDS show, so both operands of a
// row are loaded while the products of the one before run.  32,761 POIs of a
// grating of period 4: 0.260 ms at N = 40 (all 400 candidates: 2.3; the integer
// kernel, with more wavefronts, 0.20), 0.46 ms at N = 56 (784: 6.3; 0.36).
template <int CH>
__device__ __forceinline__ void mma_direct(DftWgSmem<CH, false>& sm, int wave, int lane, int N, const int (&sums)[4],
                                           int& bestI, int& peak)
{
    using Sm = DftWgSmem<CH, false>;
    constexpr int TE = CH == 3 ? 16 : 32, T = CH == 3 ? 3 : 2, KC = CH == 3 ? 1 : 2, NB = 3, REGS = TE * TE / 64;
    typedef int acc_t __attribute__((ext_vector_type(REGS)));
    uint8_t *rows = sm.ex[wave], *trows = rows + Sm::ROWS * Sm::RP;
    wave_lds_sync();
    constexpr int RQ = Sm::RP / 8, RN = Sm::ROWS * RQ, TN = Sm::ROWS * Sm::TP / 8;
#pragma unroll
    for (int k = 0; k < (RN + 63) / 64; ++k) {
        const int i = 64 * k + lane, x = 8 * (i % RQ);
        if (i < RN) {
            uint2* q = reinterpret_cast<uint2*>(rows) + i;
            auto flip = [&](int at) { return at + 4 <= N ? 0x80808080u : at >= N ? 0u : 0x8080u; };     // N is even
            *q = make_uint2(q->x ^ flip(x), q->y ^ flip(x + 4));
        }
    }
#pragma unroll
    for (int k = 0; k < (TN + 63) / 64; ++k) {
        const int i = 64 * k + lane;
        if (i < TN) {
            uint2* q = reinterpret_cast<uint2*>(trows) + i;
            *q = make_uint2(q->x ^ 0x80808080u, q->y ^ 0x80808080u);
        }
    }
    wave_lds_sync();

    const int m = lane % TE, g = lane / TE;
    // bytes 48 .. 63 of a 48-byte row: the zeros of the half spectrum's unused column 31
    const bool pad = CH == 3 && g == 3;
    const int step = pad ? 0 : Sm::RP, wrap = N * Sm::RP, end = pad ? INT_MAX : wrap;
    int ra[T], bd[NB], bs[NB];
#pragma unroll
    for (int t = 0; t < T; ++t) {
        const int kv = TE * t + m;       // reference row (y' - kv) mod N
        ra[t] = pad ? (int)(reinterpret_cast<const uint8_t*>(&sm.ta[0][0][31]) - rows)
                    : (kv > 0 && kv < N ? N - kv : 0) * Sm::RP + 16 * g;
    }
#pragma unroll
    for (int j = 0; j < NB; ++j) {
        const int o = TE * j + 16 * g + m;
        bd[j] = o >> 2;
        bs[j] = o & 3;
    }
    acc_t acc[T][T];
#pragma unroll
    for (int t = 0; t < T; ++t)
#pragma unroll
        for (int t2 = 0; t2 < T; ++t2) acc[t][t2] = acc_t{};
    v4i A[2][KC][T];
    uint32_t raw[NB][5];
    auto fetch_b = [&](int y) {
        const uint32_t* trow = reinterpret_cast<const uint32_t*>(trows + y * Sm::TP);
#pragma unroll
        for (int j = 0; j < NB; ++j)
#pragma unroll
            for (int i = 0; i < 5; ++i) raw[j][i] = trow[bd[j] + i];
    };
    auto fetch_a = [&](v4i (&d)[KC][T]) {
#pragma unroll
        for (int t = 0; t < T; ++t) {
#pragma unroll
            for (int xc = 0; xc < KC; ++xc) {
                const uint2* p = reinterpret_cast<const uint2*>(rows + ra[t] + 32 * xc);
                const uint2 a = p[0], b = p[1];
                d[xc][t] = v4i{(int)a.x, (int)a.y, (int)b.x, (int)b.y};
            }
            ra[t] += step;
            if (ra[t] >= end) ra[t] -= wrap;
        }
    };
    auto row = [&](const v4i (&cur)[KC][T], v4i (&next)[KC][T], int y) {
        v4i B[NB];
#pragma unroll
        for (int j = 0; j < NB; ++j)
#pragma unroll
            for (int i = 0; i < 4; ++i) B[j][i] = (int)__builtin_amdgcn_alignbyte(raw[j][i + 1], raw[j][i], bs[j]);
        fetch_b(min(y + 1, N - 1));
        fetch_a(next);
        __builtin_amdgcn_sched_barrier(0);
#pragma unroll
        for (int xc = 0; xc < KC; ++xc)
#pragma unroll
            for (int t = 0; t < T; ++t)
#pragma unroll
                for (int t2 = 0; t2 < T; ++t2) {
                    if constexpr (CH == 3)
                        acc[t][t2] = __builtin_amdgcn_mfma_i32_16x16x64_i8(cur[xc][t], B[xc + t2], acc[t][t2], 0, 0, 0);
                    else
                        acc[t][t2] = __builtin_amdgcn_mfma_i32_32x32x32_i8(cur[xc][t], B[xc + t2], acc[t][t2], 0, 0, 0);
                }
        __builtin_amdgcn_sched_barrier(0);
    };
    fetch_b(0);
    fetch_a(A[0]);
    for (int y = 0; y < N; y += 2) {      // N is even
        row(A[0], A[1], y);
        row(A[1], A[0], y + 1);
    }
    // the largest, of equal ones the lowest place 64 kv + ku: a lane's are visited
    // in increasing order
    int best = INT_MIN;
    peak = INT_MAX;
#pragma unroll
    for (int t = 0; t < T; ++t)
#pragma unroll
        for (int r = 0; r < REGS; ++r)
#pragma unroll
            for (int t2 = 0; t2 < T; ++t2) {
                const int kv = TE * t + 8 * (r >> 2) + 4 * g + (r & 3), ku = TE * t2 + m, v = acc[t][t2][r];
                // N > TE (T - 1): only the last tiles reach beyond the window
                const bool take = (t < T - 1 || kv < N) && (t2 < T - 1 || ku < N) && v > best;
                best = take ? v : best;
                peak = take ? 64 * kv + ku : peak;
            }
#pragma unroll
    for (int o = 32; o > 0; o >>= 1) {
        const int ov = __shfl_xor(best, o), ok = __shfl_xor(peak, o);
        const bool take = ov > best || (ov == best && ok < peak);
        best = take ? ov : best;
        peak = take ? ok : peak;
    }
    bestI = best + 128 * (sums[0] + sums[1]) - 16384 * N * N;
}

// The exact peak of one window pair whose rows are in `rows`; `next` is called
// when they and most registers are free again, to load the following pair's.
// Gives the four window sums, the number of candidates (DFT_MANY: the first N, and
// no peak) and, but for a flat window, the exact sum of R T at the peak and the
// peak's place 64 a + b.
enum { DFT_PEAK, DFT_FLAT, DFT_MANY };
template <int CH, bool FULL, class Next>
__device__ __forceinline__ int fftcc_dft_mfma_poi(DftWgSmem<CH, FULL>& sm, int wave, int lane, int N,
                                                  DftRows<CH, FULL>& rows, int (&sums)[4], int& many, int& bestI,
                                                  int& peak, Next next)
{
    using Sm = DftWgSmem<CH, FULL>;
    constexpr int WORDS = 4 * CH;
    if constexpr (FULL) N = 64;
    const int NN = N * N, m = lane & 31, h = lane >> 5;
    const uint8_t* erows = sm.ex[wave];
    const uint8_t* etrows = erows + Sm::ROWS * Sm::RP;
    dft_window(sm, wave, lane, N, rows, sums);
    const DftNorms norm(sums, NN);
    many = 0;
    if (norm.flat()) {
        next();
        return DFT_FLAT;
    }
    const h2v oa = {(_Float16)(1024 + norm.a), (_Float16)(1024 + norm.a)};
    const h2v ob = {(_Float16)(1024 + norm.b), (_Float16)(1024 + norm.b)};
    // s: a power of two, s N^2 ||r|| ||t|| in [2^13, 2^14); the tolerance in C^ units
    // (s 2^-16 N^2 C).  Below N = 64 in FP32, whose rounding the factor 1.25 over the
    // bound dwarfs (in FP64 0.534 -> 0.543 ms for 155k POIs at N = 40)
    float s, tol;
    if constexpr (FULL) {
        const double rho = sqrt((double)norm.r2 * (double)norm.t2);
        s = ldexpf(1.0f, 14 - __builtin_amdgcn_frexp_exp(4096.0 * rho));
        tol = (float)(2.0 * 1.25 * kDftBound * rho * (double)s / 65536.0);
    } else {
        const float rho = __builtin_amdgcn_sqrtf((float)norm.r2) * __builtin_amdgcn_sqrtf((float)norm.t2);
        s = ldexpf(1.0f, 14 - __builtin_amdgcn_frexp_expf((float)NN * rho));
        tol = 2.5f / 65536.f * (float)(kDftBoundN / 4096.0) * (float)NN * rho * s;
    }
    wave_lds_sync();

    const int wave_f = FULL ? wave : 0;
    // -- first pass, columns k = 0 .. 31 (column 0 = Y[.][0] + i Y[.][32]) -------
    h8 Yrr[CH], Yri[CH], Ytr[CH], Yti[CH];     // B operands, K chunk c = rows 16 c .. 16 c + 15 (accumulator order)
#pragma unroll
    for (int Mt = 0; Mt < 2; ++Mt) {
        f16x yrr = {}, yri = {}, ytr = {}, yti = {};
        const int y = FULL ? 32 * Mt + m : min(32 * Mt + m, N - 1);    // rows from N on meet zeros of the table
#pragma unroll
        for (int c = 0; c < CH; ++c) {
            const h8 Fr = sm.ta[0][c][lane], Fi = sm.ta[1][c][lane];
            const h8 Ar = centred_h8(*reinterpret_cast<const uint2*>(erows + y * Sm::RP + 16 * c + 8 * h), oa);
            const h8 At = centred_h8(*reinterpret_cast<const uint2*>(etrows + y * Sm::TP + 16 * c + 8 * h), ob);
            yrr = mfma16(Ar, Fr, yrr);
            yri = mfma16(Ar, Fi, yri);
            ytr = mfma16(At, Fr, ytr);
            yti = mfma16(At, Fi, yti);
        }
#pragma unroll
        for (int hf = 0; hf < 2 && 2 * Mt + hf < CH; ++hf) {
            Yrr[2 * Mt + hf] = to_h8(yrr, hf, 1.f);
            Yri[2 * Mt + hf] = to_h8(yri, hf, 1.f);
            Ytr[2 * Mt + hf] = to_h8(ytr, hf, 1.f);
            Yti[2 * Mt + hf] = to_h8(yti, hf, 1.f);
        }
        __builtin_amdgcn_sched_barrier(0);
    }
    // -- second pass: R^, T^ for k = 0 .. 31 and P = conj(R^) T^ s ----------------
    h8 Pre[CH], Pim[CH];                       // A operands of the first inverse pass [j chunk]
#pragma unroll
    for (int Mj = 0; Mj < 2; ++Mj) {
        f16x Rr = {}, Ri = {}, Tr = {}, Ti = {};
#pragma unroll
        for (int c = 0; c < CH; ++c) {
            const h8 Fr = sm.tb[0][Mj][c][lane], Fi = sm.tb[1][Mj][c][lane], nFi = sm.tb[2][Mj][c][lane];
            Rr = mfma16(Fr, Yrr[c], Rr);
            Ri = mfma16(Fr, Yri[c], Ri);
            Tr = mfma16(Fr, Ytr[c], Tr);
            Ti = mfma16(Fr, Yti[c], Ti);
            Rr = mfma16(nFi, Yri[c], Rr);
            Ri = mfma16(Fi, Yrr[c], Ri);
            Tr = mfma16(nFi, Yti[c], Tr);
            Ti = mfma16(Fi, Ytr[c], Ti);
        }
        if (FULL && m == 0) {                  // column 0: W_R = R^[j][0] + i R^[j][32], W_T likewise
#pragma unroll
            for (int g = 0; g < 4; ++g) {      // registers 4 g .. 4 g + 3 hold rows j0 .. j0 + 3
                const int j0 = 32 * Mj + 8 * g + 4 * h;
                *reinterpret_cast<float4*>(&sm.col0[wave_f][0][j0]) = make_float4(Rr[4 * g], Rr[4 * g + 1], Rr[4 * g + 2], Rr[4 * g + 3]);
                *reinterpret_cast<float4*>(&sm.col0[wave_f][1][j0]) = make_float4(Ri[4 * g], Ri[4 * g + 1], Ri[4 * g + 2], Ri[4 * g + 3]);
                *reinterpret_cast<float4*>(&sm.col0[wave_f][2][j0]) = make_float4(Tr[4 * g], Tr[4 * g + 1], Tr[4 * g + 2], Tr[4 * g + 3]);
                *reinterpret_cast<float4*>(&sm.col0[wave_f][3][j0]) = make_float4(Ti[4 * g], Ti[4 * g + 1], Ti[4 * g + 2], Ti[4 * g + 3]);
            }
        }
        f16x pr, pi;
#pragma unroll
        for (int i = 0; i < 16; ++i) {
            pr[i] = fmaf(Rr[i], Tr[i], Ri[i] * Ti[i]);
            pi[i] = fmaf(Rr[i], Ti[i], -(Ri[i] * Tr[i]));
        }
        // columns k >= 1 doubled for their conjugates N - k (at N = 64 column 0 is
        // rewritten below; otherwise 0 and N / 2, their own conjugates, count
        // once); 2^16 undoes the two 2^-8 of the table
        const float weight = !FULL && (m == 0 || 2 * m == N) ? 65536.f * s : 131072.f * s;
#pragma unroll
        for (int hf = 0; hf < 2 && 2 * Mj + hf < CH; ++hf) {
            Pre[2 * Mj + hf] = to_h8(pr, hf, weight);
            Pim[2 * Mj + hf] = to_h8(pi, hf, weight);
        }
        __builtin_amdgcn_sched_barrier(0);
    }
    if constexpr (FULL) {
        float (*col0)[64] = sm.col0[wave_f];
        uint32_t* xcol = sm.xcol[wave_f];
        // column 0 of P becomes P[j][0] + i P[j][32]: unpack R^[j][0] = (W[j] +
        // conj W[-j]) / 2, R^[j][32] = (W[j] - conj W[-j]) / 2i, likewise T^; lane
        // j does row j (the results for j and -j are exact conjugates), lanes m = 0
        // collect theirs
        wave_lds_sync();
        {
            const int jm = (64 - lane) & 63;
            const float4 w = make_float4(col0[0][lane], col0[1][lane], col0[2][lane], col0[3][lane]);
            const float4 wm = make_float4(col0[0][jm], col0[1][jm], col0[2][jm], col0[3][jm]);
            const float ar = 0.5f * (w.x + wm.x), ai = 0.5f * (w.y - wm.y);    // R^[j][0]
            const float br = 0.5f * (w.y + wm.y), bi = 0.5f * (wm.x - w.x);    // R^[j][32]
            const float cr = 0.5f * (w.z + wm.z), ci = 0.5f * (w.w - wm.w);    // T^[j][0]
            const float dr = 0.5f * (w.w + wm.w), di = 0.5f * (wm.z - w.z);    // T^[j][32]
            const float p0r = fmaf(ar, cr, ai * ci), p0i = fmaf(ar, ci, -(ai * cr));   // conj(R^0) T^0
            const float p1r = fmaf(br, dr, bi * di), p1i = fmaf(br, di, -(bi * dr));   // conj(R^32) T^32
            const h2v x = {(_Float16)((p0r - p1i) * (65536.f * s)), (_Float16)((p0i + p1r) * (65536.f * s))};
            xcol[lane] = __builtin_bit_cast(uint32_t, x);
        }
        wave_lds_sync();
        if (m == 0) {
#pragma unroll
            for (int Mj = 0; Mj < 2; ++Mj)
#pragma unroll
                for (int r = 0; r < 16; ++r) {
                    const h2v x = __builtin_bit_cast(h2v, xcol[32 * Mj + 8 * (r >> 2) + 4 * h + (r & 3)]);
                    Pre[2 * Mj + (r >> 3)][r & 7] = x[0];
                    Pim[2 * Mj + (r >> 3)][r & 7] = x[1];
                }
        }
    }
    // -- first inverse pass, rows k = 0 .. 31: Q[k][a] = sum_j P[j][k] conj(F[j][a])
    //    (row 0 comes out as Q[0][a] + i Q[32][a], both real) -----------------------
    h8 Qr[2][2], Qi[2][2];                     // B operands of the last pass [k chunk][a tile]
    {
        f16x qr[2] = {}, qi[2] = {};
#pragma unroll
        for (int c = 0; c < CH; ++c) {
#pragma unroll
            for (int Nc = 0; Nc < 2; ++Nc) {
                const h8 Fr = sm.tb[0][Nc][c][lane], Fi = sm.tb[1][Nc][c][lane], nFi = sm.tb[2][Nc][c][lane];
                qr[Nc] = mfma16(Pre[c], Fr, qr[Nc]);
                qi[Nc] = mfma16(Pim[c], Fr, qi[Nc]);
                qr[Nc] = mfma16(Pim[c], Fi, qr[Nc]);
                qi[Nc] = mfma16(Pre[c], nFi, qi[Nc]);
            }
        }
#pragma unroll
        for (int Nc = 0; Nc < 2; ++Nc) {
#pragma unroll
            for (int hf = 0; hf < 2; ++hf) {
                Qr[hf][Nc] = to_h8(qr[Nc], hf, 1.f);
                Qi[hf][Nc] = to_h8(qi[Nc], hf, 1.f);
            }
        }
        // N <= 60: row k = 31 is empty; a one in it lets the last pass's table
        // push the rows b >= N below every candidate
        if (!FULL && h == 1) Qr[1][0][7] = Qr[1][1][7] = (_Float16)1.f;
        __builtin_amdgcn_sched_barrier(0);
    }
    // -- last pass: C^T = Re(F* Q) + (-1)^b Q[32][a], lane -> a, register -> b ------
    f16x Cd[2][2] = {};                        // [b tile][a tile]
#pragma unroll
    for (int c = 0; c < 2; ++c) {
#pragma unroll
        for (int Md = 0; Md < 2; ++Md) {
            const h8 Fr = !FULL && c == 1 ? sm.tn[Md][lane] : sm.tb[0][Md][c][lane];
            const h8 Fi = FULL && c == 0 ? sm.tn[Md][lane] : sm.tb[1][Md][c][lane];
#pragma unroll
            for (int Nd = 0; Nd < 2; ++Nd) {
                Cd[Md][Nd] = mfma16(Fr, Qr[c][Nd], Cd[Md][Nd]);
                Cd[Md][Nd] = mfma16(Fi, Qi[c][Nd], Cd[Md][Nd]);
            }
        }
    }

    // -- candidates: every shift within tol of the approximate maximum -----------
    float gmx[2][2];                           // per 16-register group [Nd][Md]
#pragma unroll
    for (int Md = 0; Md < 2; ++Md)
#pragma unroll
        for (int Nd = 0; Nd < 2; ++Nd) {
            float g = Cd[Md][Nd][0];
#pragma unroll
            for (int r = 1; r < 16; ++r) g = fmaxf(g, Cd[Md][Nd][r]);
            gmx[Nd][Md] = !FULL && 32 * Nd + m >= N ? -FLT_MAX : g;    // columns a >= N are none
        }
    const float mx = dpp_max(fmaxf(fmaxf(gmx[0][0], gmx[0][1]), fmaxf(gmx[1][0], gmx[1][1])));
    const float thr = mx - tol;
    // bit 16 (2 Nd + Md) + r: this lane's shifts in increasing row-major index (a,
    // then b, kept as 64 a + b) (shifted in from the top bit down); a group no lane has a candidate
    // in is skipped
    uint32_t mw[2] = {0u, 0u};
#pragma unroll
    for (int Nd = 0; Nd < 2; ++Nd)
#pragma unroll
        for (int Md = 1; Md >= 0; --Md) {
            uint32_t bits = 0;
            if (gmx[Nd][Md] >= thr) {
#pragma unroll
                for (int r = 15; r >= 0; --r) bits = shift_in_ge(bits, Cd[Md][Nd][r], thr);
            }
            mw[Nd] |= bits << (16 * Md);
        }
    uint64_t mask = ((uint64_t)mw[1] << 32) | mw[0];

    next();

    // -- exact integer correlation at the candidates: the largest, of equal ones
    //    the lowest index ------------------------------------------------------
    const uint32_t* rrow = reinterpret_cast<const uint32_t*>(erows + (FULL || lane < N ? lane : 0) * Sm::RP);
    bestI = -1;
    peak = 0;
    // a lane's lowest candidate as 64 a + b
    auto lowest = [&]() {
        const int bit = __builtin_ctzll(mask | (1ull << 63));
        const int Nd = bit >> 5, Md = (bit >> 4) & 1, r = bit & 15;
        return (32 * Nd + m) * 64 + 32 * Md + 8 * (r >> 2) + 4 * h + (r & 3);
    };
    for (unsigned long long lanes; (lanes = __ballot(mask != 0)) != 0;) {
        if (++many > N && !FULL) return DFT_MANY;
        const int from = __builtin_ctzll(lanes), k = __builtin_amdgcn_readlane(lowest(), from);
        if (lane == from) mask &= mask - 1;
        const int kv = k >> 6, ku = k & 63, d = ku >> 2, sh = ku & 3;
        int ty = lane + kv;                        // row (lane + kv) mod N
        if constexpr (FULL)
            ty &= 63;
        else
            ty = lane >= N ? 0 : ty >= N ? ty - N : ty;
        const uint32_t* trow = reinterpret_cast<const uint32_t*>(etrows + ty * Sm::TP);
        // all words first: read and used one by one, each waits for LDS
        uint32_t acc = 0, tw[WORDS + 1], rw[WORDS];
#pragma unroll
        for (int j = 0; j <= WORDS; ++j) tw[j] = trow[d + j];
#pragma unroll
        for (int j = 0; j < WORDS; ++j) rw[j] = rrow[j];
        __builtin_amdgcn_sched_barrier(0);
#pragma unroll
        for (int j = 0; j < WORDS; ++j)
            acc = __builtin_amdgcn_udot4(rw[j], __builtin_amdgcn_alignbyte(tw[j + 1], tw[j], sh), acc, false);
        const int I = dpp_sum(FULL || lane < N ? (int)acc : 0);
        if (I > bestI || (I == bestI && k < peak)) {
            bestI = I;
            peak = k;
        }
    }
    return DFT_PEAK;
}

// A workgroup's wavefronts share the DFT tables in LDS; workgroup b takes the
// contiguous POI range [g n / G, (g + 1) n / G) (G workgroups), its wavefronts
// every WAVES-th POI of it.  Workgroups go to the 8 XCDs
// round-robin, so g = (b mod 8) G / 8 + b / 8 when 8 divides G: each XCD
// (and its L2) then covers one contiguous eighth of the POIs, a band of rows.
__device__ __forceinline__ void dft_tables_to_lds(DftWgSmem<4, true>& sm, const float2*, int)
{
    const h8* gb = &g_dft_tab[1][0][0][0][0];
    h8* la = &sm.ta[0][0][0];
    h8* lb = &sm.tb[0][0][0][0];
    for (int i = threadIdx.x; i < 2 * 4 * 64; i += blockDim.x)        // table 0, tile 0, parts re and im
        la[i] = g_dft_tab[0][i >> 8][0][(i >> 6) & 3][i & 63];
    for (int i = threadIdx.x; i < 3 * 2 * 4 * 64; i += blockDim.x) lb[i] = gb[i];
    for (int i = threadIdx.x; i < 2 * 64; i += blockDim.x) sm.tn[i >> 6][i & 63] = g_dft_nyq[i >> 6][i & 63];
    __syncthreads();
}

// N < 64: from the N twiddles exp(-2 pi i e / N), each rounded to fp16, zero
// where a row or column is beyond the window (or, in table 0, beyond the half
// spectrum k <= N / 2).  The upper half of the circle mirrors the lower one,
// so F[-j][y] = conj F[j][y] holds exactly, as the half spectrum needs.  tn:
// the last pass's real part of K chunk 1 with -1 at k = 31 in the rows b >= N.
template <int CH>
__device__ __forceinline__ void dft_tables_to_lds(DftWgSmem<CH, false>& sm, const float2* __restrict__ tw, int N)
{
    const uint32_t inv = (1u << 18) / (uint32_t)N + 1u;       // x / N = (x inv) >> 18 for x < 4096, N <= 64
    auto entry = [&](int row, int col, _Float16& re, _Float16& im) {
        const uint32_t x = (uint32_t)(row * col);
        const int e = (int)(x - ((x * inv) >> 18) * (uint32_t)N);
        const bool up = 2 * e > N;
        const float2 w = tw[up ? N - e : e];
        re = (_Float16)w.x;
        im = (_Float16)(up ? -w.y : w.y);
    };
    _Float16* la = reinterpret_cast<_Float16*>(&sm.ta[0][0][0]);
    _Float16* lb = reinterpret_cast<_Float16*>(&sm.tb[0][0][0][0]);
    _Float16* ln = reinterpret_cast<_Float16*>(&sm.tn[0][0]);
    const _Float16 zero = (_Float16)0.f, down = (_Float16)0.00390625f;
    constexpr int A = CH * 64 * 8, B = 2 * A;                  // entries of one part
    for (int i = threadIdx.x; i < A; i += blockDim.x) {
        const int q = i & 7, lane = (i >> 3) & 63, c = i >> 9;
        const int x = 16 * c + 8 * (lane >> 5) + q, k = lane & 31;
        _Float16 re = zero, im = zero;
        if (x < N && 2 * k <= N) entry(x, k, re, im);
        la[i] = re;
        la[A + i] = im;
    }
    for (int i = threadIdx.x; i < B; i += blockDim.x) {
        const int q = i & 7, lane = (i >> 3) & 63, c = (i >> 9) % CH, tile = (i >> 9) / CH;
        const int row = 32 * tile + (lane & 31), col = 16 * c + 8 * (q >> 2) + 4 * (lane >> 5) + (q & 3);
        _Float16 re = zero, im = zero;
        if (row < N && col < N) entry(row, col, re, im);
        lb[i] = re * down;
        lb[B + i] = im * down;
        lb[2 * B + i] = -im * down;
        if (c == 1) ln[((tile << 6) + lane) * 8 + q] = col == 31 ? (row < N ? zero : (_Float16)-1.f) : re * down;
    }
    __syncthreads();
}

__device__ __forceinline__ int dft_range_index()
{
    const int G = gridDim.x, b = blockIdx.x;
    return (G & 7) == 0 ? (b & 7) * (G >> 3) + (b >> 3) : b;
}

// A wavefront's share of the items [lo, hi): every WAVES-th.  The next item's
// rows are loaded while the current one's candidates are evaluated (of 22,600
// cycles per POI 4,100 went by waiting for its place and rows), and the
// outputs, some 100 FP64 instructions, are formed for KEPT items at a time, a lane
// each, instead of by one lane per item.  With the rows' loads in DftRows:
// 0.81 -> 0.73 ms for 157k POIs at N = 64, 0.53 -> 0.48 ms at N = 40.  src.item(i) is the window pair of item i, src.params(i)
// its outputs, src.poi(i) their index.
template <int CH, bool FULL, class Source>
__device__ __forceinline__ void fftcc_dft_run(DftWgSmem<CH, FULL>& sm, const Source& src, int N, int lo, int hi)
{
    using Sm = DftWgSmem<CH, FULL>;
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), lane = threadIdx.x & 63;
    int (*kept)[Sm::KEPT] = sm.kept[wave];
    int nkept = 0;
    auto flush = [&]() {
        wave_lds_sync();
        if (lane < nkept) {
            const int i = kept[0][lane], I = kept[5][lane], peak = kept[6][lane];
            const double sr = kept[1][lane], st = kept[2][lane], srr = kept[3][lane], stt = kept[4][lane];
            const FftccParams p = src.params(i);
            const int poi = src.poi(i);
            const double NN = (double)(N * N);
            const double nr = srr - sr * sr / NN, nt = stt - st * st / NN;
            int iu = peak & 63, iv = peak >> 6;    // wrapped to the reference's (u, v) (:316-322)
            if (iu > N / 2) iu -= N;
            if (iv > N / 2) iv -= N;
            p.u[poi] = (float)iu;
            p.v[poi] = (float)iv;
            p.zncc[poi] = (float)(((double)I - sr * st / NN) / sqrt(nr * nt));
            if (p.status) p.status[poi] = TWDIC_FFTCC_OK;
        }
        wave_lds_sync();
        nkept = 0;
    };
    auto fail = [&](int i, int status) {
        const FftccParams p = src.params(i);
        if (lane == 0 && p.status) p.status[src.poi(i)] = (uint8_t)status;
    };
    auto keep = [&](int i, const int (&sums)[4], int I, int peak) {
        if (lane == 0) {
            const int v[7] = {i, sums[0], sums[1], sums[2], sums[3], I, peak};
#pragma unroll
            for (int f = 0; f < 7; ++f) kept[f][nkept] = v[f];
        }
        if (++nkept == Sm::KEPT) flush();
    };
    int i = lo + wave, run = 0;
    while (i < hi) {
        DftRows<CH, FULL> rows;
        DftItem cur = src.item(i);
        rows.drop();
        if (cur.inside) rows.load(cur, N, lane);
        int direct = 0;                       // items from i on that are mma_direct's
        for (;;) {
            const int ni = i + Sm::WAVES;
            DftItem nx = cur;
            if (ni < hi) nx = src.item(ni);
            auto next = [&]() {
                rows.drop();
                if (ni < hi && nx.inside) rows.load(nx, N, lane);
            };
            if (cur.inside) {
                int sums[4], many, I, peak;
                const int r = fftcc_dft_mfma_poi<CH, FULL>(sm, wave, lane, N, rows, sums, many, I, peak, next);
                if (r == DFT_PEAK)
                    keep(i, sums, I, peak);
                else if (r == DFT_FLAT)
                    fail(i, TWDIC_FFTCC_FLAT);
                if constexpr (!FULL) {
                    if (2 * many > N) {
                        run = r == DFT_MANY ? kDftDirectRun : min(2 * run + 1, kDftDirectRun);
                        direct = run + (r == DFT_MANY ? 1 : 0);
                        if (r != DFT_MANY) i = ni;
                        break;
                    }
                    run = 0;
                }
            } else {
                next();
                fail(i, TWDIC_FFTCC_OUT);
            }
            i = ni;
            if (i >= hi) break;
            cur = nx;
        }
        if constexpr (!FULL) {
            // in a loop of its own, whose registers the one above does not give up
            for (; direct > 0 && i < hi; --direct, i += Sm::WAVES) {
                int l = lane;
                asm volatile("" : "+v"(l));      // (as that would: nothing that follows from the lane is kept)
                const DftItem it = src.item(i);
                if (!it.inside) {
                    fail(i, TWDIC_FFTCC_OUT);
                    continue;
                }
                rows.drop();
                rows.load(it, N, l);
                int sums[4], I, peak;
                dft_window(sm, wave, l, N, rows, sums);
                if (DftNorms(sums, N * N).flat()) {
                    fail(i, TWDIC_FFTCC_FLAT);
                } else {
                    mma_direct<CH>(sm, wave, l, N, sums, I, peak);
                    keep(i, sums, I, peak);
                }
            }
        }
    }
    flush();
}

struct DftSet {                                    // the POIs of one set
    const FftccParams& p;
    __device__ __forceinline__ DftItem item(int i) const { return dft_item(p, i); }
    __device__ __forceinline__ const FftccParams& params(int) const { return p; }
    __device__ __forceinline__ int poi(int i) const { return i; }
};

struct DftBatch {                                  // items (pair, POI) of a batch
    const PairDesc* pairs;
    const int2* items;
    __device__ __forceinline__ DftItem item(int i) const
    {
        const int2 it = items[i];
        return dft_item(const_pairs(pairs)[__builtin_amdgcn_readfirstlane(it.x)].fftcc,
                        __builtin_amdgcn_readfirstlane(it.y));
    }
    __device__ __forceinline__ FftccParams params(int i) const { return const_pairs(pairs)[items[i].x].fftcc; }
    __device__ __forceinline__ int poi(int i) const { return items[i].y; }
};

template <int CH, bool FULL>
__global__ __launch_bounds__((64 * DftWgSmem<CH, FULL>::WAVES), 1) void k_fftcc_dft_mfma(FftccParams p)
{
    __shared__ DftWgSmem<CH, FULL> sm;
    dft_tables_to_lds(sm, p.tw, p.N);
    const int g = dft_range_index();
    const int lo = (int)((long long)g * p.n / gridDim.x);
    const int hi = (int)((long long)(g + 1) * p.n / gridDim.x);
    fftcc_dft_run<CH, FULL>(sm, DftSet{p}, FULL ? 64 : p.N, lo, hi);
}

// Batched form over items (pair, POI) of pairs that share N: the same ranges
// per workgroup, each item with its pair's descriptor.
template <int CH, bool FULL>
__global__ __launch_bounds__((64 * DftWgSmem<CH, FULL>::WAVES), 1) void k_batch_fftcc_dft_mfma(
    const PairDesc* __restrict__ pairs, const int2* __restrict__ items, int count)
{
    __shared__ DftWgSmem<CH, FULL> sm;
    const FftccParams p = const_pairs(pairs)[__builtin_amdgcn_readfirstlane(items[0].x)].fftcc;
    dft_tables_to_lds(sm, p.tw, p.N);
    const int g = dft_range_index();
    const int lo = (int)((long long)g * count / gridDim.x);
    const int hi = (int)((long long)(g + 1) * count / gridDim.x);
    fftcc_dft_run<CH, FULL>(sm, DftBatch{pairs, items}, FULL ? 64 : p.N, lo, hi);
}

// workgroups for n POIs: one per compute unit (each holds one), fewer for
// small n
int dft_blocks(int n, int waves)
{
    int dev = 0;
    (void)hipGetDevice(&dev);
    const int cus = dev >= 0 && dev < 64 && g_dft_cus[dev] > 0 ? g_dft_cus[dev] : 256;
    return std::max(1, std::min(cus, (n + waves - 1) / waves));
}

template <int CH, bool FULL>
void launch_dft(const FftccParams& p, hipStream_t st)
{
    constexpr int W = DftWgSmem<CH, FULL>::WAVES;
    hipLaunchKernelGGL((k_fftcc_dft_mfma<CH, FULL>), dim3(dft_blocks(p.n, W)), dim3(64 * W), 0, st, p);
}

template <int CH, bool FULL>
void launch_batch_dft(const PairDesc* pairs, const int2* items, int count, hipStream_t st)
{
    constexpr int W = DftWgSmem<CH, FULL>::WAVES;
    hipLaunchKernelGGL((k_batch_fftcc_dft_mfma<CH, FULL>), dim3(dft_blocks(count, W)), dim3(64 * W), 0, st, pairs, items,
                       count);
}

}  // namespace

hipError_t launch_batch_fftcc_mma(const PairDesc* pairs, const int2* items, int count, int N, bool dft,
                                  hipStream_t st)
{
    if (count <= 0) return hipSuccess;
    if (dft && N == 64)
        launch_batch_dft<4, true>(pairs, items, count, st);
    else if (dft && N > 48)
        launch_batch_dft<4, false>(pairs, items, count, st);
    else if (dft)
        launch_batch_dft<3, false>(pairs, items, count, st);
    else if (N > 48)
        hipLaunchKernelGGL((k_batch_fftcc_mma<64, false, 32>), dim3(count), dim3(64), 0, st, pairs, items);
    else if (N > 32)
        hipLaunchKernelGGL((k_batch_fftcc_mma<64, false, 16>), dim3(count), dim3(64), 0, st, pairs, items);
    else
        hipLaunchKernelGGL((k_batch_fftcc_mma<32, false, 32>), dim3(count), dim3(64), 0, st, pairs, items);
    return hipGetLastError();
}

hipError_t launch_fftcc(const FftccParams& p, int variant, hipStream_t st)
{
    if (p.n <= 0) return hipSuccess;
    const int pairs = (p.n + 1) / 2;
    if (variant == kFftccDftMfma && dft_takes(p.N, p.n)) {
        if (p.N == 64)
            launch_dft<4, true>(p, st);
        else if (p.N > 48)
            launch_dft<4, false>(p, st);
        else
            launch_dft<3, false>(p, st);
    } else if (variant == kFftccMma || variant == kFftccDftMfma) {
        if (p.N == 64)
            hipLaunchKernelGGL((k_fftcc_mma<64, true, 32>), dim3(p.n), dim3(64), 0, st, p);
        else if (p.N > 48)
            hipLaunchKernelGGL((k_fftcc_mma<64, false, 32>), dim3(p.n), dim3(64), 0, st, p);
        else if (p.N > 32)
            hipLaunchKernelGGL((k_fftcc_mma<64, false, 16>), dim3(p.n), dim3(64), 0, st, p);
        else
            hipLaunchKernelGGL((k_fftcc_mma<32, false, 32>), dim3(p.n), dim3(64), 0, st, p);
    } else if (p.N == 64) {
        if (variant == 3)
            hipLaunchKernelGGL((k_fftcc_fft<16, 3>), dim3(pairs), dim3(256), 0, st, p);
        else if (variant == 4)
            hipLaunchKernelGGL((k_fftcc_fft<16, 4>), dim3(pairs), dim3(256), 0, st, p);
        else
            hipLaunchKernelGGL((k_fftcc_fft<16, 2>), dim3(pairs), dim3(256), 0, st, p);
    } else if (p.N == 32) {
        hipLaunchKernelGGL((k_fftcc_fft<8, 4>), dim3(pairs), dim3(128), 0, st, p);
    } else
        hipLaunchKernelGGL(k_fftcc_dft, dim3(p.n), dim3(kDftThreads), 0, st, p);
    return hipGetLastError();
}

hipError_t launch_batch_fftcc(const PairDesc* pairs, const int2* items, int total, int* counter, int N, int variant,
                              int blocks, hipStream_t st)
{
    if (total <= 0) return hipSuccess;
    if (N == 64) {
        if (variant == 2)
            hipLaunchKernelGGL((k_batch_fftcc<16, 2>), dim3(blocks), dim3(256), 0, st, pairs, items, total, counter);
        else if (variant == 4)
            hipLaunchKernelGGL((k_batch_fftcc<16, 4>), dim3(blocks), dim3(256), 0, st, pairs, items, total, counter);
        else
            hipLaunchKernelGGL((k_batch_fftcc<16, 3>), dim3(blocks), dim3(256), 0, st, pairs, items, total, counter);
    } else if (N == 32) {
        hipLaunchKernelGGL((k_batch_fftcc<8, 4>), dim3(blocks), dim3(128), 0, st, pairs, items, total, counter);
    } else {
        hipLaunchKernelGGL(k_batch_fftcc_dft, dim3(blocks), dim3(kDftThreads), 0, st, pairs, items, total, counter);
    }
    return hipGetLastError();
}

int persistent_blocks_fftcc(int device, int N, int variant)
{
    int cus = 0, per = 0;
    (void)hipDeviceGetAttribute(&cus, hipDeviceAttributeMultiprocessorCount, device);
    hipError_t e;
    if (N == 64)
        e = variant == 2 ? hipOccupancyMaxActiveBlocksPerMultiprocessor(&per, k_batch_fftcc<16, 2>, 256, 0)
            : variant == 4 ? hipOccupancyMaxActiveBlocksPerMultiprocessor(&per, k_batch_fftcc<16, 4>, 256, 0)
                           : hipOccupancyMaxActiveBlocksPerMultiprocessor(&per, k_batch_fftcc<16, 3>, 256, 0);
    else if (N == 32)
        e = hipOccupancyMaxActiveBlocksPerMultiprocessor(&per, k_batch_fftcc<8, 4>, 128, 0);
    else
        e = hipOccupancyMaxActiveBlocksPerMultiprocessor(&per, k_batch_fftcc_dft, kDftThreads, 0);
    if (e != hipSuccess || per < 1) per = 1;
    return (cus > 0 ? cus : 256) * per;
}

hipError_t dft_tables_init(int device)
{
    static std::mutex mu;
    static bool done[64] = {};
    if (device < 0 || device >= 64) return hipErrorInvalidDevice;
    std::lock_guard<std::mutex> lk(mu);
    if (done[device]) return hipSuccess;
    static _Float16 host[2][3][2][4][64][8];
    for (int t = 0; t < 2; ++t)
        for (int tile = 0; tile < 2; ++tile)
            for (int c = 0; c < 4; ++c)
                for (int lane = 0; lane < 64; ++lane)
                    for (int q = 0; q < 8; ++q) {
                        const int m = lane & 31, h = lane >> 5;
                        const int row = t == 0 ? 16 * c + 8 * h + q : 32 * tile + m;
                        const int col = t == 0 ? 32 * tile + m : 16 * c + 8 * (q / 4) + 4 * h + q % 4;
                        const double ang = -2.0 * M_PI * (double)((row * col) & 63) / 64.0;
                        // direct double -> fp16, nearest-even; table 1 then times 2^-8 (exact:
                        // its non-zero entries stay normal)
                        const double sc = t == 0 ? 1.0 : 1.0 / 256.0;
                        host[t][0][tile][c][lane][q] = (_Float16)((double)(_Float16)std::cos(ang) * sc);
                        host[t][1][tile][c][lane][q] = (_Float16)((double)(_Float16)std::sin(ang) * sc);
                        if (t == 0 && tile == 0 && m == 0)                        // (-1)^x: Y[.][32]
                            host[t][1][tile][c][lane][q] = (_Float16)(((16 * c + 8 * h + q) & 1) ? -1.0 : 1.0);
                        host[t][2][tile][c][lane][q] = -host[t][1][tile][c][lane][q];
                    }
    static _Float16 nyq[2][64][8];
    for (int tile = 0; tile < 2; ++tile)
        for (int lane = 0; lane < 64; ++lane)
            for (int q = 0; q < 8; ++q) {
                nyq[tile][lane][q] = host[1][1][tile][0][lane][q];
                if ((lane >> 5) == 0 && q == 0)                                   // K index 0: b = 32 tile + m
                    nyq[tile][lane][q] = (_Float16)((lane & 1) ? -1.0 / 256.0 : 1.0 / 256.0);
            }
    int cur = 0;
    hipError_t e = hipGetDevice(&cur);
    if (e == hipSuccess) e = hipDeviceGetAttribute(&g_dft_cus[device], hipDeviceAttributeMultiprocessorCount, device);
    if (e == hipSuccess) e = hipSetDevice(device);
    if (e == hipSuccess) e = hipMemcpyToSymbol(HIP_SYMBOL(g_dft_tab), host, sizeof(host));
    if (e == hipSuccess) e = hipMemcpyToSymbol(HIP_SYMBOL(g_dft_nyq), nyq, sizeof(nyq));
    if (e == hipSuccess) e = hipSetDevice(cur);
    if (e == hipSuccess) done[device] = true;
    return e;
}

hipError_t launch_fftcc_generic(const FftccParams& p, hipStream_t st)
{
    if (p.n <= 0) return hipSuccess;
    hipLaunchKernelGGL(k_fftcc_dft, dim3(p.n), dim3(kDftThreads), 0, st, p);
    return hipGetLastError();
}

}  // namespace twdic
