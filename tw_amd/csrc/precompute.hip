// precompute.hip -- POI grid, central-difference gradients, bicubic LUT and
// the per-reference IC-GN state (FP64 Hessian + Cholesky), for gfx950.
//
// All gradient and LUT values are exact in FP32 (half/quarter integers and
// sums of at most 16 integer multiples of them, below 2^14), so these kernels
// are bit-identical to the CPU path in any summation order.
#include "twdic_internal.h"

#include <algorithm>
#include <cfloat>

namespace twdic {

// ---------------------------------------------------------------------------
// POI grid: TW_utils.cpp:29-49 / TW_cuUtils.cu:116-134 (y first).
// ---------------------------------------------------------------------------
__global__ void k_poi_grid(int32_t* poi, int start_x, int start_y, int nx, int ny, int mx, int my,
                           int sx, int sy, int gx, int gy)
{
    int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= nx * ny) return;
    int iy = i / nx, ix = i - iy * nx;
    int2 yx = make_int2(start_y + my + sy + iy * gy, start_x + mx + sx + ix * gx);
    reinterpret_cast<int2*>(poi)[i] = yx;
}

hipError_t launch_poi_grid(int32_t* poi, int start_x, int start_y, int nx, int ny, int mx, int my,
                           int sx, int sy, int gx, int gy, hipStream_t st)
{
    int n = nx * ny;
    hipLaunchKernelGGL(k_poi_grid, dim3((n + 255) / 256), dim3(256), 0, st, poi, start_x, start_y,
                       nx, ny, mx, my, sx, sy, gx, gy);
    return hipGetLastError();
}

// ---------------------------------------------------------------------------
// Gradients: GradientXY_2Images_s (TW_utils.cpp:260-273), one image.
// Thread per pixel, x fastest; stores are fully coalesced.  g2 (optional)
// receives the doubled gradients (2 Gx, 2 Gy) as a packed int16 pair, the
// 4-byte-per-pixel form the IC-GN kernels read.
// ---------------------------------------------------------------------------
__global__ __launch_bounds__(256) void k_gradients(const uint8_t* __restrict__ img, int stride,
                                                   int sx0, int sy0, int rw, int rh,
                                                   float* __restrict__ gx, float* __restrict__ gy,
                                                   float* __restrict__ gxy, uint32_t* __restrict__ g2)
{
    int x = blockIdx.x * 64 + (threadIdx.x & 63);
    int y = blockIdx.y * 4 + (threadIdx.x >> 6);
    if (x >= rw || y >= rh) return;
    const uint8_t* c = img + (size_t)(y + sy0) * stride + (x + sx0);
    int l = c[-1], r = c[1], u = c[-stride], d = c[stride];
    size_t o = (size_t)y * rw + x;
    if (gx) gx[o] = 0.5f * (float)(r - l);
    if (gy) gy[o] = 0.5f * (float)(d - u);
    if (g2) g2[o] = (uint32_t)(uint16_t)(int16_t)(r - l) | ((uint32_t)(uint16_t)(int16_t)(d - u) << 16);
    if (gxy) {
        int ur = c[-stride + 1], ul = c[-stride - 1], dr = c[stride + 1], dl = c[stride - 1];
        gxy[o] = 0.25f * (float)(dr - ur - dl + ul);
    }
}

hipError_t launch_gradients(const uint8_t* img, int stride, int sx0, int sy0, int rw, int rh,
                            float* gx, float* gy, float* gxy, uint32_t* g2, hipStream_t st)
{
    dim3 grid((rw + 63) / 64, (rh + 3) / 4);
    hipLaunchKernelGGL(k_gradients, grid, dim3(256), 0, st, img, stride, sx0, sy0, rw, rh, gx, gy, gxy, g2);
    return hipGetLastError();
}

// ---------------------------------------------------------------------------
// Cubic B-spline LUT: BicubicSplineCoefficients_s (TW_utils.cpp:521-602).
// From the 4x4 neighbourhood Om (rows y-1..y+2, columns x-1..x+2):
// beta = CP Om^T CP^T with the local prefilter CP, then B beta^T B^T with the
// B-spline basis B, rotated by 180 degrees.  FP32, every product and sum
// rounded separately in the reference's order.  Every ROI pixel gets
// coefficients (the caller guarantees a 2-pixel frame right and below).
// PLANES: the y^k coefficients of all cells in plane k (float4[4][rh][rw])
// instead of 16 floats per cell.
// ---------------------------------------------------------------------------
namespace {
__device__ __forceinline__ float bsp_cp(int k, int l)
{
    constexpr float t[4][4] = {{(float)(71 / 56.0), (float)(-19 / 56.0), (float)(5 / 56.0), (float)(-1 / 56.0)},
                               {(float)(-19 / 56.0), (float)(95 / 56.0), (float)(-25 / 56.0), (float)(5 / 56.0)},
                               {(float)(5 / 56.0), (float)(-25 / 56.0), (float)(95 / 56.0), (float)(-19 / 56.0)},
                               {(float)(-1 / 56.0), (float)(5 / 56.0), (float)(-19 / 56.0), (float)(71 / 56.0)}};
    return t[k][l];
}
__device__ __forceinline__ float bsp_base(int k, int l)
{
    constexpr float t[4][4] = {{(float)(-1 / 6.0), (float)(3 / 6.0), (float)(-3 / 6.0), (float)(1 / 6.0)},
                               {(float)(3 / 6.0), (float)(-6 / 6.0), (float)(3 / 6.0), 0.f},
                               {(float)(-3 / 6.0), 0.f, (float)(3 / 6.0), 0.f},
                               {(float)(1 / 6.0), (float)(4 / 6.0), (float)(1 / 6.0), 0.f}};
    return t[k][l];
}
}  // namespace

template <bool PLANES>
__global__ __launch_bounds__(256) void k_bspline_lut(const uint8_t* __restrict__ img, int stride, int sx0, int sy0,
                                                     int rw, int rh, float* __restrict__ lut)
{
#pragma clang fp contract(off)
    const int x = blockIdx.x * 64 + (threadIdx.x & 63);
    const int y = blockIdx.y * 4 + (threadIdx.x >> 6);
    if (x >= rw || y >= rh) return;
    float om[4][4], beta[4][4], c[4][4];
#pragma unroll
    for (int k = 0; k < 4; ++k)
#pragma unroll
        for (int l = 0; l < 4; ++l)
            om[k][l] = (float)img[(size_t)(y + sy0 - 1 + k) * stride + (x + sx0 - 1 + l)];
#pragma unroll
    for (int k = 0; k < 4; ++k)
#pragma unroll
        for (int l = 0; l < 4; ++l) {
            float b = 0.f;
#pragma unroll
            for (int m = 0; m < 4; ++m)
#pragma unroll
                for (int n = 0; n < 4; ++n) b = b + bsp_cp(k, m) * bsp_cp(l, n) * om[n][m];
            beta[k][l] = b;
        }
#pragma unroll
    for (int k = 0; k < 4; ++k)
#pragma unroll
        for (int l = 0; l < 4; ++l) {
            float a = 0.f;
#pragma unroll
            for (int m = 0; m < 4; ++m)
#pragma unroll
                for (int n = 0; n < 4; ++n) a = a + bsp_base(k, m) * bsp_base(l, n) * beta[n][m];
            c[k][l] = a;
        }
    const size_t cell = (size_t)y * rw + x, at = PLANES ? cell : 4 * cell, step = PLANES ? (size_t)rw * rh : 1;
    float4* out = reinterpret_cast<float4*>(lut);
#pragma unroll
    for (int k = 0; k < 4; ++k)      // rotated by 180 degrees (:591-599)
        out[at + k * step] = make_float4(c[3 - k][3], c[3 - k][2], c[3 - k][1], c[3 - k][0]);
}

hipError_t launch_bspline_lut(const uint8_t* tar, int stride, int sx0, int sy0, int rw, int rh, float* lut,
                              hipStream_t st)
{
    dim3 grid((rw + 63) / 64, (rh + 3) / 4);
    hipLaunchKernelGGL(k_bspline_lut<false>, grid, dim3(256), 0, st, tar, stride, sx0, sy0, rw, rh, lut);
    return hipGetLastError();
}

hipError_t launch_bspline_planes(const uint8_t* tar, int stride, int sx0, int sy0, int rw, int rh, float4* planes,
                                 hipStream_t st)
{
    dim3 grid((rw + 63) / 64, (rh + 3) / 4);
    hipLaunchKernelGGL(k_bspline_lut<true>, grid, dim3(256), 0, st, tar, stride, sx0, sy0, rw, rh,
                       reinterpret_cast<float*>(planes));
    return hipGetLastError();
}

// ---------------------------------------------------------------------------
// Bicubic LUT: BicubicCoefficients_s (TW_utils.cpp:604-700), fused with the
// target gradients: tau (corner values, x/y/xy central differences) is built
// straight from the 4x4 pixel neighbourhood, alpha = M tau with the standard
// bicubic matrix (TW_utils.cpp:622-638) expanded by hand.  Layout per pixel:
// 16 contiguous floats, element 4k+l multiplies y^k x^l.  The last ROI row and
// column are written as zeros (the CPU buffer is calloc-zeroed there).
// ---------------------------------------------------------------------------
__global__ __launch_bounds__(256) void k_bicubic_lut(const uint8_t* __restrict__ tar, int stride,
                                                     int sx0, int sy0, int rw, int rh,
                                                     float* __restrict__ lut)
{
    int x = blockIdx.x * 64 + (threadIdx.x & 63);
    int y = blockIdx.y * 4 + (threadIdx.x >> 6);
    if (x >= rw || y >= rh) return;
    float4* out = reinterpret_cast<float4*>(lut + ((size_t)y * rw + x) * 16);
    if (x == rw - 1 || y == rh - 1) {
        float4 z = make_float4(0.f, 0.f, 0.f, 0.f);
        out[0] = z; out[1] = z; out[2] = z; out[3] = z;
        return;
    }
    // p[r][c] = T(y0 - 1 + r, x0 - 1 + c), r,c in 0..3
    const uint8_t* b = tar + (size_t)(y + sy0 - 1) * stride + (x + sx0 - 1);
    float p[4][4];
#pragma unroll
    for (int r = 0; r < 4; ++r)
#pragma unroll
        for (int c = 0; c < 4; ++c) p[r][c] = (float)b[r * stride + c];
    // corner values f, x/y derivatives, cross derivatives (TW_utils.cpp:265-271)
    float f00 = p[1][1], f10 = p[1][2], f01 = p[2][1], f11 = p[2][2];
    float x00 = 0.5f * (p[1][2] - p[1][0]), x10 = 0.5f * (p[1][3] - p[1][1]);
    float x01 = 0.5f * (p[2][2] - p[2][0]), x11 = 0.5f * (p[2][3] - p[2][1]);
    float y00 = 0.5f * (p[2][1] - p[0][1]), y10 = 0.5f * (p[2][2] - p[0][2]);
    float y01 = 0.5f * (p[3][1] - p[1][1]), y11 = 0.5f * (p[3][2] - p[1][2]);
    float c00 = 0.25f * (p[2][2] - p[0][2] - p[2][0] + p[0][0]);
    float c10 = 0.25f * (p[2][3] - p[0][3] - p[2][1] + p[0][1]);
    float c01 = 0.25f * (p[3][2] - p[1][2] - p[3][0] + p[1][0]);
    float c11 = 0.25f * (p[3][3] - p[1][3] - p[3][1] + p[1][1]);
    // tau = [f00 f10 f01 f11 | x00 x10 x01 x11 | y00 y10 y01 y11 | c00 c10 c01 c11]
    float a[16];
    a[0] = f00;
    a[1] = x00;
    a[2] = -3.f * f00 + 3.f * f10 - 2.f * x00 - x10;
    a[3] = 2.f * f00 - 2.f * f10 + x00 + x10;
    a[4] = y00;
    a[5] = c00;
    a[6] = -3.f * y00 + 3.f * y10 - 2.f * c00 - c10;
    a[7] = 2.f * y00 - 2.f * y10 + c00 + c10;
    a[8] = -3.f * f00 + 3.f * f01 - 2.f * y00 - y01;
    a[9] = -3.f * x00 + 3.f * x01 - 2.f * c00 - c01;
    a[10] = 9.f * f00 - 9.f * f10 - 9.f * f01 + 9.f * f11 + 6.f * x00 + 3.f * x10 - 6.f * x01 - 3.f * x11
          + 6.f * y00 - 6.f * y10 + 3.f * y01 - 3.f * y11 + 4.f * c00 + 2.f * c10 + 2.f * c01 + c11;
    a[11] = -6.f * f00 + 6.f * f10 + 6.f * f01 - 6.f * f11 - 3.f * x00 - 3.f * x10 + 3.f * x01 + 3.f * x11
          - 4.f * y00 + 4.f * y10 - 2.f * y01 + 2.f * y11 - 2.f * c00 - 2.f * c10 - c01 - c11;
    a[12] = 2.f * f00 - 2.f * f01 + y00 + y01;
    a[13] = 2.f * x00 - 2.f * x01 + c00 + c01;
    a[14] = -6.f * f00 + 6.f * f10 + 6.f * f01 - 6.f * f11 - 4.f * x00 - 2.f * x10 + 4.f * x01 + 2.f * x11
          - 3.f * y00 + 3.f * y10 - 3.f * y01 + 3.f * y11 - 2.f * c00 - c10 - 2.f * c01 - c11;
    a[15] = 4.f * f00 - 4.f * f10 - 4.f * f01 + 4.f * f11 + 2.f * x00 + 2.f * x10 - 2.f * x01 - 2.f * x11
          + 2.f * y00 - 2.f * y10 + 2.f * y01 - 2.f * y11 + c00 + c10 + c01 + c11;
    out[0] = make_float4(a[0], a[1], a[2], a[3]);
    out[1] = make_float4(a[4], a[5], a[6], a[7]);
    out[2] = make_float4(a[8], a[9], a[10], a[11]);
    out[3] = make_float4(a[12], a[13], a[14], a[15]);
}

hipError_t launch_bicubic_lut(const uint8_t* tar, int stride, int sx0, int sy0, int rw, int rh,
                              float* lut, hipStream_t st)
{
    dim3 grid((rw + 63) / 64, (rh + 3) / 4);
    hipLaunchKernelGGL(k_bicubic_lut, grid, dim3(256), 0, st, tar, stride, sx0, sy0, rw, rh, lut);
    return hipGetLastError();
}

// ---------------------------------------------------------------------------
// Row polynomials of the target for the fused bicubic interpolation.  The
// bicubic LUT above, built from central-difference corner derivatives, is the
// tensor-product Catmull-Rom spline; along one image row y, between pixels x
// and x + 1, its cubic through p0..p3 = T(y, x-1 .. x+2) is
//   R(t) = c0 + t/2 (c1 + t (c2 + t c3)),
//   c0 = p1, c1 = p2 - p0, c2 = 2 p0 - 5 p1 + 4 p2 - p3, c3 = 3 (p1 - p2) + p3 - p0,
// integers of magnitude at most 1530.  Stored as c0, c1/2, c2/2, c3/2 in fp16
// (exactly), the cubic is c0 + t (c1/2 + t (c2/2 + t c3/2)).  Entry (x, j) holds
// the coefficients (8 bytes each) of rows y = sy0 - 1 + j and y + 1 for cell column
// sx0 + x, x < rw, j <= rh; the last column (never an interior cell) is
// zero.  A cell's four neighbourhood rows are the entries (x, j) and (x, j + 2).
// ---------------------------------------------------------------------------
typedef _Float16 h8 __attribute__((ext_vector_type(8)));

// Entry (x, j) from the target rows' dwords at columns sx0 + x - 1 ..
// sx0 + x + 2: for x < rw - 1 it lies in the image (the ROI keeps a one-pixel
// frame); the buffer's range check would read anything past its last row as
// zero.  The target resource's base is the image, records (sy0 + rh + 1) rows.
__device__ __forceinline__ void row_poly_entry(__amdgpu_buffer_rsrc_t img, int stride, int sx0, int sy0, int rw,
                                               int x, int j, float4* __restrict__ rp)
{
    h8 e = {};
    if (x < rw - 1) {
        const int o = (sy0 - 1 + j) * stride + (sx0 - 1 + x);
#pragma unroll
        for (int r = 0; r < 2; ++r) {
            const uint32_t w = __builtin_amdgcn_raw_buffer_load_b32(img, o, r * stride, 0);
            const int p0 = (int)(w & 255u), p1 = (int)((w >> 8) & 255u), p2 = (int)((w >> 16) & 255u), p3 = (int)(w >> 24);
            e[4 * r] = (_Float16)(float)p1;
            e[4 * r + 1] = (_Float16)(0.5f * (float)(p2 - p0));
            e[4 * r + 2] = (_Float16)(0.5f * (float)(2 * p0 - 5 * p1 + 4 * p2 - p3));
            e[4 * r + 3] = (_Float16)(0.5f * (float)(3 * (p1 - p2) + p3 - p0));
        }
    }
    rp[(size_t)j * rw + x] = __builtin_bit_cast(float4, e);
}

__device__ __forceinline__ __amdgpu_buffer_rsrc_t row_poly_src(const uint8_t* tar, int stride, int sy0, int rh)
{
    return __builtin_amdgcn_make_buffer_rsrc((void*)tar, (short)0, (sy0 + rh + 1) * stride, 0x00020000);
}

// One entry per thread: x along the block's 256 threads and blockIdx.x, rows
// j = blockIdx.y, + gridDim.y, ...
__global__ __launch_bounds__(256) void k_row_poly(const uint8_t* __restrict__ tar, int stride, int sx0, int sy0,
                                                  int rw, int rh, float4* __restrict__ rp)
{
    const __amdgpu_buffer_rsrc_t img = row_poly_src(tar, stride, sy0, rh);
    const int x = blockIdx.x * 256 + threadIdx.x;
    if (x >= rw) return;
    for (int j = blockIdx.y; j <= rh; j += gridDim.y) row_poly_entry(img, stride, sx0, sy0, rw, x, j, rp);
}

hipError_t launch_row_poly(const uint8_t* tar, int stride, int sx0, int sy0, int rw, int rh, float4* rp,
                           hipStream_t st)
{
    const dim3 grid((rw + 255) / 256, std::min(rh + 1, 65535));
    hipLaunchKernelGGL(k_row_poly, grid, dim3(256), 0, st, tar, stride, sx0, sy0, rw, rh, rp);
    return hipGetLastError();
}

// Batched form: blockIdx.y is the pair; geometry and buffers come from its
// descriptor (read when the kernel runs, so a captured graph follows new
// targets).  Rows j = blockIdx.x, + gridDim.x, ..., the block's threads along
// x.  Pairs without a plane (rp null) are skipped.
__global__ __launch_bounds__(256) void k_batch_row_poly(const PairDesc* __restrict__ pairs)
{
    const IcgnParams P = const_pairs(pairs)[blockIdx.y].icgn;
    if (P.rp == nullptr) return;
    const __amdgpu_buffer_rsrc_t img = row_poly_src(P.tar, P.stride, P.sy0, P.rh);
    for (int j = blockIdx.x; j <= P.rh; j += gridDim.x)
        for (int x = threadIdx.x; x < P.rw; x += 256)
            row_poly_entry(img, P.stride, P.sx0, P.sy0, P.rw, x, j, const_cast<float4*>(P.rp));
}

hipError_t launch_batch_row_poly(const PairDesc* pairs, int npairs, int max_rh, hipStream_t st)
{
    if (npairs <= 0) return hipSuccess;
    const int blocks = std::max(1, std::min(max_rh + 1, 1024));
    hipLaunchKernelGGL(k_batch_row_poly, dim3(blocks, npairs), dim3(256), 0, st, pairs);
    return hipGetLastError();
}

// ---------------------------------------------------------------------------
// The LUT from the layouts IC-GN reads instead of it, once per context: when the
// LUT is handed out, its cells must be those of the target IC-GN last ran on,
// which the image buffer need no longer hold.  Once: a launch recorded into a
// graph does nothing where another has done it (done).  Bound by the 64 bytes
// written per cell.
// ---------------------------------------------------------------------------

// a[k][l], the coefficient of y^k x^l, is a small-integer combination of the row
// coefficients, exact in FP32 (multiples of 1/4 below 2^14), as k_bicubic_lut's
// sums are, so the two write the same numbers.
__global__ __launch_bounds__(256) void k_lut_of_rows(const float4* __restrict__ rp, int rw, int rh,
                                                     float4* __restrict__ lut, const int* done)
{
    if (*done) return;
    const int x = blockIdx.x * 64 + (threadIdx.x & 63), y = blockIdx.y * 4 + (threadIdx.x >> 6);
    if (x >= rw || y >= rh) return;
    float a[4][4] = {};
    if (x < rw - 1 && y < rh - 1) {               // the last row and column are zero
        // rows y - 1, y and y + 1, y + 2
        const h8 e0 = __builtin_bit_cast(h8, rp[(size_t)y * rw + x]);
        const h8 e2 = __builtin_bit_cast(h8, rp[(size_t)(y + 2) * rw + x]);
#pragma unroll
        for (int l = 0; l < 4; ++l) {
            const float q0 = (float)e0[l], q1 = (float)e0[4 + l], q2 = (float)e2[l], q3 = (float)e2[4 + l];
            a[0][l] = q1;
            a[1][l] = 0.5f * (q2 - q0);
            a[2][l] = 0.5f * (2.f * q0 - 5.f * q1 + 4.f * q2 - q3);
            a[3][l] = 0.5f * (3.f * (q1 - q2) + (q3 - q0));
        }
    }
    float4* out = lut + 4 * ((size_t)y * rw + x);
#pragma unroll
    for (int k = 0; k < 4; ++k) out[k] = make_float4(a[k][0], a[k][1], a[k][2], a[k][3]);
}

__global__ __launch_bounds__(256) void k_lut_of_planes(const float4* __restrict__ planes, int rw, int rh,
                                                       float4* __restrict__ lut, const int* done)
{
    if (*done) return;
    const int x = blockIdx.x * 64 + (threadIdx.x & 63), y = blockIdx.y * 4 + (threadIdx.x >> 6);
    if (x >= rw || y >= rh) return;
    const size_t cell = (size_t)y * rw + x, cells = (size_t)rw * rh;
#pragma unroll
    for (int k = 0; k < 4; ++k) lut[4 * cell + k] = planes[k * cells + cell];
}

__global__ void k_set(int* flag) { *flag = 1; }

hipError_t launch_lut_of_rows(const float4* rp, int rw, int rh, float* lut, int* done, hipStream_t st)
{
    hipLaunchKernelGGL(k_lut_of_rows, dim3((rw + 63) / 64, (rh + 3) / 4), dim3(256), 0, st, rp, rw, rh,
                       reinterpret_cast<float4*>(lut), done);
    hipLaunchKernelGGL(k_set, dim3(1), dim3(1), 0, st, done);
    return hipGetLastError();
}

hipError_t launch_lut_of_planes(const float4* planes, int rw, int rh, float* lut, int* done, hipStream_t st)
{
    hipLaunchKernelGGL(k_lut_of_planes, dim3((rw + 63) / 64, (rh + 3) / 4), dim3(256), 0, st, planes, rw, rh,
                       reinterpret_cast<float4*>(lut), done);
    hipLaunchKernelGGL(k_set, dim3(1), dim3(1), 0, st, done);
    return hipGetLastError();
}

// ---------------------------------------------------------------------------
// Per-reference state, one POI per group of L lanes (a wavefront, or a
// half-wavefront for large POI sets; built once per reference and POI set; the
// reference rebuilds it on m_isRefImgUpdated, TW_paDIC_cuICGN2D.cu:883-903).
// Sums follow ICGN2D_Compute's precompute (TW_paDIC_ICGN2D_CPU.cpp:516-595):
// SD = [Rx, Rx dx, Rx dy, Ry, Ry dx, Ry dy], H = sum SD^T SD.  With g = 2R the
// 35 sums are 32 moments of eight integers per pixel (gx^2, gx gy, gy^2 with
// 1, dx, dy, dx^2, dx dy, dy^2; gx, gy, gx R, gy R with 1, dx, dy; R, R^2),
// exact however they are added up.  The Cholesky factorisation is FP64.
//
// Each lane walks down columns (StripPlan), so dx is constant and the dy
// moments come from running sums (summation by parts, twice for dy^2): 19
// integer accumulators and 21 integer instructions per pixel, where the sums
// in FP64 took 35 accumulators and about 50.  A row range of at most kRefRows
// rows keeps the largest, sum sum sum gx^2, below 2^31; the ranges' moments
// are added in FP64, integers below 2^53.  The lanes' moments are then added
// through LDS, eight at a time, each lane taking one moment of eight lanes; and
// a workgroup's factorisations run side by side, one per lane, instead of once
// in every lane of a POI's group.  157,609 POIs of 41x41: 0.79 ms with FP64 sums
// per pixel and butterflies, 0.26 ms so (47k POIs 0.24 and 0.09 ms); bound by VALU
// issue.  Two rows per trip instead of four: 0.305 ms, eight 0.255 ms.
// ---------------------------------------------------------------------------
namespace {

// the moments' places in a POI's slot: 0, 6, 12 the six of gx^2, gx gy, gy^2;
// 18, 21, 24, 27 the three of gx, gy, gx R, gy R; 30, 31 R and R^2
enum { M_XX = 0, M_XY = 6, M_YY = 12, M_X = 18, M_Y = 21, M_XR = 24, M_YR = 27, M_R = 30, M_RR = 31, kMoments = 32 };
constexpr int kMomentSlot = kRefStateUsed + 1;      // odd: the factorising lanes' reads fall on distinct banks

// true when the subset at (px, py) leaves the ROI
__device__ __forceinline__ bool subset_outside(const IcgnParams& P, int px, int py)
{
    return px - P.Sx < P.sx0 || py - P.Sy < P.sy0 || px + P.Sx >= P.sx0 + P.rw || py + P.Sy >= P.sy0 + P.rh;
}

// The moments of the POI at (px, py), whose subset lies in the ROI, by the L
// lanes of its group (hl = lane % L).  red: the group's own LDS.
template <int L>
__device__ __forceinline__ void ref_moments(const IcgnParams& P, int nstrips, int px, int py, int hl, const StripLane* tab,
                                            double (*red)[L + 1], double* mom)
{
    const __amdgpu_buffer_rsrc_t imgr =
        __builtin_amdgcn_make_buffer_rsrc((void*)P.ref, (short)0, P.stride * (P.sy0 + P.rh), 0x00020000);
    const __amdgpu_buffer_rsrc_t g2r =
        __builtin_amdgcn_make_buffer_rsrc((void*)P.g2, (short)0, (int)(4u * (uint32_t)P.rw * (uint32_t)P.rh),
                                          0x00020000);
    const uint32_t gcorner = 4u * (uint32_t)((py - P.Sy - P.sy0) * P.rw + (px - P.Sx - P.sx0));
    double m[kMoments];
#pragma unroll
    for (int i = 0; i < kMoments; ++i) m[i] = 0.0;
#pragma unroll 1
    for (int k = 0; k < nstrips; ++k) {
        const StripLane e = tab[k * L + hl];
        const int full = __builtin_amdgcn_readfirstlane((int)((e.rows >> 8) & 0xffu)), rows = (int)(e.rows & 0xffu);
        if (rows == 0) continue;
        int xx[3] = {}, xy[3] = {}, yy[3] = {}, x[2] = {}, y[2] = {}, xr[2] = {}, yr[2] = {}, r1 = 0, r2 = 0;
        const int go = (int)(gcorner + e.go), ro = (py + (int)e.dy) * P.stride + px + (int)e.dx;
        int gso = 0, rso = 0;
        auto pixel = [&]() {
            const uint32_t g = __builtin_amdgcn_raw_buffer_load_b32(g2r, go, gso, 0);
            const int R = __builtin_amdgcn_raw_buffer_load_b8(imgr, ro, rso, 0);
            const int gx = (int16_t)(g & 0xffffu), gy = (int)g >> 16;
            gso += 4 * P.rw;
            rso += P.stride;
            xx[0] += __mul24(gx, gx); xx[1] += xx[0]; xx[2] += xx[1];
            xy[0] += __mul24(gx, gy); xy[1] += xy[0]; xy[2] += xy[1];
            yy[0] += __mul24(gy, gy); yy[1] += yy[0]; yy[2] += yy[1];
            x[0] += gx; x[1] += x[0];
            y[0] += gy; y[1] += y[0];
            xr[0] += __mul24(gx, R); xr[1] += xr[0];
            yr[0] += __mul24(gy, R); yr[1] += yr[0];
            r1 += R;
            r2 += __mul24(R, R);
        };
#pragma unroll 4
        for (int r = 0; r < full; ++r) pixel();
        if (rows > full) pixel();
        // with j = rows - i for row i: sum j q and sum j (j + 1) / 2 q are the
        // running sums' sums, and dy = end - j
        const double dx = (double)e.dx, end = (double)e.dy + (double)rows;
        auto fold3 = [&](const int (&q)[3], double* o) {
            const double s0 = (double)q[0], s1 = (double)q[1], s2 = (double)q[2];
            const double sy = end * s0 - s1;
            o[0] += s0;
            o[1] += dx * s0;
            o[2] += sy;
            o[3] += dx * dx * s0;
            o[4] += dx * sy;
            o[5] += end * (end * s0 - 2.0 * s1) + (2.0 * s2 - s1);
        };
        auto fold2 = [&](const int (&q)[2], double* o) {
            const double s0 = (double)q[0];
            o[0] += s0;
            o[1] += dx * s0;
            o[2] += end * s0 - (double)q[1];
        };
        fold3(xx, m + M_XX);
        fold3(xy, m + M_XY);
        fold3(yy, m + M_YY);
        fold2(x, m + M_X);
        fold2(y, m + M_Y);
        fold2(xr, m + M_XR);
        fold2(yr, m + M_YR);
        m[M_R] += (double)r1;
        m[M_RR] += (double)r2;
    }
    // the lanes' sum: eight moments at a time, lane hl takes moment hl % 8 of
    // the lanes 8 (hl / 8) .. + 7
#pragma unroll
    for (int c = 0; c < kMoments / 8; ++c) {
        wave_lds_sync();
#pragma unroll
        for (int v = 0; v < 8; ++v) red[v][hl] = m[8 * c + v];
        wave_lds_sync();
        double s = 0.0;
#pragma unroll
        for (int i = 0; i < 8; ++i) s += red[hl & 7][(hl & ~7) + i];
        s += __shfl_xor(s, 8);
        s += __shfl_xor(s, 16);
        if constexpr (L == 64) s += __shfl_xor(s, 32);
        if (hl < 8) mom[8 * c + hl] = s;
    }
}

// One POI's state (kRefStateUsed doubles) from its moments, in place.
__device__ __forceinline__ void ref_finish(const IcgnParams& P, double* slot)
{
    constexpr int kPick[3][3] = {{0, 1, 2}, {1, 3, 4}, {2, 4, 5}};       // the moment of basis product (k, q)
    double Lf[21], a[6], b[6];
    int t = 0;
#pragma unroll
    for (int k = 0; k < 6; ++k)
#pragma unroll
        for (int q = 0; q <= k; ++q)
            Lf[t++] = 0.25 * slot[(k < 3 ? M_XX : q < 3 ? M_XY : M_YY) + kPick[k % 3][q % 3]];
#pragma unroll
    for (int k = 0; k < 6; ++k) {
        a[k] = 0.5 * slot[(k < 3 ? M_X : M_Y) + k % 3];
        b[k] = 0.5 * slot[(k < 3 ? M_XR : M_YR) + k % 3];
    }
    const double sr = slot[M_R], srr = slot[M_RR];
    double mean, spread;
    mean_spread(sr, srr, (double)P.s, mean, spread);
    double flag = 0.0;
    // TW_paDIC_ICGN2D_CPU.cpp:580-595: zero mean or zero spread -> DarkSubset.
    // Both sums are exact integers, so the test is exact: all-zero or uniform.
    if (sr == 0.0 || srr * (double)P.s == sr * sr) flag = (double)TWDIC_ICGN_DARK_SUBSET;
    if (flag == 0.0) {
        // Cholesky (spotrf 'L', TW_paDIC_ICGN2D_CPU.cpp:682,688-693) in FP64
#pragma unroll
        for (int j = 0; j < 6; ++j) {
            const int jj = j * (j + 1) / 2;
            double d = Lf[jj + j];
#pragma unroll
            for (int k = 0; k < j; ++k) d -= Lf[jj + k] * Lf[jj + k];
            if (!(d > 0.0)) { flag = (double)TWDIC_ICGN_SINGULAR_HESSIAN; break; }
            d = sqrt(d);
            Lf[jj + j] = d;
#pragma unroll
            for (int i = j + 1; i < 6; ++i) {
                const int ii = i * (i + 1) / 2;
                double v = Lf[ii + j];
#pragma unroll
                for (int k = 0; k < j; ++k) v -= Lf[ii + k] * Lf[jj + k];
                Lf[ii + j] = v / d;
            }
        }
    }
#pragma unroll
    for (int i = 0; i < 21; ++i) slot[RS_L + i] = Lf[i];
#pragma unroll
    for (int i = 0; i < 6; ++i) {
        slot[RS_A + i] = a[i];
        slot[RS_B + i] = centred(b[i], mean, a[i]);
    }
    slot[RS_NORM] = spread;
    slot[RS_FLAG] = flag;
    slot[RS_MEAN] = mean;
#pragma unroll
    for (int i = 0; i < 6; ++i) slot[RS_RDIAG + i] = flag == 0.0 ? 1.0 / Lf[i * (i + 1) / 2 + i] : 0.0;
}

// The state of a subset that leaves the ROI, which the iteration kernel flags:
// well defined, and no memory outside the ROI is read for it.
__device__ __forceinline__ void ref_outside(double* slot)
{
    for (int i = 0; i < kRefStateUsed; ++i) slot[i] = i == RS_FLAG ? (double)TWDIC_ICGN_OUT_OF_ROI : 0.0;
}

}  // namespace

// R rounds of 256 / L POIs per workgroup, then their factorisations together.
template <int L, int R>
__global__ __launch_bounds__(256) void k_ref_state(IcgnParams P, RefPlan plan)
{
    constexpr int G = 256 / L, Q = G * R;
    __shared__ StripLane tab[RefPlan::kMax * L];
    __shared__ double red[G][8][L + 1];
    __shared__ double slots[Q][kMomentSlot];
    const int t = threadIdx.x, first = blockIdx.x * Q;
    fill_strips<L>(tab, plan, P, true, t, 256);
    __syncthreads();
#pragma unroll 1
    for (int r = 0; r < R; ++r) {
        const int slot = r * G + t / L, poi = first + slot;
        if (poi >= P.n) break;
        const int py = P.poi[2 * poi], px = P.poi[2 * poi + 1];
        if (!subset_outside(P, px, py)) ref_moments<L>(P, plan.count, px, py, t & (L - 1), tab, red[t / L], slots[slot]);
    }
    __syncthreads();
    if (t < Q && first + t < P.n) {
        const int py = P.poi[2 * (first + t)], px = P.poi[2 * (first + t) + 1];
        if (subset_outside(P, px, py))
            ref_outside(slots[t]);
        else
            ref_finish(P, slots[t]);
    }
    __syncthreads();
    for (int i = t; i < Q * kRefStateUsed; i += 256) {
        const int slot = i / kRefStateUsed, j = i - slot * kRefStateUsed;
        if (first + slot < P.n) P.refstate[(size_t)(first + slot) * kRefStateStride + j] = slots[slot][j];
    }
}

// Two rounds per workgroup (one factorisation pass for 16 POIs) where that
// leaves the GPU full: 0.26 ms for 157,609 POIs, as with four; one round 0.30 ms,
// eight 0.36 ms.  Smaller sets take one.
hipError_t launch_ref_state(const IcgnParams& p, const RefPlan& plan, hipStream_t st)
{
    if (p.n <= 0) return hipSuccess;
    if (ref_lanes_for(p.n) == 64)
        hipLaunchKernelGGL((k_ref_state<64, 1>), dim3((p.n + 3) / 4), dim3(256), 0, st, p, plan);
    else if (p.n < 32768)
        hipLaunchKernelGGL((k_ref_state<32, 1>), dim3((p.n + 7) / 8), dim3(256), 0, st, p, plan);
    else
        hipLaunchKernelGGL((k_ref_state<32, 2>), dim3((p.n + 15) / 16), dim3(256), 0, st, p, plan);
    return hipGetLastError();
}

// Persistent form over (pair, POI) work items, one item per wavefront grab, on
// its pair's lanes (the whole wavefront, or its lower half).
__global__ __launch_bounds__(256) void k_batch_ref_state(const PairDesc* __restrict__ pairs,
                                                         const int2* __restrict__ items, int total, int* counter)
{
    __shared__ StripLane tabs[4][RefPlan::kMax * 64];
    __shared__ double reds[4][8][64 + 1];
    __shared__ double slots[4][kMomentSlot];
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    double* slot = slots[wave];
    for (;;) {
        int i = 0;
        if (lane == 0) i = atomicAdd(counter, 1);
        i = __builtin_amdgcn_readfirstlane(__shfl(i, 0));
        if (i >= total) break;
        const int2 it = items[i];
        const int pair = __builtin_amdgcn_readfirstlane(it.x);
        const IcgnParams P = const_pairs(pairs)[pair].icgn;
        const RefPlan plan = const_pairs(pairs)[pair].ref;
        const int poi = __builtin_amdgcn_readfirstlane(it.y), py = P.poi[2 * poi], px = P.poi[2 * poi + 1];
        wave_lds_sync();
        if (!subset_outside(P, px, py)) {
            if (ref_lanes_for(P.n) == 64) {
                fill_strips<64>(tabs[wave], plan, P, true, lane, 64);
                wave_lds_sync();
                ref_moments<64>(P, plan.count, px, py, lane, tabs[wave], reds[wave], slot);
            } else {
                fill_strips<32>(tabs[wave], plan, P, true, lane, 64);
                wave_lds_sync();
                if (lane < 32)
                    ref_moments<32>(P, plan.count, px, py, lane, tabs[wave], reinterpret_cast<double (*)[33]>(reds[wave]),
                                    slot);
            }
        }
        wave_lds_sync();
        if (lane == 0) {
            if (subset_outside(P, px, py))
                ref_outside(slot);
            else
                ref_finish(P, slot);
        }
        wave_lds_sync();
        for (int j = lane; j < kRefStateUsed; j += 64) P.refstate[(size_t)poi * kRefStateStride + j] = slot[j];
    }
}

int persistent_blocks_state(int device)
{
    int cus = 0, per = 0;
    (void)hipDeviceGetAttribute(&cus, hipDeviceAttributeMultiprocessorCount, device);
    if (hipOccupancyMaxActiveBlocksPerMultiprocessor(&per, k_batch_ref_state, 256, 0) != hipSuccess || per < 1) per = 1;
    return (cus > 0 ? cus : 256) * per;
}

hipError_t launch_batch_ref_state(const PairDesc* pairs, const int2* items, int total, int* counter, int blocks,
                                  hipStream_t st)
{
    if (total <= 0) return hipSuccess;
    hipLaunchKernelGGL(k_batch_ref_state, dim3(blocks), dim3(256), 0, st, pairs, items, total, counter);
    return hipGetLastError();
}

// Zero-fill for work counters (a kernel, so it is safe inside captured graphs).
__global__ void k_fill_zero(int* p, int n)
{
    int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i < n) p[i] = 0;
}

hipError_t launch_fill_zero(int* p, int n, hipStream_t st)
{
    hipLaunchKernelGGL(k_fill_zero, dim3((n + 255) / 256), dim3(256), 0, st, p, n);
    return hipGetLastError();
}

}  // namespace twdic
