// Affine view transform and border-weight mask (gfx950).
//
// Reference: fmvd_transform.impl.cu:24-56 (transform_plane_kernel, a CUDA
// 3D-texture trilinear fetch at r + 0.5 with border address mode and
// normalised-float read), :77-224 (transform_cuda driver) and
// fmvd_transform.cu:19-89 (create_transformed_mask).
//
// Arithmetic: source coordinates and interpolation weights are evaluated in
// FP64 with a fixed operation order and no contraction, so every output
// sample equals the FP64 definition bit for bit:
//   r = ((m0 x + m1 y) + m2 z) + m3 per axis, i = floor(r), a = r - i,
//   nested lerps v*(1-a) + v'*a in x, then y, then z (texels outside -> 0),
//   out = clamp(floor(interp / (2^B-1) * 2^B + 0.5), 0, 2^B-1).
#include <hip/hip_runtime.h>

#include <algorithm>
#include <cmath>
#include <cstdint>
#include <cstdio>
#include <vector>

#include "../../include/fmvd_transform.h"
#include "hip_check.hpp"
#include "timing.hpp"
#include "transform.hpp"

namespace fmvd {

struct Mat12 {
    double m[12];
};

// Two horizontally adjacent samples (x, x + 1) of one source row as one
// 4-byte (16-bit samples) or 2-byte (8-bit samples) load; x need not be even.
template <typename S>
__device__ __forceinline__ void load_pair(const S* row, int x, double& t0, double& t1)
{
    if constexpr (sizeof(S) == 2) {
        uint32_t u;
        __builtin_memcpy(&u, row + x, 4);
        t0 = (double)(u & 0xffffu);
        t1 = (double)(u >> 16);
    } else {
        uint16_t u;
        __builtin_memcpy(&u, row + x, 2);
        t0 = (double)(u & 0xffu);
        t1 = (double)(u >> 8);
    }
}

// Samples (ix, iy, iz) and (ix + 1, iy, iz), zero outside the volume.
template <typename S>
__device__ __forceinline__ void fetch_pair(const S* __restrict__ src, int w, int h, int d, int ix, int iy, int iz,
                                           double& t0, double& t1)
{
    if (iy < 0 || iy >= h || iz < 0 || iz >= d) {
        t0 = t1 = 0.0;
        return;
    }
    const S* row = src + ((size_t)iz * h + iy) * w;
    if (ix >= 0 && ix + 1 < w) {
        load_pair<S>(row, ix, t0, t1);
    } else {
        t0 = (ix >= 0 && ix < w) ? (double)row[ix] : 0.0;
        t1 = (ix + 1 >= 0 && ix + 1 < w) ? (double)row[ix + 1] : 0.0;
    }
}

// a b + c d, each operation rounded.
__device__ __forceinline__ double mul_add(double a, double b, double c, double d)
{
#pragma clang fp contract(off)
    return a * b + c * d;
}

// One output sample at plane z of target column (x, y); axy[a] holds
// m[4a] x + m[4a+1] y (the first sum of the fixed operation order).  FP64
// with no contraction:
//   r_a = ((m[4a] x + m[4a+1] y) + m[4a+2] z) + m[4a+3], i = floor(r), f = r - i,
//   nested lerps v (1 - f) + v' f in x, then y, then z (texels outside -> 0),
//   out = clamp(floor(interp / (2^B-1) * 2^B + 0.5), 0, 2^B-1)
// (fmvd_transform.impl.cu:41-53 with FP64 coordinates and weights).
template <typename S>
__device__ __forceinline__ S transform_sample(const S* __restrict__ src, int w, int h, int d, const Mat12& M,
                                              const double* axy, int z)
{
#pragma clang fp contract(off)
    const double zd = (double)z;
    const double rx = (axy[0] + M.m[2] * zd) + M.m[3];
    const double ry = (axy[1] + M.m[6] * zd) + M.m[7];
    const double rz = (axy[2] + M.m[10] * zd) + M.m[11];
    double val = 0.0;
    if (rx > -2.0 && ry > -2.0 && rz > -2.0 && rx < (double)w + 1.0 && ry < (double)h + 1.0 &&
        rz < (double)d + 1.0) {
        const double fx = floor(rx), fy = floor(ry), fz = floor(rz);
        const double ax = rx - fx, ay = ry - fy, az = rz - fz;
        const double bx = 1.0 - ax, by = 1.0 - ay, bz = 1.0 - az;
        const int ix = (int)fx, iy = (int)fy, iz = (int)fz;
        double t000, t100, t010, t110, t001, t101, t011, t111;
        fetch_pair<S>(src, w, h, d, ix, iy, iz, t000, t100);
        fetch_pair<S>(src, w, h, d, ix, iy + 1, iz, t010, t110);
        fetch_pair<S>(src, w, h, d, ix, iy, iz + 1, t001, t101);
        fetch_pair<S>(src, w, h, d, ix, iy + 1, iz + 1, t011, t111);
        const double c00 = t000 * bx + t100 * ax;
        const double c10 = t010 * bx + t110 * ax;
        const double c01 = t001 * bx + t101 * ax;
        const double c11 = t011 * bx + t111 * ax;
        const double c0 = c00 * by + c10 * ay;
        const double c1 = c01 * by + c11 * ay;
        val = c0 * bz + c1 * az;
    }
    constexpr double maxv = (double)((1u << (8 * sizeof(S))) - 1u);
    constexpr double scale = (double)(1u << (8 * sizeof(S)));
    // yv = (val / maxv) * scale + 0.5 decides the sample only through its
    // integer part and the bounds 0 and maxv (integers).  val * (1 / maxv)
    // stays within 3 ulp of val / maxv, so the reciprocal form moves yv
    // (< 2^16) by less than 1e-10: when it lies farther than 1e-9 from an
    // integer both forms give the same sample, otherwise the division
    // decides.
    constexpr double inv_maxv = 1.0 / maxv;
    double yv = (val * inv_maxv) * scale + 0.5;
    const double fr = yv - floor(yv);
    if (!(fr > 1e-9 && fr < 1.0 - 1e-9)) yv = (val / maxv) * scale + 0.5;
    if (yv >= maxv) return (S)maxv;
    if (yv > 0.0) return (S)floor(yv);
    return (S)0;
}

// General kernel: any map.  A thread computes kGZ consecutive target planes of one
// (x, y) column; a workgroup holds 64 x 4 columns.  The trilinear fetches read the source
// straight from global memory (two samples per load).  Workgroups are taken in
// supertiles of kSX x kSY x kSZ workgroups (128 x 32 x 32 target voxels, about 1.5 MB
// of source), numbered x fastest, then y, then z, with each XCD given a
// contiguous range, so the supertiles in flight on one XCD keep their source
// rows in its L2.
constexpr int kGX = 64, kGY = 4, kGZ = 8;
constexpr unsigned kSX = 2, kSY = 8, kSZ = 4, kSuper = kSX * kSY * kSZ;

__device__ __forceinline__ unsigned xcd_block(unsigned bid, unsigned nblocks)
{
    const unsigned q = nblocks >> 3, rem = nblocks & 7u;
    const unsigned x = bid & 7u, k = bid >> 3;
    return x * q + (x < rem ? x : rem) + k;
}

template <typename S>
__global__ __launch_bounds__(256) void transform_general_kernel(const S* __restrict__ src, int w, int h, int d,
                                                        S* __restrict__ dst, int tw, int th, int z0, int nz,
                                                        Mat12 M, unsigned nbx, unsigned nby, unsigned nsx,
                                                        unsigned nsy)
{
#pragma clang fp contract(off)
    const unsigned lid = xcd_block(blockIdx.x, gridDim.x);
    const unsigned st = lid / kSuper, wi = lid % kSuper;
    const unsigned bx = (st % nsx) * kSX + wi % kSX;
    const unsigned by = ((st / nsx) % nsy) * kSY + (wi / kSX) % kSY;
    const unsigned bz = (st / (nsx * nsy)) * kSZ + wi / (kSX * kSY);
    if (bx >= nbx || by >= nby) return;
    const int x = (int)bx * kGX + (int)(threadIdx.x % kGX);
    const int y = (int)by * kGY + (int)(threadIdx.x / kGX);
    if (x >= tw || y >= th) return;
    const double xd = (double)x, yd = (double)y;
    const double axy[3] = {mul_add(M.m[0], xd, M.m[1], yd), mul_add(M.m[4], xd, M.m[5], yd),
                           mul_add(M.m[8], xd, M.m[9], yd)};
    const int zb = z0 + (int)bz * kGZ, ze = min(zb + kGZ, z0 + nz);
    if (zb >= ze) return;
    S* out = dst + ((size_t)(zb - z0) * th + y) * tw + x;
    const size_t pstride = (size_t)th * tw;
    for (int z = zb; z < ze; ++z, out += pstride) *out = transform_sample<S>(src, w, h, d, M, axy, z);
}

// ------------------------------------------------------------------ box kernel
// A workgroup computes a cube of kT^3 target voxels.  It stages the bounding box of the
// cube's texels (3.8 texels an output at +-15 degrees about each axis) in LDS with
// coalesced loads, zero outside the volume, and gathers from there without
// bounds checks.  Gathering straight from global memory costs the texture path
// about one cycle per lane and load, whatever the lanes' arrangement (40 L1 accesses a
// load; 64 x 1, 32 x 2, 16 x 4 and 8 x 8 voxels ran alike, as did aligned loads):
// 190 cycles for 64 outputs, against about 40 for the four LDS reads.  1024^2 x
// 512 voxels of 16 bits under such maps: 3.06 ms gathered, 1.34 ms here (1.6 TB/s
// of 2.1 GB).  At 2048^2 x 1024 the texture data path is busy 78 % of the time with the
// staging, the VALU issues 63 % (74 instructions an output, most of them FP64, conversions
// or byte shifts), the LDS is busy 38 %, a fifth of the cycles in bank conflicts.
// 301 x 257 x 129 voxels of 8 bits into 333 x 270 x 141: 95 -> 56 us.
//
// The arithmetic is FP64 with fewer operations than the definition: the
// coordinates as one FMA on a sum per (x, y) column, lerps as v + f (v' - v).  The result
// differs from the definition's by at most `guard` output units (transform_guard),
// so a sample farther than that from a rounding boundary is the definition's, and
// any other is evaluated by transform_sample.
constexpr int kT = 16, kBoxThreads = 512;
constexpr unsigned kBoxSuper = 4;  // supertiles of 4^3 cubes, about 1.7 MB of source; flat targets' of fewer layers

struct BoxMap {
    double guard;
    double low[3];      // least source coordinate of a cube, from its first voxel's, less a margin for rounding
    int ny, nz;         // rows and planes of the box
    int pieces;         // pieces staged per row
    int pitch, plane;   // bytes from row to row and plane to plane
    int step, step_y, step_z;  // rows staged at a time: floor(threads / pieces) = step_z ny + step_y
    unsigned magic_pieces;     // ceil(2^16 / pieces): i / pieces = i magic >> 16 for i < 512, pieces <= 150
    unsigned nx, nby, nsx, nsy;  // cubes, and supertiles, along x and y
    unsigned log_sz;             // cubes of a supertile along z
};

__device__ __forceinline__ double lerp(double a, double b, double f) { return fma(f, b - a, a); }
// Samples x, x + 1 of a staged row, `shift` bytes into the word at LDS address `at`, interpolated.
template <typename S> __device__ __forceinline__ double lerp_row(uint32_t at, uint32_t shift, double f)
{
    typedef uint32_t two __attribute__((ext_vector_type(2), aligned(4)));
    const two t = *reinterpret_cast<__attribute__((address_space(3))) const two*>(at);
    const uint32_t u = __builtin_amdgcn_alignbyte(t.y, t.x, shift);
    constexpr uint32_t bits = 8 * sizeof(S), mask = (1u << bits) - 1u;
    return lerp((double)(u & mask), (double)(u >> bits & mask), f);
}
__device__ __forceinline__ uint32_t lds_address(const void* p)
{
    return (uint32_t)(uintptr_t)(__attribute__((address_space(3))) const char*)p;
}

// The bytes of a piece from sample (x, y, z) on, zero where outside the volume.
template <typename S, typename P>
__device__ __forceinline__ P load_piece(const S* __restrict__ src, int w, int h, int d, int x, int y, int z)
{
    constexpr int n = sizeof(P) / sizeof(S);
    P p{};
    if (y < 0 || y >= h || z < 0 || z >= d || x + n <= 0 || x >= w) return p;
    const S* row = src + ((size_t)z * h + y) * w;
    if (x >= 0 && x + n <= w) {
        if constexpr (sizeof(P) == 16) p = *reinterpret_cast<const P*>(row + x);
        else __builtin_memcpy(&p, row + x, sizeof p);
    } else if constexpr (sizeof(P) == 4) {  // (16-byte pieces lie inside or outside)
        for (int i = 0; i < n; ++i)
            if (x + i >= 0 && x + i < w) p |= (uint32_t)row[x + i] << (8 * sizeof(S) * i);
    }
    return p;
}

template <typename S, typename P>
__global__ __launch_bounds__(kBoxThreads, 4) void transform_box_kernel(const S* __restrict__ src, int w, int h, int d,
                                                                       S* __restrict__ dst, int tw, int th, int z0,
                                                                       int nz, Mat12 M, BoxMap B)
{
    extern __shared__ __attribute__((aligned(16))) char box[];
    constexpr unsigned s = kBoxSuper;
    const unsigned lid = xcd_block(blockIdx.x, gridDim.x), st = lid / (s * s) >> B.log_sz, wi = lid - ((st * s * s) << B.log_sz);
    const unsigned bx = st % B.nsx * s + wi % s, by = st / B.nsx % B.nsy * s + wi / s % s,
                   bz = (st / (B.nsx * B.nsy) << B.log_sz) + wi / (s * s);
    const int x0 = (int)bx * kT, y0 = (int)by * kT, zb = z0 + (int)bz * kT, ze = z0 + nz;
    if (bx >= B.nx || by >= B.nby || zb >= ze) return;

    // first texel of the box on each axis
    int org[3];
#pragma unroll
    for (int a = 0; a < 3; ++a) {
        const double r = fma(M.m[4 * a], (double)x0, fma(M.m[4 * a + 1], (double)y0, fma(M.m[4 * a + 2], (double)zb, M.m[4 * a + 3])));
        org[a] = __builtin_amdgcn_readfirstlane((int)floor(r + B.low[a]));
    }
    constexpr int n = sizeof(P) / sizeof(S);
    if constexpr (sizeof(P) == 16) org[0] &= -n;  // rows are staged from 16-byte boundaries

    // a box that meets no texel: its samples are zero (uniform)
    if (org[0] >= w || org[0] + B.pieces * n <= 0 || org[1] >= h || org[1] + B.ny <= 0 || org[2] >= d || org[2] + B.nz <= 0) {
        const int x = x0 + (int)(threadIdx.x & 15), y = y0 + (int)(threadIdx.x >> 4 & 15);
        if (x < tw && y < th)
            for (int z = zb + (int)(threadIdx.x >> 8); z < min(zb + kT, ze); z += kBoxThreads / 256)
                dst[((size_t)(z - z0) * th + y) * tw + x] = 0;
        return;
    }

    // Staging: a thread takes piece q of the rows row, row + step, ... (iy, iz by
    // counting), four loads in flight; past the last row, and in the threads left
    // over, it repeats a row.
    const int rows = B.ny * B.nz, passes = (rows + B.step - 1) / B.step;
    int row = (int)(threadIdx.x * B.magic_pieces >> 16);
    const int q = (int)threadIdx.x - row * B.pieces;
    row = min(row < B.step ? row : 0, rows - 1);
    int iz = row / B.ny, iy = row - iz * B.ny;
    uint32_t to = iz * B.plane + iy * B.pitch + q * (int)sizeof(P);
    const uint32_t to_step = B.step_z * B.plane + B.step_y * B.pitch, to_wrap = B.plane - B.ny * B.pitch;
    const bool within = org[0] >= 0 && org[0] + B.pieces * n <= w && org[1] >= 0 && org[1] + B.ny <= h && org[2] >= 0 &&
                        org[2] + B.nz <= d;
    constexpr int U = 4;
    if (within) {  // uniform: a box inside the volume needs no checks and 32-bit offsets
        const char* from = reinterpret_cast<const char*>(src + ((size_t)org[2] * h + org[1]) * w + org[0]);
        const uint32_t row_bytes = (uint32_t)w * sizeof(S), plane_bytes = row_bytes * (uint32_t)h;
        const uint32_t step = B.step_z * plane_bytes + B.step_y * row_bytes, wrap = plane_bytes - B.ny * row_bytes;
        uint32_t off = iz * plane_bytes + iy * row_bytes + q * (uint32_t)sizeof(P);
        for (int k = 0; k < passes; k += U) {
            P p[U];
            uint32_t at[U];
#pragma unroll
            for (int u = 0; u < U; ++u) {
                at[u] = to;
                if constexpr (sizeof(P) == 16) p[u] = *reinterpret_cast<const P*>(from + off);
                else __builtin_memcpy(&p[u], from + off, sizeof(P));
                if (row + B.step < rows) {
                    row += B.step;
                    iy += B.step_y;
                    const bool over = iy >= B.ny;
                    off += step + (over ? wrap : 0);
                    to += to_step + (over ? to_wrap : 0);
                    iy -= over ? B.ny : 0;
                }
            }
#pragma unroll
            for (int u = 0; u < U; ++u) *reinterpret_cast<P*>(box + at[u]) = p[u];
        }
    } else {
        for (int k = 0; k < passes; ++k) {
            *reinterpret_cast<P*>(box + to) = load_piece<S, P>(src, w, h, d, org[0] + q * n, org[1] + iy, org[2] + iz);
            if (row + B.step >= rows) break;
            row += B.step;
            iz += B.step_z;
            iy += B.step_y;
            to += to_step;
            if (iy >= B.ny) {
                iy -= B.ny;
                ++iz;
                to += to_wrap;
            }
        }
    }
    __syncthreads();

    // wavefront: 16 x 4 columns, 8 planes
    const int x = x0 + (int)(threadIdx.x & 15), y = y0 + (int)(threadIdx.x >> 4 & 15), zw = zb + (int)(threadIdx.x >> 8) * 8;
    if (x >= tw || y >= th) return;
    const double xd = (double)x, yd = (double)y, zd = (double)zw;
    double r[3];  // source coordinates, stepped from plane to plane
    auto first_plane = [&] {
#pragma unroll
        for (int a = 0; a < 3; ++a)
            r[a] = fma(M.m[4 * a + 2], zd, fma(M.m[4 * a], xd, fma(M.m[4 * a + 1], yd, M.m[4 * a + 3])));
    };
    first_plane();
    const double pitch = (double)B.pitch, plane = (double)B.plane;
    // byte address in LDS of texel (0, 0, 0)
    const double at0 = (double)lds_address(box) -
                       fma((double)org[2], plane, fma((double)org[1], pitch, (double)(org[0] * (int)sizeof(S))));
    S* out = dst + ((size_t)(zw - z0) * th + y) * tw + x;
    const size_t pstride = (size_t)th * tw;
    double worst = 0.0;  // largest distance of an unrounded sample from its rounded value
    auto sample = [&]() -> S {
        const double fx = floor(r[0]), fy = floor(r[1]), fz = floor(r[2]);
        const uint32_t shift = (uint32_t)(int)fma(fz, plane, fma(fy, pitch, fma(fx, (double)sizeof(S), at0)));
        const uint32_t at = shift & ~3u;
        const double ax = r[0] - fx, ay = r[1] - fy, az = r[2] - fz;
        const double c0 = lerp(lerp_row<S>(at, shift, ax), lerp_row<S>(at + B.pitch, shift, ax), ay);
        const double c1 = lerp(lerp_row<S>(at + B.plane, shift, ax), lerp_row<S>(at + B.plane + B.pitch, shift, ax), ay);
        constexpr double maxv = (double)((1u << (8 * sizeof(S))) - 1u);
        const double v = lerp(c0, c1, az) * ((maxv + 1.0) / maxv), n = rint(v);  // floor(v + 1/2) off ties
        worst = fmax(worst, fabs(v - n));
#pragma unroll
        for (int a = 0; a < 3; ++a) r[a] += M.m[4 * a + 2];
        return (S)min((uint32_t)(int)n, (uint32_t)maxv);
    };
    if (zw + 8 <= ze) {  // wave-uniform
#pragma unroll
        for (int i = 0; i < 8; ++i) out[i * pstride] = sample();
    } else {
        for (int i = 0; zw + i < ze; ++i) out[i * pstride] = sample();
    }
    // Which of the 8 it was is found by computing them again: keeping the flags would cost every sample, and
    // evaluating all 8 made a wavefront wait for 8 fetches (1024^2 x 256 voxels of 8 bits shifted by
    // (1/8, 3/8, 5/8), where 0.2 % of the samples are ties: 1570 us, 1010 here, and 1414 in the general kernel).
    if (!(worst < 0.5 - B.guard)) {
        uint32_t tied = 0;
        first_plane();
#pragma unroll 1
        for (int i = 0; i < min(8, ze - zw); ++i) {
            worst = 0.0;
            (void)sample();
            if (!(worst < 0.5 - B.guard)) tied |= 1u << i;
        }
        const double axy[3] = {mul_add(M.m[0], xd, M.m[1], yd), mul_add(M.m[4], xd, M.m[5], yd),
                               mul_add(M.m[8], xd, M.m[9], yd)};
        for (; tied; tied &= tied - 1) {
            const int i = __builtin_ctz(tied);
            out[i * pstride] = transform_sample<S>(src, w, h, d, M, axy, zw + i);
        }
    }
}

__global__ __launch_bounds__(256) void mask_kernel(float* __restrict__ out, int z, int w, int h, int d,
                                                   double zspacing, int tw, int th, double border,
                                                   Mat12 M)
{
#pragma clang fp contract(off)
    const int x = blockIdx.x * blockDim.x + threadIdx.x;
    const int y = blockIdx.y * blockDim.y + threadIdx.y;
    if (x >= tw || y >= th) return;
    const double xd = (double)x, yd = (double)y, zd = (double)z;
    const double rx = ((M.m[0] * xd + M.m[1] * yd) + M.m[2] * zd) + M.m[3];
    const double ry = ((M.m[4] * xd + M.m[5] * yd) + M.m[6] * zd) + M.m[7];
    const double rz = ((M.m[8] * xd + M.m[9] * yd) + M.m[10] * zd) + M.m[11];
    float r = 0.0f;
    if (!(rx < 0 || rx >= w || ry < 0 || ry >= h || rz < 0 || rz >= d)) {
        // fmvd_transform.cu:46-64 (w/2 etc. are integer divisions)
        double dx = rx < (double)(w / 2) ? rx : (double)w - rx;
        double dy = ry < (double)(h / 2) ? ry : (double)h - ry;
        double dz = rz < (double)(d / 2) ? rz : (double)d - rz;
        dz *= zspacing;
        double v = 1.0;
        if (dx < border) v *= 0.5 * (1.0 - cos(dx / border * M_PI));
        if (dy < border) v *= 0.5 * (1.0 - cos(dy / border * M_PI));
        if (dz < border) v *= 0.5 * (1.0 - cos(dz / border * M_PI));
        r = (float)v;
    }
    out[(long)y * tw + x] = r;
}

static Mat12 to_mat(const float* m)
{
    Mat12 M;
    for (int i = 0; i < 12; ++i) M.m[i] = (double)m[i];
    return M;
}

// Bound, in output units, on the difference between the box kernel's
// arithmetic and the definition over a launch's target voxels: each coordinate is a sum of
// four terms in either, off by at most 4 roundings of the terms' magnitudes (and 8
// more from plane to plane);
// trilinear interpolation changes by at most the sample range per unit of a
// coordinate, and its own roundings are far below the 1e-9 added.
static double transform_guard(const Mat12& M, int tw, int th, int zend, double range)
{
    double sum = 0.0;
    for (int a = 0; a < 3; ++a)
        sum += std::fabs(M.m[4 * a]) * tw + std::fabs(M.m[4 * a + 1]) * th + std::fabs(M.m[4 * a + 2]) * zend +
               std::fabs(M.m[4 * a + 3]);
    return (4.0 + 12.0) * 0x1p-53 * sum * range + 1e-9;
}

// The box kernel where its box fits 64 KiB of LDS, so that one workgroup of a
// CU computes while another stages, and where the guard leaves few samples to
// evaluate twice (coordinates up to about 10^7).  Maps that shrink the
// source by more than about 2 take the general kernel, and so do one or two planes, which
// leave a workgroup little to compute behind its staging (512 x 512 voxels under
// rotations to 45 degrees, us, general and box: one plane 6.5, 10.4; two 8.5 to 10.0, 11.0 to 11.4;
// three 11.1 to 13.1, 11.2 to 11.9; eight 22 to 31, 14 to 19; of 1024 x 1024 three 27, 23).
template <typename S, typename P>
static bool launch_box(const S* src, int w, int h, int d, S* dst, int tw, int th, int z0, int nz, const Mat12& M,
                       hipStream_t s)
{
    if (nz < 3) return false;
    BoxMap B;
    B.guard = transform_guard(M, tw, th, z0 + nz, 65536.0);
    if (!(B.guard < 1e-3)) return false;
    // (a slab of a few planes, or a target that is narrower than a cube, needs less of the source:
    // 3 planes of 1024 x 1024: 36 -> 23 us together with the layers below; the general kernel 27)
    const int target[3] = {tw, th, nz};
    int n[3];
    for (int a = 0; a < 3; ++a) {
        double e = 0.0;
        B.low[a] = -1e-5;
        for (int k = 0; k < 3; ++k) {
            const double step = M.m[4 * a + k] * (std::min(kT, target[k]) - 1);
            e += std::fabs(step);
            B.low[a] += std::min(step, 0.0);
        }
        if (!(e < 140.0)) return false;
        n[a] = (int)std::ceil(e + 1e-4) + 2;
    }
    constexpr int ps = sizeof(P) / sizeof(S);
    B.pieces = (n[0] + (sizeof(P) == 16 ? 2 * ps - 2 : ps - 1)) / ps;
    B.ny = n[1];
    B.nz = n[2];
    // rows and planes an odd number of pieces apart spread over the banks
    B.pitch = (B.pieces | 1) * (int)sizeof(P);
    B.plane = (B.ny | 1) * B.pitch;
    const size_t lds = (size_t)B.plane * B.nz + 16;  // (a row's last read reaches 8 bytes past it)
    if (lds > 64 * 1024) return false;
    // 16-bit rows off the 16-byte boundaries, in a box of which only two workgroups fit a CU (160 KiB of
    // LDS): staging in 4-byte pieces is then slower than the general kernel where the 64 lanes of its
    // wavefront stay on few source rows (512 x 384 x 64 voxels from 1021 x 768 x 128, us, general and
    // box: unrotated at scale 1.7, 48.7 KB, 67, 66; at 1.8, 55.8 KB, 67, 90; turned by 3 degrees about each
    // axis at 1.7, 65.4 KB, 69, 93; but by 45 degrees about z at 1.5, 59.5 KB, 146, 93).  8 bits: 91, 85.
    if (sizeof(S) == 2 && sizeof(P) == 4 && 3 * lds > 160 * 1024 && std::fabs(M.m[4]) + std::fabs(M.m[8]) < 0.7)
        return false;
    B.step = kBoxThreads / B.pieces;
    B.step_z = B.step / B.ny;
    B.step_y = B.step % B.ny;
    B.magic_pieces = (65536u + B.pieces - 1) / B.pieces;
    B.nx = (unsigned)((tw + kT - 1) / kT);
    B.nby = (unsigned)((th + kT - 1) / kT);
    const unsigned nbz = (unsigned)((nz + kT - 1) / kT);
    // (no empty layers: 8 planes of 1024 x 1024 took 42 us with three of them launched, 29 without)
    B.log_sz = nbz >= 3 ? 2 : nbz - 1;
    const unsigned sz = 1u << B.log_sz;
    static_assert(kBoxSuper == 4);
    B.nsx = (B.nx + kBoxSuper - 1) / kBoxSuper;
    B.nsy = (B.nby + kBoxSuper - 1) / kBoxSuper;
    const unsigned long long blocks =
        (unsigned long long)B.nsx * B.nsy * ((nbz + sz - 1) / sz) * kBoxSuper * kBoxSuper * sz;
    if (blocks > 0x7fffffffull || (double)w * h * sizeof(S) * B.nz >= 4294967296.0) return false;
    launch(transform_box_kernel<S, P>, dim3((unsigned)blocks), dim3(kBoxThreads), (unsigned)lds, s, src, w, h, d, dst, tw,
           th, z0, nz, M, B);
    return true;
}

template <typename S>
static void launch_transform(const S* src, int w, int h, int d, S* dst, int tw, int th, int z0, int nz,
                             const Mat12& M, hipStream_t s)
{
    if (nz <= 0 || tw <= 0 || th <= 0) return;
    const unsigned nbx = (unsigned)((tw + kGX - 1) / kGX), nby = (unsigned)((th + kGY - 1) / kGY);
    const unsigned nbz = (unsigned)((nz + kGZ - 1) / kGZ);
    const unsigned nsx = (nbx + kSX - 1) / kSX, nsy = (nby + kSY - 1) / kSY, nsz = (nbz + kSZ - 1) / kSZ;
    const unsigned long long nblocks = (unsigned long long)nsx * nsy * nsz * kSuper;
    if (nblocks > 0x7fffffffull) throw_msg("transform: target volume too large for one launch");
    TimedScope ts(kTimeTransform, s);
    // 16-byte pieces where every row starts on a 16-byte boundary
    const bool aligned = (size_t)w * sizeof(S) % 16 == 0 && (uintptr_t)src % 16 == 0;
    if (aligned ? launch_box<S, uint4>(src, w, h, d, dst, tw, th, z0, nz, M, s)
                : launch_box<S, uint32_t>(src, w, h, d, dst, tw, th, z0, nz, M, s)) {
        FMVD_LAUNCH_CHECK();
        return;
    }
    launch(transform_general_kernel<S>, dim3((unsigned)nblocks), dim3(kGX * kGY), 0, s, src, w, h, d, dst, tw, th, z0,
           nz, M, nbx, nby, nsx, nsy);
    FMVD_LAUNCH_CHECK();
}

static void launch_mask(float* out, int w, int h, int d, int tw, int th, int td, const Mat12& M,
                        int border, float zspacing, hipStream_t s)
{
    dim3 block(64, 4);
    dim3 grid((unsigned)((tw + 63) / 64), (unsigned)((th + 3) / 4));
    mask_kernel<<<grid, block, 0, s>>>(out, td / 2, w, h, d, (double)zspacing, tw, th, (double)border, M);
    FMVD_LAUNCH_CHECK();
}

static void check_dims(int w, int h, int d, int tw, int th, int td)
{
    if (w < 1 || h < 1 || d < 1 || tw < 1 || th < 1 || td < 1)
        throw_msg("invalid transform dimensions (all extents must be >= 1)");
}

// fmvd_transform.impl.cu:77-224: whole source volume resident on the device,
// target planes computed in chunks and written to `outfile` in z order while
// the next chunk computes.
template <typename S>
static void transform_files(S** h_data, int w, int h, int d, int tw, int th, int td, const float* inv,
                            const char* outfile, int createMasks, int border, float zspacing,
                            const char* maskfile)
{
    check_dims(w, h, d, tw, th, td);
    if (!h_data || !inv || !outfile) throw_msg("transform: NULL argument");
    const Mat12 M = to_mat(inv);
    const size_t plane = (size_t)w * h, tplane = (size_t)tw * th;
    S* dsrc = nullptr;
    S* ddst = nullptr;
    S* hdst = nullptr;
    float* dmask = nullptr;
    float* hmask = nullptr;
    hipStream_t s = nullptr;
    hipEvent_t ev[2] = {nullptr, nullptr};
    FILE* out = nullptr;
    auto cleanup = [&] {
        if (s) (void)hipStreamSynchronize(s);
        if (dsrc) (void)hipFree(dsrc);
        if (ddst) (void)hipFree(ddst);
        if (hdst) (void)hipHostFree(hdst);
        if (dmask) (void)hipFree(dmask);
        if (hmask) (void)hipHostFree(hmask);
        for (auto& e : ev)
            if (e) (void)hipEventDestroy(e);
        if (s) (void)hipStreamDestroy(s);
        if (out) fclose(out);
    };
    try {
        FMVD_HIP(hipStreamCreateWithFlags(&s, hipStreamNonBlocking));
        FMVD_HIP(hipMalloc(&dsrc, sizeof(S) * plane * d));
        for (int z = 0; z < d; ++z)
            FMVD_HIP(hipMemcpy(dsrc + plane * z, h_data[z], sizeof(S) * plane, hipMemcpyHostToDevice));
        if (createMasks) {
            if (!maskfile) throw_msg("transform: mask requested without a mask file");
            FMVD_HIP(hipMalloc(&dmask, sizeof(float) * tplane));
            FMVD_HIP(hipHostMalloc(&hmask, sizeof(float) * tplane, hipHostMallocDefault));
            launch_mask(dmask, w, h, d, tw, th, td, M, border, zspacing, s);
            FMVD_HIP(hipMemcpyAsync(hmask, dmask, sizeof(float) * tplane, hipMemcpyDeviceToHost, s));
            FMVD_HIP(hipStreamSynchronize(s));
            FILE* mf = fopen(maskfile, "wb");
            if (!mf) throw_msg(std::string("cannot open mask file for writing: ") + maskfile);
            const size_t wr = fwrite(hmask, sizeof(float), tplane, mf);
            fclose(mf);
            if (wr != tplane) throw_msg("short write to mask file");
        }
        out = fopen(outfile, "wb");
        if (!out) throw_msg(std::string("cannot open output file for writing: ") + outfile);
        // chunk of target planes per launch (~64 MiB of output)
        int zc = (int)std::max<size_t>(1, ((size_t)64 << 20) / (sizeof(S) * tplane));
        zc = std::min(zc, td);
        FMVD_HIP(hipMalloc(&ddst, sizeof(S) * tplane * zc * 2));
        FMVD_HIP(hipHostMalloc(&hdst, sizeof(S) * tplane * zc * 2, hipHostMallocDefault));
        for (auto& e : ev) FMVD_HIP(hipEventCreateWithFlags(&e, hipEventDisableTiming));
        int pend_z = -1, pend_n = 0, pend_slot = 0;
        auto flush = [&](int slot, int n) {
            FMVD_HIP(hipEventSynchronize(ev[slot]));
            const size_t cnt = tplane * n;
            if (fwrite(hdst + tplane * zc * slot, sizeof(S), cnt, out) != cnt)
                throw_msg("short write to output file");
        };
        int slot = 0;
        for (int z0 = 0; z0 < td; z0 += zc) {
            const int n = std::min(zc, td - z0);
            S* dd = ddst + tplane * zc * slot;
            launch_transform<S>(dsrc, w, h, d, dd, tw, th, z0, n, M, s);
            FMVD_HIP(hipMemcpyAsync(hdst + tplane * zc * slot, dd, sizeof(S) * tplane * n,
                                    hipMemcpyDeviceToHost, s));
            FMVD_HIP(hipEventRecord(ev[slot], s));
            if (pend_z >= 0) flush(pend_slot, pend_n);
            pend_z = z0;
            pend_n = n;
            pend_slot = slot;
            slot ^= 1;
        }
        if (pend_z >= 0) flush(pend_slot, pend_n);
    } catch (...) {
        cleanup();
        throw;
    }
    cleanup();
}

void transform_volume_u16(const uint16_t* src, int w, int h, int d, uint16_t* dst, int tw, int th, int td,
                          const float* inv, hipStream_t s)
{
    check_dims(w, h, d, tw, th, td);
    if (!src || !dst || !inv) throw_msg("transform: NULL argument");
    launch_transform<uint16_t>(src, w, h, d, dst, tw, th, 0, td, to_mat(inv), s);
}

void transform_volume_u8(const uint8_t* src, int w, int h, int d, uint8_t* dst, int tw, int th, int td,
                         const float* inv, hipStream_t s)
{
    check_dims(w, h, d, tw, th, td);
    if (!src || !dst || !inv) throw_msg("transform: NULL argument");
    launch_transform<uint8_t>(src, w, h, d, dst, tw, th, 0, td, to_mat(inv), s);
}

void transform_mask(int w, int h, int d, int tw, int th, int td, const float* inv, int border, float zspacing,
                    float* out, hipStream_t s)
{
    check_dims(w, h, d, tw, th, td);
    if (!out || !inv) throw_msg("mask: NULL argument");
    launch_mask(out, w, h, d, tw, th, td, to_mat(inv), border, zspacing, s);
}

}  // namespace fmvd

extern "C" {

void transform_cuda_8(unsigned char** h_data, int w, int h, int d, int tw, int th, int td,
                      float* h_inverse, const char* outfile, int createTransformedMasks, int border,
                      float zspacing, const char* maskfile)
{
    FMVD_API_GUARD(, {
        fmvd::transform_files<uint8_t>(h_data, w, h, d, tw, th, td, h_inverse, outfile,
                                       createTransformedMasks, border, zspacing, maskfile);
    })
}

void transform_cuda_16(unsigned short** h_data, int w, int h, int d, int tw, int th, int td,
                       float* h_inverse, const char* outfile, int createTransformedMasks, int border,
                       float zspacing, const char* maskfile)
{
    FMVD_API_GUARD(, {
        fmvd::transform_files<uint16_t>(h_data, w, h, d, tw, th, td, h_inverse, outfile,
                                        createTransformedMasks, border, zspacing, maskfile);
    })
}

int fmvd_transform_device_8(const unsigned char* d_src, int w, int h, int d, unsigned char* d_dst,
                            int tw, int th, int td, const float* h_inverse, void* stream)
{
    FMVD_API_GUARD(-1, {
        fmvd::transform_volume_u8(d_src, w, h, d, d_dst, tw, th, td, h_inverse, (hipStream_t)stream);
        return 0;
    })
}

int fmvd_transform_device_16(const unsigned short* d_src, int w, int h, int d, unsigned short* d_dst,
                             int tw, int th, int td, const float* h_inverse, void* stream)
{
    FMVD_API_GUARD(-1, {
        fmvd::transform_volume_u16(d_src, w, h, d, d_dst, tw, th, td, h_inverse, (hipStream_t)stream);
        return 0;
    })
}

int fmvd_transform_mask_device(int w, int h, int d, int tw, int th, int td, const float* h_inverse,
                               int border, float zspacing, float* d_mask, void* stream)
{
    FMVD_API_GUARD(-1, {
        fmvd::transform_mask(w, h, d, tw, th, td, h_inverse, border, zspacing, d_mask, (hipStream_t)stream);
        return 0;
    })
}

}  // extern "C"
