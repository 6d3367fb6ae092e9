// The 32 -> 32 channel layers of the warm-start network on MFMA (gfx950):
// forward and input gradient.
//
// Implicit GEMM with v_mfma_f32_32x32x16_bf16, D[cout][voxel] += W[cout][cin] X[cin][voxel],
// over 27 taps x 32 input channels.  The volume is cut into columns of kCY x kCX output
// voxels; a block takes a run of consecutive (column, z) steps, dealt evenly to one block
// per CU, and walks the planes p of each column in it: the plane with its halo is staged in LDS once (the
// next one loads into registers meanwhile) and feeds the outputs z = p + 1, p, p - 1
// through the taps dz = 0, 1, 2, whose sums live in three sets of registers.  A
// wavefront computes two rows of 32 voxels: a (dy, dx, 16-channel) step reads 3 weight
// operands and 2 voxel operands from LDS for 6 MFMAs (27 LDS cycles per 32-cycle
// MFMA and SIMD), where one operand of each per MFMA would need 64.  Every output
// sums its taps in the order dz, dy, dx, channel half.
//
// The output has the voxel on the lane and four consecutive channels per register
// quad, so a voxel's channels are packed in registers and stored in 16-byte pieces.
//
// Per layer at 8 x 64 x 128 x 128 (464 GFLOP): forward 2230 -> 458 us (1.01 PFLOP/s; a
// bf16 GEMM of 8192^3 reaches 1.24 on this card), input gradient with its relu mask
// 3433 + 793 -> 646 us (3.25 GB moved, 5.0 TB/s).  Before, a wavefront loaded one
// operand of each per MFMA, the voxels' from global memory 27 times.
#include <hip/hip_runtime.h>
#include <stdint.h>

#include <algorithm>

#include "hip_check.hpp"
#include "net.hpp"
#include "net_device.hpp"

namespace fmvd {
namespace net {

constexpr int kCY = 16, kCX = 32;             // output tile of one plane
constexpr int kHY = kCY + 2, kHX = kCX + 2;   // with its halo
constexpr int kPitch = 40;                    // LDS row pitch in voxels (a multiple of 8)
constexpr int kVB = 2 * kC;                   // bytes of one voxel
constexpr int kRow = kPitch * kVB, kPlane = kHY * kRow;
constexpr int kThreads = 512;                 // 8 wavefronts x 2 rows
constexpr int kPieces = (kHY * kHX * 4 + kThreads - 1) / kThreads;
constexpr int kTapBytes = kC * kC * 2;

struct Tile {
    int n, y0, x0;
};

// Plane z of a tile with its halo: 16-byte pieces, zero outside the volume.
__device__ __forceinline__ void load_plane(uint4* r, const uint16_t* __restrict__ in, const Geo& g, const Tile& t, int z)
{
#pragma unroll
    for (int i = 0; i < kPieces; ++i) {
        const int e = threadIdx.x + kThreads * i, v = e >> 2;
        const int y = t.y0 + v / kHX - 1, x = t.x0 + v % kHX - 1;
        r[i] = make_uint4(0, 0, 0, 0);
        if (v < kHY * kHX && y >= 0 && y < g.H && x >= 0 && x < g.W)
            r[i] = reinterpret_cast<const uint4*>(in + g.vox(t.n, z, y, x) * kC)[e & 3];
    }
}
__device__ __forceinline__ void store_plane(char* plane, const uint4* r)
{
#pragma unroll
    for (int i = 0; i < kPieces; ++i) {
        const int e = threadIdx.x + kThreads * i, v = e >> 2, y = v / kHX, x = v % kHX;
        if (v < kHY * kHX) *reinterpret_cast<uint4*>(plane + y * kRow + x * kVB + (((e & 3) ^ slot_swizzle(x)) << 4)) = r[i];
    }
}

// All taps from one plane: acc[dz][t] += W X for the wavefront's rows t.
__device__ __forceinline__ void plane_taps(f32x16 (*acc)[2], const char* plane, const char* weights, const int (*xo)[2],
                                           const int* wo)
{
#pragma unroll 1
    for (int dy = 0; dy < 3; ++dy, plane += kRow, weights += 3 * kTapBytes)
#pragma unroll
        for (int dx = 0; dx < 3; ++dx)
#pragma unroll
            for (int kc = 0; kc < 2; ++kc) {
                bf16x8 x[2];
#pragma unroll
                for (int t = 0; t < 2; ++t)
                    x[t] = *reinterpret_cast<const bf16x8*>(plane + xo[dx][kc] + t * kRow);
#pragma unroll
                for (int dz = 0; dz < 3; ++dz) {
                    const bf16x8 w =
                        *reinterpret_cast<const bf16x8*>(weights + wo[kc] + (dz * 9 + dx) * kTapBytes);
#pragma unroll
                    for (int t = 0; t < 2; ++t)
                        acc[dz][t] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(w, x[t], acc[dz][t], 0, 0, 0);
                }
            }
}

// kForward:  r = relu(acc + b) in bf16, out = in + r
// kTrain:    the same, and relu[voxel] gets the bits r > 0
// kGradient: dh += acc (FP32; stored while keep_dh), out = bf16(dh) where the bits of relu are
//            set: the masked gradient of the layer below (weights given flipped and transposed)
enum ConvMode { kForward, kTrain, kGradient };
template <ConvMode MODE>
__global__ __launch_bounds__(kThreads, 2) void conv32_kernel(const uint16_t* __restrict__ in, Geo g,
                                                             const uint16_t* __restrict__ wt,
                                                             const float* __restrict__ bias, uint32_t* relu,
                                                             float* __restrict__ dh, int keep_dh,
                                                             uint16_t* __restrict__ out, int steps)
{
    __shared__ __attribute__((aligned(16))) char planes[2 * kPlane];
    __shared__ __attribute__((aligned(16))) char weights[27 * kTapBytes];
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6, m = lane & 31, kh = lane >> 5;

    for (int i = threadIdx.x; i < 27 * kTapBytes / 16; i += kThreads) {
        const int row = i >> 2;  // (tap, cout)
        *reinterpret_cast<uint4*>(weights + row * kVB + (((i & 3) ^ slot_swizzle(row & 31)) << 4)) =
            reinterpret_cast<const uint4*>(wt)[i];
    }
    // this lane's voxel operands (row 2 wave, tap dx, channel half kc) and weight operands
    int xo[3][2], wo[2];
#pragma unroll
    for (int kc = 0; kc < 2; ++kc) {
        wo[kc] = m * kVB + (((2 * kc + kh) ^ slot_swizzle(m)) << 4);
#pragma unroll
        for (int dx = 0; dx < 3; ++dx)
            xo[dx][kc] = 2 * wave * kRow + (m + dx) * kVB + (((2 * kc + kh) ^ slot_swizzle(m + dx)) << 4);
    }
    __shared__ __attribute__((aligned(16))) float bs[kC];
    if (MODE != kGradient && threadIdx.x < kC) bs[threadIdx.x] = bias[threadIdx.x];

    const unsigned b = xcd_block(blockIdx.x, gridDim.x);
    const int s0 = (int)((long)steps * b / gridDim.x), s1 = (int)((long)steps * (b + 1) / gridDim.x);
    const int nx = (g.W + kCX - 1) / kCX, ny = (g.H + kCY - 1) / kCY;
    uint4 pre[kPieces];
    uint2 res[2][4];
    f32x16 acc[3][2];
    // Step p multiplies plane p, stores plane p + 1 where plane p - 1 was (its last readers
    // passed the barrier that ended step p - 1) and completes the outputs z = p - 1, whose inputs
    // (the residual) step p - 1 kept in registers: one barrier per plane.
    for (int s = s0; s < s1;) {
        const int col = s / g.D, za = s % g.D, zb = min(g.D, za + (s1 - s));  // outputs [za, zb) of one column
        const Tile t{col / (nx * ny), (col / nx) % ny * kCY, col % nx * kCX};
        const int x = t.x0 + m, pa = max(za - 1, 0);
        s += zb - za;
        load_plane(pre, in, g, t, pa);
        __syncthreads();  // the last column's readers are done
        store_plane(planes + (pa & 1) * kPlane, pre);
#pragma unroll
        for (int i = 0; i < 3; ++i) acc[i][0] = acc[i][1] = f32x16{};
        __syncthreads();
        for (int p = pa; p <= zb; ++p) {
            const int z = p - 1;  // the output that this plane completes
            const bool next = p < zb && p + 1 < g.D;
            if (next) load_plane(pre, in, g, t, p + 1);
            // dh of the completed rows: the first row's is loaded behind the matrix
            // products, the second's (no registers left for it) behind the first's epilogue
            float4 d[2][4];
            uint32_t bits[2];
            auto load_dh = [&](int r) {
                const int y = t.y0 + 2 * wave + r;
                if (z < za || y >= g.H || x >= g.W) return;
                const long v = g.vox(t.n, z, y, x);
                bits[r] = relu[v];
#pragma unroll
                for (int q = 0; q < 4; ++q) d[r][q] = reinterpret_cast<const float4*>(dh + v * kC)[2 * q + kh];
            };
            if constexpr (MODE == kGradient) load_dh(0);
            // (at a segment's ends the sums of outputs outside it are dropped)
            if (p < g.D) plane_taps(acc, planes + (p & 1) * kPlane, weights, xo, wo);
            if (next) store_plane(planes + ((p + 1) & 1) * kPlane, pre);
            if constexpr (MODE == kGradient) load_dh(1);
            if (z >= za) {
#pragma unroll
                for (int r = 0; r < 2; ++r) {
                    const int y = t.y0 + 2 * wave + r;
                    if (y >= g.H) continue;  // wave-uniform
                    const long v = g.vox(t.n, z, y, x);
                    uint32_t c[4][2], pos = 0;
#pragma unroll
                    for (int q = 0; q < 4; ++q) {
                        uint16_t o[4];
                        if constexpr (MODE == kGradient) {
                            const float e[4] = {d[r][q].x + acc[2][r][4 * q], d[r][q].y + acc[2][r][4 * q + 1],
                                                d[r][q].z + acc[2][r][4 * q + 2], d[r][q].w + acc[2][r][4 * q + 3]};
                            if (keep_dh && x < g.W)
                                reinterpret_cast<float4*>(dh + v * kC)[2 * q + kh] = make_float4(e[0], e[1], e[2], e[3]);
#pragma unroll
                            for (int i = 0; i < 4; ++i)
                                o[i] = (bits[r] >> (8 * q + 4 * kh + i)) & 1 ? f2bf(e[i]) : (uint16_t)0;
                        } else {
                            const float4 bv = *reinterpret_cast<const float4*>(bs + 8 * q + 4 * kh);
                            const float be[4] = {bv.x, bv.y, bv.z, bv.w};
                            const uint2 h = res[r][q];
                            const uint16_t hi[4] = {(uint16_t)h.x, (uint16_t)(h.x >> 16), (uint16_t)h.y, (uint16_t)(h.y >> 16)};
#pragma unroll
                            for (int i = 0; i < 4; ++i) {
                                const uint16_t rb = f2bf(fmaxf(acc[2][r][4 * q + i] + be[i], 0.f));
                                if (MODE == kTrain && rb) pos |= 1u << (8 * q + 4 * kh + i);
                                o[i] = f2bf(bf2f(hi[i]) + bf2f(rb));
                            }
                        }
                        c[q][0] = o[0] | (uint32_t)o[1] << 16;
                        c[q][1] = o[2] | (uint32_t)o[3] << 16;
                    }
                    if constexpr (MODE == kTrain) {
                        const auto both = __builtin_amdgcn_permlane32_swap(pos, pos, false, false);
                        pos = both[0] | both[1];
                    }
                    // (lanes l and l + 32 hold one voxel: they leave together)
                    if (x < g.W) {
                        store_voxel(out + v * kC, c, kh);
                        if (MODE == kTrain && kh == 0) relu[v] = pos;
                    }
                }
            }
            if constexpr (MODE != kGradient) {
#pragma unroll
                for (int r = 0; r < 2; ++r)
#pragma unroll
                    for (int q = 0; q < 4; ++q)
                        res[r][q] = *reinterpret_cast<const uint2*>(planes + (p & 1) * kPlane + (2 * wave + r + 1) * kRow +
                                                                   (m + 1) * kVB + ((q ^ slot_swizzle(m + 1)) << 4) + 8 * kh);
            }
            acc[2][0] = acc[1][0];
            acc[2][1] = acc[1][1];
            acc[1][0] = acc[0][0];
            acc[1][1] = acc[0][1];
            acc[0][0] = acc[0][1] = f32x16{};
            if (next) __syncthreads();
        }
    }
}

template <ConvMode MODE>
static void launch_conv32(const uint16_t* in, Dims d, const uint16_t* wt, const float* bias, uint32_t* relu, float* dh,
                          bool keep_dh, uint16_t* out, hipStream_t s)
{
    const long tiles = (long)d.N * ((d.H + kCY - 1) / kCY) * ((d.W + kCX - 1) / kCX);
    if (tiles * d.D > 0x7fffffffL) throw_msg("network: volume too large");
    // a block's LDS (144 KB) allows one per CU
    const int steps = (int)(tiles * d.D), blocks = std::min(steps, 256);
    conv32_kernel<MODE><<<(unsigned)blocks, kThreads, 0, s>>>(in, geo(d), wt, bias, relu, dh, keep_dh ? 1 : 0, out, steps);
    FMVD_LAUNCH_CHECK();
}

void launch_conv32_fwd(const uint16_t* in, Dims d, const uint16_t* wf_layer, const float* bias, uint32_t* relu,
                       uint16_t* hout, hipStream_t s)
{
    if (relu) launch_conv32<kTrain>(in, d, wf_layer, bias, relu, nullptr, false, hout, s);
    else launch_conv32<kForward>(in, d, wf_layer, bias, nullptr, nullptr, false, hout, s);
}
void launch_conv32_dgrad(const uint16_t* g, Dims d, const uint16_t* wt_layer, const uint32_t* relu, float* dh,
                         bool keep_dh, uint16_t* gout, hipStream_t s)
{
    launch_conv32<kGradient>(g, d, wt_layer, nullptr, const_cast<uint32_t*>(relu), dh, keep_dh, gout, s);
}

}  // namespace net
}  // namespace fmvd
