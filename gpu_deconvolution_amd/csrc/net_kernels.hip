// Warm-start network kernels (gfx950): a 6-layer 3-D residual conv net with
// 32 channels and 3x3x3 kernels, bfloat16 weights and activations, FP32
// accumulation.  No counterpart in the reference.
//
// Layout: activations are voxel-major, channel-fastest: act[v][32] bf16 with
// v = ((n * D + z) * H + y) * W + x (n = sample of a batch).  Weights of a
// 32->32 layer are [tap][cout][cin] bf16 (tap = (dz*3 + dy)*3 + dx reads
// voxel (z+dz-1, y+dy-1, x+dx-1); zero padding at the volume faces).
//
// The four 32->32 layers (98% of the work) run on MFMA (net_conv32.hip), their
// weight gradients and those of the edge layers too (net_wgrad.hip).  The
// 2->32 input layer and the 32->1 output layer's input gradient use the FP32
// matrix instruction, the output layer the bf16 one for inference and the VALU
// for training.
#include <hip/hip_runtime.h>
#include <stdint.h>

#include <algorithm>
#include <cmath>

#include "hip_check.hpp"
#include "net.hpp"
#include "net_device.hpp"

namespace fmvd {
namespace net {

// ------------------------------------------------------------ MFMA check
// D = A (32 x 16) * B (16 x 32) for a unit test of the operand layout:
// lane l supplies A[l%32][8(l/32)+j] and B[8(l/32)+j][l%32] (j < 8) and
// receives D[8(r/4) + 4(l/32) + r%4][l%32] in element r (r < 16).
__global__ void mfma_layout_kernel(const uint16_t* __restrict__ A, const uint16_t* __restrict__ B,
                                   float* __restrict__ Dm)
{
    const int l = threadIdx.x;
    bf16x8 a, b;
    for (int j = 0; j < 8; ++j) {
        const uint16_t av = A[(l % 32) * 16 + 8 * (l / 32) + j];
        const uint16_t bv = B[(8 * (l / 32) + j) * 32 + (l % 32)];
        a[j] = __builtin_bit_cast(__bf16, av);
        b[j] = __builtin_bit_cast(__bf16, bv);
    }
    f32x16 acc = {};
    acc = __builtin_amdgcn_mfma_f32_32x32x16_bf16(a, b, acc, 0, 0, 0);
    for (int r = 0; r < 16; ++r) Dm[(8 * (r / 4) + 4 * (l / 32) + r % 4) * 32 + (l % 32)] = acc[r];
}

// ------------------------------------------------------------ input layer
// views (u16, V volumes of D x H x W per sample) -> x (bf16, 2 channels):
// mean of the even-index views, mean of the odd-index views, over scale.
__global__ void prep_input_kernel(const uint16_t* const* __restrict__ views, int nviews, Geo g,
                                  const float* __restrict__ inv_scale, uint16_t* __restrict__ x)
{
    const long per = (long)g.D * g.H * g.W;
    const long i = (long)blockIdx.x * blockDim.x + threadIdx.x;
    const int n = blockIdx.y;
    if (i >= per) return;
    float se = 0.f, so = 0.f;
    int ne = 0, no = 0;
    for (int v = 0; v < nviews; ++v) {
        const float s = (float)views[n * nviews + v][i];
        if (v & 1) {
            so += s;
            ++no;
        } else {
            se += s;
            ++ne;
        }
    }
    const float e = se / (float)ne, o = no ? so / (float)no : e;
    const float k = inv_scale[n];
    x[2 * (n * per + i)] = f2bf(e * k);
    x[2 * (n * per + i) + 1] = f2bf(o * k);
}

// The input layer and the output layer's input gradient take one dword of each neighbour
// and give 32 channels: a block stages the box of kEZ x kEY x kEX voxels with its halo
// in LDS once, and a wavefront computes rows of 32 voxels on MFMA.  Walking planes
// would save only re-reads of the halo (0.8 dwords a voxel next to the 16 and 48 written).
// Where the boxes are too few for the chip, several blocks (`parts`) stage one and share its rows: a
// wavefront would else compute 16 of them in turn (24 us before boxes, 39 with one block a box, 8.7 with
// up to 16: 2 x 16 x 32 x 32).
constexpr int kEX = 32, kEY = 16, kEZ = 4, kEThreads = 256;
constexpr int kEHX = kEX + 2, kEHY = kEY + 2, kEHZ = kEZ + 2, kEBox = kEHZ * kEHY * kEHX;

struct EdgeTile {
    int n, z, y, x, row;  // row: the block's first row
};
__device__ __forceinline__ EdgeTile edge_tile(const Geo& g, int parts)
{
    const int nx = (g.W + kEX - 1) / kEX, ny = (g.H + kEY - 1) / kEY, nz = (g.D + kEZ - 1) / kEZ;
    int b = (int)xcd_block(blockIdx.x, gridDim.x);
    EdgeTile t;
    t.row = b % parts * (kEThreads / 64);
    b /= parts;
    t.x = b % nx * kEX;
    b /= nx;
    t.y = b % ny * kEY;
    b /= ny;
    t.z = b % nz * kEZ;
    t.n = b / nz;
    return t;
}
template <typename Put>
__device__ __forceinline__ void load_box(const uint32_t* __restrict__ in, const Geo& g, const EdgeTile& t, Put put)
{
    constexpr int kLoads = (kEBox + kEThreads - 1) / kEThreads;
    uint32_t r[kLoads];
#pragma unroll
    for (int i = 0; i < kLoads; ++i) {
        const int e = threadIdx.x + kEThreads * i;
        const int z = t.z + e / (kEHY * kEHX) - 1, y = t.y + e / kEHX % kEHY - 1, x = t.x + e % kEHX - 1;
        r[i] = 0;
        if (e < kEBox && z >= 0 && z < g.D && y >= 0 && y < g.H && x >= 0 && x < g.W) r[i] = in[g.vox(t.n, z, y, x)];
    }
#pragma unroll
    for (int i = 0; i < kLoads; ++i) {
        const int e = threadIdx.x + kEThreads * i;
        if (e < kEBox) put(e, r[i]);
    }
}
// position in the box, relative to its first voxel, of the neighbour that a tap reads
__device__ constexpr int box_offset(int tap) { return (tap / 9 * kEHY + tap / 3 % 3) * kEHX + tap % 3; }

// Layer 1 (2 -> 32): h1 = relu(conv(x, W1) + b1); W1 is FP32 [27][32][2] (bf16-rounded
// values).  relu (if wanted): the bits h1 > 0.  A tap's two products and their FP32 sum are one
// v_mfma_f32_32x32x2_f32 from zero, which the VALU adds to the taps' sum in their order: the
// rounding of the definition.  (The bf16 instruction would take all 54 products in 4 steps, but it
// truncates inside a sum: 5 % of two-product sums differ in their last bit.)
// Weights and inputs are finite (taps outside the volume multiply by zero).
// At 8 x 64 x 128 x 128: 619 us on the VALU (three instructions a tap and channel, 553 us of issue),
// 470 here: a tap's 64 cycles of products and 64 of additions a wavefront do not overlap
// (368 us; issuing the next tap's products first changed nothing).  At most 128 registers,
// or the products land in accumulation registers and a copy each costs a third again (585 us).
__global__ __launch_bounds__(kEThreads, 4) void conv_in_kernel(const uint32_t* __restrict__ x, Geo g, int parts,
                                                               const float* __restrict__ w,
                                                               const float* __restrict__ b,
                                                               uint16_t* __restrict__ h, uint32_t* __restrict__ relu)
{
    __shared__ uint32_t box[2 * kEBox];  // FP32: channel 0, channel 1
    const EdgeTile t = edge_tile(g, parts);
    const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), m = lane & 31, kh = lane >> 5;
    float wk[27];
#pragma unroll
    for (int k = 0; k < 27; ++k) wk[k] = w[(k * 32 + m) * 2 + kh];
    f32x16 bias;
#pragma unroll
    for (int r = 0; r < 16; ++r) bias[r] = b[8 * (r / 4) + 4 * kh + r % 4];
    load_box(x, g, t, [&](int e, uint32_t v) {
        box[e] = v << 16;
        box[kEBox + e] = v & 0xffff0000u;
    });
    __syncthreads();
    const int xx = t.x + m;
    for (int row = t.row + wave; row < kEZ * kEY; row += kEThreads / 64 * parts) {
        const int dz = row / kEY, dy = row % kEY, zz = t.z + dz, yy = t.y + dy;
        if (zz >= g.D || yy >= g.H) continue;  // wave-uniform
        const uint32_t* v0 = box + kh * kEBox + (dz * kEHY + dy) * kEHX + m;
        f32x16 acc = bias;
#pragma unroll
        for (int k = 0; k < 27; ++k)
            acc += __builtin_amdgcn_mfma_f32_32x32x2f32(wk[k], __uint_as_float(v0[box_offset(k)]), f32x16{}, 0, 0, 0);
        uint32_t c[4][2], pos = 0;
#pragma unroll
        for (int q = 0; q < 4; ++q) {
            uint16_t o[4];
#pragma unroll
            for (int i = 0; i < 4; ++i) {
                o[i] = f2bf(fmaxf(acc[4 * q + i], 0.f));
                if (o[i]) pos |= 1u << (8 * q + 4 * kh + i);
            }
            c[q][0] = o[0] | (uint32_t)o[1] << 16;
            c[q][1] = o[2] | (uint32_t)o[3] << 16;
        }
        const auto both = __builtin_amdgcn_permlane32_swap(pos, pos, false, false);
        // (lanes l and l + 32 hold one voxel: they leave together)
        if (xx < g.W) {
            const long v = g.vox(t.n, zz, yy, xx);
            store_voxel(h + v * kC, c, kh);
            if (relu && kh == 0) relu[v] = both[0] | both[1];
        }
    }
}

// Layer 6 (32 -> 1): y = conv(h5, W6) + b6 + (x0 + x1) / 2 (FP32 out), in two variants.
//
// conv_out_kernel serves training: an output is one chain of FP32 FMAs, as the
// gradients' bf16 roundings were always fed (a last-bit change of y moves dy and flips some of
// them).  A block
// walks the planes p of a kOY x kOX column, one voxel per thread: the plane with its
// halo is staged in LDS (the next one loads meanwhile), and each of a thread's 9
// neighbours in it is read and converted once for its three taps dz, whose sums belong to
// the outputs p + 1, p, p - 1; the weights are uniform and come through scalar
// loads.  An output sums in the order dz, dy, dx, channel.  One voxel per thread with
// 27 x 64 bytes from L1 and the weights from LDS took 843 us at 8 x 64 x 128 x 128; this 425,
// of which the VALU's 1152 instructions a voxel are 246.
constexpr int kOY = 8, kOX = 32, kOHX = kOX + 2, kOHV = (kOY + 2) * kOHX, kOPitch = 40;
constexpr int kOPieces = (kOHV * 4 + 255) / 256, kOPlane = (kOY + 2) * kOPitch * 64;
__global__ __launch_bounds__(256) void conv_out_kernel(const uint16_t* __restrict__ h, const uint32_t* __restrict__ x,
                                                       Geo g, const float* __restrict__ w,
                                                       const float* __restrict__ b, float* __restrict__ y, int nseg)
{
    __shared__ __attribute__((aligned(16))) char planes[2][kOPlane];
    const int nx = (g.W + kOX - 1) / kOX, ny = (g.H + kOY - 1) / kOY;
    const unsigned bid = xcd_block(blockIdx.x, gridDim.x);
    const int seg = bid % nseg, tile = bid / nseg, n = tile / (nx * ny);
    const int y0 = (tile / nx) % ny * kOY, x0 = tile % nx * kOX;
    const int za = (int)((long)g.D * seg / nseg), zb = (int)((long)g.D * (seg + 1) / nseg);
    const int row = threadIdx.x / kOX, col = threadIdx.x % kOX;

    uint4 pre[kOPieces];
    auto load = [&](int z) {
#pragma unroll
        for (int i = 0; i < kOPieces; ++i) {
            const int e = threadIdx.x + 256 * i, v = e >> 2, yy = y0 + v / kOHX - 1, xx = x0 + v % kOHX - 1;
            pre[i] = make_uint4(0, 0, 0, 0);
            if (v < kOHV && yy >= 0 && yy < g.H && xx >= 0 && xx < g.W)
                pre[i] = reinterpret_cast<const uint4*>(h + g.vox(n, z, yy, xx) * 32)[e & 3];
        }
    };
    auto store = [&](int z) {
#pragma unroll
        for (int i = 0; i < kOPieces; ++i) {
            const int e = threadIdx.x + 256 * i, v = e >> 2, yy = v / kOHX, xx = v % kOHX;
            if (v < kOHV)
                *reinterpret_cast<uint4*>(planes[z & 1] + (yy * kOPitch + xx) * 64 + (((e & 3) ^ slot_swizzle(xx)) << 4)) =
                    pre[i];
        }
    };
    const float bias = b[0];
    float a0 = bias, a1 = bias, a2 = bias;
    const int pa = max(za - 1, 0);
    load(pa);
    store(pa);
    __syncthreads();
    for (int p = pa; p <= zb; ++p) {
        const bool next = p < zb && p + 1 < g.D;
        if (next) load(p + 1);
        if (p < g.D) {
#pragma unroll 1
            for (int dy = 0; dy < 3; ++dy)
#pragma unroll
                for (int dx = 0; dx < 3; ++dx) {
                    const char* v = planes[p & 1] + ((row + dy) * kOPitch + col + dx) * 64;
                    const float* wk = w + (dy * 3 + dx) * 32;
#pragma unroll
                    for (int q = 0; q < 4; ++q) {
                        const uint4 u = *reinterpret_cast<const uint4*>(v + ((q ^ slot_swizzle(col + dx)) << 4));
                        const uint32_t wds[4] = {u.x, u.y, u.z, u.w};
#pragma unroll
                        for (int j = 0; j < 8; ++j) {
                            const float f = bf2f((uint16_t)(wds[j / 2] >> (16 * (j & 1))));
                            a0 += f * wk[8 * q + j];
                            a1 += f * wk[9 * 32 + 8 * q + j];
                            a2 += f * wk[18 * 32 + 8 * q + j];
                        }
                    }
                }
        }
        if (next) store(p + 1);
        const int z = p - 1, yy = y0 + row, xx = x0 + col;
        if (z >= za && yy < g.H && xx < g.W) {
            const long v = g.vox(n, z, yy, xx);
            const uint32_t u = x[v];
            y[v] = a2 + 0.5f * (bf2f((uint16_t)u) + bf2f((uint16_t)(u >> 16)));
        }
        a2 = a1;
        a1 = a0;
        a0 = bias;
        if (next) __syncthreads();
    }
}

// conv_out_mfma_kernel serves inference, where y is the result (W6 is FP32 of bf16-rounded
// values, so bf16 operands are exact; the products' sums are FP32, as in the 32 -> 32 layers).
// A block walks the planes of the same columns.  For every voxel of the plane with its halo,
// v_mfma_f32_32x32x16_bf16 makes the products of its 32 channels with all 27 taps at once,
// P[tap][voxel]: a lane's operands are 16-byte pieces of a voxel, loaded from global
// memory one plane ahead.  P goes through LDS, and a thread adds the 27 that belong to the
// outputs p + 1, p, p - 1 of its voxel, in the order dz, dy, dx.  Over 96 x 300 x 260:
// 463 us with the chains, 157 here; the error of y against 64 bits falls (rms 0.97e-6 against
// 1.31e-6 at 8 x 24 x 40 with |y| to 232 and the same h5, 1.47e-6 against 2.44e-6 with another).
constexpr int kOThreads = kOY * kOX;
constexpr int kOGroups = (kOHV + 31) / 32, kOWaves = kOThreads / 64, kOPer = (kOGroups + kOWaves - 1) / kOWaves;
constexpr int kPPitch = 344;  // of P's rows: rows 4 apart (the halves of a wavefront) lie 32 banks apart
static_assert(kPPitch >= kOHV && kPPitch * 4 % 64 == 32);
__global__ __launch_bounds__(kOThreads, 4) void conv_out_mfma_kernel(const uint16_t* __restrict__ h,
                                                                     const uint32_t* __restrict__ x, Geo g,
                                                                     const float* __restrict__ w,
                                                                     const float* __restrict__ b,
                                                                     float* __restrict__ y, int nseg)
{
    __shared__ float P[27 * kPPitch];
    const int nx = (g.W + kOX - 1) / kOX, ny = (g.H + kOY - 1) / kOY;
    const unsigned bid = xcd_block(blockIdx.x, gridDim.x);
    const int seg = bid % nseg, tile = bid / nseg, n = tile / (nx * ny);
    const int y0 = (tile / nx) % ny * kOY, x0 = tile % nx * kOX;
    const int za = (int)((long)g.D * seg / nseg), zb = (int)((long)g.D * (seg + 1) / nseg);
    const int row = threadIdx.x / kOX, col = threadIdx.x % kOX;
    const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), m = lane & 31, kh = lane >> 5;

    // this lane's weights: tap m, channels 16 i + 8 kh + j
    uint4 wk[2];
#pragma unroll
    for (int i = 0; i < 2; ++i) {
        uint32_t v[4];
#pragma unroll
        for (int j = 0; j < 4; ++j) {
            const float2 f = m < 27 ? reinterpret_cast<const float2*>(w)[(m * kC + 16 * i + 8 * kh) / 2 + j]
                                    : make_float2(0.f, 0.f);
            v[j] = __float_as_uint(f.x) >> 16 | (__float_as_uint(f.y) & 0xffff0000u);
        }
        wk[i] = make_uint4(v[0], v[1], v[2], v[3]);
    }
    // the voxels of this wavefront's groups: wave, wave + kOWaves, ...
    uint4 pre[kOPer][2];
    auto load = [&](int z) {
#pragma unroll
        for (int k = 0; k < kOPer; ++k) {
            const int v = (wave + kOWaves * k) * 32 + m, yy = y0 + v / kOHX - 1, xx = x0 + v % kOHX - 1;
            pre[k][0] = pre[k][1] = make_uint4(0, 0, 0, 0);
            if (v < kOHV && yy >= 0 && yy < g.H && xx >= 0 && xx < g.W) {
                const uint4* q = reinterpret_cast<const uint4*>(h + g.vox(n, z, yy, xx) * kC);
                pre[k][0] = q[kh];
                pre[k][1] = q[2 + kh];
            }
        }
    };
    const float bias = b[0];
    float a0 = bias, a1 = bias, a2 = bias;
    const int pa = max(za - 1, 0);
    load(pa);
    for (int p = pa; p <= zb; ++p) {
        const int z = p - 1, yy = y0 + row, xx = x0 + col;  // the output that this plane completes
        const bool done = z >= za && yy < g.H && xx < g.W;
        const long vo = g.vox(n, z, yy, xx);
        const uint32_t u = done ? x[vo] : 0;
        if (p < g.D) {
            f32x16 acc[kOPer];
#pragma unroll
            for (int k = 0; k < kOPer; ++k) {
                acc[k] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(__builtin_bit_cast(bf16x8, wk[0]),
                                                                 __builtin_bit_cast(bf16x8, pre[k][0]), f32x16{}, 0, 0, 0);
                acc[k] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(__builtin_bit_cast(bf16x8, wk[1]),
                                                                 __builtin_bit_cast(bf16x8, pre[k][1]), acc[k], 0, 0, 0);
            }
            if (p < zb && p + 1 < g.D) load(p + 1);
            __syncthreads();  // the last plane's readers are done
#pragma unroll
            for (int k = 0; k < kOPer; ++k) {
                const int v = (wave + kOWaves * k) * 32 + m;
                if (v < kOHV) {
#pragma unroll
                    for (int r = 0; r < 16; ++r) {
                        const int tap = 8 * (r / 4) + 4 * kh + r % 4;
                        if (tap < 27) P[tap * kPPitch + v] = acc[k][r];
                    }
                }
            }
            __syncthreads();
            const float* v = P + row * kOHX + col;
#pragma unroll
            for (int k = 0; k < 9; ++k) {
                const int at = k / 3 * kOHX + k % 3;
                a0 += v[k * kPPitch + at];
                a1 += v[(9 + k) * kPPitch + at];
                a2 += v[(18 + k) * kPPitch + at];
            }
        }
        if (done) y[vo] = a2 + 0.5f * (bf2f((uint16_t)u) + bf2f((uint16_t)(u >> 16)));
        a2 = a1;
        a1 = a0;
        a0 = bias;
    }
}

// ------------------------------------------------------- backward helpers
// loss partials (FP64) and dy = 2 (y - t) / count
__global__ void loss_kernel(const float* __restrict__ y, const float* __restrict__ t, long count,
                            float* __restrict__ dy, double* __restrict__ partial)
{
    __shared__ double red[256];
    double s = 0.0;
    for (long i = (long)blockIdx.x * blockDim.x + threadIdx.x; i < count; i += (long)gridDim.x * blockDim.x) {
        const double d = (double)y[i] - (double)t[i];
        s += d * d;
        dy[i] = (float)(2.0 * d / (double)count);
    }
    red[threadIdx.x] = s;
    __syncthreads();
    for (int k = 128; k > 0; k >>= 1) {
        if (threadIdx.x < k) red[threadIdx.x] += red[threadIdx.x + k];
        __syncthreads();
    }
    if (threadIdx.x == 0) partial[blockIdx.x] = red[0];
}

// dh5[v][c] = sum_k dy[v - off(k)] W6[k][c]  (FP32 out), and the masked bf16 gradient of
// layer 5 (relu: its bits r > 0).  Products and sums are FP32: v_mfma_f32_32x32x2_f32, two
// taps at a time in the order dz, dy, dx.  The masks are staged too: a load between the rows
// would wait for the stores of the row before it.
// At 8 x 64 x 128 x 128 (1.68 GB moved): 719 us with a voxel per thread, whose 128 and 64 bytes
// left in pieces, 490 here (3.4 TB/s); 554 with the masks loaded row by row.
__global__ __launch_bounds__(kEThreads, 4) void out_dgrad_kernel(const uint32_t* __restrict__ dy, Geo g, int parts,
                                                                 const float* __restrict__ w,
                                                                 const uint32_t* __restrict__ relu,
                                                                 float* __restrict__ dh, uint16_t* __restrict__ gout)
{
    __shared__ uint32_t box[kEBox], mask[kEZ * kEY * kEX];
    const EdgeTile t = edge_tile(g, parts);
    const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), m = lane & 31, kh = lane >> 5;
    float wk[14];
    int off[14];
#pragma unroll
    for (int i = 0; i < 14; ++i) {
        const int tap = 2 * i + kh;
        wk[i] = tap < 27 ? w[tap * 32 + m] : 0.f;
        off[i] = kh ? box_offset(2 * i + 1 < 27 ? 25 - 2 * i : 0) : box_offset(26 - 2 * i);
    }
    uint32_t mk[kEZ * kEY * kEX / kEThreads];
#pragma unroll
    for (int i = 0; i < kEZ * kEY * kEX / kEThreads; ++i) {
        const int e = threadIdx.x + kEThreads * i, z = t.z + e / (kEY * kEX), y = t.y + e / kEX % kEY, x = t.x + e % kEX;
        mk[i] = z < g.D && y < g.H && x < g.W ? relu[g.vox(t.n, z, y, x)] : 0;
    }
    load_box(dy, g, t, [&](int e, uint32_t v) { box[e] = v; });
#pragma unroll
    for (int i = 0; i < kEZ * kEY * kEX / kEThreads; ++i) mask[threadIdx.x + kEThreads * i] = mk[i];
    __syncthreads();
    const int xx = t.x + m;
    for (int row = t.row + wave; row < kEZ * kEY; row += kEThreads / 64 * parts) {
        const int dz = row / kEY, ry = row % kEY, zz = t.z + dz, yy = t.y + ry;
        if (zz >= g.D || yy >= g.H) continue;  // wave-uniform
        const long v = g.vox(t.n, zz, yy, xx);
        const uint32_t bits = mask[row * kEX + m];
        const uint32_t* v0 = box + (dz * kEHY + ry) * kEHX + m;
        f32x16 acc = {};
#pragma unroll
        for (int i = 0; i < 14; ++i) {
            float d = __uint_as_float(v0[off[i]]);
            if (i == 13 && kh) d = 0.f;
            acc = __builtin_amdgcn_mfma_f32_32x32x2f32(wk[i], d, acc, 0, 0, 0);
        }
        uint32_t c[4][2];
#pragma unroll
        for (int q = 0; q < 4; ++q) {
            uint16_t o[4];
#pragma unroll
            for (int i = 0; i < 4; ++i) o[i] = (bits >> (8 * q + 4 * kh + i)) & 1 ? f2bf(acc[4 * q + i]) : (uint16_t)0;
            c[q][0] = o[0] | (uint32_t)o[1] << 16;
            c[q][1] = o[2] | (uint32_t)o[3] << 16;
            if (xx < g.W)
                reinterpret_cast<float4*>(dh + v * kC)[2 * q + kh] =
                    make_float4(acc[4 * q], acc[4 * q + 1], acc[4 * q + 2], acc[4 * q + 3]);
        }
        if (xx < g.W) store_voxel(gout + v * kC, c, kh);
    }
}

// Adam on FP32 master parameters; also refreshes the bf16 copies used by
// the kernels.  Bias-corrected (Kingma & Ba 2015).
__global__ void adam_kernel(float* __restrict__ p, const float* __restrict__ gr, float* __restrict__ m,
                            float* __restrict__ v, int count, float lr, float b1, float b2, float eps, float c1,
                            float c2)
{
    const int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= count) return;
    const float gg = gr[i];
    const float mm = b1 * m[i] + (1.f - b1) * gg;
    const float vv = b2 * v[i] + (1.f - b2) * gg * gg;
    m[i] = mm;
    v[i] = vv;
    p[i] -= lr * (mm / c1) / (sqrtf(vv / c2) + eps);
}

// bf16 weight copies of the 32->32 layers: forward [k][co][ci] and the
// transposed, tap-flipped copy for the input gradient [26-k][ci][co]; FP32
// bf16-rounded copies of the small layers.
__global__ void pack_weights_kernel(const float* __restrict__ p, uint16_t* __restrict__ wf, uint16_t* __restrict__ wt,
                                    float* __restrict__ small)
{
    const int i = blockIdx.x * blockDim.x + threadIdx.x;
    const int per = 27 * 32 * 32;
    if (i < 4 * per) {
        const int l = i / per, e = i % per;
        const int k = e / 1024, co = (e / 32) % 32, ci = e % 32;
        const uint16_t b = f2bf(p[off_w(l + 1) + e]);
        wf[i] = b;
        wt[l * per + ((26 - k) * 32 + ci) * 32 + co] = b;
    }
    if (i < 27 * 32 * 2) small[i] = bf2f(f2bf(p[off_w(0) + i]));
    if (i < 27 * 32) small[27 * 64 + i] = bf2f(f2bf(p[off_w(5) + i]));
}

// Network input of a sub-volume [z0, z0+r.D) x [y0, ...) x [x0, ...) of one
// sample's views (full volumes D x H x W).
__global__ void prep_region_kernel(const uint16_t* const* __restrict__ views, int nviews, int D, int H, int W, int z0,
                                   int y0, int x0, Geo r, float inv_scale, uint16_t* __restrict__ x)
{
    const long per = (long)r.D * r.H * r.W;
    const long i = (long)blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= per) return;
    const int xx = (int)(i % r.W), yy = (int)((i / r.W) % r.H), zz = (int)(i / ((long)r.W * r.H));
    const long src = ((long)(z0 + zz) * H + (y0 + yy)) * W + (x0 + xx);
    float se = 0.f, so = 0.f;
    int ne = 0, no = 0;
    for (int v = 0; v < nviews; ++v) {
        const float s = (float)views[v][src];
        if (v & 1) {
            so += s;
            ++no;
        } else {
            se += s;
            ++ne;
        }
    }
    const float e = se / (float)ne, o = no ? so / (float)no : e;
    x[2 * i] = f2bf(e * inv_scale);
    x[2 * i + 1] = f2bf(o * inv_scale);
}

// out[z0+z][y0+y][x0+x] = max(y_region[iz0+z][iy0+y][ix0+x] * scale, floor)
__global__ void scale_out_kernel(const float* __restrict__ yr, Geo r, int H, int W, int z0, int y0, int x0, int iz0,
                                 int iy0, int ix0, int nz, int ny, int nx, float scale, float floor_value,
                                 float* __restrict__ out)
{
    const long per = (long)nz * ny * nx;
    const long i = (long)blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= per) return;
    const int xx = (int)(i % nx), yy = (int)((i / nx) % ny), zz = (int)(i / ((long)nx * ny));
    const float v = yr[r.vox(0, iz0 + zz, iy0 + yy, ix0 + xx)] * scale;
    out[((long)(z0 + zz) * H + (y0 + yy)) * W + (x0 + xx)] = fmaxf(v, floor_value);
}

// ------------------------------------------------------------ launchers
static inline unsigned nblk(long n, int t) { return (unsigned)((n + t - 1) / t); }

void launch_mfma_layout_test(const uint16_t* A, const uint16_t* B, float* D, hipStream_t s)
{
    mfma_layout_kernel<<<1, 64, 0, s>>>(A, B, D);
    FMVD_LAUNCH_CHECK();
}
void launch_prep_input(const uint16_t* const* d_views, int nviews, Dims d, const float* d_inv_scale, uint16_t* x,
                       hipStream_t s)
{
    const long per = (long)d.D * d.H * d.W;
    prep_input_kernel<<<dim3(nblk(per, 256), d.N), 256, 0, s>>>(d_views, nviews, geo(d), d_inv_scale, x);
    FMVD_LAUNCH_CHECK();
}
void launch_prep_region(const uint16_t* const* d_views, int nviews, int D, int H, int W, int z0, int y0, int x0,
                        Dims r, float inv_scale, uint16_t* x, hipStream_t s)
{
    prep_region_kernel<<<nblk(r.voxels(), 256), 256, 0, s>>>(d_views, nviews, D, H, W, z0, y0, x0, geo(r), inv_scale,
                                                              x);
    FMVD_LAUNCH_CHECK();
}
void launch_pack_weights(const float* params, uint16_t* wf, uint16_t* wt, float* small, hipStream_t s)
{
    pack_weights_kernel<<<nblk(4 * kConv32, 256), 256, 0, s>>>(params, wf, wt, small);
    FMVD_LAUNCH_CHECK();
}
// boxes x parts: up to one residency of the chip (four blocks a CU), a row a wavefront at least
static unsigned edge_blocks(Dims d, int* parts)
{
    const long n = (long)d.N * ((d.D + kEZ - 1) / kEZ) * ((d.H + kEY - 1) / kEY) * ((d.W + kEX - 1) / kEX);
    if (n > 0x7fffffffL) throw_msg("network: volume too large");
    *parts = (int)std::clamp<long>(1024 / n, 1, kEZ * kEY / (kEThreads / 64));
    return (unsigned)(n * *parts);
}
void launch_conv_in(const uint16_t* x, Dims d, const float* small, const float* params, uint16_t* h,
                    uint32_t* relu, hipStream_t s)
{
    int parts;
    const unsigned blocks = edge_blocks(d, &parts);
    conv_in_kernel<<<blocks, kEThreads, 0, s>>>(reinterpret_cast<const uint32_t*>(x), geo(d), parts, small,
                                                params + off_b(0), h, relu);
    FMVD_LAUNCH_CHECK();
}
void launch_conv_out(const uint16_t* h, const uint16_t* x, Dims d, const float* small, const float* params, float* y,
                     bool training, hipStream_t s)
{
    // segments of about 16 planes: a segment reads two planes beyond its ends; of fewer planes
    // where the blocks would leave CUs idle (2 x 16 x 32 x 32: 69 us in one segment, 16 so;
    // in every voxel on its own 14)
    const long columns = (long)d.N * ((d.H + kOY - 1) / kOY) * ((d.W + kOX - 1) / kOX);
    const int planes = (int)std::clamp<long>((columns * d.D + 511) / 512, 1, 16), nseg = (d.D + planes - 1) / planes;
    const long blocks = columns * nseg;
    if (blocks > 0x7fffffffL) throw_msg("network: volume too large");
    (training ? conv_out_kernel : conv_out_mfma_kernel)<<<(unsigned)blocks, kOThreads, 0, s>>>(
        h, reinterpret_cast<const uint32_t*>(x), geo(d), small + 27 * 64, params + off_b(5), y, nseg);
    FMVD_LAUNCH_CHECK();
}
int launch_loss(const float* y, const float* t, long count, float* dy, double* partial, hipStream_t s)
{
    const int nb = (int)std::min<long>(1024, nblk(count, 256));
    loss_kernel<<<nb, 256, 0, s>>>(y, t, count, dy, partial);
    FMVD_LAUNCH_CHECK();
    return nb;
}
void launch_out_dgrad(const float* dy, Dims d, const float* small, const uint32_t* relu, float* dh, uint16_t* gout,
                      hipStream_t s)
{
    int parts;
    const unsigned blocks = edge_blocks(d, &parts);
    out_dgrad_kernel<<<blocks, kEThreads, 0, s>>>(reinterpret_cast<const uint32_t*>(dy), geo(d), parts, small + 27 * 64,
                                                  relu, dh, gout);
    FMVD_LAUNCH_CHECK();
}
void launch_adam(float* p, const float* g, float* m, float* v, int count, float lr, int step, hipStream_t s)
{
    const float b1 = 0.9f, b2 = 0.999f;
    const float c1 = (float)(1.0 - std::pow(0.9, step)), c2 = (float)(1.0 - std::pow(0.999, step));
    adam_kernel<<<nblk(count, 256), 256, 0, s>>>(p, g, m, v, count, lr, b1, b2, 1e-8f, c1, c2);
    FMVD_LAUNCH_CHECK();
}
void launch_scale_out(const float* y, Dims r, int D, int H, int W, int z0, int y0, int x0, int iz0, int iy0,
                      int ix0, int nz, int ny, int nx, float scale, float floor_value, float* out, hipStream_t s)
{
    (void)D;
    scale_out_kernel<<<nblk((long)nz * ny * nx, 256), 256, 0, s>>>(y, geo(r), H, W, z0, y0, x0, iz0, iy0, ix0, nz,
                                                                   ny, nx, scale, floor_value, out);
    FMVD_LAUNCH_CHECK();
}

}  // namespace net
}  // namespace fmvd
