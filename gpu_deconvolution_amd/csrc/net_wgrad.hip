// Weight gradients of the warm-start network (gfx950).
//
//   dW[k][co][ci] = sum_v g[v][co] a[v + off(k)][ci],   db[co] = sum_v g[v][co]
//
// is a matrix product with the voxels as the reduction dimension.  The three
// kernels below share one scheme.  The volume is cut into columns of kWY x
// kWX voxels; a block takes a run of consecutive (column, z) steps and keeps
// all its sums in registers.  At each step the LDS holds one plane of the
// unshifted operand's tile and a ring of three planes of the shifted one
// with its one-voxel halo, so that every voxel is read from memory once per
// column (1.33 times with the halo) and used for all 27 taps from LDS; the next
// step's planes load into registers while the current one multiplies.  The
// steps are dealt evenly, so the last round of blocks is as full as the
// first.  The operands stay voxel-major: a bf16 matrix operand with the voxels along
// its reduction dimension is read from them by ds_read_b64_tr_b16, which
// transposes 4 voxels x 16 channels of a 16-lane group, at any voxel
// offset, so a tap's shift costs an address and no data movement.
#include <hip/hip_runtime.h>
#include <stdint.h>

#include <algorithm>

#include "hip_check.hpp"
#include "net.hpp"
#include "net_device.hpp"

namespace fmvd {
namespace net {

constexpr int kWY = 8, kWX = 32;             // tile of one step
constexpr int kHY = kWY + 2, kHX = kWX + 2;  // with its halo
constexpr int kPitch = 40;                   // LDS row pitch of halo tiles (voxels; a multiple of 8)
constexpr int kWThreads = 512;
constexpr int kVB = 2 * kC;                  // bytes of one 32-channel voxel
constexpr int kTileBytes = kWY * kWX * kVB;

typedef short s16x4 __attribute__((ext_vector_type(4)));

// Column of steps: sample, first row, first voxel.
struct Column {
    int n, y0, x0;
};
__device__ __forceinline__ Column column_of(int col, const Geo& g)
{
    const int nx = (g.W + kWX - 1) / kWX, ny = (g.H + kWY - 1) / kWY;
    return Column{col / (nx * ny), (col / nx) % ny * kWY, col % nx * kWX};
}

// Plane z of a column's tile of 32-channel voxels: 16-byte pieces, zero
// outside the volume, first into registers, then into LDS.
constexpr int kTilePieces = kWY * kWX * 4 / kWThreads;
__device__ __forceinline__ void load_tile(uint4* r, const uint16_t* __restrict__ a, const Geo& g, const Column& c, int z)
{
#pragma unroll
    for (int i = 0; i < kTilePieces; ++i) {
        const int e = threadIdx.x + kWThreads * i, s = e & 3, x = c.x0 + ((e >> 2) & (kWX - 1)), y = c.y0 + (e >> 7);
        r[i] = make_uint4(0, 0, 0, 0);
        if (y < g.H && x < g.W) r[i] = reinterpret_cast<const uint4*>(a + g.vox(c.n, z, y, x) * kC)[s];
    }
}
__device__ __forceinline__ void store_tile(char* lds, const uint4* r)
{
#pragma unroll
    for (int i = 0; i < kTilePieces; ++i) {
        const int e = threadIdx.x + kWThreads * i, s = e & 3, v = e >> 2;
        *reinterpret_cast<uint4*>(lds + v * kVB + ((s ^ slot_swizzle(v & (kWX - 1))) << 4)) = r[i];
    }
}

// The same for a plane with its halo (z may lie outside the volume).
constexpr int kHaloPieces = (kHY * kHX * 4 + kWThreads - 1) / kWThreads;
constexpr int kHaloBytes = kHY * kPitch * kVB;
__device__ __forceinline__ void load_halo(uint4* r, const uint16_t* __restrict__ a, const Geo& g, const Column& c, int z)
{
#pragma unroll
    for (int i = 0; i < kHaloPieces; ++i) {
        const int e = threadIdx.x + kWThreads * i, s = e & 3, v = e >> 2;
        const int y = c.y0 + v / kHX - 1, x = c.x0 + v % kHX - 1;
        r[i] = make_uint4(0, 0, 0, 0);
        if (v < kHY * kHX && z >= 0 && z < g.D && y >= 0 && y < g.H && x >= 0 && x < g.W)
            r[i] = reinterpret_cast<const uint4*>(a + g.vox(c.n, z, y, x) * kC)[s];
    }
}
__device__ __forceinline__ void store_halo(char* lds, const uint4* r)
{
#pragma unroll
    for (int i = 0; i < kHaloPieces; ++i) {
        const int e = threadIdx.x + kWThreads * i, s = e & 3, v = e >> 2, y = v / kHX, x = v % kHX;
        if (v < kHY * kHX)
            *reinterpret_cast<uint4*>(lds + (y * kPitch + x) * kVB + ((s ^ slot_swizzle(x)) << 4)) = r[i];
    }
}

// Byte offset, from a row's first voxel, of this lane's part of a transposing
// read: of the 16 voxels from column c on, lanes 0-31 receive voxels 0-7 and
// lanes 32-63 voxels 8-15 of channel lane % 32, four per read (half = 0, 1).
__device__ __forceinline__ int tr_offset(int c, int half)
{
    const int l = threadIdx.x & 63, j = l & 15;
    const int col = c + 8 * (l >> 5) + 4 * half + (j >> 2), slot = 2 * ((l >> 4) & 1) + ((j >> 1) & 1);
    return col * kVB + ((slot ^ slot_swizzle(col)) << 4) + (j & 1) * 8;
}
__device__ __forceinline__ bf16x8 read_tr(const char* lds, int off0, int off1)
{
    typedef __attribute__((address_space(3))) s16x4* lds_ptr;
    const s16x4 a = __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_ptr)(lds + off0));
    const s16x4 b = __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_ptr)(lds + off1));
    return __builtin_bit_cast(bf16x8, __builtin_shufflevector(a, b, 0, 1, 2, 3, 4, 5, 6, 7));
}

// ------------------------------------------------------------ 32 -> 32 layers
// Eight wavefronts: wavefront w accumulates the taps k = w % 4 + 4 j on rows 4 (w / 4) ... + 3
// of each tile (v_mfma_f32_32x32x16_bf16, A = g, B = shifted input); tap "27" multiplies
// by one and gives the bias sums.  One operand of g serves 7 taps, so the LDS
// delivers 1.14 operands (1 KiB each, 8 cycles) per 32-cycle MFMA and SIMD: the matrix
// cores and the LDS are about equally busy.
constexpr int kNT = 7;  // taps per wavefront
// A ring of four planes and two tiles: the next step's go where no wavefront of this
// step reads, so a step needs one barrier.
constexpr int kWgradLds = 4 * kHaloBytes + 2 * kTileBytes;
static_assert(4 * kNT * 16 * 64 * 4 <= kWgradLds);  // the second row group's sums at the end
__global__ __launch_bounds__(kWThreads, 2) void wgrad32_kernel(const uint16_t* __restrict__ gin,
                                                               const uint16_t* __restrict__ a, Geo g, int steps,
                                                               float* __restrict__ partial)
{
    __shared__ __attribute__((aligned(16))) char lds[kWgradLds];
    char* const tiles = lds + 4 * kHaloBytes;
    const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int w4 = wave & 3, rows = (wave >> 2) * (kWY / 2);
    const unsigned b = xcd_block(blockIdx.x, gridDim.x);
    const int s0 = (int)((long)steps * b / gridDim.x), s1 = (int)((long)steps * (b + 1) / gridDim.x);

    // lane offsets of the shifted operand for dx = (w4 + j) % 3, and of g's
    int off[3][2], offg[2];
#pragma unroll
    for (int h = 0; h < 2; ++h) {
        offg[h] = tr_offset(0, h) + rows * kWX * kVB;
#pragma unroll
        for (int j = 0; j < 3; ++j) off[j][h] = tr_offset((w4 + j) % 3, h) + rows * kPitch * kVB;
    }
    bf16x8 one;
#pragma unroll
    for (int j = 0; j < 8; ++j) one[j] = (__bf16)1.0f;
    f32x16 acc[kNT];
#pragma unroll
    for (int j = 0; j < kNT; ++j) acc[j] = f32x16{};

    uint4 rh[kHaloPieces], rt[kTilePieces];
    Column c{};
    for (int s = s0; s < s1; ++s) {
        const int z = s % g.D;
        if (s == s0 || z == 0) {
            c = column_of(s / g.D, g);
            __syncthreads();
            for (int dz = 0; dz < 3; ++dz) {
                load_halo(rh, a, g, c, z + dz - 1);
                store_halo(lds + ((z + dz - 1) & 3) * kHaloBytes, rh);
            }
            load_tile(rt, gin, g, c, z);
            store_tile(tiles + (z & 1) * kTileBytes, rt);
            __syncthreads();
        }
        const bool next = s + 1 < s1 && z + 1 < g.D;
        if (next) {
            load_halo(rh, a, g, c, z + 2);
            load_tile(rt, gin, g, c, z + 1);
        }
        int tap[kNT];
#pragma unroll
        for (int j = 0; j < kNT; ++j) {
            const int k = min(w4 + 4 * j, 26);
            tap[j] = ((z + k / 9 - 1) & 3) * kHaloBytes + k / 3 % 3 * (kPitch * kVB);
        }
        const char* tile = tiles + (z & 1) * kTileBytes;
#pragma unroll
        for (int y = 0; y < kWY / 2; ++y)
#pragma unroll
            for (int x = 0; x < kWX; x += 16) {
                const int og = (y * kWX + x) * kVB, oa = (y * kPitch + x) * kVB;
                const bf16x8 av = read_tr(tile, offg[0] + og, offg[1] + og);
#pragma unroll
                for (int j = 0; j < kNT; ++j) {
                    bf16x8 bv = read_tr(lds, off[j % 3][0] + tap[j] + oa, off[j % 3][1] + tap[j] + oa);
                    if (j == kNT - 1 && w4 == 3) bv = one;
                    acc[j] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(av, bv, acc[j], 0, 0, 0);
                }
            }
        if (next) {
            store_halo(lds + ((z + 2) & 3) * kHaloBytes, rh);
            store_tile(tiles + ((z + 1) & 1) * kTileBytes, rt);
            __syncthreads();
        }
    }

    // second row group's sums through LDS, then D[co][ci]: lane holds ci = lane % 32,
    // co = 8 (r / 4) + 4 (lane / 32) + r % 4
    float* sums = reinterpret_cast<float*>(lds) + (size_t)w4 * kNT * 16 * 64 + lane;
    __syncthreads();
    if (wave >= 4) {
#pragma unroll
        for (int j = 0; j < kNT; ++j)
#pragma unroll
            for (int r = 0; r < 16; ++r) sums[(j * 16 + r) * 64] = acc[j][r];
    }
    __syncthreads();
    if (wave >= 4) return;
    float* p = partial + (long)blockIdx.x * (kConv32 + kC);
    const int ci = lane & 31, kh = lane >> 5;
#pragma unroll
    for (int j = 0; j < kNT; ++j) {
        const int k = w4 + 4 * j;
#pragma unroll
        for (int r = 0; r < 16; ++r) {
            const int co = 8 * (r / 4) + 4 * kh + r % 4;
            const float v = acc[j][r] + sums[(j * 16 + r) * 64];
            if (k < 27) p[(k * kC + co) * kC + ci] = v;
            else if (ci == 0) p[kConv32 + co] = v;
        }
    }
}

// A dword per voxel of a plane with its halo (thread e < kHY * kHX holds
// voxel e), zero outside the volume.
__device__ __forceinline__ uint32_t load_halo_word(const uint32_t* __restrict__ a, const Geo& g, const Column& c, int z)
{
    const int v = threadIdx.x, y = c.y0 + v / kHX - 1, x = c.x0 + v % kHX - 1;
    if (v < kHY * kHX && z >= 0 && z < g.D && y >= 0 && y < g.H && x >= 0 && x < g.W) return a[g.vox(c.n, z, y, x)];
    return 0;
}

// --------------------------------------------------------------- input layer
// 32 x (27 taps x 2 channels) with the FP32 matrix instruction, two voxels at a time: B holds
// the 54 (tap, channel) pairs, a column of ones (the bias) and zeros, in two 32-column tiles.
// The bf16 instruction takes 159 us at 8 x 64 x 128 x 128 where this takes 378 (its matrix
// instructions alone 218), but it cuts low bits off the addends of its sums: gradients with addends
// of both signs came out up to 2.8 times as far from 64 bits as FP32 sums by rows, these 0.4 to 1.0 times.
// x lies channel-major in LDS, in FP32.  A step's row of 32 voxels is summed from zero, as
// in the output layer below.
constexpr int kXPlane = kHY * 2 * kPitch;  // floats of one plane of x
constexpr int kXBytes = 3 * kXPlane * 4;
constexpr int kWgradInLds = 8 * 2 * 16 * 64 * 4;
static_assert(kXBytes + kTileBytes <= kWgradInLds);
__global__ __launch_bounds__(kWThreads, 4) void wgrad_in_kernel(const uint16_t* __restrict__ gin,
                                                                const uint32_t* __restrict__ x, Geo g, int steps,
                                                                float* __restrict__ partial)
{
    __shared__ __attribute__((aligned(16))) char lds[kWgradInLds];
    char* const tile = lds + kXBytes;
    float* const xs = reinterpret_cast<float*>(lds);
    const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const unsigned b = xcd_block(blockIdx.x, gridDim.x);
    const int s0 = (int)((long)steps * b / gridDim.x), s1 = (int)((long)steps * (b + 1) / gridDim.x);
    const int m = lane & 31, kh = lane >> 5;

    int base[2], dz[2];
#pragma unroll
    for (int t = 0; t < 2; ++t) {
        const int e = t * 32 + m, k = e < 54 ? e >> 1 : 0;
        dz[t] = k / 9;
        base[t] = ((k / 3 % 3 + wave) * 2 + (e & 1)) * kPitch + k % 3 + kh;
    }
    const bool pair = m < 22;  // of the second tile's columns: pairs 32 .. 53
    const float fill = m == 22 ? 1.f : 0.f;
    // g of voxel 2 q + kh: its slot's swizzle depends on q alone (kh is bit 0 of the column)
    const int gbase = (wave * kWX + kh) * kVB + (m & 7) * 2;
    f32x16 acc[2] = {f32x16{}, f32x16{}};

    auto put = [&](int z, uint32_t w) {
        const int v = threadIdx.x;
        if (v >= kHY * kHX) return;
        float* d = xs + (z + 3) % 3 * kXPlane + v / kHX * 2 * kPitch + v % kHX;
        d[0] = __uint_as_float(w << 16);
        d[kPitch] = __uint_as_float(w & 0xffff0000u);
    };
    uint4 rt[kTilePieces];
    Column c{};
    for (int s = s0; s < s1; ++s) {
        const int z = s % g.D;
        if (s == s0 || z == 0) {
            c = column_of(s / g.D, g);
            __syncthreads();
            for (int q = z - 1; q <= z + 1; ++q) put(q, load_halo_word(x, g, c, q));
            load_tile(rt, gin, g, c, z);
            store_tile(tile, rt);
            __syncthreads();
        }
        const bool next = s + 1 < s1 && z + 1 < g.D;
        uint32_t rw = 0;
        if (next) {
            rw = load_halo_word(x, g, c, z + 2);
            load_tile(rt, gin, g, c, z + 1);
        }
        const float* xr[2];
        f32x16 row[2] = {f32x16{}, f32x16{}};
#pragma unroll
        for (int t = 0; t < 2; ++t) xr[t] = xs + (z + dz[t] + 2) % 3 * kXPlane + base[t];
#pragma unroll
        for (int q = 0; q < kWX / 2; ++q) {
            const float gv = bf2f(*reinterpret_cast<const uint16_t*>(
                tile + gbase + 2 * q * kVB + (((m >> 3) ^ slot_swizzle(2 * q)) << 4)));
#pragma unroll
            for (int t = 0; t < 2; ++t) {
                const float xv = xr[t][2 * q];
                row[t] = __builtin_amdgcn_mfma_f32_32x32x2f32(gv, t == 1 && !pair ? fill : xv, row[t], 0, 0, 0);
            }
        }
#pragma unroll
        for (int t = 0; t < 2; ++t) acc[t] += row[t];
        if (next) {
            __syncthreads();
            put(z + 2, rw);
            store_tile(tile, rt);
            __syncthreads();
        }
    }

    float* sums = reinterpret_cast<float*>(lds);
    __syncthreads();
#pragma unroll
    for (int t = 0; t < 2; ++t)
#pragma unroll
        for (int r = 0; r < 16; ++r) sums[((wave * 2 + t) * 16 + r) * 64 + lane] = acc[t][r];
    __syncthreads();
    float* p = partial + (long)blockIdx.x * (27 * kC * 2 + kC);
    for (int i = threadIdx.x; i < 2 * 16 * 64; i += kWThreads) {
        float v = 0.f;
        for (int w = 0; w < 8; ++w) v += sums[w * 2 * 16 * 64 + i];
        const int l = i & 63, r = (i >> 6) & 15, e = (i >> 10) * 32 + (l & 31), co = 8 * (r / 4) + 4 * (l >> 5) + r % 4;
        if (e < 54) p[((e >> 1) * kC + co) * 2 + (e & 1)] = v;
        else if (e == 54) p[27 * kC * 2 + co] = v;
    }
}

// -------------------------------------------------------------- output layer
// dW6[k][ci] = sum_u dy[u - off(k)] h5[u][ci] with dy in FP32: the FP32 matrix
// instruction v_mfma_f32_32x32x2_f32 (A = 27 shifted dy of 32 rows, B = h5), two
// voxels at a time, keeps the products and sums in FP32 without splitting dy.  A step's
// row of 32 voxels is summed from zero and added to the block's sums: with S steps a block, the
// rounding error of a weight grows like sqrt(32 + S) of a product's, where one chain over
// all of a block's voxels has sqrt(32 S) (against 64 bits 3 to 5 times as far off; 225 us a launch at
// 8 x 64 x 128 x 128, 228 with the additions).
constexpr int kYPlane = kHY * kPitch;
constexpr int kYBytes = 3 * kYPlane * 4;
constexpr int kWgradOutLds = 8 * 16 * 64 * 4;
static_assert(kYBytes + kTileBytes <= kWgradOutLds);
__global__ __launch_bounds__(kWThreads, 4) void wgrad_out_kernel(const uint32_t* __restrict__ dy,
                                                                 const uint16_t* __restrict__ h5, Geo g, int steps,
                                                                 float* __restrict__ partial)
{
    __shared__ __attribute__((aligned(16))) char lds[kWgradOutLds];
    char* const tile = lds + kYBytes;
    float* const ys = reinterpret_cast<float*>(lds);
    const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const unsigned b = xcd_block(blockIdx.x, gridDim.x);
    const int s0 = (int)((long)steps * b / gridDim.x), s1 = (int)((long)steps * (b + 1) / gridDim.x);
    const int k = min(lane & 31, 26), kh = lane >> 5, ci = lane & 31;
    const int ybase = (wave + 2 - k / 3 % 3) * kPitch + 2 - k % 3 + kh;
    // h5 of voxel 2 q + kh: its slot's swizzle depends on q alone (kh is bit 0 of the column)
    const int hbase = (wave * kWX + kh) * kVB + (ci & 7) * 2;
    f32x16 acc = {};
    float bsum = 0.f;

    auto put = [&](int z, uint32_t w) {
        const int v = threadIdx.x;
        if (v < kHY * kHX) ys[(z + 3) % 3 * kYPlane + v / kHX * kPitch + v % kHX] = __uint_as_float(w);
    };
    uint4 rt[kTilePieces];
    Column c{};
    for (int s = s0; s < s1; ++s) {
        const int z = s % g.D;
        if (s == s0 || z == 0) {
            c = column_of(s / g.D, g);
            __syncthreads();
            for (int q = z - 1; q <= z + 1; ++q) put(q, load_halo_word(dy, g, c, q));
            load_tile(rt, h5, g, c, z);
            store_tile(tile, rt);
            __syncthreads();
        }
        const bool next = s + 1 < s1 && z + 1 < g.D;
        uint32_t rw = 0;
        if (next) {
            rw = load_halo_word(dy, g, c, z + 2);
            load_tile(rt, h5, g, c, z + 1);
        }
        const float* yr = ys + (z + 4 - k / 9) % 3 * kYPlane + ybase;
        f32x16 row = {};
#pragma unroll
        for (int q = 0; q < kWX / 2; ++q) {
            const uint16_t h = *reinterpret_cast<const uint16_t*>(
                tile + hbase + 2 * q * kVB + (((ci >> 3) ^ slot_swizzle(2 * q)) << 4));
            row = __builtin_amdgcn_mfma_f32_32x32x2f32(yr[2 * q], bf2f(h), row, 0, 0, 0);
        }
        acc += row;
        if (threadIdx.x < kWY * kWX)
            bsum += ys[z % 3 * kYPlane + ((threadIdx.x >> 5) + 1) * kPitch + (threadIdx.x & 31) + 1];
        if (next) {
            __syncthreads();
            put(z + 2, rw);
            store_tile(tile, rt);
            __syncthreads();
        }
    }

    float* sums = reinterpret_cast<float*>(lds);
    float* p = partial + (long)blockIdx.x * (27 * kC + 1);
    __syncthreads();
#pragma unroll
    for (int r = 0; r < 16; ++r) sums[(wave * 16 + r) * 64 + lane] = acc[r];
    __syncthreads();
    for (int i = threadIdx.x; i < 16 * 64; i += kWThreads) {
        float v = 0.f;
        for (int w = 0; w < 8; ++w) v += sums[w * 16 * 64 + i];
        const int l = i & 63, r = i >> 6, kk = 8 * (r / 4) + 4 * (l >> 5) + r % 4;
        if (kk < 27) p[kk * kC + (l & 31)] = v;
    }
    __syncthreads();
    if (threadIdx.x < kWY * kWX) sums[threadIdx.x] = bsum;
    __syncthreads();
    for (int n = kWY * kWX / 2; n > 0; n >>= 1) {
        if (threadIdx.x < n) sums[threadIdx.x] += sums[threadIdx.x + n];
        __syncthreads();
    }
    if (threadIdx.x == 0) p[27 * kC] = sums[0];
}

// Sum partials[nb][count] -> out[count] in FP64: a block takes 32 columns and
// deals the rows to 8 groups of 32 lanes.  (One thread per column left 108
// blocks with nb dependent loads each; over the six layers of a step with 512
// rows the mean was 127 us a launch, against 9.)
__global__ __launch_bounds__(256) void reduce_partials_kernel(const float* __restrict__ partial, int nb, int count,
                                                              float* __restrict__ out)
{
    __shared__ double sums[8][32];
    const int c = threadIdx.x & 31, q = threadIdx.x >> 5, i = blockIdx.x * 32 + c;
    double s = 0.0;
    if (i < count) {
#pragma unroll 8
        for (int r = q; r < nb; r += 8) s += (double)partial[(long)r * count + i];
    }
    sums[q][c] = s;
    __syncthreads();
    if (q == 0 && i < count) {
        for (int k = 1; k < 8; ++k) s += sums[k][c];
        out[i] = (float)s;
    }
}

// ------------------------------------------------------------ launchers
static int wgrad_steps(Dims d)
{
    const long s = (long)d.N * ((d.H + kWY - 1) / kWY) * ((d.W + kWX - 1) / kWX) * d.D;
    if (s > 0x7fffffffL) throw_msg("network: training volume too large");
    return (int)s;
}

// Blocks (rows of partial sums, added in FP64): one or more per CU, and no fewer than (n, z)
// planes, so that a partial sum covers at most about one plane of voxels.
int wgrad_blocks(Dims d)
{
    const long planes = (long)d.N * d.D;
    const long nb = (std::max<long>(planes, 256) + 255) / 256 * 256;
    return (int)std::min<long>(nb, wgrad_steps(d));
}

void launch_wgrad_in(const uint16_t* g, const uint16_t* x, Dims d, float* partial, hipStream_t s)
{
    wgrad_in_kernel<<<wgrad_blocks(d), kWThreads, 0, s>>>(g, reinterpret_cast<const uint32_t*>(x), geo(d),
                                                          wgrad_steps(d), partial);
    FMVD_LAUNCH_CHECK();
}
void launch_wgrad_out(const float* dy, const uint16_t* h5, Dims d, float* partial, hipStream_t s)
{
    wgrad_out_kernel<<<wgrad_blocks(d), kWThreads, 0, s>>>(reinterpret_cast<const uint32_t*>(dy), h5, geo(d),
                                                           wgrad_steps(d), partial);
    FMVD_LAUNCH_CHECK();
}
void launch_wgrad32(const uint16_t* g, const uint16_t* a, Dims d, float* partial, hipStream_t s)
{
    wgrad32_kernel<<<wgrad_blocks(d), kWThreads, 0, s>>>(g, a, geo(d), wgrad_steps(d), partial);
    FMVD_LAUNCH_CHECK();
}
void launch_reduce_partials(const float* partial, int nb, int count, float* out, hipStream_t s)
{
    reduce_partials_kernel<<<(unsigned)((count + 31) / 32), 256, 0, s>>>(partial, nb, count, out);
    FMVD_LAUNCH_CHECK();
}

}  // namespace net
}  // namespace fmvd
