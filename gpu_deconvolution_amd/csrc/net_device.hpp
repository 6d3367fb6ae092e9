// Device helpers shared by the warm-start network's kernels.
#pragma once
#include <hip/hip_runtime.h>
#include <stdint.h>

#include "net.hpp"

namespace fmvd {
namespace net {

typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
typedef float f32x16 __attribute__((ext_vector_type(16)));

__device__ __forceinline__ float bf2f(uint16_t b) { return __uint_as_float((uint32_t)b << 16); }
// round to nearest even (finite inputs)
__device__ __forceinline__ uint16_t f2bf(float f)
{
    const uint32_t u = __float_as_uint(f);
    return (uint16_t)((u + 0x7FFFu + ((u >> 16) & 1u)) >> 16);
}

struct Geo {
    int N, D, H, W;  // batch, depth, height, width
    __device__ __forceinline__ long vox(int n, int z, int y, int x) const
    {
        return (((long)n * D + z) * H + y) * W + x;
    }
};
static inline Geo geo(Dims d) { return Geo{d.N, d.D, d.H, d.W}; }

// Blocks are dispatched round-robin over the 8 XCDs; give each XCD a
// contiguous range of logical block ids so that neighbouring tiles, which
// share their halos, share its L2.
__device__ __forceinline__ unsigned xcd_block(unsigned bid, unsigned nblocks)
{
    const unsigned q = nblocks >> 3, rem = nblocks & 7u;
    const unsigned x = bid & 7u, k = bid >> 3;
    return x * q + (x < rem ? x : rem) + k;
}

// LDS tiles of 32-channel bf16 voxels (64 bytes each): the 16-byte slot s
// (channels 8s .. 8s+7) of the voxel in column c is stored at slot
// s ^ slot_swizzle(c).  The LDS serves 128 bytes per cycle; with a row pitch
// that is a multiple of 8 voxels, 8 consecutive voxels' equal slots (a row
// operand of an MFMA tile) and slots 2h, 2h+1 of 4 consecutive voxels (a
// transposing read) then lie in distinct banks, and the swizzle depends on
// the column alone, so rows are immediate offsets.
__device__ __forceinline__ int slot_swizzle(int c) { return (c & 2) | ((c >> 2) & 1); }

// A voxel's 32 channels, held as bf16 pairs c[q][i] = channels 8 q + 4 (lane / 32) + 2 i, + 1 by
// the lanes l and l + 32: each lane gets two 16-byte pieces (channels 8 q .. 8 q + 7 for q =
// lane / 32 and 2 + lane / 32) and stores them.
__device__ __forceinline__ void store_voxel(uint16_t* __restrict__ v, const uint32_t (*c)[2], int kh)
{
#pragma unroll
    for (int h = 0; h < 2; ++h) {
        const auto a = __builtin_amdgcn_permlane32_swap(c[2 * h][0], c[2 * h + 1][0], false, false);
        const auto b = __builtin_amdgcn_permlane32_swap(c[2 * h][1], c[2 * h + 1][1], false, false);
        reinterpret_cast<uint4*>(v)[2 * h + kh] = make_uint4(a[0], b[0], a[1], b[1]);
    }
}

}  // namespace net
}  // namespace fmvd
