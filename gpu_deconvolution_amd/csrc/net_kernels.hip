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
// 2->32 input layer and the 32->1 output layer have too few channels for MFMA
// tiles and run on the VALU, still with FP32 accumulation.
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

// The edge layers run on the VALU.

// Layer 1 (2 -> 32): h1 = relu(conv(x, W1) + b1); W1 is FP32 [27][32][2]
// (bf16-rounded values).  One thread per voxel; relu (if wanted): the bits h1 > 0.
// Bound by the VALU: 27 x 32 x 3 instructions a voxel (two products, rounded
// separately, and their sum) are 553 us at 8 x 64 x 128 x 128, measured 634; reading the
// weights through scalar loads, or walking planes with 96 sums a thread to
// read a neighbour once, measured 656 and 734.
__global__ void conv_in_kernel(const uint16_t* __restrict__ x, Geo g, const float* __restrict__ w,
                               const float* __restrict__ b, uint16_t* __restrict__ h,
                               uint32_t* __restrict__ relu)
{
    __shared__ float ws[27 * 32 * 2 + 32];
    for (int i = threadIdx.x; i < 27 * 64 + 32; i += blockDim.x) ws[i] = i < 27 * 64 ? w[i] : b[i - 27 * 64];
    __syncthreads();
    const long per = (long)g.D * g.H * g.W;
    const long i = (long)blockIdx.x * blockDim.x + threadIdx.x;
    const int n = blockIdx.y;
    if (i >= per) return;
    const int xx = (int)(i % g.W), yy = (int)((i / g.W) % g.H), zz = (int)(i / ((long)g.W * g.H));
    float acc[32];
#pragma unroll
    for (int c = 0; c < 32; ++c) acc[c] = ws[27 * 64 + c];
    for (int k = 0; k < 27; ++k) {
        const int z = zz + k / 9 - 1, y = yy + (k / 3) % 3 - 1, xi = xx + k % 3 - 1;
        if (z < 0 || z >= g.D || y < 0 || y >= g.H || xi < 0 || xi >= g.W) continue;
        const long v = g.vox(n, z, y, xi);
        const float x0 = bf2f(x[2 * v]), x1 = bf2f(x[2 * v + 1]);
#pragma unroll
        for (int c = 0; c < 32; ++c) acc[c] += x0 * ws[(k * 32 + c) * 2] + x1 * ws[(k * 32 + c) * 2 + 1];
    }
    uint16_t* o = h + (n * per + i) * 32;
    uint32_t pos = 0;
#pragma unroll
    for (int c = 0; c < 32; ++c) {
        const uint16_t r = f2bf(fmaxf(acc[c], 0.f));
        if (r) pos |= 1u << c;
        o[c] = r;
    }
    if (relu) relu[n * per + i] = pos;
}

// Layer 6 (32 -> 1): y = conv(h5, W6) + b6 + (x0 + x1) / 2 (FP32 out).  A block
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

// dh5[v][c] = sum_k dy[v - off(k)] W6[k][c]  (FP32 out), and the masked bf16
// gradient of layer 5 (relu: its bits r > 0)
__global__ void out_dgrad_kernel(const float* __restrict__ dy, Geo g, const float* __restrict__ w,
                                 const uint32_t* __restrict__ relu, float* __restrict__ dh,
                                 uint16_t* __restrict__ gout)
{
    __shared__ float ws[27 * 32];
    for (int i = threadIdx.x; i < 27 * 32; i += blockDim.x) ws[i] = w[i];
    __syncthreads();
    const long per = (long)g.D * g.H * g.W;
    const long i = (long)blockIdx.x * blockDim.x + threadIdx.x;
    const int n = blockIdx.y;
    if (i >= per) return;
    const int xx = (int)(i % g.W), yy = (int)((i / g.W) % g.H), zz = (int)(i / ((long)g.W * g.H));
    float acc[32];
#pragma unroll
    for (int c = 0; c < 32; ++c) acc[c] = 0.f;
    for (int k = 0; k < 27; ++k) {
        const int z = zz - (k / 9 - 1), y = yy - ((k / 3) % 3 - 1), xi = xx - (k % 3 - 1);
        if (z < 0 || z >= g.D || y < 0 || y >= g.H || xi < 0 || xi >= g.W) continue;
        const float d = dy[g.vox(n, z, y, xi)];
#pragma unroll
        for (int c = 0; c < 32; ++c) acc[c] += d * ws[k * 32 + c];
    }
    float* o = dh + (n * per + i) * 32;
    uint16_t* go = gout + (n * per + i) * 32;
    const uint32_t bits = relu[n * per + i];
#pragma unroll
    for (int c = 0; c < 32; ++c) {
        o[c] = acc[c];
        go[c] = (bits >> c) & 1 ? f2bf(acc[c]) : (uint16_t)0;
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
void launch_conv_in(const uint16_t* x, Dims d, const float* small, const float* params, uint16_t* h,
                    uint32_t* relu, hipStream_t s)
{
    const long per = (long)d.D * d.H * d.W;
    conv_in_kernel<<<dim3(nblk(per, 256), d.N), 256, 0, s>>>(x, geo(d), small, params + off_b(0), h, relu);
    FMVD_LAUNCH_CHECK();
}
void launch_conv_out(const uint16_t* h, const uint16_t* x, Dims d, const float* small, const float* params, float* y,
                     hipStream_t s)
{
    // segments of about 16 planes: a segment reads two planes beyond its ends
    const int nseg = (d.D + 15) / 16;
    const long blocks = (long)d.N * ((d.H + kOY - 1) / kOY) * ((d.W + kOX - 1) / kOX) * nseg;
    if (blocks > 0x7fffffffL) throw_msg("network: volume too large");
    conv_out_kernel<<<(unsigned)blocks, 256, 0, s>>>(h, reinterpret_cast<const uint32_t*>(x), geo(d), small + 27 * 64,
                                                     params + off_b(5), y, nseg);
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
    const long per = (long)d.D * d.H * d.W;
    out_dgrad_kernel<<<dim3(nblk(per, 256), d.N), 256, 0, s>>>(dy, geo(d), small + 27 * 64, relu, dh, gout);
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
