// unet.hip -- kernels of the learned initial estimate: a 3-level 3D U-Net
// (16/32/64 channels, 3^3 convolutions, ReLU) in BF16 on MFMA with FP32
// accumulation, forward and backward.
//
// Tensors are channels-last bf16 [n][z][y][x][c] with the channel count padded
// to a multiple of 16; a tensor view is (pointer, channel stride, channel
// offset), so a skip concatenation is two producers writing disjoint channel
// ranges of one buffer.  Convolution weights are [tap][cout][cin] (cin
// contiguous), master copies FP32, compute copies bf16.
//
// The MFMA kernels are in unet_conv.hip (convolutions, forward and data
// gradient) and unet_wgrad.hip (weight and bias gradients).
#include <hip/hip_runtime.h>

#include <cstdint>

#include "unet.hpp"

namespace mvr {

__device__ __forceinline__ float bf2f(uint16_t b) { return __uint_as_float((uint32_t)b << 16); }
__device__ __forceinline__ uint16_t f2bf(float f) {
  const uint32_t u = __float_as_uint(f);
  return (uint16_t)((u + 0x7FFFu + ((u >> 16) & 1u)) >> 16);  // round to nearest even
}

// ------------------------------------------------------------------ elementwise pieces
// All work on units of 8 channels (16 bytes); channel counts, strides and offsets are multiples of 16.
typedef __attribute__((ext_vector_type(8))) unsigned short u16x8;

__device__ __forceinline__ void unpack8(const u16x8& u, float f[8]) {
#pragma unroll
  for (int k = 0; k < 8; ++k) f[k] = bf2f(u[k]);
}
__device__ __forceinline__ u16x8 pack8(const float f[8]) {
  u16x8 u;
#pragma unroll
  for (int k = 0; k < 8; ++k) u[k] = f2bf(f[k]);
  return u;
}
template <typename T>
__device__ __forceinline__ const u16x8& at8(const T* p) { return *reinterpret_cast<const u16x8*>(p); }
__device__ __forceinline__ u16x8& at8w(uint16_t* p) { return *reinterpret_cast<u16x8*>(p); }

// Index spaces: row kernels run on grid (ceil(W * U / block), H, N * D) of the tensor they iterate
// over, U = C / 8 units per voxel, so all index arithmetic is 32-bit; work-groups as large as a row, up to 256.
struct RowIdx {
  int x, c, y, z, n;
  bool ok;
};
__device__ __forceinline__ RowIdx row_idx(int U, int W, int D) {
  RowIdx r;
  const int xu = blockIdx.x * blockDim.x + threadIdx.x;
  r.ok = xu < W * U;
  r.x = xu / U;
  r.c = (xu - r.x * U) * 8;
  r.y = blockIdx.y;
  r.z = blockIdx.z % D;
  r.n = blockIdx.z / D;
  return r;
}
__device__ __forceinline__ size_t vox(int n, int z, int y, int x, int D, int H, int W) {
  return (((size_t)n * D + z) * H + y) * W + x;
}

// ReLU backward: the gradient where the activation was positive, else 0
__device__ __forceinline__ u16x8 relu_bwd(u16x8 g, u16x8 post) {
#pragma unroll
  for (int k = 0; k < 8; ++k)
    if (bf2f(post[k]) <= 0.f) g[k] = 0;
  return g;
}

// 2x2x2 average pooling (forward) over channels [0, C) of in -> out; grid over the output (D, H, W)
__global__ void k_pool_fwd(const uint16_t* __restrict__ in, int ics, int ico, uint16_t* __restrict__ out, int ocs,
                           int C, int D, int H, int W) {
  const RowIdx r = row_idx(C / 8, W, D);
  if (!r.ok) return;
  float s[8] = {0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f};
#pragma unroll
  for (int k = 0; k < 8; ++k) {
    const size_t vi = vox(r.n, 2 * r.z + (k >> 2), 2 * r.y + ((k >> 1) & 1), 2 * r.x + (k & 1), 2 * D, 2 * H, 2 * W);
    float f[8];
    unpack8(at8(in + vi * ics + ico + r.c), f);
#pragma unroll
    for (int q = 0; q < 8; ++q) s[q] += f[q];
  }
#pragma unroll
  for (int q = 0; q < 8; ++q) s[q] *= 0.125f;
  at8w(out + vox(r.n, r.z, r.y, r.x, D, H, W) * ocs + r.c) = pack8(s);
}

// pooling backward: din[2v + k] += dout[v] / 8, then the ReLU of the layer below (post: its activations, strided as
// din); grid over the fine tensor (2D, 2H, 2W)
__global__ void k_pool_bwd(const uint16_t* __restrict__ dout, int ocs, uint16_t* __restrict__ din, int ics, int ico,
                           int C, int D, int H, int W, const uint16_t* __restrict__ post) {  // dims of the pooled tensor
  const RowIdx r = row_idx(C / 8, 2 * W, 2 * D);
  if (!r.ok) return;
  float gval[8], cur[8];
  unpack8(at8(dout + vox(r.n, r.z / 2, r.y / 2, r.x / 2, D, H, W) * ocs + r.c), gval);
  const size_t at = vox(r.n, r.z, r.y, r.x, 2 * D, 2 * H, 2 * W) * ics + ico + r.c;
  unpack8(at8(din + at), cur);
#pragma unroll
  for (int q = 0; q < 8; ++q) cur[q] += 0.125f * gval[q];
  at8w(din + at) = relu_bwd(pack8(cur), at8(post + at));
}

// nearest-neighbour x2 upsampling into channels [oco, oco + C) of out; grid over the fine tensor
__global__ void k_up_fwd(const uint16_t* __restrict__ in, int ics, uint16_t* __restrict__ out, int ocs, int oco, int C,
                         int D, int H, int W) {  // D, H, W of the coarse tensor
  const RowIdx r = row_idx(C / 8, 2 * W, 2 * D);
  if (!r.ok) return;
  at8w(out + vox(r.n, r.z, r.y, r.x, 2 * D, 2 * H, 2 * W) * ocs + oco + r.c) =
      at8(in + vox(r.n, r.z / 2, r.y / 2, r.x / 2, D, H, W) * ics + r.c);
}

// upsampling backward: dcoarse[v] = sum of the 8 fine gradients, through the ReLU of the coarse activations (post, strided
// as dcoarse); grid over the coarse tensor
__global__ void k_up_bwd(const uint16_t* __restrict__ dfine, int fcs, int fco, uint16_t* __restrict__ dcoarse, int ccs,
                         int C, int D, int H, int W, const uint16_t* __restrict__ post) {  // coarse dims
  const RowIdx r = row_idx(C / 8, W, D);
  if (!r.ok) return;
  float s[8] = {0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f};
#pragma unroll
  for (int k = 0; k < 8; ++k) {
    const size_t vf = vox(r.n, 2 * r.z + (k >> 2), 2 * r.y + ((k >> 1) & 1), 2 * r.x + (k & 1), 2 * D, 2 * H, 2 * W);
    float f[8];
    unpack8(at8(dfine + vf * fcs + fco + r.c), f);
#pragma unroll
    for (int q = 0; q < 8; ++q) s[q] += f[q];
  }
  const size_t at = vox(r.n, r.z, r.y, r.x, D, H, W) * ccs + r.c;
  at8w(dcoarse + at) = relu_bwd(pack8(s), at8(post + at));
}

// network input: channels 0..V-1 = w_v * img_v / scale, channel V = their weighted mean
// sum_v w_v img_v / (scale * sum_v w_v) (0 where no view has weight), rest 0; returns the mean
__device__ __forceinline__ float pack_values(const float* const* img, const float* const* w, int V, size_t gi,
                                             float inv_scale, float (&val)[16]) {
  float s = 0.f, sw = 0.f;
#pragma unroll
  for (int c = 0; c < 16; ++c) val[c] = 0.f;
#pragma unroll
  for (int c = 0; c < kNetMaxViews; ++c) {  // unrolled over the packer's view slots
    if (c < V) {
      const float wv = w[c][gi];
      val[c] = img[c][gi] * wv * inv_scale;
      s += val[c];
      sw += wv;
    }
  }
  const float mean = sw > 0.f ? s / sw : 0.f;
#pragma unroll
  for (int c = 0; c < 16; ++c)
    if (c == V) val[c] = mean;
  return mean;
}

// one sample: the region [x0, x0 + W) x [y0, ...) x [z0, ...) of volumes of dims N3.  Positions past the
// volume's last voxel (a region padded up to a multiple of 4) repeat that voxel.
__global__ void k_pack_input(InputArgs a) {
  const int x = blockIdx.x * blockDim.x + threadIdx.x, y = blockIdx.y, z = blockIdx.z;
  if (x >= a.W) return;
  const size_t v = ((size_t)z * a.H + y) * a.W + x;
  const int gx = min(a.x0 + x, a.N3[0] - 1), gy = min(a.y0 + y, a.N3[1] - 1), gz = min(a.z0 + z, a.N3[2] - 1);
  const size_t gi = ((size_t)gz * a.N3[1] + gy) * a.N3[0] + gx;
  float val[16];
  const float mean = pack_values(a.img, a.w, a.V, gi, a.inv_scale, val);
  uint16_t* o = a.out + v * a.out_cs;
  at8w(o) = pack8(val);
  if (a.out_cs == 16) at8w(o + 8) = pack8(val + 8);
  if (a.avg_out) a.avg_out[v] = mean;
}

// the patches of a training batch, their targets normalised alike (one launch: four patches of 64^3 in eight launches of
// a quarter of the lanes took 46 us and their gaps, so 25)
__global__ __launch_bounds__(256) void k_pack_patches(PatchArgs a) {
  const PatchArgs::Patch& p = a.p[blockIdx.y];
  const unsigned total = (unsigned)a.P * a.P * a.P, v = blockIdx.x * 256u + threadIdx.x;
  if (v >= total) return;
  const unsigned row = v / a.P, x = v - row * a.P, z = row / a.P, y = row - z * a.P;
  const size_t gi = ((size_t)(p.o[2] + z) * p.N3[1] + (p.o[1] + y)) * p.N3[0] + (p.o[0] + x);
  float val[16];
  const float mean = pack_values(p.img, p.w, a.V, gi, p.inv_scale, val);
  const size_t at = (size_t)blockIdx.y * total + v;
  at8w(a.out + at * 16) = pack8(val);
  at8w(a.out + at * 16 + 8) = pack8(val + 8);
  a.avg_out[at] = mean;
  a.target_out[at] = p.target[gi] * p.inv_scale;
}

// output head of a training step (an inference fuses it into the last convolution): r[v] = sum_c wo[c] d1[v][c] + bo;
// pred = avg[v] + r; loss partials of (pred - target)^2 and dr[v] = 2 (pred - target) / count
__global__ __launch_bounds__(256) void k_head(HeadArgs a) {
  __shared__ double red[256];
  double ls = 0.0;
  for (size_t v = (size_t)blockIdx.x * blockDim.x + threadIdx.x; v < a.nvox; v += (size_t)gridDim.x * blockDim.x) {
    float r = a.bias[0], f[16];
    unpack8(at8(a.d1 + v * a.d1_cs), f);
    unpack8(at8(a.d1 + v * a.d1_cs + 8), f + 8);
#pragma unroll
    for (int c = 0; c < 16; ++c) r += a.wo[c] * f[c];
    const float e = a.avg[v] + r - a.target[v];
    ls += (double)e * e;
    a.dr[v] = 2.f * e / (float)a.nvox;
  }
  red[threadIdx.x] = ls;
  __syncthreads();
  for (int off = 128; off > 0; off >>= 1) {
    if ((int)threadIdx.x < off) red[threadIdx.x] += red[threadIdx.x + off];
    __syncthreads();
  }
  if (threadIdx.x == 0) a.loss_partial[blockIdx.x] = red[0];
}

// head backward: d_d1[v][c] = dr[v] * wo[c] through the ReLU of d1; partials of dwo[c] = sum dr d1[v][c], dbo = sum dr
__global__ __launch_bounds__(256) void k_head_bwd(HeadArgs a, uint16_t* __restrict__ dd1, float* __restrict__ partial) {
  __shared__ float red[4][17];
  float acc[17];
#pragma unroll
  for (int c = 0; c < 17; ++c) acc[c] = 0.f;
  for (size_t v = (size_t)blockIdx.x * blockDim.x + threadIdx.x; v < a.nvox; v += (size_t)gridDim.x * blockDim.x) {
    const float dr = a.dr[v];
    float f[16], g[16];
    unpack8(at8(a.d1 + v * a.d1_cs), f);
    unpack8(at8(a.d1 + v * a.d1_cs + 8), f + 8);
#pragma unroll
    for (int c = 0; c < 16; ++c) {
      acc[c] += dr * f[c];
      g[c] = f[c] <= 0.f ? 0.f : dr * a.wo[c];
    }
    at8w(dd1 + v * 16) = pack8(g);
    at8w(dd1 + v * 16 + 8) = pack8(g + 8);
    acc[16] += dr;
  }
#pragma unroll
  for (int c = 0; c < 17; ++c) {
    for (int off = 32; off > 0; off >>= 1) acc[c] += __shfl_down(acc[c], off);
    if ((threadIdx.x & 63) == 0) red[threadIdx.x >> 6][c] = acc[c];
  }
  __syncthreads();
  if (threadIdx.x < 17) {
    float s = 0.f;
    for (int k = 0; k < 4; ++k) s += red[k][threadIdx.x];
    partial[(size_t)blockIdx.x * 17 + threadIdx.x] = s;
  }
}

// Adam on FP32 master weights; refreshes the bf16 compute copy and, for 3^3 layers,
// the flipped/transposed copy used by the data gradient (wt[26 - tap][ci][co] = w[tap][co][ci]).
// All of a network's tensors in one launch (21 launches took 101 us and their gaps, one 11).
__global__ __launch_bounds__(256) void k_adam(AdamArgs a) {
  int k = 0;
  while (k + 1 < a.n && blockIdx.x >= a.t[k + 1].first) ++k;
  const AdamTensor& t = a.t[k];
  const unsigned j = (blockIdx.x - t.first) * 256u + threadIdx.x;
  if (j >= t.count) return;
  const float g = t.grad[j];
  const float m = a.beta1 * t.m[j] + (1.f - a.beta1) * g;
  const float v = a.beta2 * t.v[j] + (1.f - a.beta2) * g * g;
  t.m[j] = m;
  t.v[j] = v;
  const float mh = m * a.c1, vh = v * a.c2;
  const float w = t.w[j] - a.lr * mh / (sqrtf(vh) + a.eps);
  t.w[j] = w;
  if (t.wbf) t.wbf[j] = f2bf(w);
  if (t.wt) {
    const unsigned per = (unsigned)(t.cout * t.cin);
    const unsigned tap = j / per, rem = j - tap * per;
    const unsigned co = rem / t.cin, ci = rem - co * t.cin;
    t.wt[((size_t)(t.taps - 1 - (int)tap) * t.cin + ci) * t.cout + co] = f2bf(w);
  }
}

// normalisation of the network input: partial[b] = {sum w_v img_v, sum w_v} (FP64) over a
// grid-stride share of the voxels and all views; the scale is the ratio of the totals
__global__ __launch_bounds__(256) void k_wsum_partials(InputArgs a, size_t n, double2* __restrict__ partial) {
  __shared__ double red[256], redw[256];
  double s = 0.0, sw = 0.0;
  const size_t stride = (size_t)gridDim.x * blockDim.x;
  const size_t t0 = (size_t)blockIdx.x * blockDim.x + threadIdx.x;
  // Four voxels per step with 16-byte loads when every volume is 16-byte aligned: all views' loads are issued
  // before the sums (views beyond V read view 0 and are not summed), and each voxel's float sums run over the
  // views in order, as in the scalar loop below that takes the rest.
  bool vec = true;
  for (int c = 0; c < a.V; ++c) vec = vec && !(((uintptr_t)a.img[c] | (uintptr_t)a.w[c]) & 15);
  const size_t n4 = vec ? n / 4 : 0;
  for (size_t i = t0; i < n4; i += stride) {
    float4 im[kNetMaxViews], wv[kNetMaxViews];
#pragma unroll
    for (int c = 0; c < kNetMaxViews; ++c) {
      const int cc = c < a.V ? c : 0;
      im[c] = reinterpret_cast<const float4*>(a.img[cc])[i];
      wv[c] = reinterpret_cast<const float4*>(a.w[cc])[i];
    }
    float4 t = make_float4(0.f, 0.f, 0.f, 0.f), tw = t;
#pragma unroll
    for (int c = 0; c < kNetMaxViews; ++c) {
      if (c >= a.V) break;
      t.x += im[c].x * wv[c].x;
      t.y += im[c].y * wv[c].y;
      t.z += im[c].z * wv[c].z;
      t.w += im[c].w * wv[c].w;
      tw.x += wv[c].x;
      tw.y += wv[c].y;
      tw.z += wv[c].z;
      tw.w += wv[c].w;
    }
    s += (double)t.x;
    s += (double)t.y;
    s += (double)t.z;
    s += (double)t.w;
    sw += (double)tw.x;
    sw += (double)tw.y;
    sw += (double)tw.z;
    sw += (double)tw.w;
  }
  for (size_t i = 4 * n4 + t0; i < n; i += stride) {
    float t = 0.f, tw = 0.f;
    for (int c = 0; c < a.V; ++c) {
      t += a.img[c][i] * a.w[c][i];
      tw += a.w[c][i];
    }
    s += (double)t;
    sw += (double)tw;
  }
  red[threadIdx.x] = s;
  redw[threadIdx.x] = sw;
  __syncthreads();
  for (int off = 128; off > 0; off >>= 1) {
    if ((int)threadIdx.x < off) {
      red[threadIdx.x] += red[threadIdx.x + off];
      redw[threadIdx.x] += redw[threadIdx.x + off];
    }
    __syncthreads();
  }
  if (threadIdx.x == 0) partial[blockIdx.x] = make_double2(red[0], redw[0]);
}

// ------------------------------------------------------------------ launchers
static inline dim3 row_block(int units) { return dim3(units <= 64 ? 64 : units <= 128 ? 128 : 256); }
static inline dim3 row_grid(int units, int H, int ND) { return dim3((units + row_block(units).x - 1) / row_block(units).x, H, ND); }
static inline int grid1(size_t n, int cap = 8192) {
  const size_t b = (n + 255) / 256;
  return (int)(b < 1 ? 1 : (b > (size_t)cap ? (size_t)cap : b));
}

void launch_pool_fwd(const uint16_t* in, int ics, int ico, uint16_t* out, int ocs, int C, int N, int D, int H, int W,
                     hipStream_t s) {
  const int units = W * (C / 8);
  hipLaunchKernelGGL(k_pool_fwd, row_grid(units, H, N * D), row_block(units), 0, s, in, ics, ico, out, ocs, C, D, H, W);
}
void launch_pool_bwd(const uint16_t* dout, int ocs, uint16_t* din, int ics, int ico, int C, int N, int D, int H, int W,
                     const uint16_t* post, hipStream_t s) {
  const int units = 2 * W * (C / 8);
  hipLaunchKernelGGL(k_pool_bwd, row_grid(units, 2 * H, N * 2 * D), row_block(units), 0, s, dout, ocs, din, ics, ico, C, D, H, W, post);
}
void launch_up_fwd(const uint16_t* in, int ics, uint16_t* out, int ocs, int oco, int C, int N, int D, int H, int W,
                   hipStream_t s) {
  const int units = 2 * W * (C / 8);
  hipLaunchKernelGGL(k_up_fwd, row_grid(units, 2 * H, N * 2 * D), row_block(units), 0, s, in, ics, out, ocs, oco, C, D, H, W);
}
void launch_up_bwd(const uint16_t* dfine, int fcs, int fco, uint16_t* dcoarse, int ccs, int C, int N, int D, int H,
                   int W, const uint16_t* post, hipStream_t s) {
  const int units = W * (C / 8);
  hipLaunchKernelGGL(k_up_bwd, row_grid(units, H, N * D), row_block(units), 0, s, dfine, fcs, fco, dcoarse, ccs, C, D, H, W, post);
}
void launch_pack_patches(const PatchArgs& a, int n, hipStream_t s) {
  const unsigned total = (unsigned)a.P * a.P * a.P;
  hipLaunchKernelGGL(k_pack_patches, dim3((total + 255) / 256, n), dim3(256), 0, s, a);
}
void launch_pack_input(const InputArgs& a, hipStream_t s) {
  hipLaunchKernelGGL(k_pack_input, dim3((a.W + 255) / 256, a.H, a.D), dim3(256), 0, s, a);
}
int launch_head(const HeadArgs& a, hipStream_t s) {
  const int nb = grid1(a.nvox, 1024);
  hipLaunchKernelGGL(k_head, dim3(nb), dim3(256), 0, s, a);
  return nb;
}
int launch_head_bwd(const HeadArgs& a, uint16_t* dd1, float* partial, hipStream_t s) {
  const int nb = grid1(a.nvox, 512);
  hipLaunchKernelGGL(k_head_bwd, dim3(nb), dim3(256), 0, s, a, dd1, partial);
  return nb;
}
void launch_adam(const AdamArgs& a, hipStream_t s) {
  AdamArgs b = a;
  unsigned nwg = 0;
  for (int k = 0; k < b.n; ++k) {
    b.t[k].first = nwg;
    nwg += (b.t[k].count + 255) / 256;
  }
  hipLaunchKernelGGL(k_adam, dim3(nwg), dim3(256), 0, s, b);
}
int launch_wsum_partials(const InputArgs& a, size_t n, double2* partial, hipStream_t s) {
  const int nb = grid1(n, 1024);
  hipLaunchKernelGGL(k_wsum_partials, dim3(nb), dim3(256), 0, s, a, n, partial);
  return nb;
}
}  // namespace mvr
