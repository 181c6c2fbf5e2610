// unet_wgrad.hip -- weight and bias gradients of the U-Net's 3^3 convolutions on BF16 MFMA.
//
// dw[tap][co][ci] = sum_v dout[v][co] in[v + off(tap)][ci] and db[co] = sum_v dout[v][co], zero padding,
// channels-last bf16 tensors (see unet.hip): a matrix product over the voxels for each tap.  A work-group owns NCO
// 16-channel blocks of dout and one 16-channel block of the input (grid.y) and walks a contiguous range of tiles of
// TX x TY = 128 voxels of one z plane (grid.x partitions):
//   - the tile of dout and the halo 3 x (TY+2) x (TX+2) of the input go into LDS as they are in HBM, [voxel][16],
//     with 16-byte accesses; the next tile's values are requested into registers before the products of this one;
//   - the products need 8 voxels of one channel per lane, the transpose of that layout: ds_read_b64_tr_b16
//     transposes 4 voxels x 16 channels per 16 lanes on the way out of LDS, so a tap's shift is only a voxel offset
//     of the read.  Two such reads (voxels 4g..4g+3 and 16 + 4g.. of a 32-voxel step, g = lane / 16) fill one operand
//     of v_mfma_f32_16x16x32_bf16; the sum over K pairs both operands' slots the same way;
//   - each of the four waves holds 7 of the 27 taps; the 28th slot takes an operand of ones: its product is the bias
//     gradient, without another pass over dout.
// Partial sums per work-group (FP32) are added by k_sum_partials in a fixed order.
//
// Bound by the LDS reads of the transposed fragments (1 KB per MFMA of 16 clocks) and the staging latency.  The ten
// layers of a 4 x 64^3 training step (124 GFLOP): 0.47 ms, with fragments straight from L1/L2 (2-byte loads) 7.0 ms
// and 0.38 ms of bias sums; the whole step 9.96 -> 2.06 ms, the sums of partials below included.
#include <hip/hip_runtime.h>

#include <algorithm>
#include <cstdint>

#include "unet.hpp"

namespace mvr {

namespace {

typedef __attribute__((ext_vector_type(4))) short s16x4;
typedef __attribute__((ext_vector_type(8))) short s16x8;
typedef __attribute__((ext_vector_type(8))) __bf16 bf16x8;
typedef __attribute__((ext_vector_type(4))) float f32x4;

constexpr int kWgTile = 128;  // voxels per tile: four K = 32 steps
constexpr int kWgTaps = 7;    // taps per wave

// 8 voxels of the lane's channel: transposed reads at `p` (voxels k) and at `p` + 16 voxels' worth of `step` elements
__device__ __forceinline__ bf16x8 tr_read(const uint16_t* p, int step) {
  typedef __attribute__((address_space(3))) s16x4 lds_s16x4;
  const s16x4 lo = __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_s16x4*)(p));
  const s16x4 hi = __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_s16x4*)(p + step));
  const s16x8 v = __builtin_shufflevector(lo, hi, 0, 1, 2, 3, 4, 5, 6, 7);
  return __builtin_bit_cast(bf16x8, v);
}

template <int TX, int NCO>
__global__ __launch_bounds__(256) void k_conv_wgrad(WgradArgs a, int nbx, int nby, int ntiles) {
  constexpr int TY = kWgTile / TX;
  constexpr int HX = TX + 2, HY = TY + 2;
  constexpr int HV = 3 * HY * HX;             // halo voxels
  constexpr int NL = (HV * 2 + 255) / 256;    // halo loads (16 bytes) per thread
  __shared__ __attribute__((aligned(16))) uint16_t inT[NL * 256 * 8];
  __shared__ __attribute__((aligned(16))) uint16_t doT[NCO * kWgTile * 16];

  const int wave = threadIdx.x >> 6, lane = threadIdx.x & 63;
  const int nib = a.cin / 16;
  const int ib = blockIdx.y % nib, cb = (blockIdx.y / nib) * NCO;
  const int t0 = (int)((long long)ntiles * blockIdx.x / gridDim.x);
  const int t1 = (int)((long long)ntiles * (blockIdx.x + 1) / gridDim.x);

  // staging: this thread's 16-byte unit u = threadIdx.x + 256 k is half (u & 1) of halo voxel u >> 1
  const int half = threadIdx.x & 1;
  uint4 hbuf[NL], dbuf[NCO];
  auto issue = [&](int t) {
    const int bx = t % nbx;
    int r = t / nbx;
    const int by = r % nby;
    r /= nby;
    const int z = r % a.D, n = r / a.D;
    const int x0 = bx * TX, y0 = by * TY;
    const int zb = max(z - 1, 0);  // a valid plane: lanes outside the volume read its first voxel and take zeros
    const uint16_t* src = a.in + ((size_t)n * a.D + zb) * a.H * a.W * a.in_cs + ib * 16 + half * 8;
    int hx = (threadIdx.x >> 1) % HX, hy = ((threadIdx.x >> 1) / HX) % HY, hz = (threadIdx.x >> 1) / (HX * HY);
    constexpr int DX = 128 % HX, DY = (128 / HX) % HY, DZ = 128 / (HX * HY);
#pragma unroll
    for (int k = 0; k < NL; ++k) {
      if (k) {  // advance by 128 halo voxels
        hx += DX;
        const int cy = hx >= HX;
        hx -= cy ? HX : 0;
        hy += DY + cy;
        const int cz = hy >= HY;
        hy -= cz ? HY : 0;
        hz += DZ + cz;
      }
      const int xx = x0 + hx - 1, yy = y0 + hy - 1, zz = z + hz - 1;
      const bool ok = hz < 3 && (unsigned)xx < (unsigned)a.W && (unsigned)yy < (unsigned)a.H &&
                      (unsigned)zz < (unsigned)a.D;
      const size_t gv = ((size_t)(zz - zb) * a.H + yy) * a.W + xx;
      hbuf[k] = *reinterpret_cast<const uint4*>(src + (ok ? gv * a.in_cs : 0));
      if (!ok) hbuf[k] = make_uint4(0u, 0u, 0u, 0u);
    }
    const int v = threadIdx.x >> 1, xx = x0 + v % TX, yy = y0 + v / TX;
    const bool ok = xx < a.W && yy < a.H;
    const uint16_t* dsrc = a.dout + ((size_t)n * a.D + z) * a.H * a.W * a.dout_cs + a.dout_co + cb * 16 + half * 8 +
                           (ok ? ((size_t)yy * a.W + xx) * a.dout_cs : 0);
#pragma unroll
    for (int c = 0; c < NCO; ++c) {
      dbuf[c] = *reinterpret_cast<const uint4*>(dsrc + c * 16);
      if (!ok) dbuf[c] = make_uint4(0u, 0u, 0u, 0u);
    }
  };
  auto park = [&]() {
#pragma unroll
    for (int k = 0; k < NL; ++k) *reinterpret_cast<uint4*>(inT + (threadIdx.x + 256 * k) * 8) = hbuf[k];
#pragma unroll
    for (int c = 0; c < NCO; ++c) *reinterpret_cast<uint4*>(doT + (c * 256 + threadIdx.x) * 8) = dbuf[c];
  };

  // fragment addresses: lane l reads 8 bytes of voxel kv = 4 (l / 16) + (l % 16) / 4 of a step, channels 4 (l % 4)..+3;
  // the step's second 16 voxels and the steps lie at constant offsets
  const int kv = 4 * (lane >> 4) + ((lane & 15) >> 2), c4 = (lane & 3) * 4;
  const uint16_t* da = doT + kv * 16 + c4;
  constexpr int ROWS16 = 16 / TX;  // rows that 16 voxels cover (0: half a row of 32)
  const uint16_t* ba = inT + ((kv / TX) * HX + kv % TX) * 16 + c4;
  constexpr int HI = (ROWS16 ? ROWS16 * HX : 16) * 16;   // halo elements from voxel k to voxel k + 16
  constexpr int STEP = (32 / TX) * HX * 16;              // and to the next step
  const uint16_t* bt[kWgTaps];
#pragma unroll
  for (int j = 0; j < kWgTaps; ++j) {
    const int tap = min(kWgTaps * wave + j, 26);
    bt[j] = ba + ((tap / 9 * HY + tap / 3 % 3) * HX + tap % 3) * 16;
  }
  const bool ones = wave == 3;  // the wave's last slot is the bias gradient's
  const short one = 0x3F80;     // 1.0 in bf16
  const bf16x8 vones = __builtin_bit_cast(bf16x8, s16x8{one, one, one, one, one, one, one, one});

  f32x4 acc[kWgTaps][NCO];
#pragma unroll
  for (int j = 0; j < kWgTaps; ++j)
#pragma unroll
    for (int c = 0; c < NCO; ++c) acc[j][c] = f32x4{0.f, 0.f, 0.f, 0.f};

  if (t0 < t1) issue(t0);
  for (int t = t0; t < t1; ++t) {
    if (t != t0) __syncthreads();  // the previous tile's reads are done
    park();
    __syncthreads();
    if (t + 1 < t1) issue(t + 1);
#pragma unroll
    for (int ks = 0; ks < kWgTile / 32; ++ks) {
      bf16x8 av[NCO];
#pragma unroll
      for (int c = 0; c < NCO; ++c) av[c] = tr_read(da + (c * kWgTile + ks * 32) * 16, 16 * 16);
#pragma unroll
      for (int j = 0; j < kWgTaps; ++j) {
        bf16x8 bv = tr_read(bt[j] + ks * STEP, HI);
        if (j == kWgTaps - 1 && ones) bv = vones;
#pragma unroll
        for (int c = 0; c < NCO; ++c)
          acc[j][c] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(av[c], bv, acc[j][c], 0, 0, 0);
      }
    }
  }

  // D: lane l holds dw[co = 4 (l / 16) + r][ci = l % 16]
  const int i = lane & 15, g = lane >> 4;
#pragma unroll
  for (int j = 0; j < kWgTaps; ++j) {
    const int tap = kWgTaps * wave + j;
#pragma unroll
    for (int c = 0; c < NCO; ++c) {
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        const int co = (cb + c) * 16 + 4 * g + r;
        if (tap < 27)
          a.partial[(((size_t)blockIdx.x * 27 + tap) * a.cout + co) * a.cin + ib * 16 + i] = acc[j][c][r];
        else if (ib == 0 && i == 0)
          a.bias_partial[(size_t)blockIdx.x * a.cout + co] = acc[j][c][r];
      }
    }
  }
}

// Sums of partials in a fixed order: grad[j] = sum_p partial[p][j] for j < count and, in the last work-group,
// bgrad[j] = sum_p bpartial[p][j] for j < bcount <= 64.  A work-group takes 64 consecutive j, its 16 waves every
// 16th partial each (8 loads in flight per lane): with one thread per j the 256 loads of a small layer ran one after
// the other on a few CUs (53 us per sum, 21 sums in a training step; now 7 us, 11 sums).
constexpr int kSumWaves = 16;
__global__ __launch_bounds__(64 * kSumWaves) void k_sum_partials(const float* __restrict__ partial, int nparts,
                                                                 size_t count, float* __restrict__ grad,
                                                                 const float* __restrict__ bpartial, int bcount,
                                                                 float* __restrict__ bgrad) {
  __shared__ float red[kSumWaves][64];
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  const bool isBias = (size_t)blockIdx.x * 64 >= count;
  const float* src = isBias ? bpartial : partial;
  const size_t n = isBias ? (size_t)bcount : count;
  const size_t j = isBias ? (size_t)lane : (size_t)blockIdx.x * 64 + lane;
  float s = 0.f;
  if (j < n) {
    int p = wave;
    for (; p + 7 * kSumWaves < nparts; p += 8 * kSumWaves) {
      float v[8];
#pragma unroll
      for (int k = 0; k < 8; ++k) v[k] = src[(size_t)(p + k * kSumWaves) * n + j];
#pragma unroll
      for (int k = 0; k < 8; ++k) s += v[k];
    }
    for (; p < nparts; p += kSumWaves) s += src[(size_t)p * n + j];
  }
  red[wave][lane] = s;
  __syncthreads();
  if (wave == 0 && j < n) {
    float t = 0.f;
#pragma unroll
    for (int k = 0; k < kSumWaves; ++k) t += red[k][lane];
    (isBias ? bgrad : grad)[j] = t;
  }
}

template <int TX>
void launch_tx(const WgradArgs& a, int nbx, int nby, int ntiles, int nparts, hipStream_t s) {
  const int nib = a.cin / 16, ncb = a.cout / 16;
  if (ncb % 2 == 0)
    hipLaunchKernelGGL((k_conv_wgrad<TX, 2>), dim3(nparts, nib * ncb / 2), dim3(256), 0, s, a, nbx, nby, ntiles);
  else
    hipLaunchKernelGGL((k_conv_wgrad<TX, 1>), dim3(nparts, nib * ncb), dim3(256), 0, s, a, nbx, nby, ntiles);
}

// voxels of all tiles of width tx, padding included
long long tiled_voxels(const WgradArgs& a, int tx) {
  const int ty = kWgTile / tx;
  return (long long)((a.W + tx - 1) / tx) * ((a.H + ty - 1) / ty) * kWgTile;
}

}  // namespace

int launch_conv_wgrad(const WgradArgs& a, int maxParts, hipStream_t s) {
  // the tile shape that pads the plane least (the widest of equals: its halo rows are the longest runs)
  int tx = 32;
  for (const int c : {16, 8})
    if (tiled_voxels(a, c) < tiled_voxels(a, tx)) tx = c;
  const int ty = kWgTile / tx;
  const int nbx = (a.W + tx - 1) / tx, nby = (a.H + ty - 1) / ty;
  const int ntiles = nbx * nby * a.D * a.N;
  // at least two tiles per partition
  const int nparts = std::max(1, std::min(wgrad_max_parts(a.cin, a.cout, maxParts), (ntiles + 1) / 2));
  if (tx == 32) launch_tx<32>(a, nbx, nby, ntiles, nparts, s);
  else if (tx == 16) launch_tx<16>(a, nbx, nby, ntiles, nparts, s);
  else launch_tx<8>(a, nbx, nby, ntiles, nparts, s);
  return nparts;
}

void launch_sum_partials(const float* partial, int nparts, size_t count, float* grad, const float* bpartial,
                         int bcount, float* bgrad, hipStream_t s) {
  const unsigned nb = (unsigned)((count + 63) / 64) + (bcount > 0 ? 1 : 0);
  hipLaunchKernelGGL(k_sum_partials, dim3(nb), dim3(64 * kSumWaves), 0, s, partial, nparts, count, grad, bpartial,
                     bcount, bgrad);
}

}  // namespace mvr
