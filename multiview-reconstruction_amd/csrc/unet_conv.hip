// unet_conv.hip -- 3^3 convolutions of the U-Net on BF16 MFMA (forward and data gradient).
//
// out[v][co] = act( sum_tap sum_ci in[v + off(tap)][ci] * w[tap][co][ci] + bias[co] ), zero padding,
// channels-last bf16 tensors (see unet.hip).  A work-group computes a column of 16 x 16 voxel tiles (consecutive z
// planes) for NG x 16 output channels (grid.y selects the channel group):
//   - an input may be a concatenation [up(coarse), fine] whose first part is read from the coarse
//     tensor at half the coordinates (nearest x2 upsampling fused into the staging);
//   - the input goes through LDS one 16-channel chunk and one 18 x 18 halo plane at a time, in a ring of five planes
//     (one chunk) or six (several): while the products of one output plane run on three of them, LDS-DMA loads
//     (global_load_lds_dwordx4: 16 bytes per lane straight into LDS at the wave's base + 16 lane) fill the others with
//     the planes that come next, so each input plane crosses LDS once per work-group.  Halo voxels outside the volume read a zero in device memory.  Each
//     plane is stored as two 8-channel halves [half][voxel][8], so that the 16 lanes reading one half of 16
//     consecutive voxels touch 256 contiguous bytes (no bank conflicts);
//   - v_mfma_f32_16x16x32_bf16 takes K = 32 as two taps x 16 channels: lanes 0-31 carry tap 2p,
//     lanes 32-63 tap 2p+1 (tap 27 = zero weights on tap 26's voxel), eight channels per lane;
//   - the weights of the chunk stay in registers (14 fragments per output group): only the voxel fragments are read
//     from LDS;
//   - the weights are the first operand, the voxels the second: lane l of the result holds channels 4(l/16)..+3 of
//     voxel l%16, stored with one 8-byte access.
// The sum over K pairs both operands' slots the same way, so the kernel relies only on the M/N placement:
// lane l holds rows/columns l%16 of A/B, and D[4(l/16)+r][l%16].
//
// One-chunk layers (cin = 16) march a column of planes with one plane's accumulators; layers of several chunks keep
// the accumulators of ZP planes and take the chunks one after the other (every sum runs over the chunks in order,
// and over the tap pairs in order within a chunk).
//
// Bound by the LDS reads of the voxel fragments: a fragment (1 KB, 8 clocks of the CU's LDS) feeds NG products of 16
// clocks, so 16 -> 16 layers that read one for each product take 0.75 us at least per plane tile and CU (191 us at
// 252 x 250 x 254; 272 measured, 520 with the weights read from LDS and three halo planes staged per output plane); the
// wide layers lose the rest to the weight reloads between chunks.  Of the 56 fragments that a wave reads per output plane
// more than half repeat values of the same input plane (25 are distinct over the three outputs it serves); taking each once
// needs three outputs' accumulators at a time, in the same order of every sum.  One inference at 252 x 250 x 254, 6 views: 4.75 -> 3.05 ms, with the skip tensors
// stored without the upsampled channels beside them (the pooled layer 734 -> 312 us) and the head fused behind the last
// layer.
#include <hip/hip_runtime.h>

#include <algorithm>
#include <cstdint>

#include "unet.hpp"

namespace mvr {

namespace {

typedef __attribute__((ext_vector_type(8))) __bf16 bf16x8;
typedef __attribute__((ext_vector_type(4))) float f32x4;

__device__ __forceinline__ uint16_t f2bf_rne(float f) {
  const uint32_t u = __float_as_uint(f);
  return (uint16_t)((u + 0x7FFFu + ((u >> 16) & 1u)) >> 16);
}
__device__ __forceinline__ float bf2f(uint32_t b) { return __uint_as_float(b << 16); }

constexpr int TX = 16, TY = 16;               // output tile (one 16-voxel segment per row, four rows per wave)
constexpr int HX = TX + 2, HY = TY + 2;
constexpr int HVP = HX * HY;                  // halo voxels of a plane
constexpr int kDma = 3;                       // DMA instructions per wave and plane: 2 halves x 6 over four waves
constexpr int kPlane = 2 * HVP * 8;           // elements of one ring plane
static_assert(HVP > 5 * 64 && HVP <= 6 * 64, "six DMA instructions per half");

__device__ __attribute__((aligned(16))) uint16_t g_zero[8];  // what halo voxels outside the volume read

// DMA instruction id of a plane fills half id / 6, voxels dma_voxel(id)..+63; a half's last instruction starts early and
// repeats voxels of the one before it (the same values), so that every lane of every instruction writes
__device__ __forceinline__ int dma_voxel(int id) { return min(id % 6 * 64, HVP - 64); }

// a 16-channel chunk's source and this lane's halo voxels in it
struct RingSrc {
  const uint16_t* base;   // the sample's first plane
  size_t plane;           // elements between planes
  int sh;                 // 1: the upsampled (coarse) source
  int off[kDma];          // element offsets in a plane, -1: zeros (outside the xy extent, or channels not stored)
};

__device__ __forceinline__ RingSrc ring_src(const ConvArgs& a, int n, int x0, int y0, int cb, int wave, int lane) {
  RingSrc s;
  const bool up = cb * 16 < a.up_c;
  s.sh = up ? 1 : 0;
  const int sH = a.H >> s.sh, sW = a.W >> s.sh, cs = up ? a.up_cs : a.in_cs;
  const int halves = !up && a.in_half ? 1 : 2;
  s.plane = (size_t)sH * sW * cs;
  s.base = (up ? a.up_in + cb * 16 : a.in + (cb * 16 - a.up_c)) + (size_t)n * (a.D >> s.sh) * s.plane;
#pragma unroll
  for (int j = 0; j < kDma; ++j) {
    const int id = wave * kDma + j, v = dma_voxel(id) + lane;
    const int xx = x0 + v % HX - 1, yy = y0 + v / HX - 1;
    const bool ok = (unsigned)xx < (unsigned)a.W && (unsigned)yy < (unsigned)a.H && id / 6 < halves;
    s.off[j] = ok ? ((yy >> s.sh) * sW + (xx >> s.sh)) * cs + (id / 6) * 8 : -1;
  }
  return s;
}

// DMA of the halo of input plane z into the ring plane `dst`: kDma instructions of every wave
__device__ __forceinline__ void ring_issue(const RingSrc& s, int z, int D, int wave, uint16_t* __restrict__ dst) {
  const bool zok = (unsigned)z < (unsigned)D;
  const uint16_t* src = s.base + (zok ? (size_t)(z >> s.sh) * s.plane : 0);
#pragma unroll
  for (int j = 0; j < kDma; ++j) {
    const int id = wave * kDma + j;
    const uint16_t* p = zok && s.off[j] >= 0 ? src + s.off[j] : g_zero;
    __builtin_amdgcn_global_load_lds((const void*)p,
                                     (__attribute__((address_space(3))) void*)(dst + (id / 6 * HVP + dma_voxel(id)) * 8),
                                     16, 0, 0);
  }
}

// The products of one output plane: ring planes s0, s1, s2 (dz = -1, 0, 1) with the weights wf into acc.  Called with
// the ring planes that DMA loads may be filling as further restrict parameters, so that the compiler can tell the DMA's
// writes from this plane's reads and does not wait for the DMA before them.  Every fragment address is one of a few
// per-lane bases plus a constant: the odd tap of a pair lies one voxel, or one row less two voxels, beyond the even
// one, or is the first tap of the next plane.  LAST: the next chunk's weights replace each pair's after its last use
// (wnext: the next chunk's weights).
struct Weights {
  const uint16_t* base;    // the layer's weights
  int lane0, lane1;        // this lane's byte offsets for pair 13 (tap 26 and the zero tap) and the others
  int chunk;               // byte offset of the output group and chunk (uniform)
  int pair, group;         // bytes between tap pairs, between 16-channel output blocks
};
template <int NG>
__device__ __forceinline__ void load_pair(const Weights& w, int p, bf16x8 (&wf)[NG]) {
  // a buffer load: the uniform part of the address in a scalar, so that the pairs' addresses take no vector registers
  const __amdgpu_buffer_rsrc_t r =
      __builtin_amdgcn_make_buffer_rsrc(const_cast<uint16_t*>(w.base), 0, 0xffffffff, 0x00020000);
  typedef unsigned u32x4 __attribute__((ext_vector_type(4)));
#pragma unroll
  for (int t = 0; t < NG; ++t) {
    u32x4 v = __builtin_amdgcn_raw_buffer_load_b128(r, p < 13 ? w.lane1 : w.lane0, w.chunk + p * w.pair + t * w.group, 0);
    if (p == 13 && (threadIdx.x & 32)) v = u32x4{0u, 0u, 0u, 0u};
    wf[t] = __builtin_bit_cast(bf16x8, v);
  }
}

template <int NG, bool LAST, int AHEAD>
__device__ __forceinline__ void ring_products(const uint16_t* __restrict__ s0, const uint16_t* __restrict__ s1,
                                              const uint16_t* __restrict__ s2, bf16x8 (&wf)[14][NG],
                                              f32x4 (&acc)[4][NG], const Weights& wnext) {
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), lane = threadIdx.x & 63;
  const int hi = lane >> 5, hsel = (lane >> 4) & 1;
  int lb = hsel * HVP + 4 * wave * HX + (lane & 15);
  asm volatile("" : "+v"(lb));  // the addresses are formed here, not kept in registers for every ring position
  auto frag = [&](int p, int m) {
    const int t0 = 2 * p, t1 = t0 < 26 ? t0 + 1 : t0;  // tap 27 has zero weights: it reads tap 26
    const int d0 = t0 / 9, d1 = t1 / 9;
    const uint16_t* q0 = d0 == 0 ? s0 : d0 == 1 ? s1 : s2;
    const int sh0 = (t0 / 3 % 3) * HX + t0 % 3, sh1 = (t1 / 3 % 3) * HX + t1 % 3;
    const uint16_t* q;
    if (d0 == d1) {
      q = q0 + (lb + hi * (sh1 - sh0) + sh0) * 8;
    } else {
      const uint16_t* q1 = d1 == 1 ? s1 : s2;
      q = hi ? q1 + (lb + sh1) * 8 : q0 + (lb + sh0) * 8;
    }
    return *reinterpret_cast<const bf16x8*>(q + m * HX * 8);
  };
  bf16x8 vf[14][4];
#pragma unroll
  for (int p = 0; p < 14; ++p)
#pragma unroll
    for (int m = 0; m < 4; ++m) vf[p][m] = frag(p, m);
#pragma unroll
  for (int p = 0; p < 14; ++p) {
#pragma unroll
    for (int m = 0; m < 4; ++m)
#pragma unroll
      for (int t = 0; t < NG; ++t)
        acc[m][t] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(wf[p][t], vf[p][m], acc[m][t], 0, 0, 0);
    if (LAST) load_pair<NG>(wnext, p, wf[p]);
  }
  // The reads run AHEAD to AHEAD + 1 pairs ahead of the products (left to itself the compiler waits for each read at
  // its product: 1037 -> 926-968 us for the 48 -> 16 layer at 252 x 250 x 254).  AHEAD = 0 leaves it so: at three
  // work-groups per CU the registers of reads in flight spill, and the others' reads fill the gaps (16 -> 16 layer: 272 us,
  // 304 us with two work-groups and reads two pairs ahead).
  if constexpr (AHEAD > 0) {
    __builtin_amdgcn_sched_group_barrier(0x100, 4 * AHEAD, 0);  // LDS reads
#pragma unroll
    for (int p = 0; p < 14 - AHEAD; ++p) {
      __builtin_amdgcn_sched_group_barrier(0x100, 4, 0);
      __builtin_amdgcn_sched_group_barrier(0x008, 4 * NG, 0);  // MFMA
    }
    __builtin_amdgcn_sched_group_barrier(0x008, 4 * NG * AHEAD, 0);
  }
  // the products belong before the wait that follows (nothing else orders them with it)
#pragma unroll
  for (int m = 0; m < 4; ++m)
#pragma unroll
    for (int t = 0; t < NG; ++t) asm volatile("" : "+v"(acc[m][t]));
}

// the weights of a chunk: lane l holds output channel l%16 of tap 2p + l/32, channels 8 (l/16 % 2)..+7
__device__ __forceinline__ Weights ring_weights(const ConvArgs& a, int co0, int cb) {
  const int lane = threadIdx.x & 63;
  Weights w;
  w.base = a.w;
  w.lane0 = 2 * ((lane & 15) * a.cin + ((lane >> 4) & 1) * 8);
  w.lane1 = w.lane0 + 2 * (lane >> 5) * a.cout * a.cin;
  w.chunk = 2 * (co0 * a.cin + cb * 16);
  w.pair = 4 * a.cout * a.cin;
  w.group = 32 * a.cin;
  return w;
}

// bias and ReLU of output plane z, bf16 stores, and what is fused behind them:
//   - the 2x2x2 pooling: even lanes sum the stored values of their voxel pair (the odd voxel's from the next lane) in
//     the order of k_pool_fwd, z, then y, then x, so the fused pooling rounds exactly as the pooling kernel; pool[ky]
//     carries the sums from an even plane to the odd one after it;
//   - the output head of an inference (NG = 1, 16 channels): psi of voxel (row 4 wave + l/16, l%16) per lane, the
//     activations themselves not stored;
//   - the ReLU of a backward pass: values whose activation (mask_values) was not positive
//     are stored as zeros (ten passes over the gradients before, 121 us of a step of four 64^3 patches).
enum Epilogue { kPlain, kPool, kHead, kMask };

// this lane's activations of output plane z, in the order of ring_store
template <int NG>
__device__ __forceinline__ void mask_values(const ConvArgs& a, int n, int z, int x0, int y0, int co0,
                                            uint2 (&act)[4][NG]) {
  const int wave = threadIdx.x >> 6, lane = threadIdx.x & 63;
  const int x = min(x0 + (lane & 15), a.W - 1);
  const uint16_t* plane = a.mask + ((size_t)n * a.D + z) * a.H * a.W * a.mask_cs + co0 + 4 * (lane >> 4);
#pragma unroll
  for (int m = 0; m < 4; ++m) {
    const int y = min(y0 + 4 * wave + m, a.H - 1);
#pragma unroll
    for (int t = 0; t < NG; ++t)
      act[m][t] = *reinterpret_cast<const uint2*>(plane + ((size_t)y * a.W + x) * a.mask_cs + t * 16);
  }
}

template <int NG, int EPI>
__device__ __forceinline__ void ring_store(const ConvArgs& a, int n, int z, int x0, int y0, int co0,
                                           const f32x4 (&acc)[4][NG], const f32x4 (&bias)[NG], const f32x4& hw,
                                           float hb, float avg, float (*pool)[NG][4], const uint2 (*act)[NG]) {
  const int wave = threadIdx.x >> 6, lane = threadIdx.x & 63;
  const int i = lane & 15, g = lane >> 4;
  const int x = x0 + i;
  uint16_t* outPlane = a.out + ((size_t)n * a.D + z) * a.H * a.W * a.out_cs + a.out_co + co0 + 4 * g;
  constexpr bool pooling = EPI == kPool;
  if (pooling && !(z & 1)) {
#pragma unroll
    for (int ky = 0; ky < 2; ++ky)
#pragma unroll
      for (int t = 0; t < NG; ++t)
#pragma unroll
        for (int r = 0; r < 4; ++r) pool[ky][t][r] = 0.f;
  }
  float head = 0.f;
#pragma unroll
  for (int m = 0; m < 4; ++m) {
    const int y = y0 + 4 * wave + m;
    const bool ok = y < a.H && x < a.W;
#pragma unroll
    for (int t = 0; t < NG; ++t) {
      uint32_t b[4];
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        float v = acc[m][t][r] + bias[t][r];
        if (a.relu) v = fmaxf(v, 0.f);
        b[r] = f2bf_rne(v);
        if constexpr (EPI == kMask) {
          const uint32_t p = r < 2 ? act[m][t].x : act[m][t].y;
          if (bf2f(r & 1 ? p >> 16 : p & 0xffffu) <= 0.f) b[r] = 0;
        }
      }
      if constexpr (EPI == kHead) {
        float h = 0.f;
#pragma unroll
        for (int r = 0; r < 4; ++r) h += hw[r] * bf2f(b[r]);
        h += __shfl_xor(h, 16, 64);
        h += __shfl_xor(h, 32, 64);
        head = m == g ? h : head;
        continue;
      }
      if (ok)
        *reinterpret_cast<uint2*>(outPlane + ((size_t)y * a.W + x) * a.out_cs + t * 16) =
            make_uint2(b[0] | (b[1] << 16), b[2] | (b[3] << 16));
      if (pooling) {
#pragma unroll
        for (int r = 0; r < 4; ++r) {
          const int own = __float_as_int(bf2f(b[r]));
          const float next = __int_as_float(__builtin_amdgcn_update_dpp(0, own, 0xB1, 0xf, 0xf, true));  // lane ^ 1
          pool[m >> 1][t][r] += __int_as_float(own);
          pool[m >> 1][t][r] += next;
        }
      }
    }
  }
  if constexpr (EPI == kHead) {
    const int y = y0 + 4 * wave + g;
    if (y < a.psi.oy && x < a.psi.ox && z >= a.psi.zlo && z < a.psi.oz) {
      const float pred = avg + (head + hb);
      a.psi.out[((size_t)z * a.psi.oy + y) * a.psi.ox + x] = fmaxf(a.psi.minValue, a.psi.scale * pred);
    }
  }
  if (pooling && (z & 1)) {
    // the plane pair is complete: output voxel (z / 2, y / 2, x / 2) of the pooled tensor (D, H, W even)
    const int H2 = a.H / 2, W2 = a.W / 2, x2 = x / 2;
    uint16_t* pp = a.pool_out + ((size_t)n * (a.D / 2) + z / 2) * H2 * W2 * a.pool_cs + co0 + 4 * g;
#pragma unroll
    for (int ky = 0; ky < 2; ++ky) {
      const int y2 = (y0 + 4 * wave) / 2 + ky;
      if ((i & 1) || y2 >= H2 || x2 >= W2) continue;
#pragma unroll
      for (int t = 0; t < NG; ++t) {
        uint32_t b[4];
#pragma unroll
        for (int r = 0; r < 4; ++r) b[r] = f2bf_rne(pool[ky][t][r] * 0.125f);
        *reinterpret_cast<uint2*>(pp + ((size_t)y2 * W2 + x2) * a.pool_cs + t * 16) =
            make_uint2(b[0] | (b[1] << 16), b[2] | (b[3] << 16));
      }
    }
  }
}

struct RingTile {
  int x0, y0, zs, n;
};
// work-group -> (n, z group of zp planes, y block, x block); x block fastest.  Consecutive work-groups go to the 8 XCDs
// in turn, so the tile order is remapped to give each XCD a contiguous range of tiles (whole z planes and their
// neighbours stay in that XCD's L2).
__device__ __forceinline__ RingTile ring_tile(const ConvArgs& a, int zp) {
  const int nbx = (a.W + TX - 1) / TX, nby = (a.H + TY - 1) / TY, nzg = (a.D + zp - 1) / zp;
  const int nbt = (int)gridDim.x;
  int b = nbt % 8 == 0 ? (int)(blockIdx.x % 8) * (nbt / 8) + (int)(blockIdx.x / 8) : (int)blockIdx.x;
  RingTile t;
  t.x0 = (b % nbx) * TX;
  b /= nbx;
  t.y0 = (b % nby) * TY;
  b /= nby;
  t.zs = (b % nzg) * zp;
  t.n = b / nzg;
  return t;
}

template <int NG>
__device__ __forceinline__ void ring_bias(const ConvArgs& a, int co0, f32x4 (&bias)[NG]) {
  const int g = (threadIdx.x & 63) >> 4;
#pragma unroll
  for (int t = 0; t < NG; ++t)
#pragma unroll
    for (int r = 0; r < 4; ++r) bias[t][r] = a.bias ? a.bias[co0 + t * 16 + 4 * g + r] : 0.f;
}

template <int NG>
__device__ __forceinline__ void zero_acc(f32x4 (&acc)[4][NG]) {
#pragma unroll
  for (int m = 0; m < 4; ++m)
#pragma unroll
    for (int t = 0; t < NG; ++t) acc[m][t] = f32x4{0.f, 0.f, 0.f, 0.f};
}

// All but the wave's last `YOUNGER` memory operations have completed (its DMA among them, in issue order); after the
// barrier that holds for every wave, and every wave is done with the planes it has read.  The wait is the wave's own
// s_waitcnt: the barrier's fence would wait for the DMA still wanted in flight.
template <int YOUNGER>
__device__ __forceinline__ void ring_wait() {
  static_assert(YOUNGER < 16, "low vmcnt bits");
  __builtin_amdgcn_sched_barrier(0);
  asm volatile("" ::: "memory");
  __builtin_amdgcn_s_waitcnt(0x0070 | YOUNGER);  // vmcnt(YOUNGER) lgkmcnt(0), no export wait
  __builtin_amdgcn_s_barrier();
  asm volatile("" ::: "memory");
  __builtin_amdgcn_sched_barrier(0);
}

// One step of a column: the DMA of input plane zn into `nxt`, the products, the wait for the plane the next step needs
// (its DMA went out a step earlier; `nxt` stays in flight), the stores, which drain during the next step.
template <int NG, int EPI>
__device__ __forceinline__ void column_step(const ConvArgs& a, const RingSrc& src, const RingTile& T, int z, int ze,
                                            int co0, const uint16_t* __restrict__ s0, const uint16_t* __restrict__ s1,
                                            const uint16_t* __restrict__ s2, const uint16_t* __restrict__ s3,
                                            uint16_t* __restrict__ nxt, bf16x8 (&wf)[14][NG],
                                            const f32x4 (&bias)[NG], const f32x4& hw, float hb, float (*pool)[NG][4]) {
  (void)s3;  // in flight or landed: distinct from the others for the compiler
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), lane = threadIdx.x & 63;
  f32x4 acc[4][NG];
  zero_acc<NG>(acc);
  float avg = 0.f;
  if constexpr (EPI == kHead) {
    const int y = T.y0 + 4 * wave + (lane >> 4), x = T.x0 + (lane & 15);
    avg = a.psi.avg[((size_t)z * a.H + min(y, a.H - 1)) * a.W + min(x, a.W - 1)];
  }
  const bool more = z + 2 < ze;
  if (more) ring_issue(src, z + 3, a.D, wave, nxt);
  __builtin_amdgcn_sched_barrier(0);  // the DMA goes out before the products, not behind them
  ring_products<NG, false, NG == 1 ? 0 : 1>(s0, s1, s2, wf, acc, Weights{});
  uint2 act[4][NG];
  if constexpr (EPI == kMask) mask_values<NG>(a, T.n, z, T.x0, T.y0, co0, act);  // ahead of them its registers spill
  if (more)
    ring_wait<kDma>();
  else if (z + 1 < ze)
    ring_wait<0>();
  ring_store<NG, EPI>(a, T.n, z, T.x0, T.y0, co0, acc, bias, hw, hb, avg, pool, act);
}

// One chunk: a column of zp planes through a ring of five (unrolled by five, so that the ring positions are known at
// compile time).
template <int NG, int EPI>
__global__ __launch_bounds__(256, NG == 1 ? 3 : 2) void k_conv_column(ConvArgs a, int zp) {
  __shared__ __attribute__((aligned(16))) uint16_t r0[kPlane];
  __shared__ __attribute__((aligned(16))) uint16_t r1[kPlane];
  __shared__ __attribute__((aligned(16))) uint16_t r2[kPlane];
  __shared__ __attribute__((aligned(16))) uint16_t r3[kPlane];
  __shared__ __attribute__((aligned(16))) uint16_t r4[kPlane];
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), lane = threadIdx.x & 63;
  const RingTile T = ring_tile(a, zp);
  const int co0 = blockIdx.y * NG * 16, ze = min(a.D, T.zs + zp);
  bf16x8 wf[14][NG];
  f32x4 bias[NG];
  float pool[2][NG][4];
  const RingSrc src = ring_src(a, T.n, T.x0, T.y0, 0, wave, lane);
  ring_issue(src, T.zs - 1, a.D, wave, r0);
  ring_issue(src, T.zs, a.D, wave, r1);
  ring_issue(src, T.zs + 1, a.D, wave, r2);
  ring_issue(src, T.zs + 2, a.D, wave, r3);
  const Weights w = ring_weights(a, co0, 0);
#pragma unroll
  for (int p = 0; p < 14; ++p) load_pair<NG>(w, p, wf[p]);
  ring_bias<NG>(a, co0, bias);
  f32x4 hw{};
  float hb = 0.f;
  if constexpr (EPI == kHead) {
#pragma unroll
    for (int r = 0; r < 4; ++r) hw[r] = a.psi.w[4 * (lane >> 4) + r];
    hb = a.psi.w[16];
  }
  ring_wait<0>();
  for (int z = T.zs;; z += 5) {
    column_step<NG, EPI>(a, src, T, z, ze, co0, r0, r1, r2, r3, r4, wf, bias, hw, hb, pool);
    if (z + 1 >= ze) break;
    column_step<NG, EPI>(a, src, T, z + 1, ze, co0, r1, r2, r3, r4, r0, wf, bias, hw, hb, pool);
    if (z + 2 >= ze) break;
    column_step<NG, EPI>(a, src, T, z + 2, ze, co0, r2, r3, r4, r0, r1, wf, bias, hw, hb, pool);
    if (z + 3 >= ze) break;
    column_step<NG, EPI>(a, src, T, z + 3, ze, co0, r3, r4, r0, r1, r2, wf, bias, hw, hb, pool);
    if (z + 4 >= ze) break;
    column_step<NG, EPI>(a, src, T, z + 4, ze, co0, r4, r0, r1, r2, r3, wf, bias, hw, hb, pool);
    if (z + 5 >= ze) break;
  }
}

// Several chunks, NG = 1: the accumulators of four planes stay in registers while the chunks' six input planes each
// pass through a ring of six, the next chunk's planes and weights requested during the current one.
__device__ __forceinline__ void chunk_planes4(const ConvArgs& a, const RingSrc& cur, const RingSrc& nx, bool more,
                                              int zs, uint16_t* __restrict__ r0, uint16_t* __restrict__ r1,
                                              uint16_t* __restrict__ r2, uint16_t* __restrict__ r3,
                                              uint16_t* __restrict__ r4, uint16_t* __restrict__ r5,
                                              bf16x8 (&wf)[14][1], f32x4 (&acc)[4][4][1], const Weights& wnext) {
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  ring_issue(cur, zs + 2, a.D, wave, r3);
  ring_issue(cur, zs + 3, a.D, wave, r4);
  ring_issue(cur, zs + 4, a.D, wave, r5);
  __builtin_amdgcn_sched_barrier(0);
  ring_products<1, false, 2>(r0, r1, r2, wf, acc[0], wnext);
  ring_wait<2 * kDma>();
  if (more) ring_issue(nx, zs - 1, a.D, wave, r0);
  __builtin_amdgcn_sched_barrier(0);
  ring_products<1, false, 2>(r1, r2, r3, wf, acc[1], wnext);
  ring_wait<kDma>();
  if (more) ring_issue(nx, zs, a.D, wave, r1);
  __builtin_amdgcn_sched_barrier(0);
  ring_products<1, false, 2>(r2, r3, r4, wf, acc[2], wnext);
  ring_wait<0>();
  if (more) ring_issue(nx, zs + 1, a.D, wave, r2);
  __builtin_amdgcn_sched_barrier(0);
  ring_products<1, true, 2>(r3, r4, r5, wf, acc[3], wnext);
  ring_wait<0>();
}

template <int NCHUNK>
__global__ __launch_bounds__(256, 2) void k_conv_chunks4(ConvArgs a) {
  __shared__ __attribute__((aligned(16))) uint16_t r0[kPlane];
  __shared__ __attribute__((aligned(16))) uint16_t r1[kPlane];
  __shared__ __attribute__((aligned(16))) uint16_t r2[kPlane];
  __shared__ __attribute__((aligned(16))) uint16_t r3[kPlane];
  __shared__ __attribute__((aligned(16))) uint16_t r4[kPlane];
  __shared__ __attribute__((aligned(16))) uint16_t r5[kPlane];
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), lane = threadIdx.x & 63;
  const RingTile T = ring_tile(a, 4);
  const int co0 = blockIdx.y * 16;
  bf16x8 wf[14][1];
  f32x4 acc[4][4][1];
#pragma unroll
  for (int o = 0; o < 4; ++o) zero_acc<1>(acc[o]);
  RingSrc cur = ring_src(a, T.n, T.x0, T.y0, 0, wave, lane);
  ring_issue(cur, T.zs - 1, a.D, wave, r0);
  ring_issue(cur, T.zs, a.D, wave, r1);
  ring_issue(cur, T.zs + 1, a.D, wave, r2);
  const Weights w = ring_weights(a, co0, 0);
#pragma unroll
  for (int p = 0; p < 14; ++p) load_pair<1>(w, p, wf[p]);
  ring_wait<0>();
#pragma unroll
  for (int cb = 0; cb < NCHUNK; ++cb) {
    const int nb = cb + 1 < NCHUNK ? cb + 1 : cb;
    const RingSrc nx = ring_src(a, T.n, T.x0, T.y0, nb, wave, lane);
    chunk_planes4(a, cur, nx, cb + 1 < NCHUNK, T.zs, r0, r1, r2, r3, r4, r5, wf, acc, ring_weights(a, co0, nb));
    cur = nx;
  }
  f32x4 bias[1];
  ring_bias<1>(a, co0, bias);
#pragma unroll
  for (int o = 0; o < 4; ++o)
    if (T.zs + o < a.D) ring_store<1, kPlain>(a, T.n, T.zs + o, T.x0, T.y0, co0, acc[o], bias, f32x4{}, 0.f, 0.f, nullptr, nullptr);
}

// Several chunks, NG = 2: two planes' accumulators; a chunk's four input planes take the ring positions 4 c .. 4 c + 3
// modulo six, so three chunks are unrolled.
__device__ __forceinline__ void chunk_planes2(const ConvArgs& a, const RingSrc& cur, const RingSrc& nx, bool more,
                                              int zs, uint16_t* __restrict__ r0, uint16_t* __restrict__ r1,
                                              uint16_t* __restrict__ r2, uint16_t* __restrict__ r3,
                                              uint16_t* __restrict__ r4, uint16_t* __restrict__ r5,
                                              bf16x8 (&wf)[14][2], f32x4 (&acc)[2][4][2], const Weights& wnext) {
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  ring_issue(cur, zs + 2, a.D, wave, r3);
  if (more) {
    ring_issue(nx, zs - 1, a.D, wave, r4);
    ring_issue(nx, zs, a.D, wave, r5);
  }
  __builtin_amdgcn_sched_barrier(0);
  ring_products<2, false, 1>(r0, r1, r2, wf, acc[0], wnext);
  if (more)
    ring_wait<2 * kDma>();
  else
    ring_wait<0>();
  if (more) ring_issue(nx, zs + 1, a.D, wave, r0);
  __builtin_amdgcn_sched_barrier(0);
  ring_products<2, false, 1>(r1, r2, r3, wf, acc[1], wnext);
  if (more) {
#pragma unroll
    for (int p = 0; p < 14; ++p) load_pair<2>(wnext, p, wf[p]);
  }
  ring_wait<0>();
}

template <int NCHUNK, int EPI>
__global__ __launch_bounds__(256, 2) void k_conv_chunks2(ConvArgs a) {
  __shared__ __attribute__((aligned(16))) uint16_t r0[kPlane];
  __shared__ __attribute__((aligned(16))) uint16_t r1[kPlane];
  __shared__ __attribute__((aligned(16))) uint16_t r2[kPlane];
  __shared__ __attribute__((aligned(16))) uint16_t r3[kPlane];
  __shared__ __attribute__((aligned(16))) uint16_t r4[kPlane];
  __shared__ __attribute__((aligned(16))) uint16_t r5[kPlane];
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), lane = threadIdx.x & 63;
  const RingTile T = ring_tile(a, 2);
  const int co0 = blockIdx.y * 32;
  bf16x8 wf[14][2];
  f32x4 acc[2][4][2];
  zero_acc<2>(acc[0]);
  zero_acc<2>(acc[1]);
  RingSrc cur = ring_src(a, T.n, T.x0, T.y0, 0, wave, lane);
  ring_issue(cur, T.zs - 1, a.D, wave, r0);
  ring_issue(cur, T.zs, a.D, wave, r1);
  ring_issue(cur, T.zs + 1, a.D, wave, r2);
  const Weights w = ring_weights(a, co0, 0);
#pragma unroll
  for (int p = 0; p < 14; ++p) load_pair<2>(w, p, wf[p]);
  ring_wait<0>();
#pragma unroll
  for (int cb = 0; cb < NCHUNK; ++cb) {
    const int nb = cb + 1 < NCHUNK ? cb + 1 : cb;
    const RingSrc nx = ring_src(a, T.n, T.x0, T.y0, nb, wave, lane);
    const Weights wn = ring_weights(a, co0, nb);
    if (cb % 3 == 0) chunk_planes2(a, cur, nx, cb + 1 < NCHUNK, T.zs, r0, r1, r2, r3, r4, r5, wf, acc, wn);
    else if (cb % 3 == 1) chunk_planes2(a, cur, nx, cb + 1 < NCHUNK, T.zs, r4, r5, r0, r1, r2, r3, wf, acc, wn);
    else chunk_planes2(a, cur, nx, cb + 1 < NCHUNK, T.zs, r2, r3, r4, r5, r0, r1, wf, acc, wn);
    cur = nx;
  }
  f32x4 bias[2];
  ring_bias<2>(a, co0, bias);
  float pool[2][2][4];
#pragma unroll
  for (int o = 0; o < 2; ++o) {
    if (T.zs + o >= a.D) continue;
    uint2 act[4][2];
    if constexpr (EPI == kMask) mask_values<2>(a, T.n, T.zs + o, T.x0, T.y0, co0, act);
    ring_store<2, EPI>(a, T.n, T.zs + o, T.x0, T.y0, co0, acc[o], bias, f32x4{}, 0.f, 0.f, pool, act);
  }
}

template <int NG>
void launch_ng(const ConvArgs& a, hipStream_t s) {
  const long long tiles = (long long)((a.W + TX - 1) / TX) * ((a.H + TY - 1) / TY) * a.N;
  const int groups = a.cout / (16 * NG);
  auto columns = [&](int zp) { return (unsigned)(tiles * ((a.D + zp - 1) / zp)); };
  if (a.cin == 16) {
    // planes per work-group: the longest columns (the first three planes of a column are not overlapped) that still
    // give every CU its three (NG = 1) or two work-groups a few times over; even, for the pooling's plane pairs
    int zp = 16;
    while (zp > 2 && (long long)columns(zp) * groups < 1024) zp /= 2;
    const dim3 grid(columns(zp), groups);
    if (a.psi.out)
      hipLaunchKernelGGL((k_conv_column<1, kHead>), grid, dim3(256), 0, s, a, zp);
    else if (a.pool_out)
      hipLaunchKernelGGL((k_conv_column<1, kPool>), grid, dim3(256), 0, s, a, zp);
    else if (a.mask)
      hipLaunchKernelGGL((k_conv_column<1, kMask>), grid, dim3(256), 0, s, a, zp);
    else
      hipLaunchKernelGGL((k_conv_column<NG, kPlain>), grid, dim3(256), 0, s, a, zp);
    return;
  }
  if constexpr (NG == 1) {
    const dim3 grid(columns(4), groups);
    if (a.cin == 32)
      hipLaunchKernelGGL((k_conv_chunks4<2>), grid, dim3(256), 0, s, a);
    else
      hipLaunchKernelGGL((k_conv_chunks4<3>), grid, dim3(256), 0, s, a);
  } else {
    const dim3 grid(columns(2), groups);
    if (a.pool_out)
      hipLaunchKernelGGL((k_conv_chunks2<2, kPool>), grid, dim3(256), 0, s, a);
    else if (a.mask && a.cin == 32)
      hipLaunchKernelGGL((k_conv_chunks2<2, kMask>), grid, dim3(256), 0, s, a);
    else if (a.mask)
      hipLaunchKernelGGL((k_conv_chunks2<4, kMask>), grid, dim3(256), 0, s, a);
    else if (a.cin == 32)
      hipLaunchKernelGGL((k_conv_chunks2<2, kPlain>), grid, dim3(256), 0, s, a);
    else if (a.cin == 64)
      hipLaunchKernelGGL((k_conv_chunks2<4, kPlain>), grid, dim3(256), 0, s, a);
    else
      hipLaunchKernelGGL((k_conv_chunks2<6, kPlain>), grid, dim3(256), 0, s, a);
  }
}

}  // namespace

// pooling is fused into the layers of 16 inputs and 16 outputs and of 32 inputs and an even number of output blocks
bool conv_fuses_pool(const ConvArgs& a) {
  return a.pool_out && !((a.D | a.H | a.W) & 1) && ((a.cin == 16 && a.cout == 16) || (a.cin == 32 && a.cout % 32 == 0));
}

// The network's 3^3 convolutions: cout a multiple of 16; cin 16, or 32 and 48 for an odd number of 16-channel output
// blocks, 32, 64 and 96 for an even one
bool launch_conv_tiled(const ConvArgs& a, hipStream_t s) {
  const bool pairs = a.cout % 32 == 0;
  const bool known = a.cin == 16 || a.cin == 32 || (pairs ? a.cin == 64 || a.cin == 96 : a.cin == 48);
  if (a.taps != 27 || !known || a.cout % 16 != 0 || a.in_cs % (a.in_half ? 8 : 16) != 0) return false;
  // 32-bit offsets within a plane (and the limit callers are told: three planes)
  if (3ll * a.H * a.W * std::max(a.in_half ? 16 : a.in_cs, a.up_cs) >= (1ll << 31)) return false;
  if (a.up_c && (a.up_c % 16 != 0 || a.up_cs % 16 != 0 || !a.up_in || (a.W | a.H | a.D) & 1)) return false;
  if (a.in_half && a.cin != 16) return false;
  if (a.pool_out && !conv_fuses_pool(a)) return false;
  // the backward ReLU behind the layers of 16, 32 or 64 inputs and as many outputs (the kernel of 48 inputs has none)
  if (a.mask && (a.cin != a.cout || a.cin == 48 || a.cin > 64 || a.pool_out || a.psi.out || a.mask_cs % 4 != 0)) return false;
  if (a.psi.out && (a.cin != 16 || a.cout != 16 || a.N != 1)) return false;
  if (pairs)
    launch_ng<2>(a, s);
  else
    launch_ng<1>(a, s);
  return true;
}

}  // namespace mvr
