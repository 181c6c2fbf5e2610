// xpasses.hpp -- x (real axis) passes with the two-step register FFT.
//
// A work-group owns RW rows of one x-pass.  The length-M complex transform of a row (M = P0/2, real FFT by the
// even/odd split) runs as M = A x B with one LDS exchange: one side of it by A lanes per row, the other by B.
//
// The passes are bound by their vector instructions as much as by HBM (at M = 432 these took 75 % of the update's time,
// 65 % of the quotient's), so lanes are packed: where it holds more rows than rows at multiples of 16 or 32 lanes would,
// a wave of the A side holds rows side by side (a row never straddles a wave), and the B side's tasks lie densely over
// the work-group then, and on long rows (B > 16) where that leaves a wave without any.  Elsewhere the aligned rows are
// faster, at M = 225 by 10 %: their exchange has fewer LDS conflicts.  Values next to one another in the real rows move in pairs; whether a pair
// lies inside the row is a question of the register index, not of the lane, except at the row's ends.  Measured, one
// iteration of two views: M = 200 1.08 x, 288 1.06; M = 432, 767 x 700 x 321: forward 197 -> 144 us, quotient 852 -> 690,
// update 851 -> 701 (2.9 -> 3.3 TB/s).  Long rows (B > 16), 2 M - 30 wide, 27300 rows, with the quotient and the update on
// the registers that the inverse leaves and aligned rows, and so (us a launch, and the whole iteration):
//   M           360    400    432    450    480    512    540    576    600    640
//   forward     54 32  59 38  57 42  63 45  66 45  76 56  80 58  78 54  82 55  85 56
//   quotient    93 70  99 81 107 91 118 96 120 108 136 127 131 108 134 132 174 128 178 131
//   update     105 83 119 90 118 104 126 104 140 113 112 110 152 119 160 146 183 156 193 161
//   iteration  1.12x  1.12x  1.08x  1.07x  1.07x  1.02x  1.10x  1.05x  1.11x  1.11x  (M = 300 1.05x, 320 1.07x, 384 1.01x)
//
// The R2C post-processing and the C2R pre-processing combine
// the values k and M - k of a row; after the second forward step (before the first inverse step) lane q holds
// index q + A k2 in register k2, and M - (q + A k2) = (A - q) + A (B - 1 - k2), so the partner is lane A - q,
// register B - 1 - k2 of the same row: the pairs are swapped with wave shuffles, and spectra go between HBM
// and registers directly, coalesced across the row's lanes.  Real-valued data is read into the first forward step
// directly; the quotient and the psi update work on rows parked in LDS.  Index arithmetic that depends on
// runtime sizes is done once per row (row tables in LDS), never per element with '/' or '%'.
#pragma once
#include <algorithm>
#include <type_traits>

#include "passes.hpp"

namespace mvr {

// exact n / d for n < 2^32 / d (d >= 1)
struct FastDiv {
  unsigned d, m;
  __host__ __device__ FastDiv() : d(1), m(0) {}
  __host__ __device__ explicit FastDiv(unsigned dd) : d(dd), m((unsigned)((0x100000000ull + dd - 1) / dd)) {}
  __device__ __forceinline__ unsigned div(unsigned n) const {
    return d == 1 ? n : (unsigned)(((unsigned long long)n * m) >> 32);
  }
};

template <int NT>
constexpr int reduce_width() {
  return NT <= 256 ? 256 : NT <= 512 ? 512 : 1024;  // power of two >= NT
}

// {sum, max} of a work-group of NT threads (NT <= 1024) in the caller's LDS: rs and rm hold
// reduce_width<NT>() doubles each.  Every thread must be done with that memory before the call.
template <int NT>
__device__ __forceinline__ void block_reduce_stats_nt(double s, double mx, double2* out, double* rs, double* rm) {
  constexpr int P = reduce_width<NT>();
  rs[threadIdx.x] = s;
  rm[threadIdx.x] = mx;
  for (int i = NT + (int)threadIdx.x; i < P; i += NT) {
    rs[i] = 0.0;
    rm[i] = -1.0;
  }
  __syncthreads();
#pragma unroll
  for (int off = P / 2; off > 0; off >>= 1) {
    if ((int)threadIdx.x < off) {
      rs[threadIdx.x] += rs[threadIdx.x + off];
      rm[threadIdx.x] = java_max(rm[threadIdx.x], rm[threadIdx.x + off]);
    }
    __syncthreads();
  }
  if (threadIdx.x == 0) *out = make_double2(rs[0], rm[0]);
}

// Where a row's value k lies: rows of HxP consecutive values, or (TR, planar spectra) one value per hx plane, the row
// (y, z) at z P1 + y of every plane.
template <bool TR>
__device__ __forceinline__ size_t x2_row(const Dom& d, int row) {
  return TR ? (size_t)row : (size_t)row * d.HxP;
}
template <bool TR>
__device__ __forceinline__ unsigned x2_at(int k, unsigned cs) {
  return TR ? (unsigned)k * cs : (unsigned)k;
}

constexpr long long kOuterRow = -(1ll << 62);
constexpr size_t kNoRow = ~(size_t)0;

template <int M>
struct XCfg {
  static constexpr Split2 S = split2(M);
  static constexpr int A = S.A, B = S.B;
  static constexpr int NT = 256;             // threads per work-group
  static constexpr int T = A <= 16 ? 16 : A <= 32 ? 32 : 64;  // lanes of a row that start at a multiple of them
  static constexpr int RPW = 64 / A;         // rows per wave on the A side
  static constexpr int TA = RPW > 64 / T ? A : T;             // lanes from row to row
  static constexpr int RW = NT / 64 * RPW;   // rows per work-group
  static constexpr int TQ = NT / RW;         // lanes per row where rows are walked with every thread (>= A >= B)
  // lanes from row to row on the B side: dense where the A side is, and on long rows if that leaves a wave without tasks
  static constexpr int TB = TA == A || (B > 16 && (RW * B + 63) / 64 < NT / 64) ? B : T;
  static constexpr int RS = M + 5;                 // LDS row stride (complex): M used, +5 against bank conflicts
  static constexpr int PX = 2 * M;
  // the exchange rows, at least as large as the stats reduction that reuses them (2 x 256 doubles)
  static constexpr int BUF = RW * RS > 512 ? RW * RS : 512;
  // Twiddle tables (2M + 1 complex) stay in LDS unless leaving them in global memory (read through L1) fits one
  // more work-group per CU into the 160 KB of LDS; the other LDS is the exchange rows and 16-24 B of row tables
  // per row (the stats reduction reuses the rows), plus the x gather map in the forward pass.
  static constexpr int LDS_ROWS = RW * RS * 8 + RW * 24;
  static constexpr int LDS_TW = (2 * M + 1) * 8;
  static constexpr bool TWL = (160 * 1024) / (LDS_ROWS + LDS_TW) >= (160 * 1024) / LDS_ROWS;
  // The forward and quotient passes follow the same rule on long rows (B > 16; at M = 576 global twiddles gave
  // both a third work-group per CU and 2-5 %) and keep LDS twiddles on shorter rows (at M = 150 global twiddles
  // were slower despite the extra work-group).
  static constexpr bool long_rows = B > 16;
  // The forward pass exchanges in two rounds (half of the second step's lanes per round), so its rows hold
  // half a transform: at M = 150 8 instead of 6 work-groups per CU, at M = 576 4 instead of 3.
  static constexpr int AH = (A + 1) / 2;
  static constexpr int RS_FWD = AH * B + 5;
  static constexpr int BUF_FWD = RW * RS_FWD;
  static constexpr int BUF_TR = (M + 1) * (RW + 1);  // the rows' spectra of a planar store
  static constexpr int LDS_ROWS_FWD = RW * RS_FWD * 8 + RW * 24;
  static constexpr bool TWL_FWD = !long_rows || (160 * 1024) / (LDS_ROWS_FWD + PX * 4 + LDS_TW) >=
                                                   (160 * 1024) / (LDS_ROWS_FWD + PX * 4);
  static constexpr bool TWL_RATIO = !long_rows || TWL;
  // The quotient pass at M = 100, 120, 150, 200 compiles to 81 VGPRs (this ROCm), one over what 6 waves per
  // SIMD allow; bounded to 6 waves it takes 80 without spilling (x_ratio 4 % faster at M = 150).  Other lengths
  // either fit already or would spill under the bound.
  static constexpr int MINW_RATIO = (M == 100 || M == 120 || M == 150 || M == 200) ? 6 : 1;
  // The update at M = 432, 450, 480 compiles to 130, 130 and 148 VGPRs (this ROCm), over the 128 that 4 waves per SIMD allow;
  // bounded to 4 waves it takes 128 and spills one (113 -> 104, 114 -> 104, 123 -> 113 us for 27300 rows; M = 432, 225000
  // rows: 778 -> 701).  The other long rows: M = 300 to 400, 512 and 540 take 96-126 without a bound; 576 and 600 (162, 160)
  // would spill 22 (146 -> 157 us, 156 -> 156); 640 fits 3 work-groups per CU by its LDS.
  static constexpr int MINW_UPDATE = (M == 432 || M == 450 || M == 480) ? 4 : 1;
};

template <int M>
__host__ __device__ constexpr bool x2_ok() {
  return split2(M).A > 0 && split2(M).B > 1;
}

// A thread's place on the two sides of a transform: row ra, index qa < A; row rb, index qb < B.  Idle threads have
// qa = A, qb = B (and a valid row).
template <int M>
struct XLane {
  int ra, qa, rb, qb;
  __device__ __forceinline__ XLane() {
    using C = XCfg<M>;
    const int lane = (int)(threadIdx.x & 63), w = (int)(threadIdx.x >> 6), r = lane / C::TA;
    const bool a = C::TA == C::T || r < C::RPW, b = C::TB == C::T || (int)threadIdx.x < C::RW * C::B;
    ra = w * C::RPW + (a ? r : 0);
    qa = a ? lane - r * C::TA : C::A;
    rb = b ? (int)threadIdx.x / C::TB : 0;
    qb = b ? (int)threadIdx.x % C::TB : C::B;
    if (C::TA == C::T && C::TB == C::T) {  // the same lanes on both sides, in the same registers
      ra = rb;
      qa = qb;
    }
  }
};

// two consecutive values at any multiple of 4 bytes, in one access
typedef float PairValue __attribute__((ext_vector_type(2), aligned(4)));
__device__ __forceinline__ float2 ld_pair(const float* p) {
  const PairValue v = *reinterpret_cast<const PairValue*>(p);
  return make_float2(v.x, v.y);
}
__device__ __forceinline__ void st_pair(float* p, float2 v) {
  PairValue u;
  u.x = v.x;
  u.y = v.y;
  *reinterpret_cast<PairValue*>(p) = u;
}

// The x positions of a register index on the B side, [2 B a, 2 B (a + 1)) over the lanes, against a range [lo, hi): the
// same for every lane, so that only the register indices at the range's ends test their positions one by one.
template <int B>
struct XSpan {
  int lo, hi;
  __device__ __forceinline__ bool inside(int a) const { return 2 * B * a >= lo && 2 * B * (a + 1) <= hi; }
  __device__ __forceinline__ bool outside(int a) const { return 2 * B * (a + 1) <= lo || 2 * B * a >= hi; }
};

__device__ __forceinline__ float2 shfl2(float2 v, int src) {
  return make_float2(__shfl(v.x, src, 64), __shfl(v.y, src, 64));
}

// For values V[q + A k2] held as v[k2] by lane q < A of a row (and V[M] as vM in lane 0): out[k2] = V[M - (q + A k2)].
// Lane q > 0 gets them from lane A - q (register B - 1 - k2), lane 0 from itself (M - A k2 = A (B - k2)).
// Every lane of the wave must call it (wave shuffle); idle lanes (q >= A) read themselves.
template <int M>
__device__ __forceinline__ void x2_mirror_pairs(const float2* v, float2 vM, int q, float2* out) {
  using C = XCfg<M>;
  const int lane = (int)(threadIdx.x & 63);
  const int src = q > 0 && q < C::A ? lane - q + (C::A - q) : lane;
#pragma unroll
  for (int k2 = 0; k2 < C::B; ++k2) {
    const float2 t = shfl2(v[C::B - 1 - k2], src);
    out[k2] = q != 0 ? t : (k2 == 0 ? vM : v[(C::B - k2) % C::B]);
  }
}

// forward transform of rows of `buf` (RS values apart) whose first-step inputs v[a] = z[qb + B a] (lanes qb < B) are in
// registers; the rows are only written -> out[k2] = Z[qa + A k2] (lanes qa < A)
template <int M>
__device__ __forceinline__ void x2_forward_regs(float2* buf, const float2* tw, const XLane<M>& l, float2* v, float2* out) {
  using C = XCfg<M>;
  constexpr int A = C::A, B = C::B;
  if (l.qb < B) {
    float2* rb = buf + l.rb * C::RS;
    const int q = l.qb;
    rdft<A, -1>(v);
#pragma unroll
    for (int k1 = 0; k1 < A; ++k1) rb[q + B * k1] = k1 == 0 ? v[k1] : cmul(v[k1], tw[q * k1]);
  }
  __syncthreads();
  if (l.qa < A) {
    const float2* rb = buf + l.ra * C::RS;
#pragma unroll
    for (int b = 0; b < B; ++b) out[b] = rb[b + B * l.qa];
    rdft<B, -1>(out);
  } else {
#pragma unroll
    for (int b = 0; b < B; ++b) out[b] = make_float2(0.f, 0.f);
  }
}

// x2_forward_regs with the exchange in two rounds through rows of AH * B values (RS_FWD apart): round r carries the
// first-step results k1 in [r AH, r AH + AH), read by the lanes qa = k1 of that range
template <int M>
__device__ __forceinline__ void x2_forward_regs_half(float2* buf, const float2* tw, const XLane<M>& l, float2* v,
                                                     float2* out) {
  using C = XCfg<M>;
  constexpr int A = C::A, B = C::B, AH = C::AH;
  const int q = l.qb, qa = l.qa;
  float2* wb = buf + l.rb * C::RS_FWD;
  const float2* rb = buf + l.ra * C::RS_FWD;
  if (q < B) {
    rdft<A, -1>(v);
#pragma unroll
    for (int k1 = 1; k1 < A; ++k1) v[k1] = cmul(v[k1], tw[q * k1]);
  }
#pragma unroll
  for (int b = 0; b < B; ++b) out[b] = make_float2(0.f, 0.f);
#pragma unroll
  for (int r = 0; r < 2; ++r) {
    const int k0 = r * AH, kn = r == 0 ? AH : A - AH;
    if (r > 0) __syncthreads();  // the first round's readers are done
    if (q < B) {
#pragma unroll
      for (int j = 0; j < AH; ++j)
        if (j < kn) wb[q + B * j] = v[k0 + j];
    }
    __syncthreads();
    if (qa >= k0 && qa < k0 + kn) {
#pragma unroll
      for (int b = 0; b < B; ++b) out[b] = rb[b + B * (qa - k0)];
    }
  }
  if (qa < A) rdft<B, -1>(out);
}

// forward transform of the rows of `buf` (natural order) -> out[k2] = Z[qa + A k2] (lanes qa < A)
template <int M>
__device__ __forceinline__ void x2_forward(float2* buf, const float2* tw, const XLane<M>& l, float2* out) {
  using C = XCfg<M>;
  float2 v[C::A];
  if (l.qb < C::B) {
    const float2* rb = buf + l.rb * C::RS;
#pragma unroll
    for (int a = 0; a < C::A; ++a) v[a] = rb[l.qb + C::B * a];
  }
  __syncthreads();  // every lane has read its values before the rows are overwritten
  x2_forward_regs<M>(buf, tw, l, v, out);
}

// R2C post-processing of a row whose complex transform Z lane q holds as z[k2] = Z[q + A k2]:
// X[k] = (Z[k] + Z*[M - k]) / 2 + W_P0^k (Z[k] - Z*[M - k]) / 2i for k = q + A k2, and X[M] (lane 0), written
// to dst (the row's start in HBM; cs: values per hx plane) when rowOk
// (VIA_LDS, planar spectra: through the work-group's LDS `buf`, (M + 1) (RW + 1) values, and from there with lanes along
// the rows: rowAt[r] is row r's place in a plane, kNoRow: not stored.  Stored by the lanes of a row, a plane gets runs of
// 64 / A values: the forward pass of 24 blocks on 120-point grids, 169 MB, takes 78 us so, 60 through the LDS; the
// quotient pass gains nothing by it, 58 and 61)
template <int M, bool TR, bool VIA_LDS>
__device__ __forceinline__ void x2_post_store_regs(const float2* z, const XLane<M>& l, const float2* twr,
                                                   float2* __restrict__ dst, bool rowOk, float2* buf,
                                                   const size_t* rowAt, unsigned cs) {
  using C = XCfg<M>;
  const int q = l.qa;
  float2 zc[C::B];
  x2_mirror_pairs<M>(z, z[0], q, zc);  // Z[M] = Z[0]
  constexpr int TS = C::RW + 1;
  if (VIA_LDS) __syncthreads();  // the rows' exchange values have been read
  if ((VIA_LDS || rowOk) && q < C::A) {
    auto put = [&](int k, float2 zk, float2 c) {
      const float2 e = make_float2(0.5f * (zk.x + c.x), 0.5f * (zk.y + c.y));
      const float2 dd = csub(zk, c);
      const float2 od = make_float2(0.5f * dd.y, -0.5f * dd.x);
      const float2 x = cadd(e, cmul(twr[k], od));
      if (VIA_LDS)
        buf[k * TS + l.ra] = x;
      else
        dst[x2_at<TR>(k, cs)] = x;
    };
#pragma unroll
    for (int k2 = 0; k2 < C::B; ++k2) put(q + C::A * k2, z[k2], cconj(zc[k2]));
    if (q == 0) put(M, z[0], cconj(z[0]));
  }
  if (VIA_LDS) {
    __syncthreads();
    for (int i = threadIdx.x; i < (M + 1) * C::RW; i += C::NT) {
      const int k = i / C::RW, r = i % C::RW;
      const size_t at = rowAt[r];
      if (at != kNoRow) dst[(size_t)k * cs + at] = buf[k * TS + r];
    }
  }
}

// inverse of the half spectrum X[0..M] of one row (src: its start in HBM; null: a row of zeros), read straight
// into registers by the lanes qa of row ra: the C2R pre-processing Z[k] = E[k] + i O[k] combines X[k] and X*[M - k];
// returns z[qb + B n1] of row rb in out[n1] (lanes qb < B)
// PF: the transforms' coprime splits by the prime-factor algorithm (false: Cooley-Tukey throughout, which the
// update pass on short rows runs 3 % faster at M = 150)
template <int M, bool TR, bool PF = true>
__device__ __forceinline__ void x2_inverse_half_regs(const float2* __restrict__ src, float2* buf, const float2* tw,
                                                     const float2* twr, const XLane<M>& l, float2* out, unsigned cs) {
  using C = XCfg<M>;
  constexpr int A = C::A, B = C::B;
  const int q = l.qa;
  float2* wb = buf + l.ra * C::RS;
  const float2* rb = buf + l.rb * C::RS;
  float2 x[B];
  float2 xM = make_float2(0.f, 0.f);
  const bool ld = src != nullptr && q < A;
#pragma unroll
  for (int k2 = 0; k2 < B; ++k2) x[k2] = ld ? src[x2_at<TR>(q + A * k2, cs)] : make_float2(0.f, 0.f);
  if (ld && q == 0) xM = src[x2_at<TR>(M, cs)];
  float2 xc[B];
  x2_mirror_pairs<M>(x, xM, q, xc);
  float2 u[B];
  const int qq = q < A ? q : 0;  // idle lanes compute on a valid twiddle index and store nothing
#pragma unroll
  for (int k2 = 0; k2 < B; ++k2) {
    const int k = qq + A * k2;
    const float2 a = x[k2];
    const float2 b = cconj(xc[k2]);
    const float2 e = make_float2(0.5f * (a.x + b.x), 0.5f * (a.y + b.y));
    const float2 o = cmul(make_float2(0.5f * (a.x - b.x), 0.5f * (a.y - b.y)), cconj(twr[k]));
    u[k2] = make_float2(e.x - o.y, e.y + o.x);
  }
  rdft<B, 1, PF>(u);
  __syncthreads();  // the row buffer is free (previous readers are done)
  if (q < A) {
#pragma unroll
    for (int n2 = 0; n2 < B; ++n2) wb[q + A * n2] = n2 == 0 ? u[n2] : cmul(u[n2], cconj(tw[n2 * q]));
  }
  __syncthreads();
  if (l.qb < B) {
#pragma unroll
    for (int k1 = 0; k1 < A; ++k1) out[k1] = rb[k1 + A * l.qb];
    rdft<A, 1, PF>(out);
  }
}

template <int M>
__device__ __forceinline__ void x2_load_twiddles(float2* tw, float2* twr, const float2* twM, const float2* wr) {
  using C = XCfg<M>;
  for (int i = threadIdx.x; i < M; i += C::NT) tw[i] = twM[i];
  for (int i = threadIdx.x; i <= M; i += C::NT) twr[i] = wr[i];
}

// the inverse result z[qb + B n1] (lanes qb < B, register n1) into the LDS rows in natural order
template <int M>
__device__ __forceinline__ void x2_park_inverse(float2* buf, const XLane<M>& l, const float2* z) {
  using C = XCfg<M>;
  __syncthreads();  // every lane has read the rows' exchange values
  if (l.qb < C::B) {
    float2* rb = buf + l.rb * C::RS;
#pragma unroll
    for (int n1 = 0; n1 < C::A; ++n1) rb[l.qb + C::B * n1] = z[n1];
  }
  __syncthreads();
}

// ------------------------------------------------------------------ forward with gather
// work-group `wg` of the transform of one source into one spectrum
template <int M, bool TR>
__device__ __forceinline__ void x2_fwd_body(const Dom& d, const GatherParams& g, float2* __restrict__ S,
                                            const float2* __restrict__ twM, const float2* __restrict__ wr, int wg) {
  using C = XCfg<M>;
  __shared__ float2 buf[TR && C::BUF_TR > C::BUF_FWD ? C::BUF_TR : C::BUF_FWD];
  __shared__ float2 twS[C::TWL_FWD ? M : 1];
  __shared__ float2 twrS[C::TWL_FWD ? M + 1 : 1];
  const float2* tw = C::TWL_FWD ? twS : twM;
  const float2* twr = C::TWL_FWD ? twrS : wr;
  __shared__ int xmap[C::PX];
  __shared__ long long srcRow[C::RW];
  __shared__ size_t dstRow[C::RW];
  if (C::TWL_FWD) x2_load_twiddles<M>(twS, twrS, twM, wr);
  const int nrows = d.P[1] * d.P[2];
  // batched blocks: this work-group's block, its gather origin (output region origin - m) and spectrum
  int org[3] = {g.org[0], g.org[1], g.org[2]};
  if (d.btab) {
    const int b = blockIdx.x / d.wgPerBlock;
    wg -= b * d.wgPerBlock;
    const int* t = d.btab + kBlockTabInts * b;
    for (int k = 0; k < 3; ++k) org[k] = t[k] - d.m[k];
    S += (size_t)b * d.blockStride;
  }
  const int row0 = wg * C::RW;
  const XLane<M> l;
  // rows with source values only: row index -> grid row (-org1 + i % N1, -org2 + i / N1), the kernel's rows around 0
  const bool uniq = g.uniqueRows;
  const int nrowsRun = uniq ? g.N[1] * g.N[2] : nrows;
  // source index of FFT position x of a row: row start (srcRow, -1: no source row) + xmap[x] (-1: outside),
  // else g.value.  Mirror: the volume mirrored at its faces; value: the volume, `value` outside; kernel
  // placement: K[(p + K/2) mod P], 0 beyond K (GATHER_KERNEL, value 0).
  const bool kern = g.mode == GATHER_KERNEL;
  const float fill = kern ? 0.f : g.value;
  for (int x = threadIdx.x; x < C::PX; x += C::NT) {
    int gx;
    if (kern) {
      gx = (x + g.N[0] / 2) % d.P[0];
      if (gx >= g.N[0]) gx = -1;
    } else {
      const int p = org[0] + x;
      gx = g.mode == GATHER_MIRROR ? mirror_index(p, g.N[0]) : ((unsigned)p < (unsigned)g.N[0] ? p : -1);
    }
    xmap[x] = gx;
  }
  if (threadIdx.x < C::RW) {
    int row = row0 + threadIdx.x;
    long long off = -1;
    const bool live = row < nrowsRun;
    if (uniq && live) {
      int y = row % g.N[1], zz = row / g.N[1];
      y += kern ? (y < g.N[1] / 2 ? d.P[1] : 0) - g.N[1] / 2 : -org[1];
      zz += kern ? (zz < g.N[2] / 2 ? d.P[2] : 0) - g.N[2] / 2 : -org[2];
      row = zz * d.P[1] + y;
    }
    if (live) {
      const int y = row % d.P[1], zz = row / d.P[1];
      if (kern) {
        const int jy = (y + g.N[1] / 2) % d.P[1], jz = (zz + g.N[2] / 2) % d.P[2];
        if (jy < g.N[1] && jz < g.N[2]) off = ((long long)jz * g.N[1] + jy) * g.N[0];
      } else {
        int gy = org[1] + y, gz = org[2] + zz;
        if (g.mode == GATHER_MIRROR) {
          gy = mirror_index(gy, g.N[1]);
          gz = mirror_index(gz, g.N[2]);
          off = ((long long)gz * g.N[1] + gy) * g.N[0];
        } else if ((unsigned)gy < (unsigned)g.N[1] && (unsigned)gz < (unsigned)g.N[2]) {
          off = ((long long)gz * g.N[1] + gy) * g.N[0];
        }
      }
    }
    srcRow[threadIdx.x] = off;   // row start in src (>= 0), -1: no source row
    dstRow[threadIdx.x] = live ? x2_row<TR>(d, row) : kNoRow;
  }
  __syncthreads();
  // the first transform step reads its values z[q + B a] = (x[2n], x[2n + 1]) straight from the source
  float2 v[C::A];
  if (l.qb < C::B) {
    const long long off = srcRow[l.rb];
    const float* row = g.src + (off + org[0] + 2 * l.qb);  // the value of position x of an inner register index
    const XSpan<C::B> src{-org[0], g.N[0] - org[0]};
    const bool plain = !kern && !__any(off < 0);
#pragma unroll
    for (int a = 0; a < C::A; ++a) {
      if (plain && src.inside(a)) {
        v[a] = ld_pair(row + 2 * C::B * a);
      } else {
        const int x = 2 * (l.qb + C::B * a);
        const int g0 = xmap[x], g1 = xmap[x + 1];
        v[a].x = off >= 0 && g0 >= 0 ? g.src[off + g0] : fill;
        v[a].y = off >= 0 && g1 >= 0 ? g.src[off + g1] : fill;
      }
    }
  }
  float2 z[C::B];
  x2_forward_regs_half<M>(buf, tw, l, v, z);
  const size_t o = dstRow[l.ra];
  x2_post_store_regs<M, TR, TR>(z, l, twr, TR ? S : S + (o == kNoRow ? 0 : o), o != kNoRow, buf, dstRow,
                            (unsigned)(d.P[1] * d.P[2]));
}

template <int M, bool TR>
__global__ __launch_bounds__(XCfg<M>::NT) void k_x2_fwd(Dom d, GatherParams g, float2* __restrict__ S,
                                                         const float2* __restrict__ twM,
                                                         const float2* __restrict__ wr) {
  x2_fwd_body<M, TR>(d, g, S, twM, wr, blockIdx.x);
}

// two groups of sources (n1 work-groups for the first), wgEntry work-groups per source of a group
template <int M>
__global__ __launch_bounds__(XCfg<M>::NT) void k_x2_fwd_groups(Dom d, XFwdGroup g1, XFwdGroup g2, unsigned n1,
                                                                unsigned wgEntry1, unsigned wgEntry2,
                                                                const float2* __restrict__ twM,
                                                                const float2* __restrict__ wr) {
  const bool second = blockIdx.x >= n1;
  const XFwdGroup& u = second ? g2 : g1;
  const unsigned id = second ? blockIdx.x - n1 : blockIdx.x, per = second ? wgEntry2 : wgEntry1;
  const unsigned b = id / per;
  GatherParams g = u.g;
  g.src += b * u.srcStride;
  x2_fwd_body<M, true>(d, g, u.S + b * u.dstStride, twM, wr, (int)(id - b * per));
}

// ------------------------------------------------------------------ inverse, quotient, forward
// ratio = img > 0 ? img / blurred : 1 on the quotient region, 1 elsewhere
// (DeconvolutionMethods.computeQuotient, D/iteration/sequential/DeconvolutionMethods.java:46-98)
template <int M, bool TR>
__global__ __launch_bounds__(XCfg<M>::NT, XCfg<M>::MINW_RATIO) void k_x2_ratio(
    const float2* __restrict__ Sin, float2* __restrict__ Sout, const float2* __restrict__ twM,
    const float2* __restrict__ wr, Dom d, RatioPass q_, ViewOffsets views) {
  using C = XCfg<M>;
  __shared__ float2 buf[C::BUF];
  __shared__ float2 twS[C::TWL_RATIO ? M : 1];
  __shared__ float2 twrS[C::TWL_RATIO ? M + 1 : 1];
  const float2* tw = C::TWL_RATIO ? twS : twM;
  const float2* twr = C::TWL_RATIO ? twrS : wr;
  // img index of FFT position x is imgRow + x (may be negative: x starts at m0); kOuterRow: ratio row of ones
  __shared__ long long imgRow[C::RW];
  __shared__ size_t outOff[C::RW];   // spectrum row (read and written; kNoRow: beyond the grid)
  if (C::TWL_RATIO) x2_load_twiddles<M>(twS, twrS, twM, wr);
  const int nrows = d.P[1] * d.P[2];
  // batched blocks: this work-group's block, its output region and spectra
  int wg = blockIdx.x;
  int o[3] = {q_.o[0], q_.o[1], q_.o[2]}, D[3] = {d.D[0], d.D[1], d.D[2]};
  if (d.btab) {
    const int b = blockIdx.x / d.wgPerBlock;
    wg -= b * d.wgPerBlock;
    const int* t = d.btab + kBlockTabInts * b;
    for (int k = 0; k < 3; ++k) { o[k] = t[k]; D[k] = t[3 + k]; }
    Sin += (size_t)b * d.blockStride;
    Sout += (size_t)b * d.blockStride;
  }
  const float* img = q_.img;
  if (views.n > 1) {  // batched views: this work-group's spectrum and image
    const int b = wg / d.wgPerBlock;
    wg -= b * d.wgPerBlock;
    img += views.at[b];
    Sin += (size_t)b * d.blockStride;
    Sout += (size_t)b * d.blockStride;
  }
  const int row0 = wg * C::RW;
  if (threadIdx.x < C::RW) {
    // skipOnes: the work-groups cover the quotient rows only, index i -> grid row (rowLo1 + i % rowN1,
    // rowLo2 + i / rowN1)
    int row = row0 + threadIdx.x;
    int lo1 = q_.rowLo[1], n1 = q_.rowN[1], lo2 = q_.rowLo[2], n2 = q_.rowN[2];
    if (q_.skipOnes && d.btab) {  // this block's quotient rows
      lo1 = d.m[1] + max(-q_.qlo[1], -o[1]);
      n1 = d.m[1] + min(D[1] + q_.qhi[1], q_.N[1] - o[1]) - lo1;
      lo2 = d.m[2] + max(-q_.qlo[2], -o[2]);
      n2 = d.m[2] + min(D[2] + q_.qhi[2], q_.N[2] - o[2]) - lo2;
    }
    const bool live = row < (q_.skipOnes ? n1 * n2 : nrows);
    if (q_.skipOnes && live) row = (lo2 + row / n1) * d.P[1] + lo1 + row % n1;
    long long ir = kOuterRow;
    if (live) {
      // quotient rows: the output region widened by qlo / qhi, inside the volume
      const int ly = row % d.P[1] - d.m[1], lz = row / d.P[1] - d.m[2];
      if (ly >= -q_.qlo[1] && ly < D[1] + q_.qhi[1] && lz >= -q_.qlo[2] && lz < D[2] + q_.qhi[2] &&
          (unsigned)(o[1] + ly) < (unsigned)q_.N[1] && (unsigned)(o[2] + lz) < (unsigned)q_.N[2])
        ir = ((long long)(o[2] + lz) * q_.N[1] + (o[1] + ly)) * q_.N[0] + o[0] - d.m[0];
    }
    imgRow[threadIdx.x] = ir;
    outOff[threadIdx.x] = live ? x2_row<TR>(d, row) : kNoRow;
  }
  __syncthreads();
  const XLane<M> l;
  const bool rowOnes = imgRow[l.ra] == kOuterRow;
  const size_t so = outOff[l.ra];
  // FFT positions x of the row whose image value is read: the quotient region, inside the volume
  const int x0f = d.m[0] + max(-q_.qlo[0], -o[0]), x1f = d.m[0] + min(D[0] + q_.qhi[0], q_.N[0] - o[0]);
  // rows outside the quotient region are a row of ones after the quotient: their blurred values are not read
  float2 z[C::A];
  const unsigned cs = (unsigned)(d.P[1] * d.P[2]);
  x2_inverse_half_regs<M, TR>(!rowOnes ? Sin + so : nullptr, buf, tw, twr, l, z, cs);
  // park the blurred rows in LDS, form the quotient there with TQ lanes per row, all of a lane's image values in flight
  // at once at offsets from the lane's row pointers known at compile time, and run the forward transform from LDS.
  // Positions x = q + TQ i, or on long rows pairs (at M = 432 16 % faster than the quotient on the B side's registers, 1-27 % at the other lengths above;
  // at M = 150 and 225 pairs are 3-5 % slower, a flat mapping over the work-group 4 %, a wave walking its rows 9 %)
  x2_park_inverse<M>(buf, l, z);
  const int r = (int)threadIdx.x / C::TQ, q = (int)threadIdx.x % C::TQ;
  if (C::RW * C::TQ == C::NT || r < C::RW) {
    const long long ir = imgRow[r];
    const bool rowIn = ir != kOuterRow;
    const float* imr = img + (rowIn ? ir : 0);  // image value of FFT position x: imr[x], x in [x0f, x1f)
    if constexpr (!C::long_rows) {
      float* fr = reinterpret_cast<float*>(buf + r * C::RS);
      constexpr int NI = (C::PX + C::TQ - 1) / C::TQ;
      float im[NI];
#pragma unroll
      for (int i = 0; i < NI; ++i) {
        const int x = q + C::TQ * i;
        im[i] = rowIn && x >= x0f && x < x1f ? imr[x] : 0.f;
      }
#pragma unroll
      for (int i = 0; i < NI; ++i) {
        const int x = q + C::TQ * i;
        if (x < C::PX) fr[x] = im[i] > 0.f ? im[i] / fr[x] : 1.f;
      }
    } else {
      float2* fr = buf + r * C::RS + q;
      if (rowIn) imr += 2 * q;
      constexpr int NI = (M + C::TQ - 1) / C::TQ;
      const XSpan<C::TQ> quot{x0f, x1f};
      const bool plain = __all(rowIn);
      float2 im[NI];
#pragma unroll
      for (int i = 0; i < NI; ++i) {
        const int x = 2 * (q + C::TQ * i);
        im[i] = make_float2(0.f, 0.f);
        if (quot.outside(i)) continue;
        if (plain && quot.inside(i)) {
          im[i] = ld_pair(imr + 2 * C::TQ * i);
        } else if (rowIn) {
          if (x >= x0f && x < x1f) im[i].x = imr[2 * C::TQ * i];
          if (x + 1 >= x0f && x + 1 < x1f) im[i].y = imr[2 * C::TQ * i + 1];
        }
      }
#pragma unroll
      for (int i = 0; i < NI; ++i) {
        if (C::TQ * (i + 1) > M && q + C::TQ * i >= M) continue;
        float2 f = make_float2(1.f, 1.f);
        if (!quot.outside(i)) {
          const float2 b = fr[C::TQ * i];
          f.x = im[i].x > 0.f ? im[i].x / b.x : 1.f;
          f.y = im[i].y > 0.f ? im[i].y / b.y : 1.f;
        }
        fr[C::TQ * i] = f;
      }
    }
  }
  __syncthreads();
  float2 zf[C::B];
  x2_forward<M>(buf, tw, l, zf);
  x2_post_store_regs<M, TR, false>(zf, l, twr, Sout + (so == kNoRow ? 0 : so),
                                   so != kNoRow && !(q_.skipOnes && rowOnes), buf, outOff, cs);
}

// ------------------------------------------------------------------ inverse + psi update (output rows only)
template <int M, bool TR>
__global__ __launch_bounds__(XCfg<M>::NT, XCfg<M>::MINW_UPDATE) void k_x2_update(Dom d, UpdateParams u, FastDiv divPairs,
                                                            const float2* __restrict__ S,
                                                            const float2* __restrict__ twM,
                                                            const float2* __restrict__ wr) {
  using C = XCfg<M>;
  __shared__ float2 buf[C::BUF];
  __shared__ float2 twS[C::TWL ? M : 1];
  __shared__ float2 twrS[C::TWL ? M + 1 : 1];
  const float2* tw = C::TWL ? twS : twM;
  const float2* twr = C::TWL ? twrS : wr;
  __shared__ long long psiRow[C::RW];
  __shared__ size_t rowOff[C::RW];
  if (C::TWL) x2_load_twiddles<M>(twS, twrS, twM, wr);
  // batched blocks: this work-group's block, its output region and spectrum
  int wg = blockIdx.x;
  int o[3] = {u.o[0], u.o[1], u.o[2]}, D[3] = {d.D[0], d.D[1], d.D[2]};
  if (d.btab) {
    const int b = blockIdx.x / d.wgPerBlock;
    wg -= b * d.wgPerBlock;
    const int* t = d.btab + kBlockTabInts * b;
    for (int k = 0; k < 3; ++k) { o[k] = t[k]; D[k] = t[3 + k]; }
    S += (size_t)b * d.blockStride;
    if (D[0] != d.D[0]) divPairs = FastDiv((unsigned)(D[0] + 1) / 2);  // a tail block's row length
  }
  const int nrows = D[1] * D[2];
  const int row0 = wg * C::RW;
  if (threadIdx.x < C::RW) {
    const int row = row0 + threadIdx.x;
    long long pr = -1;
    size_t so = kNoRow;
    if (row < nrows) {
      const int ly = row % D[1], lz = row / D[1];
      pr = ((long long)(o[2] + lz) * u.N[1] + (o[1] + ly)) * u.N[0] + o[0];
      so = x2_row<TR>(d, (d.m[2] + lz) * d.P[1] + (d.m[1] + ly));
    }
    psiRow[threadIdx.x] = pr;   // >= 0 for output rows (the output region lies inside the volume)
    rowOff[threadIdx.x] = so;
  }
  __syncthreads();
  const XLane<M> l;
  const size_t so = rowOff[l.ra];
  float2 z[C::A];
  x2_inverse_half_regs<M, TR, C::long_rows>(so != kNoRow ? S + so : nullptr, buf, tw, twr, l, z,
                                            (unsigned)(d.P[1] * d.P[2]));
  double sum = 0.0;
  float mx = -1.f;
  const RLConsts rc = rl_consts(u.lambda, u.minValue, u.maxI);
  const int DX = D[0];
  // park the rows in LDS and update pairs of positions there, U pairs in flight (the last pair of an odd row holds one)
  x2_park_inverse<M>(buf, l, z);
  const float* fb = reinterpret_cast<const float*>(buf) + d.m[0];
  auto one = [&](float last, float integral, float weight) {
    const float next = rl_next_value(last, integral, weight, rc), ch = next - last;
    sum += (double)ch;
    mx = java_maxf(mx, ch);
    return next;
  };
  constexpr int U = 4;
  if constexpr (C::long_rows) {
    // long rows: TQ lanes per row at offsets uniform over the work-group; only a row's last pairs test their positions.
    // At M = 432 778 us for 225 000 rows, 807 with the flat mapping below, 855 on the B side's registers (the other lengths:
    // the head of this file)
    const int r = (int)threadIdx.x / C::TQ, q = (int)threadIdx.x % C::TQ;
    const long long pr = C::RW * C::TQ == C::NT || r < C::RW ? psiRow[r] : -1;
    if (pr >= 0) {
      const float* f = fb + r * 2 * C::RS + 2 * q;
      float* psi = u.psi + (pr + 2 * q);
      const float* w = u.w + (pr + 2 * q);
      for (int i0 = 0; 2 * C::TQ * i0 < DX; i0 += U) {
        float2 last[U], wt[U];
#pragma unroll
        for (int j = 0; j < U; ++j) {
          const int at = 2 * C::TQ * (i0 + j), lx = at + 2 * q;
          last[j] = wt[j] = make_float2(0.f, 0.f);
          if (at + 2 * C::TQ <= DX) {
            last[j] = ld_pair(psi + at);
            wt[j] = ld_pair(w + at);
          } else {
            if (lx < DX) { last[j].x = psi[at]; wt[j].x = w[at]; }
            if (lx + 1 < DX) { last[j].y = psi[at + 1]; wt[j].y = w[at + 1]; }
          }
        }
#pragma unroll
        for (int j = 0; j < U; ++j) {
          const int at = 2 * C::TQ * (i0 + j), lx = at + 2 * q;
          if (lx >= DX) continue;
          float2 next;
          next.x = one(last[j].x, f[at], wt[j].x);
          if (lx + 1 < DX) {
            next.y = one(last[j].y, f[at + 1], wt[j].y);
            st_pair(psi + at, next);
          } else {
            psi[at] = next.x;
          }
        }
      }
    }
  } else {
    // short rows: a flat mapping of the pairs over every thread (at M = 150 35 % faster than on the B side's registers,
    // 12 % faster than TQ lanes per row, 12-37 % than a wave walking its rows)
    const unsigned perRow = divPairs.d, total = (unsigned)C::RW * perRow;
    auto update_rows = [&](auto odd) {
      for (unsigned base = threadIdx.x; base < total; base += U * C::NT) {
        float2 last[U], wt[U];
        size_t gi[U];
        unsigned at[U];  // the pair's first value in the rows
        bool ok[U], two[U];
#pragma unroll
        for (int j = 0; j < U; ++j) {
          const unsigned e = base + j * C::NT, r = min(divPairs.div(e), (unsigned)C::RW - 1);
          const unsigned lx = 2 * (e - r * perRow);
          const long long pr = psiRow[r];
          ok[j] = e < total && pr >= 0;
          two[j] = !odd || (ok[j] && (int)lx + 1 < DX);
          gi[j] = ok[j] ? (size_t)(pr + lx) : 0;
          at[j] = r * 2 * C::RS + lx;
          if (two[j]) {
            last[j] = ld_pair(u.psi + gi[j]);
            wt[j] = ld_pair(u.w + gi[j]);
          } else {
            last[j] = make_float2(u.psi[gi[j]], 0.f);
            wt[j] = make_float2(u.w[gi[j]], 0.f);
          }
        }
#pragma unroll
        for (int j = 0; j < U; ++j) {
          if (!ok[j]) continue;
          const float* f = fb + at[j];
          const float2 next = make_float2(rl_next_value(last[j].x, f[0], wt[j].x, rc),
                                          two[j] ? rl_next_value(last[j].y, f[1], wt[j].y, rc) : 0.f);
          const float c0 = next.x - last[j].x, c1 = next.y - last[j].y;
          sum += (double)c0;
          mx = java_maxf(mx, c0);
          if (two[j]) {
            st_pair(u.psi + gi[j], next);
            sum += (double)c1;
            mx = java_maxf(mx, c1);
          } else {
            u.psi[gi[j]] = next.x;
          }
        }
      }
    };
    if (DX & 1)
      update_rows(std::true_type{});
    else
      update_rows(std::false_type{});
  }
  // the stats reduction reuses the row buffer once every thread has read its rows
  static_assert(C::BUF * sizeof(float2) >= 2 * reduce_width<C::NT>() * sizeof(double),
                "the row buffer holds the reduction");
  __syncthreads();
  double* red = reinterpret_cast<double*>(buf);
  block_reduce_stats_nt<C::NT>(sum, mx, u.partial + blockIdx.x, red, red + reduce_width<C::NT>());
}

// ------------------------------------------------------------------ inverse + store of the output region
template <int M, bool TR>
__global__ __launch_bounds__(XCfg<M>::NT) void k_x2_store(Dom d, StoreParams st, const float2* __restrict__ S,
                                                           const float2* __restrict__ twM,
                                                           const float2* __restrict__ wr) {
  using C = XCfg<M>;
  __shared__ float2 buf[C::BUF];
  __shared__ float2 twS[C::TWL ? M : 1];
  __shared__ float2 twrS[C::TWL ? M + 1 : 1];
  const float2* tw = C::TWL ? twS : twM;
  const float2* twr = C::TWL ? twrS : wr;
  __shared__ size_t rowOff[C::RW];
  if (C::TWL) x2_load_twiddles<M>(twS, twrS, twM, wr);
  const int nrows = d.D[1] * d.D[2];
  unsigned wg = blockIdx.x;
  if (st.n > 1) {  // this work-group's spectrum and output array
    const unsigned b = wg / d.wgPerBlock;
    wg -= b * d.wgPerBlock;
    S += b * d.blockStride;
    st.out += (size_t)b * d.D[0] * nrows;
  }
  const int row0 = wg * C::RW;
  if (threadIdx.x < C::RW) {
    const int row = row0 + threadIdx.x;
    size_t so = kNoRow;
    if (row < nrows) {
      const int ly = row % d.D[1], lz = row / d.D[1];
      so = x2_row<TR>(d, (d.m[2] + lz) * d.P[1] + (d.m[1] + ly));
    }
    rowOff[threadIdx.x] = so;
  }
  __syncthreads();
  const XLane<M> l;
  const size_t so = rowOff[l.ra];
  float2 z[C::A];
  x2_inverse_half_regs<M, TR>(so != kNoRow ? S + so : nullptr, buf, tw, twr, l, z, (unsigned)(d.P[1] * d.P[2]));
  const int row = row0 + l.rb, q = l.qb;
  if (q < C::B && row < nrows) {
    const int DX = d.D[0], m0 = d.m[0];
    float* out = st.out + (size_t)row * DX;
    const XSpan<C::B> span{m0, m0 + DX};
#pragma unroll
    for (int a = 0; a < C::A; ++a) {
      const int lx = 2 * (q + C::B * a) - m0;
      if (span.inside(a)) {
        st_pair(out + lx, z[a]);
      } else {
        if (lx >= 0 && lx < DX) out[lx] = z[a].x;
        if (lx + 1 >= 0 && lx + 1 < DX) out[lx + 1] = z[a].y;
      }
    }
  }
}

// ------------------------------------------------------------------ host launchers
// Batched launches (d.btab set) run d.nb blocks of wgPerBlock work-groups each: work-group w serves block
// w / wgPerBlock; rows of a block beyond its own extent are skipped inside the kernels.
template <int M, bool TR>
void launch_x_fwd(const Dom& d, const GatherParams& g, float2* S, const float2* twM, const float2* wr,
                  hipStream_t s) {
  static_assert(x2_ok<M>(), "every compiled x length has a two-step split");
  using C = XCfg<M>;
  Dom dd = d;
  const int rows = g.uniqueRows ? g.N[1] * g.N[2] : d.P[1] * d.P[2];
  dd.wgPerBlock = (rows + C::RW - 1) / C::RW;
  const int nb = d.btab ? d.nb : 1;
  hipLaunchKernelGGL((k_x2_fwd<M, TR>), dim3(dd.wgPerBlock * nb), dim3(C::NT), 0, s, dd, g, S, twM, wr);
}
template <int M>
void launch_x_fwd_groups(const Dom& d, const XFwdGroup* u, int n, const float2* twM, const float2* wr, hipStream_t s) {
  using C = XCfg<M>;
  unsigned per[2] = {1, 1}, wgs[2] = {0, 0};
  for (int i = 0; i < n; ++i) {
    const int rows = u[i].g.uniqueRows ? u[i].g.N[1] * u[i].g.N[2] : d.P[1] * d.P[2];
    per[i] = (unsigned)((rows + C::RW - 1) / C::RW);
    wgs[i] = per[i] * (unsigned)u[i].n;
  }
  hipLaunchKernelGGL(k_x2_fwd_groups<M>, dim3(wgs[0] + wgs[1]), dim3(C::NT), 0, s, d, u[0], u[n - 1], wgs[0], per[0],
                     per[1], twM, wr);
}
template <int M, bool TR>
void launch_x_ratio(const Dom& d, const RatioParams& q, const float2* Sin, float2* Sout, const float2* twM,
                    const float2* wr, hipStream_t s) {
  static_assert(x2_ok<M>(), "every compiled x length has a two-step split");
  using C = XCfg<M>;
  Dom dd = d;
  const int rows = q.skipOnes ? q.rowN[1] * q.rowN[2] : d.P[1] * d.P[2];
  if (rows == 0) return;  // no quotient rows: every row is a row of ones, put in by the z pass
  dd.wgPerBlock = (rows + C::RW - 1) / C::RW;
  const int nb = d.btab ? d.nb : std::max(1, q.views.n);
  hipLaunchKernelGGL((k_x2_ratio<M, TR>), dim3(dd.wgPerBlock * nb), dim3(C::NT), 0, s, Sin, Sout, twM, wr, dd, q, q.views);
}
template <int M, bool TR>
int launch_x_update(const Dom& d, const UpdateParams& u, const float2* S, const float2* twM, const float2* wr,
                    hipStream_t s) {
  static_assert(x2_ok<M>(), "every compiled x length has a two-step split");
  using C = XCfg<M>;
  Dom dd = d;
  const int rows = d.D[1] * d.D[2];
  dd.wgPerBlock = (rows + C::RW - 1) / C::RW;
  const int nwg = dd.wgPerBlock * (d.btab ? d.nb : 1);
  hipLaunchKernelGGL((k_x2_update<M, TR>), dim3(nwg), dim3(C::NT), 0, s, dd, u, FastDiv((unsigned)(d.D[0] + 1) / 2), S,
                     twM, wr);
  return nwg;
}
template <int M, bool TR>
void launch_x_store(const Dom& d, const StoreParams& st, const float2* S, const float2* twM, const float2* wr,
                    hipStream_t s) {
  static_assert(x2_ok<M>(), "every compiled x length has a two-step split");
  using C = XCfg<M>;
  Dom dd = d;
  const int rows = d.D[1] * d.D[2];
  dd.wgPerBlock = (rows + C::RW - 1) / C::RW;
  hipLaunchKernelGGL((k_x2_store<M, TR>), dim3(dd.wgPerBlock * st.n), dim3(C::NT), 0, s, dd, st, S, twM, wr);
}

}  // namespace mvr
