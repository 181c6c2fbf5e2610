// plane.hip -- the y and z transforms of a small FFT grid in one pass.
//
// For one x frequency, the y-z plane of a grid of up to 128 x 128 fits the LDS of a CU (131 KB at most), so the
// convolution's z transform, y transform, spectrum product and the two inverse transforms, three passes over the
// spectrum on larger grids, are one: a work-group loads a plane, transforms it in place, and stores the rows the next
// x pass reads.  The spectra of such plans are planar, [hx][z][y]: a work-group's plane is contiguous.
//
// The transforms are those of the strided passes: two register steps per pencil, L = A x B, in place.  Step 1 of the
// forward transform takes positions b + B a and leaves the values of k1 at b + B k1; step 2 takes the B consecutive
// positions of a k1 and leaves X[k1 + A k2] at B k1 + k2.  That slot order is kept through the spectrum product (the
// kernel spectrum is stored in it, [hx][y slot][z slot]) and undone by the inverse steps.  Rows of the plane are
// padded by one value, so that both directions' accesses (lanes along y or along z) are free of bank conflicts.
//
// Bound by the LDS round trips (eleven over a plane) and, at one plane per CU, by their latency: an 80 x 72 plane takes
// 12 us on its CU, of which its VALU work is 5.  A 48 x 40 x 33 convolution with its kernel: 43.6 us with three strided
// passes per transform and direction, 35.0 with this one, 17.3 with the kernel's plane transformed beside the data's.
// Two views of 64 x 60 x 52, 5 iterations: 533 -> 492 us; 24 batched blocks on 120-point grids, 340 MB: 141 -> 80 us per
// convolution.  One cubic grid at a time gains 2-12 % up to 96 points and loses 2-3 % at 120 and 128 (kPlaneMaxSingle,
// where grids short along x are listed too); 128 is what the LDS holds.
#include <type_traits>

#include "passes.hpp"

namespace mvr {

namespace {

// lengths with compiled plane transforms: f(integral_constant<L>)
template <typename F>
__device__ __forceinline__ void with_length(int L, F f) {
  switch (L) {
#define MVR_LEN(N) case N: f(std::integral_constant<int, N>{}); break;
    MVR_LEN(16) MVR_LEN(20) MVR_LEN(24) MVR_LEN(32) MVR_LEN(40) MVR_LEN(48) MVR_LEN(60) MVR_LEN(64) MVR_LEN(72)
    MVR_LEN(80) MVR_LEN(96) MVR_LEN(100) MVR_LEN(120) MVR_LEN(128)
#undef MVR_LEN
  }
}

// task t of `n` pencils: t = j n + pencil, lanes along the pencils (exact for t < 2^16; m from the host)
struct PencilDiv {
  unsigned n, m;
  __device__ __forceinline__ unsigned div(unsigned t) const { return n == 1 ? t : __umulhi(t, m); }
};
// the divisors of a launch: pencils along z (Py of them), along y (Pz), and the stored columns y
struct PlaneDivs {
  PencilDiv y, z, s;
};

// The steps on pencils of LDS: element i of pencil p at base + p * ps + i * es; all pencils [p0, p0 + n) of the plane, and
// (second > 0) of another one `second` values behind it.
template <int L, int DIR, bool FIRST, int NT>
__device__ __forceinline__ void plane_step(float2* base, int p0, PencilDiv d, int ps, int es, const float2* tw,
                                           int second = 0) {
  constexpr int A = split2(L).A, B = split2(L).B;
  // FIRST forward and second inverse: A-point transforms over positions j + B i; the others: B-point ones over B j + i
  constexpr bool OUTER = FIRST == (DIR < 0);
  constexpr int R = OUTER ? A : B, NJ = OUTER ? B : A;
  const int n = (int)d.n;
  const unsigned tasks = (unsigned)(n * NJ);
  for (unsigned k = threadIdx.x; k < (second ? 2 * tasks : tasks); k += NT) {
    const unsigned t = k < tasks ? k : k - tasks;
    const int j = (int)d.div(t);
    float2* x = base + (k < tasks ? 0 : second) + (p0 + (int)t - j * n) * ps + (OUTER ? j : B * j) * es;
    const int st = (OUTER ? B : 1) * es;
    float2 v[R];
#pragma unroll
    for (int i = 0; i < R; ++i) v[i] = x[i * st];
    rdft<R, DIR>(v);
    if constexpr (FIRST) {
#pragma unroll
      for (int i = 1; i < R; ++i) v[i] = cmul(v[i], DIR < 0 ? tw[j * i] : cconj(tw[j * i]));
    }
#pragma unroll
    for (int i = 0; i < R; ++i) x[i * st] = v[i];
  }
}

// PAIR: the kernel's and the data's plane lie side by side in the LDS and are transformed together, with half the barriers
// and twice the tasks for a step's threads, and the kernel's spectrum is not written: a convolution on device memory takes
// 12 in place of 14.5 us on a 16-point grid, 17.3 of 20.6 on 64 x 48 x 48 and 27 of 31 on 96 points, as far as two
// planes fit.  Otherwise the kernel's plane goes first.
template <int NT, int CAP, bool PAIR>
__global__ __launch_bounds__(NT) void k_plane(PlaneGeom g, PlaneDivs dv, const float2* in, float2* out,
                                              const float2* spec, const float2* __restrict__ twY,
                                              const float2* __restrict__ twZ) {
  __shared__ float2 lds[CAP];
  const int Py = g.Py, Pz = g.Pz, rp = Py + 1;
  float2* tile = lds;                  // [z][y], rows of Py + 1
  float2* ty = lds + (size_t)(PAIR ? 2 : 1) * Pz * rp;  // twiddles
  float2* tz = ty + Py;
  // work-group -> (plane, batch entry), batch entries of a plane next to one another on one XCD (they share its spectrum)
  unsigned id = blockIdx.x;
  if (gridDim.x % 8 == 0) id = (id % 8) * (gridDim.x / 8) + id / 8;
  const int hx = (int)(id / g.nb), b = (int)(id % g.nb);
  const size_t plane = (size_t)hx * Py * Pz;
  for (int i = threadIdx.x; i < Py; i += NT) ty[i] = twY[i];
  for (int i = threadIdx.x; i < Pz; i += NT) tz[i] = twZ[i];
  __syncthreads();
  const int second = PAIR ? Pz * rp : 0;
  const float2* ksrc = g.kin + b * g.kStride + plane;
  const float2* dsrc = in + (g.inIdx ? g.inIdx[b] : b) * g.inStride + plane;
  // values that were not written: zeros beyond the kernel's rows (1), constant rows (2), mirror copies (3), which are read
  // at their source
  const int dfill = g.ones ? 2 : g.mirN[0] > 0 ? 3 : 0;
  const float2 one = make_float2(hx == 0 ? g.onesDC : 0.f, 0.f);
  int lo0 = g.onesLo[0], hi0 = g.onesHi[0], lo1 = g.onesLo[1], hi1 = g.onesHi[1];
  if (g.ones && g.onesTab) {
    const int* t = g.onesTab + 4 * b;
    lo0 = t[0]; hi0 = t[1]; lo1 = t[2]; hi1 = t[3];
  }
  // pass 0: the kernel's plane, 1: the data's (PAIR: both in pass 1)
  for (int pass = !PAIR && g.kin ? 0 : 1; pass < (in ? 2 : 1); ++pass) {
    with_length(Pz, [&](auto len) {
      constexpr int L = decltype(len)::value, A = split2(L).A, B = split2(L).B;
      const unsigned tasks = (unsigned)(Py * B);
      for (unsigned k = threadIdx.x; k < (PAIR ? 2 * tasks : tasks); k += NT) {
        const bool kern = PAIR ? k >= tasks : pass == 0;
        const unsigned t = PAIR && kern ? k - tasks : k;
        const int fill = kern ? 1 : dfill;
        const float2* src = kern ? ksrc : dsrc;
        const int j = (int)dv.y.div(t), y = (int)t - j * Py;
        float2 v[A];
        if (fill == 2) {
          const bool yin = y >= lo0 && y < hi0;
#pragma unroll
          for (int a = 0; a < A; ++a) {
            const int z = j + B * a;
            v[a] = yin && z >= lo1 && z < hi1 ? src[z * Py + y] : one;
          }
        } else if (fill == 3) {
          const int yy = g.mir[0] + mirror_index(y - g.mir[0], g.mirN[0]);
#pragma unroll
          for (int a = 0; a < A; ++a) v[a] = src[(g.mir[1] + mirror_index(j + B * a - g.mir[1], g.mirN[1])) * Py + yy];
        } else if (fill == 1) {
          int yk = y + g.kK[0] / 2;
          yk -= yk >= Py ? Py : 0;
#pragma unroll
          for (int a = 0; a < A; ++a) {
            int zk = j + B * a + g.kK[1] / 2;
            zk -= zk >= Pz ? Pz : 0;
            v[a] = yk < g.kK[0] && zk < g.kK[1] ? src[(j + B * a) * Py + y] : make_float2(0.f, 0.f);
          }
        } else {
#pragma unroll
          for (int a = 0; a < A; ++a) v[a] = src[(j + B * a) * Py + y];
        }
        rdft<A, -1>(v);
#pragma unroll
        for (int i = 1; i < A; ++i) v[i] = cmul(v[i], tz[j * i]);
        float2* to = tile + (PAIR && kern ? second : 0) + y;
#pragma unroll
        for (int i = 0; i < A; ++i) to[(j + B * i) * rp] = v[i];
      }
    });
    __syncthreads();
    with_length(Pz, [&](auto len) { plane_step<decltype(len)::value, -1, false, NT>(tile, 0, dv.y, 1, rp, tz, second); });
    __syncthreads();
    with_length(Py, [&](auto len) { plane_step<decltype(len)::value, -1, true, NT>(tile, 0, dv.z, rp, 1, ty, second); });
    __syncthreads();
    if (pass == 1) break;
    // the scaled kernel spectrum in slot order
    float2* so = g.specOut + b * g.kStride + plane;
    with_length(Py, [&](auto len) {
      constexpr int L = decltype(len)::value, A = split2(L).A, B = split2(L).B;
      for (unsigned t = threadIdx.x; t < (unsigned)(Pz * A); t += NT) {
        const int j = (int)dv.z.div(t), z = (int)t - j * Pz;
        float2 v[B];
#pragma unroll
        for (int i = 0; i < B; ++i) v[i] = tile[z * rp + B * j + i];
        rdft<B, -1>(v);
#pragma unroll
        for (int i = 0; i < B; ++i) so[(B * j + i) * Pz + z] = cscale(v[i], g.kScale);
      }
    });
    __syncthreads();  // the tile is free; each thread reads back below only what it has written itself
  }
  if (!in) return;
  float2* dst = out + (size_t)b * g.outStride + plane;
  const float2* sp = g.kin ? g.specOut + b * g.kStride + plane
                           : spec + (g.views.n ? g.views.at[b] : (long long)((g.specIdx ? g.specIdx[b] : 0) * g.specStride)) + plane;
  with_length(Py, [&](auto len) {
    constexpr int L = decltype(len)::value, A = split2(L).A, B = split2(L).B;
    for (unsigned t = threadIdx.x; t < (unsigned)(Pz * A); t += NT) {
      const int j = (int)dv.z.div(t), z = (int)t - j * Pz;
      float2 kv[B], v[B];
      if constexpr (PAIR) {
#pragma unroll
        for (int i = 0; i < B; ++i) kv[i] = tile[second + z * rp + B * j + i];
        rdft<B, -1>(kv);
#pragma unroll
        for (int i = 0; i < B; ++i) kv[i] = cscale(kv[i], g.kScale);
      } else {
#pragma unroll
        for (int i = 0; i < B; ++i) kv[i] = sp[(B * j + i) * Pz + z];
      }
#pragma unroll
      for (int i = 0; i < B; ++i) v[i] = tile[z * rp + B * j + i];
      rdft<B, -1>(v);
#pragma unroll
      for (int i = 0; i < B; ++i) v[i] = cmul(v[i], kv[i]);
      rdft<B, 1>(v);
#pragma unroll
      for (int i = 0; i < B; ++i) tile[z * rp + B * j + i] = i == 0 ? v[i] : cmul(v[i], cconj(ty[j * i]));
    }
  });
  __syncthreads();
  with_length(Py, [&](auto len) { plane_step<decltype(len)::value, 1, false, NT>(tile, 0, dv.z, rp, 1, ty); });
  __syncthreads();
  // z inverse of the columns y the next pass reads, rows z stored
  const int y0 = g.lo[0], ny = g.hi[0] - g.lo[0];
  if (ny <= 0) return;
  with_length(Pz, [&](auto len) { plane_step<decltype(len)::value, 1, true, NT>(tile, y0, dv.s, 1, rp, tz); });
  __syncthreads();
  with_length(Pz, [&](auto len) {
    constexpr int L = decltype(len)::value, A = split2(L).A, B = split2(L).B;
    for (unsigned t = threadIdx.x; t < (unsigned)(ny * B); t += NT) {
      const int j = (int)dv.s.div(t), y = y0 + (int)t - j * ny;
      float2 v[A];
#pragma unroll
      for (int i = 0; i < A; ++i) v[i] = tile[(j + B * i) * rp + y];
      rdft<A, 1>(v);
#pragma unroll
      for (int i = 0; i < A; ++i) {
        const int z = j + B * i;
        if (z >= g.lo[1] && z < g.hi[1]) dst[z * Py + y] = v[i];
      }
    }
  });
}

PencilDiv pencils(int n) { return {(unsigned)n, n > 0 ? 0xffffffffu / (unsigned)n + 1 : 0}; }

// complex values of LDS for p x p planes
constexpr int cap(int p, int planes = 1) { return planes * p * (p + 1) + 2 * p; }

}  // namespace

template <int NT, int CAP, bool PAIR = false>
static void launch(const PlaneGeom& g, const float2* in, float2* out, const float2* spec, const float2* twY,
                   const float2* twZ, hipStream_t s) {
  const dim3 grid((unsigned)(g.ncols * g.nb));
  const PlaneDivs dv{pencils(g.Py), pencils(g.Pz), pencils(g.hi[0] - g.lo[0])};
  if (g.evStart)  // timed: the events hold the kernel's own start and stop
    hipExtLaunchKernelGGL((k_plane<NT, CAP, PAIR>), grid, dim3(NT), 0, s, g.evStart, g.evStop, 0u, g, dv, in, out, spec, twY, twZ);
  else
    hipLaunchKernelGGL((k_plane<NT, CAP, PAIR>), grid, dim3(NT), 0, s, g, dv, in, out, spec, twY, twZ);
}

void launch_plane(const PlaneGeom& g, const float2* in, float2* out, const float2* spec,
                  const float2* twY, const float2* twZ, hipStream_t s) {
  const int need = g.Pz * (g.Py + 1) + g.Py + g.Pz;
  if (g.kin && !g.specOut) {  // plane_pairs
    if (need + g.Pz * (g.Py + 1) <= cap(64, 2))
      launch<1024, cap(64, 2), true>(g, in, out, spec, twY, twZ, s);
    else
      launch<1024, cap(kPlanePairMax, 2), true>(g, in, out, spec, twY, twZ, s);
    return;
  }
  if (need <= cap(64))
    launch<512, cap(64)>(g, in, out, spec, twY, twZ, s);
  else if (need <= cap(96))
    launch<1024, cap(96)>(g, in, out, spec, twY, twZ, s);
  else
    launch<1024, cap(128)>(g, in, out, spec, twY, twZ, s);
}

}  // namespace mvr
