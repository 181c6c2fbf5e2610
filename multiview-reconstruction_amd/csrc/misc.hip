// misc.hip -- pointwise and reduction kernels of the deconvolution engine.
#include "passes.hpp"

namespace mvr {

__global__ void k_fill(float* __restrict__ dst, size_t n, float v) {
  for (size_t i = (size_t)blockIdx.x * blockDim.x + threadIdx.x; i < n; i += (size_t)gridDim.x * blockDim.x) dst[i] = v;
}

void launch_fill(float* dst, size_t n, float v, hipStream_t s) {
  const int nb = (int)std::min<size_t>((n + kThreads - 1) / kThreads, 4096);
  hipLaunchKernelGGL(k_fill, dim3(nb > 0 ? nb : 1), dim3(kThreads), 0, s, dst, n, v);
}

// Deterministic final reduction of per-work-group {sum, max} partials
// (IterationStatistics accumulation, ComputeBlockSeqThreadCPU.java:159-166).
__global__ void k_reduce_stats(const double2* __restrict__ partial, int n, double2* __restrict__ out) {
  __shared__ double ss[kThreads], sm[kThreads];
  double s = 0.0, m = -1.0;
  for (int i = threadIdx.x; i < n; i += kThreads) { s += partial[i].x; m = java_max(m, partial[i].y); }
  ss[threadIdx.x] = s;
  sm[threadIdx.x] = m;
  __syncthreads();
  for (int off = kThreads / 2; off > 0; off >>= 1) {
    if (threadIdx.x < off) {
      ss[threadIdx.x] += ss[threadIdx.x + off];
      sm[threadIdx.x] = java_max(sm[threadIdx.x], sm[threadIdx.x + off]);
    }
    __syncthreads();
  }
  if (threadIdx.x == 0) *out = make_double2(ss[0], sm[0]);
}

void launch_reduce_stats(const double2* partial, int n, double2* out, hipStream_t s) {
  hipLaunchKernelGGL(k_reduce_stats, dim3(1), dim3(kThreads), 0, s, partial, n, out);
}

// The same reduction for up to 32 view updates at once (work-group v: partials [v * stride, v * stride + n[v]),
// result out[v]): one launch per iteration instead of one per view update.
struct PartialCounts { int n[32]; };
__global__ void k_reduce_stats_batched(const double2* __restrict__ partial, size_t stride, PartialCounts c,
                                       double2* __restrict__ out) {
  __shared__ double ss[kThreads], sm[kThreads];
  const double2* p = partial + (size_t)blockIdx.x * stride;
  const int n = c.n[blockIdx.x];
  double s = 0.0, m = -1.0;
  for (int i = threadIdx.x; i < n; i += kThreads) { s += p[i].x; m = java_max(m, p[i].y); }
  ss[threadIdx.x] = s;
  sm[threadIdx.x] = m;
  __syncthreads();
  for (int off = kThreads / 2; off > 0; off >>= 1) {
    if (threadIdx.x < off) {
      ss[threadIdx.x] += ss[threadIdx.x + off];
      sm[threadIdx.x] = java_max(sm[threadIdx.x], sm[threadIdx.x + off]);
    }
    __syncthreads();
  }
  if (threadIdx.x == 0) out[blockIdx.x] = make_double2(ss[0], sm[0]);
}

void launch_reduce_stats_batched(const double2* partial, size_t stride, const int* counts, int nUpdates, double2* out,
                                 hipStream_t s) {
  PartialCounts c{};
  for (int v = 0; v < nUpdates && v < 32; ++v) c.n[v] = counts[v];
  hipLaunchKernelGGL(k_reduce_stats_batched, dim3(nUpdates), dim3(kThreads), 0, s, partial, stride, c, out);
}

// Divided as the host normalises, (float)((double)x / sum), and mirrored as the host mirrors: an even axis leaves its middle
// pair in place (Mirror.mirror, D/util/Mirror.java:55-132).
__device__ __forceinline__ int psf_mirror(int i, int n) {
  return n % 2 == 0 && (i == n / 2 || i == n / 2 - 1) ? i : n - 1 - i;
}
__global__ __launch_bounds__(kThreads) void k_psf_kernels(const float* __restrict__ given, const double* __restrict__ sums,
                                                          int V, int3 K, float* __restrict__ out) {
  const size_t nk = (size_t)K.x * K.y * K.z, i = (size_t)blockIdx.x * kThreads + threadIdx.x, v = blockIdx.y;
  if (i >= nk) return;
  const int x = (int)(i % K.x), y = (int)(i / K.x % K.y), z = (int)(i / K.x / K.y);
  const size_t m = ((size_t)psf_mirror(z, K.z) * K.y + psf_mirror(y, K.y)) * K.x + psf_mirror(x, K.x);
  const float a = given[v * nk + i], b = given[v * nk + m];
  const double sum = sums[v];
  out[(V - 1 + v) * nk + i] = (float)((double)a / sum);
  out[(2 * V - 1 + v) * nk + i] = (float)((double)b / sum);
  if (v > 0) {
    out[(v - 1) * nk + i] = a;
    out[(3 * V - 2 + v) * nk + i] = b;
  }
}

void launch_psf_kernels(const float* given, const double* sums, int V, const int K[3], float* out, hipStream_t s) {
  const size_t nk = (size_t)K[0] * K[1] * K[2];
  hipLaunchKernelGGL(k_psf_kernels, dim3((unsigned)((nk + kThreads - 1) / kThreads), V), dim3(kThreads), 0, s, given, sums,
                     V, make_int3(K[0], K[1], K[2]), out);
}

__global__ __launch_bounds__(kThreads) void k_psf_products(const float* first, const float* __restrict__ factors, int nf,
                                                           size_t nk, float* out) {
  const size_t i = (size_t)blockIdx.x * kThreads + threadIdx.x, v = blockIdx.y;
  if (i >= nk) return;
  float r = first[v * nk + i];  // first may be out
  for (int j = 0; j < nf; ++j) r = factors[(v * nf + j) * nk + i] * r;
  out[v * nk + i] = r;
}

void launch_psf_products(const float* first, const float* factors, int V, int nf, size_t nk, float* out, hipStream_t s) {
  hipLaunchKernelGGL(k_psf_products, dim3((unsigned)((nk + kThreads - 1) / kThreads), V), dim3(kThreads), 0, s, first,
                     factors, nf, nk, out);
}

// PsiInitAvgPrecise per voxel (D/init/PsiInitAvgPreciseThread.java:127-155): the
// mean of the positive view values is summed (double) over voxels with any
// positive value; max of the positive values per view.  Per-work-group
// partials are reduced on the host in a fixed order.
constexpr int kMaxViews = 32;
struct ViewPtrs { const float* p[kMaxViews]; };

// Bound by HBM: the views' maxima stay in registers (VM views at most, V rounded up) and the values of two voxels are in
// flight at once.  256^3, 6 views: 285 us with the maxima in scratch memory, 175 so (the double division
// per voxel is most of the rest).
template <int VM>
__global__ __launch_bounds__(kThreads) void k_psi_init(ViewPtrs imgs, int V, size_t n, double* __restrict__ psum,
                                                       unsigned long long* __restrict__ pcount,
                                                       float* __restrict__ pmax) {
  __shared__ double ssum[kThreads / 64];
  __shared__ unsigned long long scnt[kThreads / 64];
  __shared__ float smax[kThreads / 64][VM];
  double sum = 0.0;
  unsigned long long cnt = 0;
  float mx[VM];
#pragma unroll
  for (int v = 0; v < VM; ++v) mx[v] = 0.f;
  const size_t stride = (size_t)gridDim.x * kThreads;
  for (size_t i = (size_t)blockIdx.x * kThreads + threadIdx.x; i < n; i += 2 * stride) {
    const bool two = i + stride < n;
    float val[2][VM];
#pragma unroll
    for (int v = 0; v < VM; ++v) {
      if (v >= V) continue;
      val[0][v] = imgs.p[v][i];
      val[1][v] = two ? imgs.p[v][i + stride] : 0.f;
    }
#pragma unroll
    for (int h = 0; h < 2; ++h) {
      double s = 0.0;
      int c = 0;
#pragma unroll
      for (int v = 0; v < VM; ++v) {
        if (v >= V) continue;
        if (val[h][v] > 0.f) { mx[v] = fmaxf(mx[v], val[h][v]); s += (double)val[h][v]; ++c; }
      }
      if (c > 0) { sum += s / (double)c; ++cnt; }
    }
  }
  for (int off = 32; off > 0; off >>= 1) {
    sum += __shfl_down(sum, off);
    cnt += __shfl_down(cnt, off);
#pragma unroll
    for (int v = 0; v < VM; ++v) mx[v] = fmaxf(mx[v], __shfl_down(mx[v], off));
  }
  const int lane = threadIdx.x & 63, wv = threadIdx.x >> 6;
  if (lane == 0) {
    ssum[wv] = sum;
    scnt[wv] = cnt;
#pragma unroll
    for (int v = 0; v < VM; ++v) smax[wv][v] = mx[v];
  }
  __syncthreads();
  if (threadIdx.x == 0) {
    double a = 0.0;
    unsigned long long b = 0;
    for (int i = 0; i < kThreads / 64; ++i) { a += ssum[i]; b += scnt[i]; }
    psum[blockIdx.x] = a;
    pcount[blockIdx.x] = b;
    for (int v = 0; v < V; ++v) {
      float m = 0.f;
      for (int i = 0; i < kThreads / 64; ++i) m = fmaxf(m, smax[i][v]);
      pmax[(size_t)blockIdx.x * V + v] = m;
    }
  }
}

int launch_psi_init_partials(const float* const* imgs, int V, size_t n, double* psum, unsigned long long* pcount,
                             float* pmax, hipStream_t s) {
  ViewPtrs vp{};
  for (int v = 0; v < V && v < kMaxViews; ++v) vp.p[v] = imgs[v];
  const int nb = (int)std::min<size_t>((n + kThreads - 1) / kThreads, 1024);
  auto launch = [&](auto kernel) {
    hipLaunchKernelGGL(kernel, dim3(nb), dim3(kThreads), 0, s, vp, V, n, psum, pcount, pmax);
  };
  V <= 4 ? launch(k_psi_init<4>) : V <= 8 ? launch(k_psi_init<8>) : V <= 16 ? launch(k_psi_init<16>) : launch(k_psi_init<kMaxViews>);
  return nb;
}

// PsiInitAvgApproxThread.call (D/init/PsiInitAvgApproxThread.java:57-85): min/max/sum over the hyperslice
// x = nx / 2 of one view (all values, zeros included).  The reference visits that slice once per
// dimension and divides by the tripled count, which is the slice mean.  Partials per work-group:
// {sum, max}; the host reduces them in a fixed order.
__global__ __launch_bounds__(kThreads) void k_psi_approx_slice(const float* __restrict__ img, int3 N,
                                                               double2* __restrict__ partial) {
  __shared__ double ss[kThreads], sm[kThreads];
  const int x = N.x / 2;
  const size_t n = (size_t)N.y * N.z;
  double sum = 0.0, mx = -1.0e308;
  for (size_t i = (size_t)blockIdx.x * kThreads + threadIdx.x; i < n; i += (size_t)gridDim.x * kThreads) {
    const double v = (double)img[i * N.x + x];  // i = z * ny + y
    sum += v;
    mx = fmax(mx, v);
  }
  ss[threadIdx.x] = sum;
  sm[threadIdx.x] = mx;
  __syncthreads();
  for (int off = kThreads / 2; off > 0; off >>= 1) {
    if (threadIdx.x < off) {
      ss[threadIdx.x] += ss[threadIdx.x + off];
      sm[threadIdx.x] = fmax(sm[threadIdx.x], sm[threadIdx.x + off]);
    }
    __syncthreads();
  }
  if (threadIdx.x == 0) partial[blockIdx.x] = make_double2(ss[0], sm[0]);
}

int launch_psi_approx_slice(const float* img, const int N[3], double2* partial, hipStream_t s) {
  const size_t n = (size_t)N[1] * N[2];
  const int nb = (int)std::max<size_t>(1, std::min<size_t>((n + kThreads - 1) / kThreads, 256));
  hipLaunchKernelGGL(k_psi_approx_slice, dim3(nb), dim3(kThreads), 0, s, img, make_int3(N[0], N[1], N[2]), partial);
  return nb;
}

// FusedNonZeroRandomAccess.get (D/util/FusedNonZeroRandomAccess.java:57-96): the weighted mean of the
// positive view values, sum(I w) / sum(w) in double, 0 where no positive view has weight.
struct ViewPtrs2 { const float* img[kMaxViews]; const float* w[kMaxViews]; };
__global__ void k_fused_nonzero(ViewPtrs2 vp, int V, size_t n, float* __restrict__ out) {
  for (size_t i = (size_t)blockIdx.x * blockDim.x + threadIdx.x; i < n; i += (size_t)gridDim.x * blockDim.x) {
    double sI = 0.0, sW = 0.0;
    for (int v = 0; v < V; ++v) {
      const double val = (double)vp.img[v][i];
      if (val > 0.0) {
        const double wt = (double)vp.w[v][i];
        sI += val * wt;
        sW += wt;
      }
    }
    out[i] = sW > 0.0 ? (float)(sI / sW) : 0.f;
  }
}

void launch_fused_nonzero(const float* const* imgs, const float* const* ws, int V, size_t n, float* out,
                          hipStream_t s) {
  ViewPtrs2 vp{};
  for (int v = 0; v < V && v < kMaxViews; ++v) { vp.img[v] = imgs[v]; vp.w[v] = ws[v]; }
  const int nb = (int)std::max<size_t>(1, std::min<size_t>((n + kThreads - 1) / kThreads, 8192));
  hipLaunchKernelGGL(k_fused_nonzero, dim3(nb), dim3(kThreads), 0, s, vp, V, n, out);
}

// One axis of a separable symmetric convolution with mirror-single extension (the Gaussian blur of
// PsiInitBlurredFused, D/init/PsiInitBlurredFused.java:113-114): out[p] = sum_{|j| < H} k[|j|] in[mirror(p + j)]
// along `axis`, accumulated in double; mirror-single has period 2n - 2 along the axis.
__global__ void k_sym_conv_axis(const float* __restrict__ in, float* __restrict__ out, int3 N, int axis,
                                const double* __restrict__ half, int H) {
  const size_t n = (size_t)N.x * N.y * N.z;
  const int len = axis == 0 ? N.x : axis == 1 ? N.y : N.z;
  const size_t stride = axis == 0 ? 1 : axis == 1 ? (size_t)N.x : (size_t)N.x * N.y;
  for (size_t i = (size_t)blockIdx.x * blockDim.x + threadIdx.x; i < n; i += (size_t)gridDim.x * blockDim.x) {
    const int pos = (int)((i / stride) % (size_t)len);
    const float* base = in + (i - (size_t)pos * stride);
    double acc = half[0] * (double)base[(size_t)pos * stride];
    for (int j = 1; j < H; ++j) {
      const int a = mirror_index(pos - j, len), b = mirror_index(pos + j, len);
      acc += half[j] * ((double)base[(size_t)a * stride] + (double)base[(size_t)b * stride]);
    }
    out[i] = (float)acc;
  }
}

void launch_sym_conv_axis(const float* in, float* out, const int N[3], int axis, const double* half, int H,
                          hipStream_t s) {
  const size_t n = (size_t)N[0] * N[1] * N[2];
  const int nb = (int)std::max<size_t>(1, std::min<size_t>((n + kThreads - 1) / kThreads, 8192));
  hipLaunchKernelGGL(k_sym_conv_axis, dim3(nb), dim3(kThreads), 0, s, in, out, make_int3(N[0], N[1], N[2]), axis, half,
                     H);
}

// Mul-scheme update (DeconvolutionMethods.computeNextValueMul,
// D/iteration/sequential/DeconvolutionMethods.java:370-419): geometric mean of the
// per-view integrals (double product, pow 1/V), min(1, sum of weights).
struct ViewPtrsW { const float* t2[kMaxViews]; const float* w[kMaxViews]; };

// x^(1/V), V >= 2, of a double to about its last place: x = m 2^(V k) with m in [1/2, 2^V), a float estimate of m's root
// and two Newton steps (relative errors 1e-7 -> 1e-14 -> rounding).  0, infinities, NaN and negative x as pow has them.
__device__ __forceinline__ double nth_root(double x, int V, double invV) {
  int e;
  const double mant = frexp(x, &e);
  const int k = (int)floorf((float)e * (float)invV);
  const double m = ldexp(mant, e - V * k);
  double y = (double)exp2f(log2f((float)m) * (float)invV);
#pragma unroll
  for (int step = 0; step < 2; ++step) {
    double p = y;
    for (int j = 1; j < V; ++j) p = p * y;
    y = y + y * ((m - p) * __builtin_amdgcn_rcp(p)) * invV;
  }
  y = ldexp(y, k);
  if (x > 0.0 && x < __builtin_inf()) return y;
  return x == 0.0 ? 0.0 : x == -__builtin_inf() ? -x : x < 0.0 ? __builtin_nan("") : x;
}

// Bound by HBM (4 (2 V + 2) bytes a voxel): the views' values are loaded four views at a time ahead of their products, and
// the root takes a fifth of pow's instructions.
// 160 x 150 x 140, 4 views: 53.7 us with pow and a coordinate division per voxel, 27.7 (4.8 TB/s) so.
__global__ __launch_bounds__(kThreads) void k_update_mul(float* __restrict__ psi, ViewPtrsW vp, int V, size_t n,
                                                         double lambda, float minI, float maxI,
                                                         double2* __restrict__ partial) {
  // Java rounds every float and double operation: no FMA contraction in the update
#pragma clang fp contract(off)
  double sumc = 0.0;
  float mxc = -1.f;
  const double invV = 1.0 / (double)V;
  const RLConsts rc = rl_consts(lambda, minI, maxI);
  for (size_t i = (size_t)blockIdx.x * kThreads + threadIdx.x; i < n; i += (size_t)gridDim.x * kThreads) {
    const float last = psi[i];
    double sumW = 0.0, prod = 1.0;
    for (int v0 = 0; v0 < V; v0 += 4) {
      float t[4], w[4];
#pragma unroll
      for (int j = 0; j < 4; ++j) {
        const int v = min(v0 + j, V - 1);
        t[j] = vp.t2[v][i];
        w[j] = vp.w[v][i];
      }
#pragma unroll
      for (int j = 0; j < 4; ++j)
        if (v0 + j < V) {
          prod = prod * (double)t[j];
          sumW = sumW + (double)w[j];
        }
    }
    if (V > 1) prod = nth_root(prod, V, invV);
    sumW = fmin(1.0, sumW);
    const float next = rl_tikhonov_adjust(last * (float)prod, rc);
    const float res = last + (next - last) * (float)sumW;
    psi[i] = res;
    const float ch = res - last;
    sumc += (double)ch;
    mxc = java_maxf(mxc, ch);
  }
  block_reduce_stats(sumc, mxc, partial + blockIdx.x);
}

void launch_update_mul(float* psi, const float* const* T2, const float* const* w, int V, size_t n, double lambda,
                       float minValue, float maxI, double2* partial, int* nPartialOut, hipStream_t s) {
  ViewPtrsW vp{};
  for (int v = 0; v < V && v < kMaxViews; ++v) { vp.t2[v] = T2[v]; vp.w[v] = w[v]; }
  const int nb = (int)std::min<size_t>((n + kThreads - 1) / kThreads, 2048);
  hipLaunchKernelGGL(k_update_mul, dim3(nb), dim3(kThreads), 0, s, psi, vp, V, n, lambda, minValue, maxI, partial);
  *nPartialOut = nb;
}

// Block.copyBlock from a zero-extended volume (C/Block.java:158-197 with Views.extendZero, as the image and weight
// blocks of MultiViewDeconvolutionSeq.java:115-126): dst (B voxels) = src (N voxels) at volume coordinate
// off + local position, 0 outside the volume.  One thread per destination voxel, rows of B.x consecutive
// threads so that the loads of a row are contiguous.
__global__ void k_copy_block_zero(const float* __restrict__ src, int3 N, int3 off, float* __restrict__ dst, int3 B) {
  const size_t n = (size_t)B.x * B.y * B.z;
  for (size_t i = (size_t)blockIdx.x * blockDim.x + threadIdx.x; i < n; i += (size_t)gridDim.x * blockDim.x) {
    const int x = (int)(i % (size_t)B.x);
    const size_t r = i / (size_t)B.x;
    const int y = (int)(r % (size_t)B.y), z = (int)(r / (size_t)B.y);
    const long long gx = (long long)off.x + x, gy = (long long)off.y + y, gz = (long long)off.z + z;
    float v = 0.f;
    if (gx >= 0 && gy >= 0 && gz >= 0 && gx < N.x && gy < N.y && gz < N.z)
      v = src[((size_t)gz * N.y + (size_t)gy) * N.x + (size_t)gx];
    dst[i] = v;
  }
}

void launch_copy_block_zero(const float* src, const int N[3], const long long off[3], float* dst, const int B[3],
                            hipStream_t s) {
  const size_t n = (size_t)B[0] * B[1] * B[2];
  const int nb = (int)std::max<size_t>(1, std::min<size_t>((n + kThreads - 1) / kThreads, 16384));
  // offsets beyond +-2^31 would place the block wholly outside any volume the library holds: clamp to a value
  // that is still outside (the copy is then all zeros)
  auto c = [](long long v) { return (int)std::max<long long>(-(1ll << 30), std::min<long long>(v, 1ll << 30)); };
  hipLaunchKernelGGL(k_copy_block_zero, dim3(nb), dim3(kThreads), 0, s, src, make_int3(N[0], N[1], N[2]),
                     make_int3(c(off[0]), c(off[1]), c(off[2])), dst, make_int3(B[0], B[1], B[2]));
}

// DeconView.blockContainsContent (D/DeconView.java:232-274) for many blocks at once: flags[b] = 1 when the weights
// hold a non-zero value inside block b's interval (entry b of tab: {offset[3], size[3]}, zero outside the
// volume); flags must be zero before the launch.  Work-group (x, b) scans a strided share of block b.
__global__ void k_blocks_with_content(const float* __restrict__ w, int3 N, const int* __restrict__ tab,
                                      int* __restrict__ flags) {
  const int* t = tab + 6 * blockIdx.y;
  const int x0 = max(t[0], 0), y0 = max(t[1], 0), z0 = max(t[2], 0);
  const int x1 = min(t[0] + t[3], N.x), y1 = min(t[1] + t[4], N.y), z1 = min(t[2] + t[5], N.z);
  if (x1 <= x0 || y1 <= y0 || z1 <= z0) return;
  const int nx = x1 - x0, ny = y1 - y0;
  const size_t n = (size_t)nx * ny * (z1 - z0);
  bool any = false;
  for (size_t i = (size_t)blockIdx.x * blockDim.x + threadIdx.x; i < n && !any; i += (size_t)gridDim.x * blockDim.x) {
    const int x = (int)(i % nx);
    const size_t r = i / nx;
    const int y = (int)(r % ny), z = (int)(r / ny);
    any = w[((size_t)(z0 + z) * N.y + (y0 + y)) * N.x + (x0 + x)] != 0.f;
  }
  if (any) flags[blockIdx.y] = 1;  // every writer stores the same value
}

void launch_blocks_with_content(const float* w, const int N[3], const int* tab, int nblocks, int* flags,
                                hipStream_t s) {
  if (nblocks <= 0) return;
  hipLaunchKernelGGL(k_blocks_with_content, dim3(64, nblocks), dim3(kThreads), 0, s, w, make_int3(N[0], N[1], N[2]),
                     tab, flags);
}

// DeconvolutionMethods.computeQuotient (D/iteration/sequential/DeconvolutionMethods.java:46-98) over a flat array:
// blurred[i] = img[i] > 0 ? img[i] / blurred[i] : 1.
__global__ void k_quotient(const float* __restrict__ img, float* __restrict__ blurred, size_t n) {
  for (size_t i = (size_t)blockIdx.x * blockDim.x + threadIdx.x; i < n; i += (size_t)gridDim.x * blockDim.x) {
    const float im = img[i];
    blurred[i] = im > 0.f ? im / blurred[i] : 1.f;
  }
}

void launch_quotient(const float* img, float* blurred, size_t n, hipStream_t s) {
  const int nb = (int)std::max<size_t>(1, std::min<size_t>((n + kThreads - 1) / kThreads, 8192));
  hipLaunchKernelGGL(k_quotient, dim3(nb), dim3(kThreads), 0, s, img, blurred, n);
}

// DeconvolutionMethods.computeFinalValues (D/iteration/sequential/DeconvolutionMethods.java:103-182) over a flat
// array: psi[i] = computeNextValue(psi[i], integral[i], weight[i]); per work-group {sum, max} of the change.
__global__ __launch_bounds__(kThreads) void k_final_values(float* __restrict__ psi, const float* __restrict__ integral,
                                                           const float* __restrict__ weight, size_t n, double lambda,
                                                           float minI, float maxI, double2* __restrict__ partial) {
  double sumc = 0.0;
  float mxc = -1.f;
  const RLConsts rc = rl_consts(lambda, minI, maxI);
  for (size_t i = (size_t)blockIdx.x * kThreads + threadIdx.x; i < n; i += (size_t)gridDim.x * kThreads) {
    const float last = psi[i];
    const float next = rl_next_value(last, integral[i], weight[i], rc);
    psi[i] = next;
    const float ch = next - last;
    sumc += (double)ch;
    mxc = java_maxf(mxc, ch);
  }
  block_reduce_stats(sumc, mxc, partial + blockIdx.x);
}

int launch_final_values(float* psi, const float* integral, const float* weight, size_t n, double lambda,
                        float minValue, float maxI, double2* partial, int maxPartials, hipStream_t s) {
  const int nb = (int)std::max<size_t>(1, std::min<size_t>((n + kThreads - 1) / kThreads, (size_t)maxPartials));
  hipLaunchKernelGGL(k_final_values, dim3(nb), dim3(kThreads), 0, s, psi, integral, weight, n, lambda, minValue, maxI,
                     partial);
  return nb;
}

// Distance of psi to a reference volume in FP64: per work-group {sum (a - b)^2, sum b^2},
// then one work-group sums the partials in a fixed order.
__global__ __launch_bounds__(kThreads) void k_rel_l2_partials(const float* __restrict__ a, const float* __restrict__ b,
                                                              size_t n, double2* __restrict__ partial) {
  __shared__ double sd[kThreads], sr[kThreads];
  double d = 0.0, r = 0.0;
  for (size_t i = (size_t)blockIdx.x * blockDim.x + threadIdx.x; i < n; i += (size_t)gridDim.x * blockDim.x) {
    const double e = (double)a[i] - (double)b[i];
    d += e * e;
    r += (double)b[i] * (double)b[i];
  }
  sd[threadIdx.x] = d;
  sr[threadIdx.x] = r;
  __syncthreads();
  for (int off = kThreads / 2; off > 0; off >>= 1) {
    if (threadIdx.x < off) {
      sd[threadIdx.x] += sd[threadIdx.x + off];
      sr[threadIdx.x] += sr[threadIdx.x + off];
    }
    __syncthreads();
  }
  if (threadIdx.x == 0) partial[blockIdx.x] = make_double2(sd[0], sr[0]);
}

__global__ void k_sum2(const double2* __restrict__ partial, int n, double2* __restrict__ out) {
  __shared__ double sd[kThreads], sr[kThreads];
  double d = 0.0, r = 0.0;
  for (int i = threadIdx.x; i < n; i += kThreads) { d += partial[i].x; r += partial[i].y; }
  sd[threadIdx.x] = d;
  sr[threadIdx.x] = r;
  __syncthreads();
  for (int off = kThreads / 2; off > 0; off >>= 1) {
    if (threadIdx.x < off) {
      sd[threadIdx.x] += sd[threadIdx.x + off];
      sr[threadIdx.x] += sr[threadIdx.x + off];
    }
    __syncthreads();
  }
  if (threadIdx.x == 0) *out = make_double2(sd[0], sr[0]);
}

// partial must hold 1024 entries; out receives {sum (a - b)^2, sum b^2}
void launch_rel_l2(const float* a, const float* b, size_t n, double2* partial, double2* out, hipStream_t s) {
  const int nb = (int)std::max<size_t>(1, std::min<size_t>((n + kThreads - 1) / kThreads, 1024));
  hipLaunchKernelGGL(k_rel_l2_partials, dim3(nb), dim3(kThreads), 0, s, a, b, n, partial);
  hipLaunchKernelGGL(k_sum2, dim3(1), dim3(kThreads), 0, s, partial, nb, out);
}

}  // namespace mvr
