// psf.cpp -- kernel normalisation and the four iteration schemes' second kernels.
#include <algorithm>
#include <cmath>

#include "host.hpp"

namespace mvr {

namespace {

// FusionTools.divideIntoPortions (F/FusionTools.java:1287-1329); nT stands for
// Threads.numThreads() (Threads.java:40), a numeric parameter of the result.
struct Portion { size_t start, len; };
std::vector<Portion> portions(size_t n, int nT) {
  std::vector<Portion> out;
  if (n == 0) return out;
  long long np = (long long)n <= nT ? (long long)n : std::max<long long>(nT, (long long)(n / (64ull * 64ull * 64ull)));
  size_t chunk = n / np;
  while (chunk == 0) { --np; chunk = n / np; }
  const size_t mod = n % np;
  for (long long i = 0; i < np; ++i) out.push_back({(size_t)i * chunk, i == np - 1 ? chunk + mod : chunk});
  return out;
}

// compensated double accumulation (imglib2 RealSum)
struct Kahan {
  double s = 0, c = 0;
  void add(double v) { double y = v - c; double t = s + y; c = (t - s) - y; s = t; }
};

}  // namespace

// AdjustInput.sumImg (D/normalization/AdjustInput.java:71-122): the total
// starts with the first portion's sum and then adds every portion's sum.
double sum_img_quirk(const float* a, size_t n, int nT) {
  // eight portions at a time: a compensated sum alone waits out four additions per value (150 us for 31^3 values)
  const auto ps = portions(n, nT);
  std::vector<double> sums;
  for (size_t i = 0; i < ps.size(); i += 8) {
    const size_t m = std::min<size_t>(8, ps.size() - i);
    Kahan k[8];
    size_t at[8], len = ps[i].len;
    for (size_t p = 0; p < 8; ++p) at[p] = ps[i + std::min(p, m - 1)].start;
    for (size_t p = 0; p < m; ++p) len = std::min(len, ps[i + p].len);
    for (size_t j = 0; j < len; ++j)
      for (int p = 0; p < 8; ++p) k[p].add((double)a[at[p] + j]);
    for (size_t p = 0; p < m; ++p) {
      for (size_t j = len; j < ps[i + p].len; ++j) k[p].add((double)a[at[p] + j]);
      sums.push_back(k[p].s);
    }
  }
  Kahan total;
  if (!sums.empty()) total.add(sums[0]);
  for (double s : sums) total.add(s);
  return total.s;
}

// AdjustInput.normToSum1 (D/normalization/AdjustInput.java:52-58)
void norm_to_sum1(float* a, size_t n, int nT) {
  const double sum = sum_img_quirk(a, n, nT);
  for (size_t i = 0; i < n; ++i) a[i] = (float)((double)a[i] / sum);
}

// Mirror.mirror on every axis (D/util/Mirror.java:55-132), sequential order:
// pairs (i, n-1-i) with i <= n/2 are swapped in flat order, so an even axis
// leaves its middle pair in place.
void mirror_all(float* a, const int dim[3]) {
  // the source of each position along an axis after its swaps; the axes are independent of one another
  std::vector<int> from[3];
  for (int d = 0; d < 3; ++d) {
    const int n = dim[d];
    from[d].resize(n);
    for (int i = 0; i < n; ++i) from[d][i] = i;
    for (int i = 0; i <= n / 2 && i < n; ++i) std::swap(from[d][i], from[d][n - 1 - i]);
  }
  const std::vector<float> src(a, a + (size_t)dim[0] * dim[1] * dim[2]);
  for (int z = 0; z < dim[2]; ++z)
    for (int y = 0; y < dim[1]; ++y, a += dim[0]) {
      const float* row = src.data() + ((size_t)from[2][z] * dim[1] + from[1][y]) * dim[0];
      for (int x = 0; x < dim[0]; ++x) a[x] = row[from[0][x]];
    }
}

// Products of same-size convolutions (the FFTConvolution chains of DeconViewPSF.init, :132-195, :196-242): with a the
// V kernels, b the mirrored ones and (*) zero-extended,
//   twice:  out_v = b_v prod_{w != v} ((b_v (*) a_w) (*) b_w)        otherwise:  out_v = a_v prod_{w != v} (a_v (*) b_w)
// multiplied in the order of w.  kernels holds a then b, 2 V arrays on the device; out V arrays.
//
// On grids transformed plane by plane all pairs run in one launch per pass: the 2 V kernel spectra and the V data
// spectra are transformed once and shared by the pairs.  The pairs of as many views as fit kPairBytes go together.
// Six 31^3 kernels, twice (60 convolutions): the set-up of a 192 x 176 x 128 frame takes 17.5 ms with allocations and
// copies for each pair, 1.62 ms so (110 us of it these kernels).
// Larger grids run pair by pair in two spectra, as does a device without the memory for the batch.
class PsfProducts {
 public:
  PsfProducts(const int* K, int V, bool twice) : V(V), twice(twice), nk((size_t)K[0] * K[1] * K[2]) {
    for (int d = 0; d < 3; ++d) this->K[d] = K[d];
  }
  ~PsfProducts() {
    if (mem) (void)hipFree(mem);
  }
  int run(const float* kernels, float* out, hipStream_t s) {
    if (plan.create(K, K)) return -1;
    const size_t n = plan.ncpx(), pairBytes = (size_t)(V - 1) * (n * 8 + nk * 4);
    const int views = (int)std::max<size_t>(1, std::min<size_t>(V, kPairBytes / pairBytes));
    const size_t batch = 3 * (size_t)V * n * 8 + views * pairBytes + 3 * (size_t)V * (V - 1) * sizeof(int);
    if (plan.planar) {
      if (hipMalloc(&mem, batch) == hipSuccess) return batched(kernels, out, views, s);
      (void)hipGetLastError();
      mem = nullptr;
    }
    MVR_HIP(hipMalloc(&mem, 2 * n * 8 + 2 * nk * 4));
    return pair_by_pair(kernels, out, s);
  }

 private:
  static constexpr size_t kPairBytes = 256u << 20;
  GatherParams data_gather(const float* src) const {
    GatherParams g{};
    g.src = src;
    for (int d = 0; d < 3; ++d) { g.N[d] = K[d]; g.org[d] = -plan.dom.m[d]; }
    g.mode = GATHER_VALUE;
    return g;
  }

  int batched(const float* kernels, float* out, int views, hipStream_t s) {
    const size_t n = plan.ncpx();
    const int nf = V - 1, npairs = V * nf;
    float2* kspec = static_cast<float2*>(mem);
    float2* dspec = kspec + 2 * V * n;
    float2* work = dspec + V * n;
    float* o = reinterpret_cast<float*>(work + (size_t)views * nf * n);
    int* tab = reinterpret_cast<int*>(o + (size_t)views * nf * nk);
    std::vector<int> h(3 * npairs);  // of each pair: its data, its first and its second kernel
    for (int v = 0, p = 0; v < V; ++v)
      for (int w = 0; w < V; ++w)
        if (w != v) {
          h[p] = v;
          h[npairs + p] = twice ? w : V + w;
          h[2 * npairs + p++] = V + w;
        }
    MVR_HIP(hipMemcpyAsync(tab, h.data(), h.size() * sizeof(int), hipMemcpyHostToDevice, s));
    // spectra of the kernels (once: of the mirrored ones only) and of the data
    const int k0 = twice ? 0 : V;
    GatherParams g = data_gather(kernels + (twice ? V * nk : 0));
    const Plan::Mid conv = plan.convolve_geometry(g);
    const XFwdGroup first[2] = {{plan.kernel_gather(kernels + k0 * nk), kspec + k0 * n, 2 * V - k0, nk, n},
                                {g, dspec, V, nk, n}};
    plan.xfg(plan.dom, first, 2, plan.twM, plan.wr, s);
    plan.kernel_planes(kspec + k0 * n, 2 * V - k0, s);
    Dom dom = plan.dom;
    dom.blockStride = n;
    for (int v = 0; v < V; v += views) {
      const int np = std::min(views, V - v) * nf;
      const StoreParams st{o, np};
      PlaneGeom pl = conv.pl;
      pl.nb = np;
      pl.inStride = pl.outStride = pl.specStride = n;
      pl.inIdx = tab + v * nf;
      pl.specIdx = tab + npairs + v * nf;
      launch_plane(pl, dspec, work, kspec, plan.twY, plan.twZ, s);
      plan.xs(dom, st, work, plan.twM, plan.wr, s);
      if (twice) {
        g.src = o;
        const XFwdGroup again{g, work, np, nk, n};
        plan.xfg(plan.dom, &again, 1, plan.twM, plan.wr, s);
        pl.inIdx = nullptr;
        pl.specIdx = tab + 2 * npairs + v * nf;
        launch_plane(pl, work, work, kspec, plan.twY, plan.twZ, s);
        plan.xs(dom, st, work, plan.twM, plan.wr, s);
      }
      launch_psf_products(kernels + ((twice ? V : 0) + v) * nk, o, np / nf, nf, nk, out + v * nk, s);
    }
    MVR_HIP(hipGetLastError());
    MVR_HIP(hipStreamSynchronize(s));  // h and the destructor
    return 0;
  }

  int pair_by_pair(const float* kernels, float* out, hipStream_t s) {
    const size_t n = plan.ncpx();
    float2* spec = static_cast<float2*>(mem);
    float2* work = spec + n;
    float* o1 = reinterpret_cast<float*>(work + n);
    float* o2 = o1 + nk;
    const float* mirrored = kernels + V * nk;
    for (int v = 0; v < V; ++v) {
      const float* data = (twice ? mirrored : kernels) + v * nk;
      const float* acc = data;
      for (int w = 0; w < V; ++w) {
        if (w == v) continue;
        const float* o = o1;
        if (plan.convolve_once((twice ? kernels : mirrored) + w * nk, data_gather(data), spec, work, o1, s)) return -1;
        if (twice) {
          if (plan.convolve_once(mirrored + w * nk, data_gather(o1), spec, work, o2, s)) return -1;
          o = o2;
        }
        launch_psf_products(acc, o, 1, 1, nk, out + v * nk, s);
        acc = out + v * nk;
      }
    }
    MVR_HIP(hipGetLastError());
    MVR_HIP(hipStreamSynchronize(s));
    return 0;
  }

  Plan plan;
  int K[3], V;
  bool twice;
  size_t nk;
  void* mem = nullptr;
};

// the products of the kernels k1 and their mirrored copies, in out
static int psf_products(const std::vector<std::vector<float>>& k1, const std::vector<std::vector<float>>& inv,
                        const int K[3], bool twice, std::vector<std::vector<float>>& out, hipStream_t s) {
  const int V = (int)k1.size();
  const size_t nk = (size_t)K[0] * K[1] * K[2];
  std::vector<float> h(2 * V * nk);
  for (int v = 0; v < V; ++v) {
    std::copy(k1[v].begin(), k1[v].end(), h.begin() + v * nk);
    std::copy(inv[v].begin(), inv[v].end(), h.begin() + (V + v) * nk);
  }
  float* dev = nullptr;
  MVR_HIP(hipMalloc(&dev, 3 * V * nk * 4));
  int rc = -1;
  if (hipMemcpyAsync(dev, h.data(), 2 * V * nk * 4, hipMemcpyHostToDevice, s) != hipSuccess)
    set_error("init_psfs: copy failed");
  else
    rc = PsfProducts(K, V, twice).run(dev, dev + 2 * V * nk, s);
  if (!rc && (hipMemcpyAsync(h.data(), dev + 2 * V * nk, V * nk * 4, hipMemcpyDeviceToHost, s) != hipSuccess ||
              hipStreamSynchronize(s) != hipSuccess)) {
    set_error("init_psfs: readback failed");
    rc = -1;
  }
  if (rc) (void)hipStreamSynchronize(s);
  (void)hipFree(dev);
  if (rc) return rc;
  for (int v = 0; v < V; ++v) out[v].assign(h.begin() + v * nk, h.begin() + (v + 1) * nk);
  return 0;
}

int init_psfs(int dev, std::vector<std::vector<float>>& k1, const int K[3], int psfType, int nT,
              std::vector<std::vector<float>>& k2, hipStream_t s) {
  (void)dev;
  const int V = (int)k1.size();
  const size_t nk = (size_t)K[0] * K[1] * K[2];
  k2.assign(V, {});
  auto inverted = [&](const std::vector<float>& a) {
    std::vector<float> r(a);
    mirror_all(r.data(), K);
    return r;
  };
  std::vector<std::vector<float>> inv(V);
  for (int v = 0; v < V; ++v) {
    norm_to_sum1(k1[v].data(), nk, nT);
    inv[v] = inverted(k1[v]);
  }
  if (V == 1 || psfType == PSF_INDEPENDENT) {
    k2 = inv;
  } else if (psfType == PSF_EFFICIENT_BAYESIAN || psfType == PSF_OPT_I) {
    // P_v^compound = P_v^* prod_{w != v} (P_v^* (*) P_w (*) P_w^*)   (:132-195)
    // (P_v prod_{w != v} (P_v (*) P_w^*))^*                           (:196-242)
    const bool bayesian = psfType == PSF_EFFICIENT_BAYESIAN;
    if (psf_products(k1, inv, K, bayesian, k2, s)) return -1;
    for (int v = 0; v < V; ++v) {
      norm_to_sum1(k2[v].data(), nk, nT);
      if (!bayesian) mirror_all(k2[v].data(), K);
    }
  } else {
    // (P_v^V)^*, iterated float multiply   (:243-253, :276-284)
    for (int v = 0; v < V; ++v) {
      std::vector<float> e(k1[v]);
      for (size_t i = 0; i < nk; ++i) {
        float r = k1[v][i];
        for (int p = 1; p < V; ++p) r *= k1[v][i];
        e[i] = r;
      }
      norm_to_sum1(e.data(), nk, nT);
      k2[v] = inverted(e);
    }
  }
  return 0;
}

}  // namespace mvr
