// psf.cpp -- kernel normalisation and the four iteration schemes' second kernels.
#include <algorithm>
#include <cmath>
#include <cstring>

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
// (returns the sum it divided by)
double norm_to_sum1(float* a, size_t n, int nT) {
  const double sum = sum_img_quirk(a, n, nT);
  for (size_t i = 0; i < n; ++i) a[i] = (float)((double)a[i] / sum);
  return sum;
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

// kernels of V views that PsfProducts uses
static int psf_kernel_count(int V) { return 4 * V - 2; }

// Products of same-size convolutions (the FFTConvolution chains of DeconViewPSF.init, :132-195, :196-242): with a the
// V kernels, b the mirrored ones and (*) zero-extended,
//   twice:  out_v = b_v prod_{w != v} ((b_v (*) a_w) (*) b_w)        otherwise:  out_v = a_v prod_{w != v} (a_v (*) b_w)
// multiplied in the order of w.  A view's kernel is normalised when its turn comes: a_v, b_v and those of w < v are
// normalised, those of w > v as they were given.  Their scale goes with the final normalisation, but it decides where the
// float products leave their range.  kernels holds, on the device, the given a_1.., the normalised a_0.., the normalised
// b_0.. and the given b_1.., psf_kernel_count(V) arrays; out V arrays.
//
// On grids transformed plane by plane all pairs run in one launch per pass: the kernel spectra (of both scales) and the V
// data spectra are transformed once and shared by the pairs.  The pairs of as many views as fit kPairBytes go together.
// Planar spectra need no row pitch, so they are Hx planes, not HxP (allocations above 64 MiB take 0.35 ms more here).
// Six 31^3 kernels, twice (60 convolutions): the set-up of a 192 x 176 x 128 frame takes 17.5 ms with allocations and
// copies for each pair, 1.40 ms so.
// Larger grids run pair by pair in two spectra, as does a device without the memory for the batch.
class PsfProducts {
 public:
  PsfProducts(const int* K, int V, bool twice) : V(V), twice(twice), nk((size_t)K[0] * K[1] * K[2]) {
    for (int d = 0; d < 3; ++d) this->K[d] = K[d];
  }
  ~PsfProducts() {
    if (mem) (void)hipFree(mem);
  }
  // given: the kernels' normalising sums (V doubles) and the V kernels, replaced by the products
  int run(std::vector<float>& given, hipStream_t s) {
    if (plan.create(K, K)) return -1;
    // what is given, the kernels of both scales and the results lie before the spectra, in one allocation
    const size_t kernN = psf_kernel_count(V) * nk, head = ((given.size() + kernN + V * nk) * 4 + 255) / 256 * 256;
    int views = 0;
    if (plan.planar) {
      const size_t n = planes(), pairBytes = (size_t)(V - 1) * (n * 8 + nk * 4);
      views = (int)std::max<size_t>(1, std::min<size_t>(V, kPairBytes / pairBytes));
      const size_t batch = (size_t)(nkern() + V) * n * 8 + views * pairBytes + 3 * (size_t)V * (V - 1) * sizeof(int);
      if (hipMalloc(&mem, head + batch) != hipSuccess) {
        (void)hipGetLastError();
        mem = nullptr;
        views = 0;
      }
    }
    if (!mem) MVR_HIP(hipMalloc(&mem, head + 2 * plan.ncpx() * 8 + 2 * nk * 4));
    spectra = reinterpret_cast<float2*>(static_cast<char*>(mem) + head);
    float* dgiven = static_cast<float*>(mem);
    float* kernels = dgiven + given.size();
    float* out = kernels + kernN;
    MVR_HIP(hipMemcpyAsync(dgiven, given.data(), given.size() * 4, hipMemcpyHostToDevice, s));
    launch_psf_kernels(dgiven + 2 * V, reinterpret_cast<const double*>(dgiven), V, K, kernels, s);
    if (views ? batched(kernels, out, views, s) : pair_by_pair(kernels, out, s)) {
      (void)hipStreamSynchronize(s);  // given is in use
      return -1;
    }
    MVR_HIP(hipMemcpyAsync(given.data(), out, V * nk * 4, hipMemcpyDeviceToHost, s));
    MVR_HIP(hipStreamSynchronize(s));
    return 0;
  }

 private:
  static constexpr size_t kPairBytes = 256u << 20;
  // places of the kernels of view w in the pairs of view v, and of its data; the kernels in use (once: the mirrored ones)
  int kernel_at(int v, int w) const { return w > v ? w - 1 : V - 1 + w; }
  int mirrored_at(int v, int w) const { return w > v ? 3 * V - 2 + w : 2 * V - 1 + w; }
  int data_at(int v) const { return (twice ? 2 * V - 1 : V - 1) + v; }
  int kern0() const { return twice ? 0 : 2 * V - 1; }
  int nkern() const { return psf_kernel_count(V) - kern0(); }
  size_t planes() const { return (size_t)plan.Hx * plan.dom.P[1] * plan.dom.P[2]; }
  GatherParams data_gather(const float* src) const {
    GatherParams g{};
    g.src = src;
    for (int d = 0; d < 3; ++d) { g.N[d] = K[d]; g.org[d] = -plan.dom.m[d]; }
    g.mode = GATHER_VALUE;
    return g;
  }

  int batched(const float* kernels, float* out, int views, hipStream_t s) {
    const size_t n = planes();
    const int nf = V - 1, npairs = V * nf, k0 = kern0(), nkernels = nkern();
    float2* kspec = spectra;
    float2* dspec = kspec + nkernels * n;
    float2* work = dspec + V * n;
    float* o = reinterpret_cast<float*>(work + (size_t)views * nf * n);
    int* tab = reinterpret_cast<int*>(o + (size_t)views * nf * nk);
    std::vector<int> h(3 * npairs);  // of each pair: its data, its first and its second kernel
    for (int v = 0, p = 0; v < V; ++v)
      for (int w = 0; w < V; ++w)
        if (w != v) {
          h[p] = v;
          h[npairs + p] = (twice ? kernel_at(v, w) : mirrored_at(v, w)) - k0;
          h[2 * npairs + p++] = mirrored_at(v, w) - k0;
        }
    MVR_HIP(hipMemcpyAsync(tab, h.data(), h.size() * sizeof(int), hipMemcpyHostToDevice, s));
    // spectra of the kernels and of the data
    GatherParams g = data_gather(kernels + data_at(0) * nk);
    const Plan::Mid conv = plan.convolve_geometry(g);
    const XFwdGroup first[2] = {{plan.kernel_gather(kernels + k0 * nk), kspec, nkernels, nk, n},
                                {g, dspec, V, nk, n}};
    plan.xfg(plan.dom, first, 2, plan.twM, plan.wr, s);
    plan.kernel_planes(kspec, nkernels, n, s);
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
      launch_psf_products(kernels + data_at(v) * nk, o, np / nf, nf, nk, out + v * nk, s);
    }
    MVR_HIP(hipGetLastError());
    MVR_HIP(hipStreamSynchronize(s));  // h and the destructor
    return 0;
  }

  int pair_by_pair(const float* kernels, float* out, hipStream_t s) {
    const size_t n = plan.ncpx();
    float2* spec = spectra;
    float2* work = spec + n;
    float* o1 = reinterpret_cast<float*>(work + n);
    float* o2 = o1 + nk;
    for (int v = 0; v < V; ++v) {
      const float* data = kernels + data_at(v) * nk;
      const float* acc = data;
      for (int w = 0; w < V; ++w) {
        if (w == v) continue;
        const float* o = o1;
        const float* k2 = kernels + mirrored_at(v, w) * nk;
        if (plan.convolve_once(twice ? kernels + kernel_at(v, w) * nk : k2, data_gather(data), spec, work, o1, s)) return -1;
        if (twice) {
          if (plan.convolve_once(k2, data_gather(o1), spec, work, o2, s)) return -1;
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
  float2* spectra = nullptr;
};

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
  const bool bayesian = psfType == PSF_EFFICIENT_BAYESIAN, products = V > 1 && (bayesian || psfType == PSF_OPT_I);
  std::vector<float> given;
  given.reserve(products ? 2 * V + V * nk : 0);
  given.resize(products ? 2 * V : 0);
  for (int v = 0; v < V; ++v) {
    if (products) given.insert(given.end(), k1[v].begin(), k1[v].end());
    const double sum = norm_to_sum1(k1[v].data(), nk, nT);
    if (products) std::memcpy(given.data() + 2 * v, &sum, sizeof(sum));
  }
  if (V == 1 || psfType == PSF_INDEPENDENT) {
    for (int v = 0; v < V; ++v) k2[v] = inverted(k1[v]);
  } else if (products) {
    // P_v^compound = P_v^* prod_{w != v} (P_v^* (*) P_w (*) P_w^*)   (:132-195)
    // (P_v prod_{w != v} (P_v (*) P_w^*))^*                           (:196-242)
    if (PsfProducts(K, V, bayesian).run(given, s)) return -1;
    for (int v = 0; v < V; ++v) {
      k2[v].assign(given.begin() + v * nk, given.begin() + (v + 1) * nk);
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
