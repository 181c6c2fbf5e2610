// plan.cpp -- FFT-convolution plans, error state and pass timers.
#include <algorithm>
#include <cmath>
#include <vector>

#include "host.hpp"

namespace mvr {

static thread_local std::string g_err;
void set_error(const std::string& msg) { g_err = msg; }
const char* last_error() { return g_err.c_str(); }

bool device_memory_of(const void* p, int dev, bool managed) {
  hipPointerAttribute_t a{};
  if (hipPointerGetAttributes(&a, p) != hipSuccess) {
    (void)hipGetLastError();  // an unknown (pageable host) pointer: clear the error it leaves
    return false;
  }
  if (a.type == hipMemoryTypeManaged || a.isManaged) return managed;
  return a.type == hipMemoryTypeDevice && a.device == dev;
}

static int pick_length(int need, bool half) {
  for (const int* p = strided_lengths(); *p; ++p) {
    if (*p < need) continue;
    if (half) {
      bool ok = false;
      for (const int* h = half_lengths(); *h; ++h) ok |= (*h * 2 == *p);
      if (!ok) continue;
    }
    return *p;
  }
  return -1;
}

int Plan::create(const int D[3], const int Kd[3], const int* Pmin) {
  if (create_geometry(D, Kd, Pmin)) return -1;
  twM = twiddle_table(M);
  wr = twiddle_table(dom.P[0]);
  twY = twiddle_table(dom.P[1]);
  twZ = twiddle_table(dom.P[2]);
  if (!twM || !wr || !twY || !twZ) { set_error("plan: twiddle tables not found on the device"); return -1; }
  return 0;
}

int Plan::create_geometry(const int D[3], const int Kd[3], const int* Pmin) {
  for (int d = 0; d < 3; ++d) {
    if (D[d] < 1 || Kd[d] < 1) { set_error("plan: empty domain or kernel"); return -1; }
    K[d] = Kd[d];
    dom.D[d] = D[d];
    dom.m[d] = K[d] - 1 - K[d] / 2;
    int need = D[d] + K[d] - 1;
    if (Pmin && Pmin[d] > need) need = Pmin[d];
    const int P = pick_length(need, d == 0);
    if (P < 0) { set_error("plan: no compiled FFT length >= " + std::to_string(need)); return -1; }
    dom.P[d] = P;
  }
  M = dom.P[0] / 2;
  Hx = M + 1;
  dom.HxP = (Hx + 15) / 16 * 16;
  planar = dom.P[1] <= planeMax && dom.P[2] <= planeMax && M <= kPlanarMaxM;
  xf = get_x_fwd(M, planar);
  xfg = planar ? get_x_fwd_groups(M) : nullptr;
  xr = get_x_ratio(M, planar);
  xu = get_x_update(M, planar);
  xs = get_x_store(M, planar);
  sy = get_strided(dom.P[1]);
  sz = get_strided(dom.P[2]);
  if (!xf || !xr || !xu || !xs || !sy || !sz) { set_error("plan: missing kernel instantiation"); return -1; }
  // the strided passes address a lane's column and pencil position with a 32-bit byte offset from the plane
  if (((size_t)get_strided_span(dom.P[1]) * dom.HxP + 16) * sizeof(float2) > 0xffffffffull ||
      ((size_t)get_strided_span(dom.P[2]) * dom.P[1] * dom.HxP + 16) * sizeof(float2) > 0xffffffffull) {
    set_error("plan: xy plane of the FFT grid too large for 32-bit lane offsets");
    return -1;
  }
  return 0;
}

Plan::Mid Plan::mid() const {
  Mid m;
  m.y.planeStride = (size_t)dom.P[1] * dom.HxP;
  m.y.lineStride = dom.HxP;
  m.y.ncols = Hx;
  m.y.nplanes = dom.P[2];
  m.y.width = wy;
  m.zf.planeStride = dom.HxP;
  m.zf.lineStride = (size_t)dom.P[1] * dom.HxP;
  m.zf.ncols = Hx;
  m.zf.nplanes = dom.P[1];
  m.zf.width = wz;
  m.zi = m.zf;
  m.pl.Py = dom.P[1];
  m.pl.Pz = dom.P[2];
  m.pl.ncols = Hx;
  m.pl.lo[0] = m.pl.lo[1] = 0;
  m.pl.hi[0] = dom.P[1];
  m.pl.hi[1] = dom.P[2];
  return m;
}

void Plan::set_blocks(Mid& m, int nb, size_t blockStride) const {
  for (StridedGeom* g : {&m.zf, &m.y, &m.zi}) {
    g->blockPlanes = g->nplanes;
    g->nplanes *= nb;
    g->blockStride = blockStride;
  }
  m.pl.nb = nb;
  m.pl.inStride = m.pl.outStride = blockStride;
}

void Plan::set_views(Mid& m, int nb, float2* const* specs, bool shared) const {
  set_blocks(m, nb, ncpx());
  m.y.views.n = m.pl.views.n = nb;
  for (int b = 0; b < nb; ++b) m.y.views.at[b] = m.pl.views.at[b] = specs[b] - specs[0];
  m.y.views.inShared = shared;
  if (shared) m.pl.inStride = 0;
}

void Plan::restrict_rows(const int lo[3], const int hi[3], Mid& m) const {
  int a[3], b[3];
  for (int k = 1; k < 3; ++k) {
    a[k] = std::max(0, dom.m[k] - lo[k]);
    b[k] = std::min(dom.P[k], dom.m[k] + dom.D[k] + hi[k]);
    m.pl.lo[k - 1] = a[k];
    m.pl.hi[k - 1] = b[k];
  }
  m.y.storeLo = a[1];
  m.y.storeHi = b[1];
  const int nb = m.zi.blockPlanes ? m.zi.nplanes / m.zi.blockPlanes : 1;
  m.zi.plane0 = a[1];
  m.zi.nplanes = (b[1] - a[1]) * nb;
  if (m.zi.blockPlanes) m.zi.blockPlanes = b[1] - a[1];
  m.zi.storeLo = a[2];
  m.zi.storeHi = b[2];
}

void Plan::skip_ones_rows(RatioParams& q, Mid& m, const int* blockRows) const {
  if (blockRows) {
    q.skipOnes = 1;
    for (int k = 1; k < 3; ++k) q.rowN[k] = std::min(dom.P[k], dom.D[k] + q.qlo[k] + q.qhi[k]);
    m.pl.ones = true;
    m.pl.onesDC = (float)dom.P[0];
    m.pl.onesTab = blockRows;
    return;
  }
  // quotient rows (y, z) in grid coordinates, as the quotient pass selects them
  int lo[3], hi[3];
  for (int k = 1; k < 3; ++k) {
    lo[k] = std::max(dom.m[k] - q.qlo[k], dom.m[k] - q.o[k]);
    hi[k] = std::min(dom.m[k] + dom.D[k] + q.qhi[k], dom.m[k] - q.o[k] + q.N[k]);
  }
  q.skipOnes = 1;
  for (int k = 1; k < 3; ++k) {
    q.rowLo[k] = lo[k];
    q.rowN[k] = std::max(0, hi[k] - lo[k]);
  }
  constant_rows(lo, hi, 1.f, m);
}

void Plan::constant_rows(const int lo[3], const int hi[3], float value, Mid& m) const {
  for (int k = 1; k < 3; ++k) {
    m.pl.onesLo[k - 1] = lo[k];
    m.pl.onesHi[k - 1] = hi[k];
  }
  m.pl.ones = m.zf.ones = m.y.ones = true;
  m.pl.onesDC = m.zf.onesDC = value * (float)dom.P[0];  // the x transform of a constant row
  m.zf.onesPlaneLo = lo[1];
  m.zf.onesPlaneHi = hi[1];
  m.zf.onesLo = lo[2];
  m.zf.onesHi = hi[2];
  const int nb = m.zf.blockPlanes ? m.zf.nplanes / m.zf.blockPlanes : 1;
  m.zf.plane0 = lo[1];
  m.zf.nplanes = std::max(0, hi[1] - lo[1]) * nb;
  if (m.zf.blockPlanes) m.zf.blockPlanes = std::max(0, hi[1] - lo[1]);
  m.y.onesDC = value * (float)dom.P[0] * (float)dom.P[2];  // the xz transform of a constant plane
  m.y.onesDCPlane = 0;
  m.y.onesPlaneLo = 0;
  m.y.onesPlaneHi = dom.P[2];
  m.y.onesLo = lo[1];
  m.y.onesHi = hi[1];
}

void Plan::value_rows(GatherParams& g, Mid& m) const {
  g.uniqueRows = 1;
  const int lo[3] = {0, -g.org[1], -g.org[2]}, hi[3] = {0, g.N[1] - g.org[1], g.N[2] - g.org[2]};
  constant_rows(lo, hi, g.value, m);
}

void Plan::mirror_rows(GatherParams& g, Mid& m) const {
  // the strided passes read the mirror copies with 32-bit byte offsets from the plane: the z pencil's span, the
  // whole spectrum, must fit them (otherwise every row is transformed and read as written)
  if ((ncpx() + 16) * sizeof(float2) > 0xffffffffull) return;
  g.uniqueRows = 1;
  // unique rows: FFT positions [-org, -org + N) per axis, inside the grid
  m.zf.plane0 = -g.org[1];
  m.zf.nplanes = g.N[1];
  m.zf.mirM = -g.org[2];
  m.zf.mirN = g.N[2];
  m.y.mirM = -g.org[1];
  m.y.mirN = g.N[1];
  for (int k = 0; k < 2; ++k) {
    m.pl.mir[k] = -g.org[k + 1];
    m.pl.mirN[k] = g.N[k + 1];
  }
}

// geometry of a launch whose kernel execution is timed under category c (untimed without a timer, or when c is off)
template <typename G>
static G timed(Timer* t, G g, int c) {
  if (t) t->kernel(c, &g.evStart, &g.evStop);
  return g;
}

void Plan::mid_forward(const Mid& m, float2* S, hipStream_t s, Timer* t) const {
  if (planar) {
    if (t) t->zForward += t->views;
    return;
  }
  sz(timed(t, m.zf, PASS_Z_FWD), 0, S, S, nullptr, 1.f, twZ, s);
}

void Plan::mid_rest(const Mid& m, const float2* in, float2* out, const float2* spec, hipStream_t s, Timer* t) const {
  if (planar) {
    PlaneGeom g = m.pl;
    if (t) {
      const int passes[3] = {PASS_Y_CONV, PASS_Z_INV, PASS_Z_FWD}, times[3] = {t->views, t->views, t->zForward};
      t->kernel(passes, times, 3, &g.evStart, &g.evStop);
      t->zForward = 0;
    }
    launch_plane(g, in, out, spec, twY, twZ, s);
    return;
  }
  sy(timed(t, m.y, PASS_Y_CONV), 2, in, out, spec, 1.f, twY, s);
  sz(timed(t, m.zi, PASS_Z_INV), 1, out, out, nullptr, 1.f, twZ, s);
}

void Plan::kernel_planes(float2* spec, int n, size_t stride, hipStream_t s) const {
  PlaneGeom g = mid().pl;
  g.nb = n;
  g.kStride = stride;
  g.kin = g.specOut = spec;
  g.kScale = inv_scale();
  g.kK[0] = K[1];
  g.kK[1] = K[2];
  launch_plane(g, nullptr, nullptr, nullptr, twY, twZ, s);
}

GatherParams Plan::kernel_gather(const float* dKernel) const {
  GatherParams g{};
  g.src = dKernel;
  for (int d = 0; d < 3; ++d) { g.N[d] = K[d]; g.org[d] = 0; }
  g.mode = GATHER_KERNEL;
  g.uniqueRows = 1;  // the passes after it take zeros for the other rows
  return g;
}

int Plan::kernel_spectrum(const float* dKernel, float2* spec, hipStream_t s) const {
  xf(dom, kernel_gather(dKernel), spec, twM, wr, s);
  if (planar) {
    kernel_planes(spec, 1, ncpx(), s);
  } else {
    Mid m = mid();
    m.y.plane0 = dom.P[2] - K[2] / 2;  // the kernel's z planes, around 0
    m.y.planeMod = dom.P[2];
    m.y.nplanes = K[2];
    m.y.wrapN = K[1];
    m.zf.wrapN = K[2];
    sy(m.y, 0, spec, spec, nullptr, 1.f, twY, s);
    sz(m.zf, 3, spec, spec, nullptr, inv_scale(), twZ, s);
  }
  MVR_HIP(hipGetLastError());
  return 0;
}

Plan::Mid Plan::convolve_geometry(GatherParams& g) const {
  // the store reads the output rows only
  const int zero[3] = {0, 0, 0};
  Mid m = mid();
  restrict_rows(zero, zero, m);
  if (g.mode == GATHER_MIRROR)
    mirror_rows(g, m);
  else if (g.mode == GATHER_VALUE)
    value_rows(g, m);
  return m;
}

int Plan::convolve(const GatherParams& g, const float2* spec, float2* work, float* out, hipStream_t s) const {
  GatherParams gg = g;
  const Mid m = convolve_geometry(gg);
  xf(dom, gg, work, twM, wr, s);
  mid_forward(m, work, s);
  mid_rest(m, work, work, spec, s);
  StoreParams st{out};
  xs(dom, st, work, twM, wr, s);
  MVR_HIP(hipGetLastError());
  return 0;
}

int Plan::convolve_once(const float* dKernel, const GatherParams& g, float2* spec, float2* work, float* out,
                        hipStream_t s) const {
  if (!planar) return kernel_spectrum(dKernel, spec, s) || convolve(g, spec, work, out, s) ? -1 : 0;
  GatherParams gg = g;
  Mid m = convolve_geometry(gg);
  const XFwdGroup groups[2] = {{kernel_gather(dKernel), spec, 1, 0, 0}, {gg, work, 1, 0, 0}};
  xfg(dom, groups, 2, twM, wr, s);
  m.pl.kin = spec;
  m.pl.specOut = dom.P[1] <= kPlanePairMax && dom.P[2] <= kPlanePairMax ? nullptr : spec;
  m.pl.kScale = inv_scale();
  m.pl.kK[0] = K[1];
  m.pl.kK[1] = K[2];
  launch_plane(m.pl, work, work, nullptr, twY, twZ, s);
  StoreParams st{out};
  xs(dom, st, work, twM, wr, s);
  MVR_HIP(hipGetLastError());
  return 0;
}

// ------------------------------------------------------------------ timers
void Timer::grow() {
  if (used + 2 <= ev.size()) return;
  const size_t old = ev.size();
  ev.resize(old + 256);
  for (size_t i = old; i < ev.size(); ++i) (void)hipEventCreate(&ev[i]);
}
void Timer::begin(hipStream_t s, int c) {
  pending = false;
  if (!on || !((mask >> c) & 1u)) return;
  for (int i = 0; i < views; ++i)
    if (seen[c]++ % every == 0) {
      shots.push_back({used, c, 1.0 / views});
      pending = true;
    }
  if (!pending) return;
  grow();
  (void)hipEventRecord(ev[used], s);
}
void Timer::kernel(const int* c, const int* times, int n, hipEvent_t* start, hipEvent_t* stop) {
  *start = *stop = nullptr;
  if (!on) return;
  const size_t before = shots.size();
  int all = 0;
  for (int i = 0; i < n; ++i) all += times[i];
  for (int i = 0; i < n; ++i)
    for (int j = 0; j < times[i]; ++j)
      if (((mask >> c[i]) & 1u) && seen[c[i]]++ % every == 0) shots.push_back({used, c[i], 1.0 / all});
  if (shots.size() == before) return;
  grow();
  *start = ev[used];
  *stop = ev[used + 1];
  used += 2;
}
void Timer::end(hipStream_t s) {
  if (!pending) return;
  (void)hipEventRecord(ev[used + 1], s);
  used += 2;
  pending = false;
}
void Timer::reset(unsigned m, int e) {
  mask = m;
  on = m != 0;
  every = e < 1 ? 1 : e;
  for (int c = 0; c < PASS_COUNT; ++c) { ms[c] = 0; cnt[c] = 0; seen[c] = 0; }
}
int Timer::collect(double* outMs, long long* outN) {
  if (used > 0) {
    (void)hipEventSynchronize(ev[used - 1]);
    for (const Shot& s : shots) {
      float t = 0.f;
      (void)hipEventElapsedTime(&t, ev[s.ev], ev[s.ev + 1]);
      ms[s.cat] += t * s.share;
      cnt[s.cat] += 1;
    }
    used = 0;
    shots.clear();
  }
  for (int c = 0; c < PASS_COUNT; ++c) {
    if (outMs) outMs[c] = ms[c];
    if (outN) outN[c] = cnt[c];
  }
  return 0;
}
void Timer::release() {
  for (auto& e : ev) (void)hipEventDestroy(e);
  ev.clear();
  shots.clear();
  used = 0;
}

}  // namespace mvr
