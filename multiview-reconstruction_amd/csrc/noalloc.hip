// noalloc.hip -- mvr_fft_convolve_noalloc: one FFT convolution (util.FFTConvolution semantics, as
// mvr_fft_convolve) that allocates no device memory.
//
// The kernel spectrum and the work spectrum live in `scratch`, a static device array of MVR_NOALLOC_SCRATCH_BYTES
// that every GPU the library runs on holds until the process ends; the twiddle tables are the library's own.  In
// host code the array's name is only a stand-in for the symbol: its device address is looked up once per device
// (hipGetSymbolAddress with that device current) and that address is what the kernels receive.  Nothing in the
// array has to start at zero: the forward x pass writes the rows that hold source or kernel values, and the passes
// after it read those only (mirror copies from their sources, constants and zeros without a read), apart from the
// row pitch's padding columns, whose results are not stored.  All calls on one GPU share its array, so calls that
// overlap on one GPU race; the caller serialises them (one stream).
#include <mutex>
#include <string>

#include "../../include/mvr_hip.h"
#include "host.hpp"

static __device__ __align__(256) unsigned char scratch[MVR_NOALLOC_SCRATCH_BYTES];

namespace mvr {
namespace {

constexpr int kMaxDevices = 64;
std::mutex g_mu;
unsigned char* g_scratch[kMaxDevices] = {};  // device address of `scratch` per device, set on first use

// the device address of `scratch` on `dev` (which must be current)
int scratch_address(int dev, unsigned char** out) {
  std::lock_guard<std::mutex> lk(g_mu);
  if (!g_scratch[dev]) {
    void* p = nullptr;
    const hipError_t e = hipGetSymbolAddress(&p, HIP_SYMBOL(scratch));
    if (e != hipSuccess || p == nullptr) {
      set_error(std::string("scratch address lookup failed: ") + hipGetErrorString(e));
      return -1;
    }
    g_scratch[dev] = static_cast<unsigned char*>(p);
  }
  *out = g_scratch[dev];
  return 0;
}

constexpr size_t align256(size_t b) { return (b + 255) / 256 * 256; }

}  // namespace
}  // namespace mvr

using namespace mvr;

extern "C" int mvr_fft_convolve_noalloc(int dev, const float* img, const int n[3], int ext, float extValue,
                                        const float* kernel, const int k[3], float* out, void* stream) {
  if (!img || !kernel || !out || !n || !k) { set_error("null argument"); return -1; }
  if (ext != MVR_EXT_MIRROR_SINGLE && ext != MVR_EXT_VALUE) { set_error("unknown extension"); return -1; }
  if (dev < 0 || dev >= kMaxDevices) { set_error("bad device"); return -1; }
  // geometry and the scratch layout first, on the host: sizes beyond the array are refused before device work
  Plan plan;
  if (plan.create_geometry(n, k)) return -1;
  // (the limit counts four twiddle tables with the two spectra, as it did when the array held them: callers choose
  // this entry point or mvr_fft_convolve by what it refuses)
  const size_t oWork = align256(plan.ncpx() * 8);
  const size_t tables = align256((size_t)plan.M * 8) + align256((size_t)(plan.M + 1) * 8) +
                        align256((size_t)plan.dom.P[1] * 8) + align256((size_t)plan.dom.P[2] * 8);
  const size_t total = tables + 2 * oWork;
  if (total > (size_t)MVR_NOALLOC_SCRATCH_BYTES) {
    set_error("mvr_fft_convolve_noalloc: the FFT grid " + std::to_string(plan.dom.P[0]) + "x" +
              std::to_string(plan.dom.P[1]) + "x" + std::to_string(plan.dom.P[2]) + " needs " +
              std::to_string(total) + " bytes of scratch, more than the " +
              std::to_string((long long)MVR_NOALLOC_SCRATCH_BYTES) + " available (use mvr_fft_convolve)");
    return -1;
  }
  MVR_HIP(hipSetDevice(dev));
  if (!device_memory_of(img, dev, true) || !device_memory_of(kernel, dev, true) || !device_memory_of(out, dev, true)) {
    set_error("mvr_fft_convolve_noalloc: img, kernel and out must be device memory of the given device");
    return -1;
  }
  unsigned char* base = nullptr;
  if (scratch_address(dev, &base)) return -1;
  hipStream_t s = static_cast<hipStream_t>(stream);
  if (plan.create(n, k)) return -1;  // finds the twiddle tables, static too
  float2* spec = reinterpret_cast<float2*>(base);
  float2* work = reinterpret_cast<float2*>(base + oWork);
  GatherParams g{};
  g.src = img;
  for (int d = 0; d < 3; ++d) { g.N[d] = n[d]; g.org[d] = -plan.dom.m[d]; }
  g.mode = ext == MVR_EXT_MIRROR_SINGLE ? GATHER_MIRROR : GATHER_VALUE;
  g.value = extValue;
  return plan.convolve_once(kernel, g, spec, work, out, s);
}
