// engine.hpp -- shared declarations of the HIP deconvolution engine.
//
// Geometry of one convolution plan ("domain"):
//   * the output region is D[0] x D[1] x D[2] voxels of a source volume,
//     starting at volume coordinate o;
//   * the FFT grid is P[0] x P[1] x P[2] (P[d] >= D[d] + K[d] - 1); FFT
//     position p corresponds to volume coordinate o + p - m, m[d] = K[d]-1-K[d]/2
//     (the left reach of the kernel), so the output region is p in [m, m + D);
//   * the half spectrum is stored [z][y][hx], hx < P[0]/2 + 1, with row pitch HxP; small grids (Plan::planar)
//     store it [hx][z][y].
// A linear convolution evaluated this way is exact on the output region for
// any extension of the input outside it (util/FFTConvolution.java:508-543 pads
// to at least N + K - 1 for the same reason).
#pragma once
#include <hip/hip_runtime.h>
#include <cstddef>
#include <cstdint>

namespace mvr {

struct Dom {
  int P[3];
  int HxP;
  int D[3];
  int m[3];
  // Batched blocks: when btab is set, one launch runs nb blocks that share P, HxP and m.  Entry b of btab
  // (device memory, 6 ints) is {o[3], D[3]}: the volume coordinate of the block's output region and its size
  // (at most D above); the block's spectrum starts at b * blockStride complex values.  The launchers set
  // wgPerBlock (work-groups per block of an x pass).
  const int* btab = nullptr;
  int nb = 1;
  int wgPerBlock = 0;
  size_t blockStride = 0;
};
constexpr int kBlockTabInts = 6;

enum GatherMode : int { GATHER_MIRROR = 0, GATHER_VALUE = 1, GATHER_KERNEL = 2 };

// Source of the forward transform: value at FFT position p is
//   MIRROR: src[mirror(org + p)]                (extendMirrorSingle)
//   VALUE : src[org + p] inside the volume, `value` outside (extendValue / extendZero)
//   KERNEL: K[(p + K/2) mod P] if < K, else 0    (kernel centre moved to the origin)
struct GatherParams {
  const float* src;
  int N[3];
  int org[3];
  int mode;
  float value;
  // transform only the rows (y, z) that hold source values, FFT positions [-org, -org + N) per axis (KERNEL: the
  // kernel's rows); the passes after it read mirror copies from their sources and put constant rows in
  int uniqueRows;
};

// One group of forward x transforms with planar spectra: n sources, srcStride values apart, into spectra dstStride
// complex values apart.
struct XFwdGroup {
  GatherParams g;
  float2* S;
  int n;
  size_t srcStride, dstStride;
};

// Inverse-transform epilogues.  `o` is the volume coordinate of the output
// region's first voxel; N are the dims of the volume that img/psi/w index.
// The quotient is formed on the output region widened by qlo / qhi voxels per side (the reach of the second
// kernel, for domains whose neighbourhood lies inside the volume: blocks), within the volume; 1 elsewhere.
// skipOnes: rows outside the quotient region (a row of ones, whose x spectrum is P0 at frequency 0 and 0
// elsewhere) are not written; the z pass that reads the result puts them in itself (StridedGeom ones*), and
// the work-groups are dealt over the quotient rows only: grid rows (y, z) in [rowLo, rowLo + rowN) per axis
// (k = 1, 2), which are exactly the rows the quotient region selects.  For batched blocks (planar spectra only) each
// block's rows are formed from its entry in the block table, and rowN are the most rows of any block.
// Batched views: n > 0 of them, the data of view b at at[b] values from the first's.  (Offsets, so that the compiler knows
// global memory, and a kernel argument of its own: a struct that is indexed stays in memory with all its members, whose
// loads then wait one by one; 2 % of a y pass.)
constexpr int kViewBatch = 8;  // the most views of one launch
struct ViewOffsets {
  int n = 0;
  bool inShared = false;  // all read the same input
  long long at[kViewBatch];
};

struct RatioPass {
  const float* img;
  int N[3];
  int o[3];
  int qlo[3];
  int qhi[3];
  int skipOnes;
  int rowLo[3], rowN[3];
};
struct RatioParams : RatioPass {
  ViewOffsets views;  // of their images; their spectra lie Dom::blockStride apart
};

struct UpdateParams {
  float* psi;
  const float* w;
  int N[3];
  int o[3];
  double lambda;
  float minValue;
  float maxI;
  double2* partial;  // per work-group {sum change, max change}
};

struct StoreParams {
  float* out;        // compact D[0]*D[1]*D[2] array
  int n = 1;         // n > 1: as many spectra, Dom::blockStride apart, into arrays of D[0]*D[1]*D[2] back to back
};

typedef void (*XFwdFn)(const Dom&, const GatherParams&, float2* S, const float2* twM, const float2* wr,
                       hipStream_t s);
// ngroups <= 2 groups in one launch (planar spectra)
typedef void (*XFwdGroupsFn)(const Dom&, const XFwdGroup* groups, int ngroups, const float2* twM, const float2* wr,
                             hipStream_t s);
typedef void (*XRatioFn)(const Dom&, const RatioParams&, const float2* Sin, float2* Sout, const float2* twM,
                         const float2* wr, hipStream_t s);
typedef int (*XUpdateFn)(const Dom&, const UpdateParams&, const float2* S, const float2* twM, const float2* wr,
                         hipStream_t s);  // returns #work-groups (= #partials)
typedef void (*XStoreFn)(const Dom&, const StoreParams&, const float2* S, const float2* twM, const float2* wr,
                         hipStream_t s);
// strided passes: y (plane = z) or z (plane = y)
struct StridedPass {
  size_t planeStride;  // complex elements between consecutive planes
  size_t lineStride;   // complex elements between consecutive pencil elements
  int ncols;           // valid columns (hx) per line
  int nplanes;
  int width = 0;       // tile width in columns (8 or 16; 0 = the default for the length)
  // batched blocks: planes [b * blockPlanes, (b + 1) * blockPlanes) belong to block b, whose data starts at
  // b * blockStride; the kernel spectrum is shared (indexed by the plane within the block).  0 = one block.
  int blockPlanes = 0;
  size_t blockStride = 0;
  // Only what the next pass reads: planes [plane0, plane0 + nplanes) (per block) are transformed, and the inverse
  // modes (1, 2) store only the pencil positions [storeLo, storeHi).  The defaults cover the whole grid.
  int plane0 = 0;
  int storeLo = 0, storeHi = 1 << 30;
  // Forward mode over data whose rows outside planes [onesPlaneLo, onesPlaneHi) x positions [onesLo, onesHi) are
  // spectra of constant rows (or planes), never written: the pass reads none of them and uses onesDC at column 0,
  // 0 at the other columns; with onesDCPlane >= 0 onesDC is on that plane only, 0 on the others.  Off unless ones.
  bool ones = false;
  float onesDC = 0.f;
  int onesPlaneLo = 0, onesPlaneHi = 0, onesLo = 0, onesHi = 0, onesDCPlane = -1;
  // Forward modes over data that is a mirror extension along the pencil (mirN > 0): position n holds what
  // position mirM + mirror(n - mirM, mirN) holds, and only those positions were written; the loads read them
  // (byte offsets from the plane up to L lineStride 8 must fit 32 bits).
  int mirM = 0, mirN = 0;
  // Forward modes 0 and 3 over a kernel placed around the origin (wrapN > 0): only the positions n with (n + wrapN / 2)
  // mod L < wrapN were written, the others are zero and not read.  planeMod > 0: planes are counted from plane0 modulo
  // planeMod.
  int wrapN = 0, planeMod = 0;
  // timing: when set, the launch records the kernel's own start and stop in these events
  hipEvent_t evStart = nullptr, evStop = nullptr;
};
struct StridedGeom : StridedPass {
  ViewOffsets views;  // batched views, as blocks: of their kernel spectra
};
// mode: 0 forward, 1 inverse, 2 forward * spec * inverse (spec layout = data layout),
// 3 forward then scale
typedef void (*StridedFn)(const StridedGeom&, int mode, const float2* in, float2* out, const float2* spec,
                          float scale, const float2* tw, hipStream_t s);

// One pass of y and z transforms over planar spectra [hx][z][y] (plane.hip), in place or not: forward, times spec
// ([hx][y slot][z slot]), inverse.  With a kernel (kin) its x transform is first turned into that spectrum, scaled, in
// specOut (which may be kin), to be used as spec or, without data (in null), on its own; or, for planes of at most
// kPlanePairMax, with specOut null, used and dropped.
struct PlaneGeom {
  int Py, Pz;          // at most kPlaneMax each
  int ncols;           // planes (hx)
  int nb = 1;          // batch entries: entry b reads in + inIdx[b] inStride (null: b) and spec + specIdx[b] specStride
  size_t inStride = 0, outStride = 0, specStride = 0;   // (null: the shared spectrum), writes out + b outStride
  const int* inIdx = nullptr;
  const int* specIdx = nullptr;
  const float2* kin = nullptr;             // entry b: kin + b kStride, specOut + b kStride
  float2* specOut = nullptr;
  size_t kStride = 0;
  float kScale = 1.f;
  int kK[2] = {0, 0};                      // kernel sizes along y, z: only its rows were written (StridedGeom's wrapN)
  int mir[2] = {0, 0}, mirN[2] = {0, 0};   // mirror extension along y, z (StridedGeom's mirM, mirN), off at 0
  bool ones = false;                       // rows outside [onesLo, onesHi) (y, z) are constant, as in StridedGeom
  float onesDC = 0.f;
  int onesLo[2] = {0, 0}, onesHi[2] = {0, 0};
  const int* onesTab = nullptr;            // per batch entry {yLo, yHi, zLo, zHi} instead
  int lo[2] = {0, 0}, hi[2] = {1 << 30, 1 << 30};  // rows (y, z) stored
  hipEvent_t evStart = nullptr, evStop = nullptr;
  ViewOffsets views;                       // batched views: entry b takes spec + views.at[b] instead
};
constexpr int kPlaneMax = 128;     // y and z lengths
// the largest for iterations on one grid at a time: 5 view updates with strided passes and planar take, at 96^3 points, 528
// and 508 us, at 120^3 626 and 646, at 128^3 681 and 695.  The rules look at y and z alone, though a launch has a plane per
// x frequency, at most P0 / 2 + 1 of them.  8 view updates, us, strided and planar, at P0 points along x:
//   64 x 64 points (y, z): P0 = 16 362 and 328, 32 387 and 355, 64 399 and 376, 128 459 and 438, 256 529 and 494
//   96 x 96:               16 398 and 412, 32 445 and 434, 48 452 and 455, 64 473 and 464, 128 578 and 556, 256 773 and 708
// One convolution, as far as kPlaneMax: 96 x 96 30.5 and 22.1 at P0 = 16, 36.0 and 24.8 at 64; 128 x 128 33.6 and 36.8 at
// 16, 37.0 and 39.1 at 32, 44.2 and 42.2 at 64, 57.4 and 49.6 at 128.  So nine planes of 96 x 96 (batches of views and
// blocks multiply the planes) and up to 17 of 128 x 128 would be 3-9 % faster with strided passes.
constexpr int kPlaneMaxSingle = 96;
constexpr int kPlanePairMax = 96;  // the largest for a kernel's and the data's plane in the LDS together
constexpr int kPlanarMaxM = 128;   // x passes with planar spectra are compiled for half lengths up to this
void launch_plane(const PlaneGeom& g, const float2* in, float2* out, const float2* spec, const float2* twY,
                   const float2* twZ, hipStream_t s);

// planar: spectra [hx][z][y] instead of rows [z][y][hx]
XFwdFn get_x_fwd(int M, bool planar);
XFwdGroupsFn get_x_fwd_groups(int M);
XRatioFn get_x_ratio(int M, bool planar);
XUpdateFn get_x_update(int M, bool planar);
XStoreFn get_x_store(int M, bool planar);
StridedFn get_strided(int L);
// the largest pencil position a lane of the length-L strided pass addresses with its 32-bit offset, plus one
int get_strided_span(int L);
// lengths with compiled kernels, ascending; terminated by 0
const int* strided_lengths();
const int* half_lengths();
// exp(-2 pi i k / n), k < n, for every length of the two lists, in the current device's memory (null: no such length, or
// the device failed)
const float2* twiddle_table(int n);

// misc kernels (misc.hip)
void launch_fill(float* dst, size_t n, float v, hipStream_t s);
void launch_reduce_stats(const double2* partial, int n, double2* out, hipStream_t s);
// nUpdates <= 32 reductions in one launch: update v's partials at partial + v * stride, counts[v] of them
void launch_reduce_stats_batched(const double2* partial, size_t stride, const int* counts, int nUpdates, double2* out,
                                 hipStream_t s);
int launch_psi_init_partials(const float* const* imgs, int V, size_t n, double* psum, unsigned long long* pcount,
                             float* pmax, hipStream_t s);  // returns #partials
void launch_update_mul(float* psi, const float* const* T2, const float* const* w, int V, size_t n, double lambda,
                       float minValue, float maxI, double2* partial, int* nPartialOut, hipStream_t s);
void launch_copy_block_zero(const float* src, const int N[3], const long long off[3], float* dst, const int B[3],
                            hipStream_t s);
void launch_blocks_with_content(const float* w, const int N[3], const int* tab, int nblocks, int* flags,
                                hipStream_t s);
void launch_quotient(const float* img, float* blurred, size_t n, hipStream_t s);
int launch_final_values(float* psi, const float* integral, const float* weight, size_t n, double lambda,
                        float minValue, float maxI, double2* partial, int maxPartials, hipStream_t s);
// The kernels of the second kernels' products, arrays of dims K: of V given ones those as given of the views 1.., those
// divided by sums[v] of the views 0.., the same mirrored, and those as given mirrored.
void launch_psf_kernels(const float* given, const double* sums, int V, const int K[3], float* out, hipStream_t s);
// out[v] = factors[v][nf - 1] * ... * factors[v][0] * first[v], multiplied in the order of the factors, arrays of nk
void launch_psf_products(const float* first, const float* factors, int V, int nf, size_t nk, float* out, hipStream_t s);
void launch_rel_l2(const float* a, const float* b, size_t n, double2* partial, double2* out, hipStream_t s);
int launch_psi_approx_slice(const float* img, const int N[3], double2* partial, hipStream_t s);
void launch_fused_nonzero(const float* const* imgs, const float* const* ws, int V, size_t n, float* out,
                          hipStream_t s);
void launch_sym_conv_axis(const float* in, float* out, const int N[3], int axis, const double* half, int H,
                          hipStream_t s);

}  // namespace mvr
