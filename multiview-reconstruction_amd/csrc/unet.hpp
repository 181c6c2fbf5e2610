// unet.hpp -- argument blocks and host declarations of the U-Net kernels.
#pragma once
#include <hip/hip_runtime.h>

#include <cstddef>
#include <cstdint>

namespace mvr {

// output head of an inference: psi[v] = max(minValue, scale * (avg[v] + sum_c w[c] d1[v][c] + w[16]))
struct PsiArgs {
  float* out;            // psi, dims (ox, oy, oz), or null
  const float* w;        // 16 weights and the bias
  const float* avg;      // normalised average channel [D][H][W]
  float scale, minValue;
  int ox, oy, oz;        // output volume dims, <= net dims; psi holds planes [zlo, oz) of them
  int zlo;
};

struct ConvArgs {
  const uint16_t* in;  // [n][z][y][x][in_cs], channels [0, cin)
  int in_cs;
  int cin;             // multiple of 16
  int in_half;         // 1: a one-chunk input whose channels 8..15 are zero and not stored (in_cs a multiple of 8)
  const uint16_t* w;   // [taps][cout][cin]
  const float* bias;   // [cout] or null
  uint16_t* out;       // [n][z][y][x][out_cs], channels [out_co, out_co + cout)
  int out_cs, out_co;
  int cout;            // multiple of 16
  int N, D, H, W;
  int taps;            // 27 (3^3, zero padding 1)
  int relu;
  // optional fused nearest x2 upsampling: input channels [0, up_c) are read from up_in (channel stride
  // up_cs) at half the coordinates, channels [up_c, cin) from in (its channel 0 = input channel up_c)
  const uint16_t* up_in;
  int up_cs, up_c;
  // optional fused 2x2x2 average pooling of the stored (bf16) output into pool_out [n][D/2][H/2][W/2][pool_cs],
  // channels [0, cout): done where conv_fuses_pool(args) holds, else left to the caller
  uint16_t* pool_out;
  int pool_cs;
  // optional ReLU of a backward pass: the activations [n][z][y][x][mask_cs], channels [0, cout), behind the output; cin and
  // cout 16, 32 or 64 alike
  const uint16_t* mask;
  int mask_cs;
  PsiArgs psi;           // optional fused output head (psi.out set; 16 -> 16 channels, one sample): out is not written
};

struct WgradArgs {
  const uint16_t* in;    // forward input of the layer
  int in_cs, cin;
  const uint16_t* dout;  // gradient of the layer output (after the ReLU mask)
  int dout_cs, dout_co, cout;
  int N, D, H, W;
  float* partial;        // [parts][27][cout][cin]
  float* bias_partial;   // [parts][cout]
};

// views the network takes: V view channels + their weighted mean fit the 16 input channels; the input
// packer holds up to 8 view pointers
constexpr int kNetMaxViews = 8;

struct InputArgs {
  const float* img[kNetMaxViews];
  const float* w[kNetMaxViews];
  int V;
  int N3[3];             // dims of the source volumes (x, y, z)
  int x0, y0, z0;        // origin of the sample region
  int W, H, D;           // sample region
  float inv_scale;
  uint16_t* out;         // [D][H][W][out_cs], out_cs 16 or (V < 8) 8
  int out_cs;
  float* avg_out;        // [D][H][W] (normalised average channel) or null
};

// output head of a training step
struct HeadArgs {
  const uint16_t* d1;    // [nvox][d1_cs], 16 channels
  int d1_cs;
  const float* wo;       // 16
  const float* bias;     // 1
  const float* avg;      // normalised average channel
  const float* target;   // normalised target
  float* dr;             // gradient of r
  double* loss_partial;  // per work-group sum of squared errors
  size_t nvox;
};

// one tensor of an Adam step
struct AdamTensor {
  float* w;
  float* m;
  float* v;
  const float* grad;
  uint16_t* wbf;   // bf16 copy [taps][cout][cin] or null
  uint16_t* wt;    // flipped transpose [taps][cin][cout] or null
  unsigned count, first;   // elements; its first work-group (set by the launch)
  int taps, cout, cin;
};
constexpr int kAdamTensors = 24;
struct AdamArgs {
  AdamTensor t[kAdamTensors];
  int n;
  float lr, beta1, beta2, eps, c1, c2;  // c1 = 1/(1-beta1^t), c2 = 1/(1-beta2^t)
};

// patches of P^3 voxels of training volumes as network input and target, up to kPatches in a launch
constexpr int kPatches = 8;
struct PatchArgs {
  struct Patch {
    const float* img[kNetMaxViews];
    const float* w[kNetMaxViews];
    const float* target;
    int N3[3], o[3];     // dims of the volume, origin of the patch (inside it)
    float inv_scale;
  } p[kPatches];
  int V, P;
  uint16_t* out;         // of the first patch: [P][P][P][16]
  float* avg_out;        // [P][P][P]
  float* target_out;
};

// 3^3 convolution (unet_conv.hip); false when the shape is not one it covers, nothing launched
bool launch_conv_tiled(const ConvArgs& a, hipStream_t s);
bool conv_fuses_pool(const ConvArgs& a);  // the launch also writes the pooled output (pool_out set, even dimensions)
// weight and bias gradient partials of a 3^3 layer (cin and cout multiples of 16); returns how many partitions
// (at most maxParts) it wrote
int launch_conv_wgrad(const WgradArgs& a, int maxParts, hipStream_t s);
// the most partitions launch_conv_wgrad takes for a layer: enough work-groups for two to six per CU over all of the
// layer's channel blocks
inline int wgrad_max_parts(int cin, int cout, int maxParts) {
  const int p = 1536 / ((cin / 16) * (cout % 32 == 0 ? cout / 32 : cout / 16));
  return p < maxParts ? p : maxParts;
}
// grad[j] = sum_p partial[p][j], j < count; with bcount > 0 (at most 64) also bgrad from bpartial
void launch_sum_partials(const float* partial, int nparts, size_t count, float* grad, const float* bpartial,
                         int bcount, float* bgrad, hipStream_t s);
void launch_pool_fwd(const uint16_t* in, int ics, int ico, uint16_t* out, int ocs, int C, int N, int D, int H, int W,
                     hipStream_t s);
void launch_pool_bwd(const uint16_t* dout, int ocs, uint16_t* din, int ics, int ico, int C, int N, int D, int H, int W,
                     const uint16_t* post, hipStream_t s);
void launch_up_fwd(const uint16_t* in, int ics, uint16_t* out, int ocs, int oco, int C, int N, int D, int H, int W,
                   hipStream_t s);
void launch_up_bwd(const uint16_t* dfine, int fcs, int fco, uint16_t* dcoarse, int ccs, int C, int N, int D, int H,
                   int W, const uint16_t* post, hipStream_t s);
void launch_pack_patches(const PatchArgs& a, int n, hipStream_t s);
void launch_pack_input(const InputArgs& a, hipStream_t s);
int launch_head(const HeadArgs& a, hipStream_t s);
int launch_head_bwd(const HeadArgs& a, uint16_t* dd1, float* partial, hipStream_t s);
void launch_adam(const AdamArgs& a, hipStream_t s);
int launch_wsum_partials(const InputArgs& a, size_t n, double2* partial, hipStream_t s);

}  // namespace mvr
