// unet.cpp -- host side of the learned initial estimate (U-Net training and inference).
#include "unet_host.hpp"

#include <algorithm>
#include <cmath>
#include <cstring>
#include <random>

namespace mvr {

#define UCHECK(cond, msg) \
  do {                    \
    if (!(cond)) {        \
      set_error(msg);     \
      return -1;          \
    }                     \
  } while (0)

// layer table: input channels (padded), output channels, taps
static const int kCin[kLayers] = {16, 16, 16, 32, 32, 64, 96, 32, 48, 16};
static const int kCout[kLayers] = {16, 16, 32, 32, 64, 64, 32, 32, 16, 16};

size_t UNet::wcount(int l) const { return (size_t)27 * kCout[l] * kCin[l]; }

int UNet::create(int dev_, int V_, unsigned long long seed) {
  dev = dev_;
  UCHECK(V_ >= 1 && V_ <= kNetMaxViews, "the network takes 1..8 views");
  V = V_;
  MVR_HIP(hipSetDevice(dev));
  MVR_HIP(hipStreamCreateWithFlags(&stream, hipStreamNonBlocking));
  // master weights, moments and gradients, each in the order of copy_params
  for (int l = 0; l < kLayers; ++l) {
    layer[l].count = wcount(l);
    bias[l].count = kCout[l];
  }
  head.count = 17;  // 16 weights + bias
  const size_t section = (param_count() + 63) / 64 * 64;
  MVR_HIP(hipMalloc(&params, 4 * section * 4));
  MVR_HIP(hipMemset(params, 0, 4 * section * 4));
  size_t at = 0;
  auto place = [&](Param& p, bool conv) -> int {
    p.w = params + at;
    p.m = p.w + section;
    p.v = p.m + section;
    p.g = p.v + section;
    at += p.count;
    if (conv) {
      MVR_HIP(hipMalloc(&p.wbf, p.count * 2));
      MVR_HIP(hipMalloc(&p.wt, p.count * 2));
    }
    return 0;
  };
  for (int l = 0; l < kLayers; ++l)
    if (place(layer[l], true) || place(bias[l], false)) return -1;
  if (place(head, false)) return -1;
  std::mt19937_64 rng(seed);
  for (int l = 0; l < kLayers; ++l) {
    Param& p = layer[l];
    std::vector<float> h(p.count, 0.f);
    const int fanin = 27 * (l == 0 ? (V + 1) : kCin[l]);
    std::normal_distribution<float> nd(0.f, std::sqrt(2.f / (float)fanin));
    for (int t = 0; t < 27; ++t)
      for (int co = 0; co < kCout[l]; ++co)
        for (int ci = 0; ci < kCin[l]; ++ci) {
          const bool real = l != 0 || ci < V + 1;
          h[((size_t)t * kCout[l] + co) * kCin[l] + ci] = real ? nd(rng) : 0.f;
        }
    MVR_HIP(hipMemcpy(p.w, h.data(), p.count * 4, hipMemcpyHostToDevice));
  }
  {
    std::vector<float> h(17, 0.f);
    std::normal_distribution<float> nd(0.f, 0.01f);
    for (int c = 0; c < 16; ++c) h[c] = nd(rng);
    MVR_HIP(hipMemcpy(head.w, h.data(), 17 * 4, hipMemcpyHostToDevice));
  }
  return refresh_copies();
}

// a parameter tensor (of layer l, or -1: without compute copies) of an Adam step
void UNet::add_tensor(AdamArgs& a, const Param& p, int l) {
  static_assert(2 * kLayers + 1 <= kAdamTensors, "every tensor in one launch");
  AdamTensor& t = a.t[a.n++];
  t.w = p.w; t.m = p.m; t.v = p.v; t.grad = p.g; t.wbf = p.wbf; t.wt = p.wt; t.count = (unsigned)p.count;
  t.taps = 27; t.cout = l >= 0 ? kCout[l] : 0; t.cin = l >= 0 ? kCin[l] : 0;
}

// bf16 compute copies of the FP32 masters (an Adam step with learning rate 0 does exactly that)
int UNet::refresh_copies() {
  AdamArgs a{};
  a.lr = 0.f; a.beta1 = 1.f; a.beta2 = 1.f; a.eps = 1.f; a.c1 = 0.f; a.c2 = 0.f;
  for (int l = 0; l < kLayers; ++l) add_tensor(a, layer[l], l);
  launch_adam(a, stream);
  MVR_HIP(hipGetLastError());
  MVR_HIP(hipStreamSynchronize(stream));
  return 0;
}

size_t UNet::param_count() const {
  size_t n = head.count;
  for (int l = 0; l < kLayers; ++l) n += layer[l].count + bias[l].count;
  return n;
}

int UNet::copy_params(float* hostOut, const float* hostIn, bool grads) {
  MVR_HIP(hipSetDevice(dev));
  float* p = grads ? layer[0].g : layer[0].w;
  if (hostOut) MVR_HIP(hipMemcpy(hostOut, p, param_count() * 4, hipMemcpyDeviceToHost));
  if (hostIn) MVR_HIP(hipMemcpy(p, hostIn, param_count() * 4, hipMemcpyHostToDevice));
  if (hostIn && !grads) return refresh_copies();
  return 0;
}

// ------------------------------------------------------------------ activations
int UNet::Acts::alloc(int N_, int D_, int H_, int W_, int views, bool grads) {
  N = N_; D = D_; H = H_; W = W_;
  Dcap = D_;
  // Training keeps the concatenations (the weight gradients read them) with the skip tensors behind the upsampled
  // channels; an inference reads the upsampled part from the coarse tensor, so the skip tensors stand alone, and the
  // input's channels beyond the first eight are not stored where they are all zero.
  cs1 = grads ? 48 : 16;
  cs2 = grads ? 96 : 32;
  csIn = !grads && views + 1 <= 8 ? 8 : 16;
  const size_t v0 = (size_t)N * D * H * W, v1 = v0 / 8, v2 = v0 / 64;
  struct B { uint16_t** p; uint16_t** gp; size_t n; };
  const B bufs[] = {{&x0, nullptr, v0 * csIn}, {&a1, &g_a1, v0 * 16},  {&cat1, &g_cat1, v0 * cs1},
                    {&p1, &g_p1, v1 * 16},     {&a2, &g_a2, v1 * 32},  {&cat2, &g_cat2, v1 * cs2},
                    {&p2, &g_p2, v2 * 32},     {&a3, &g_a3, v2 * 64},  {&b3, &g_b3, v2 * 64},
                    {&a4, &g_a4, v1 * 32},     {&d2, &g_d2, v1 * 32},  {&a5, &g_a5, v0 * 16},
                    {&d1, &g_d1, v0 * 16}};
  for (const B& b : bufs) {
    if (b.p == &d1 && !grads) continue;  // an inference turns the last activations into psi without storing them
    MVR_HIP(hipMalloc(b.p, b.n * 2));
    if (grads && b.gp) MVR_HIP(hipMalloc(b.gp, b.n * 2));
  }
  MVR_HIP(hipMalloc(&avg, v0 * 4));
  if (grads) {
    MVR_HIP(hipMalloc(&target, v0 * 4));
    MVR_HIP(hipMalloc(&dr, v0 * 4));
  }
  return 0;
}

void UNet::Acts::release() {
  uint16_t** all[] = {&x0, &a1, &cat1, &p1, &a2, &cat2, &p2, &a3, &b3, &a4, &d2, &a5, &d1,
                      &g_a1, &g_cat1, &g_p1, &g_a2, &g_cat2, &g_p2, &g_a3, &g_b3, &g_a4, &g_d2, &g_a5, &g_d1};
  for (auto p : all)
    if (*p) { (void)hipFree(*p); *p = nullptr; }
  for (float** p : {&avg, &target, &dr})
    if (*p) { (void)hipFree(*p); *p = nullptr; }
  N = D = H = W = Dcap = 0;
}

int UNet::ensure_acts(Acts& a, int N_, int D_, int H_, int W_, bool grads) {
  UCHECK(D_ % 4 == 0 && H_ % 4 == 0 && W_ % 4 == 0 && D_ >= 4 && H_ >= 4 && W_ >= 4,
         "network input dims must be multiples of 4");
  if (a.N == N_ && a.Dcap >= D_ && a.H == H_ && a.W == W_ && (!grads || a.g_a1)) {
    a.D = D_;  // the buffers hold Dcap planes per sample; the tensors use the first D
    return 0;
  }
  a.release();
  return a.alloc(N_, D_, H_, W_, V, grads);
}

bool UNet::conv(int l, const uint16_t* in, int in_cs, int in_co, uint16_t* out, int out_cs, int out_co, int N, int D,
                int H, int W, bool relu, const uint16_t* up, int up_cs, int up_c, uint16_t* pool, int pool_cs,
                const PsiArgs* psi) {
  ConvArgs c{};
  if (psi) c.psi = *psi;
  c.up_in = up;
  c.up_cs = up_cs;
  c.up_c = up ? up_c : 0;
  c.in = in + in_co;
  c.in_cs = in_cs;
  c.cin = kCin[l];
  c.in_half = l == 0 && in_cs == 8;
  c.w = layer[l].wbf;
  c.bias = bias[l].w;
  c.out = out;
  c.out_cs = out_cs;
  c.out_co = out_co;
  c.cout = kCout[l];
  c.N = N; c.D = D; c.H = H; c.W = W;
  c.taps = 27;
  c.relu = relu ? 1 : 0;
  c.pool_out = pool;
  c.pool_cs = pool_cs;
  const bool fused = pool && conv_fuses_pool(c);
  if (!fused) c.pool_out = nullptr;
  if (!launch_conv_tiled(c, stream)) convFailed = true;
  return fused;
}

// data gradient of layer l: din = conv(dout, flipped transposed weights), no bias
// and, with the layer's input activations `post` (strided as din), the backward ReLU below it
void UNet::dgrad(int l, const uint16_t* dout, int dout_cs, int dout_co, uint16_t* din, int din_cs, int N, int D, int H,
                 int W, const uint16_t* post) {
  ConvArgs c{};
  c.in = dout + dout_co;
  c.in_cs = dout_cs;
  c.cin = kCout[l];
  c.w = layer[l].wt;
  c.bias = nullptr;
  c.out = din;
  c.out_cs = din_cs;
  c.mask = post;
  c.mask_cs = din_cs;
  c.cout = kCin[l];
  c.N = N; c.D = D; c.H = H; c.W = W;
  c.taps = 27;
  c.relu = 0;
  if (!launch_conv_tiled(c, stream)) convFailed = true;
}

void UNet::wgrad(int l, const uint16_t* in, int in_cs, const uint16_t* dout, int dout_cs, int dout_co, int N, int D,
                 int H, int W) {
  WgradArgs a{};
  a.in = in; a.in_cs = in_cs; a.cin = kCin[l];
  a.dout = dout; a.dout_cs = dout_cs; a.dout_co = dout_co; a.cout = kCout[l];
  a.N = N; a.D = D; a.H = H; a.W = W;
  a.partial = wpart;
  a.bias_partial = bpart;
  const int nparts = launch_conv_wgrad(a, kWgradParts, stream);
  launch_sum_partials(wpart, nparts, layer[l].count, layer[l].g, bpart, kCout[l], bias[l].g, stream);
}

// ------------------------------------------------------------------ forward / backward
int UNet::forward(Acts& a, bool training, const float* psiScale, float* psiOut, const int* outDims, float minValue) {
  const int N = a.N, D0 = a.D, H0 = a.H, W0 = a.W;
  const int D1 = D0 / 2, H1 = H0 / 2, W1 = W0 / 2, D2 = D0 / 4, H2 = H0 / 4, W2 = W0 / 4;
  convFailed = false;
  // the skip tensors' channels of cat1 and cat2
  const int cs1 = a.cs1, co1 = cs1 - 16, cs2 = a.cs2, co2 = cs2 - 32;
  conv(0, a.x0, a.csIn, 0, a.a1, 16, 0, N, D0, H0, W0, true);
  // e1, pooled into p1 by the convolution where it can
  if (!conv(1, a.a1, 16, 0, a.cat1, cs1, co1, N, D0, H0, W0, true, nullptr, 0, 0, a.p1, 16))
    launch_pool_fwd(a.cat1, cs1, co1, a.p1, 16, 16, N, D1, H1, W1, stream);
  conv(2, a.p1, 16, 0, a.a2, 32, 0, N, D1, H1, W1, true);
  // e2, pooled into p2
  if (!conv(3, a.a2, 32, 0, a.cat2, cs2, co2, N, D1, H1, W1, true, nullptr, 0, 0, a.p2, 32))
    launch_pool_fwd(a.cat2, cs2, co2, a.p2, 32, 32, N, D2, H2, W2, stream);
  conv(4, a.p2, 32, 0, a.a3, 64, 0, N, D2, H2, W2, true);
  conv(5, a.a3, 64, 0, a.b3, 64, 0, N, D2, H2, W2, true);
  // decoder: training materialises the concatenations (the weight gradients read them); inference
  // reads the upsampled part straight from the coarse tensor inside the convolution's staging
  if (training) {
    launch_up_fwd(a.b3, 64, a.cat2, 96, 0, 64, N, D2, H2, W2, stream);      // up(b3) -> cat2[0:64)
    conv(6, a.cat2, 96, 0, a.a4, 32, 0, N, D1, H1, W1, true);
  } else {
    conv(6, a.cat2, cs2, 0, a.a4, 32, 0, N, D1, H1, W1, true, a.b3, 64, 64);
  }
  conv(7, a.a4, 32, 0, a.d2, 32, 0, N, D1, H1, W1, true);
  if (training) {
    launch_up_fwd(a.d2, 32, a.cat1, 48, 0, 32, N, D1, H1, W1, stream);      // up(d2) -> cat1[0:32)
    conv(8, a.cat1, 48, 0, a.a5, 16, 0, N, D0, H0, W0, true);
  } else {
    conv(8, a.cat1, cs1, 0, a.a5, 16, 0, N, D0, H0, W0, true, a.d2, 32, 32);
  }
  if (!training) {
    // the output head is fused into the last convolution, whose activations are not stored
    PsiArgs h{};
    h.out = psiOut;
    h.w = head.w;
    h.avg = a.avg;
    h.scale = *psiScale;
    h.minValue = minValue;
    h.ox = outDims[0]; h.oy = outDims[1]; h.oz = outDims[2]; h.zlo = outDims[3];
    conv(9, a.a5, 16, 0, nullptr, 16, 0, N, D0, H0, W0, true, nullptr, 0, 0, nullptr, 0, &h);
    UCHECK(!convFailed, "U-Net convolution refused: three x-y planes of the input exceed 32-bit offsets");
    MVR_HIP(hipGetLastError());
    return 0;
  }
  conv(9, a.a5, 16, 0, a.d1, 16, 0, N, D0, H0, W0, true);
  UCHECK(!convFailed, "U-Net convolution refused: three x-y planes of the input exceed 32-bit offsets");
  HeadArgs h{};
  h.d1 = a.d1; h.d1_cs = 16;
  h.wo = head.w; h.bias = head.w + 16;
  h.avg = a.avg;
  h.nvox = (size_t)N * D0 * H0 * W0;
  h.target = a.target;
  h.dr = a.dr;
  h.loss_partial = lossPart;
  lossParts = launch_head(h, stream);
  MVR_HIP(hipGetLastError());
  return 0;
}

// the loss of the last training forward pass, waiting for everything enqueued since
int UNet::read_loss(const Acts& a, double* loss) {
  std::vector<double> lp(lossParts);
  MVR_HIP(hipMemcpyAsync(lp.data(), lossPart, lossParts * 8, hipMemcpyDeviceToHost, stream));
  MVR_HIP(hipStreamSynchronize(stream));
  double s = 0;
  for (double x : lp) s += x;
  *loss = s / (double)((size_t)a.N * a.D * a.H * a.W);
  return 0;
}

int UNet::backward(Acts& a) {
  const int N = a.N, D0 = a.D, H0 = a.H, W0 = a.W;
  const int D1 = D0 / 2, H1 = H0 / 2, W1 = W0 / 2, D2 = D0 / 4, H2 = H0 / 4, W2 = W0 / 4;
  const size_t v0 = (size_t)N * D0 * H0 * W0;
  convFailed = false;
  HeadArgs h{};
  h.d1 = a.d1; h.d1_cs = 16; h.wo = head.w; h.bias = head.w + 16; h.avg = a.avg; h.dr = a.dr; h.nvox = v0;
  const int hb = launch_head_bwd(h, a.g_d1, bpart, stream);
  launch_sum_partials(bpart, hb, 17, head.g, nullptr, 0, nullptr, stream);
  // decoder level 1
  wgrad(9, a.a5, 16, a.g_d1, 16, 0, N, D0, H0, W0);
  dgrad(9, a.g_d1, 16, 0, a.g_a5, 16, N, D0, H0, W0, a.a5);
  wgrad(8, a.cat1, 48, a.g_a5, 16, 0, N, D0, H0, W0);
  dgrad(8, a.g_a5, 16, 0, a.g_cat1, 48, N, D0, H0, W0);
  // decoder level 2
  launch_up_bwd(a.g_cat1, 48, 0, a.g_d2, 32, 32, N, D1, H1, W1, a.d2, stream);
  wgrad(7, a.a4, 32, a.g_d2, 32, 0, N, D1, H1, W1);
  dgrad(7, a.g_d2, 32, 0, a.g_a4, 32, N, D1, H1, W1, a.a4);
  wgrad(6, a.cat2, 96, a.g_a4, 32, 0, N, D1, H1, W1);
  dgrad(6, a.g_a4, 32, 0, a.g_cat2, 96, N, D1, H1, W1);
  // bottleneck
  launch_up_bwd(a.g_cat2, 96, 0, a.g_b3, 64, 64, N, D2, H2, W2, a.b3, stream);
  wgrad(5, a.a3, 64, a.g_b3, 64, 0, N, D2, H2, W2);
  dgrad(5, a.g_b3, 64, 0, a.g_a3, 64, N, D2, H2, W2, a.a3);
  wgrad(4, a.p2, 32, a.g_a3, 64, 0, N, D2, H2, W2);
  dgrad(4, a.g_a3, 64, 0, a.g_p2, 32, N, D2, H2, W2);
  // encoder level 2: e2 receives the skip gradient (g_cat2[64:96)) plus the pooled path
  launch_pool_bwd(a.g_p2, 32, a.g_cat2, 96, 64, 32, N, D2, H2, W2, a.cat2, stream);
  wgrad(3, a.a2, 32, a.g_cat2, 96, 64, N, D1, H1, W1);
  dgrad(3, a.g_cat2, 96, 64, a.g_a2, 32, N, D1, H1, W1, a.a2);
  wgrad(2, a.p1, 16, a.g_a2, 32, 0, N, D1, H1, W1);
  dgrad(2, a.g_a2, 32, 0, a.g_p1, 16, N, D1, H1, W1);
  // encoder level 1
  launch_pool_bwd(a.g_p1, 16, a.g_cat1, 48, 32, 16, N, D1, H1, W1, a.cat1, stream);
  wgrad(1, a.a1, 16, a.g_cat1, 48, 32, N, D0, H0, W0);
  dgrad(1, a.g_cat1, 48, 32, a.g_a1, 16, N, D0, H0, W0, a.a1);
  wgrad(0, a.x0, 16, a.g_a1, 16, 0, N, D0, H0, W0);
  UCHECK(!convFailed, "U-Net convolution refused: three x-y planes of the input exceed 32-bit offsets");
  MVR_HIP(hipGetLastError());
  return 0;
}

int UNet::adam_step(float lr) {
  ++step;
  const float b1 = 0.9f, b2 = 0.999f;
  const float c1 = 1.f / (1.f - std::pow(b1, (float)step)), c2 = 1.f / (1.f - std::pow(b2, (float)step));
  AdamArgs a{};
  a.lr = lr; a.beta1 = b1; a.beta2 = b2; a.eps = 1e-8f; a.c1 = c1; a.c2 = c2;
  for (int l = 0; l < kLayers; ++l) {
    add_tensor(a, layer[l], l);
    add_tensor(a, bias[l], -1);
  }
  add_tensor(a, head, -1);
  launch_adam(a, stream);
  MVR_HIP(hipGetLastError());
  return 0;
}

int UNet::ensure_scratch() {
  if (!wpart) {
    size_t maxc = 0;
    // the widest layers take 1536 / groups partitions (unet_wgrad.hip), the others up to kWgradParts
    for (int l = 0; l < kLayers; ++l) maxc = std::max(maxc, wgrad_max_parts(kCin[l], kCout[l], kWgradParts) * wcount(l));
    MVR_HIP(hipMalloc(&wpart, maxc * 4));
    MVR_HIP(hipMalloc(&bpart, (size_t)1024 * 64 * 4));
    MVR_HIP(hipMalloc(&lossPart, 2048 * 8));  // 1024 double2
  }
  return 0;
}

// ------------------------------------------------------------------ training volumes and steps
int UNet::add_volume(const float* const* imgs, const float* const* ws, const float* target, const int N3[3]) {
  MVR_HIP(hipSetDevice(dev));
  TrainVolume tv;
  for (int d = 0; d < 3; ++d) tv.N[d] = N3[d];
  const size_t n = (size_t)N3[0] * N3[1] * N3[2];
  for (int v = 0; v < V; ++v) {
    float *a = nullptr, *b = nullptr;
    MVR_HIP(hipMalloc(&a, n * 4));
    MVR_HIP(hipMalloc(&b, n * 4));
    MVR_HIP(hipMemcpy(a, imgs[v], n * 4, hipMemcpyDefault));
    MVR_HIP(hipMemcpy(b, ws[v], n * 4, hipMemcpyDefault));
    tv.img.push_back(a);
    tv.w.push_back(b);
  }
  double mean = 0;
  if (weighted_mean(tv.img, tv.w, n, &mean)) return -1;
  tv.scale = (float)std::max(1e-6, mean);
  MVR_HIP(hipMalloc(&tv.target, n * 4));
  MVR_HIP(hipMemcpy(tv.target, target, n * 4, hipMemcpyDefault));
  vols.push_back(tv);
  return (int)vols.size() - 1;
}

int UNet::pack(Acts& a, const std::vector<float*>& img, const std::vector<float*>& w, const int N3[3],
               const int o[3], float invScale) {
  InputArgs in{};
  for (int v = 0; v < V; ++v) { in.img[v] = img[v]; in.w[v] = w[v]; }
  in.V = V;
  for (int d = 0; d < 3; ++d) in.N3[d] = N3[d];
  in.x0 = o[0]; in.y0 = o[1]; in.z0 = o[2];
  in.W = a.W; in.H = a.H; in.D = a.D;
  in.inv_scale = invScale;
  in.out = a.x0;
  in.out_cs = a.csIn;
  in.avg_out = a.avg;
  launch_pack_input(in, stream);
  return 0;
}

int UNet::train_step(const int* volIdx, const int* origins, int batch, int P, float lr, double* loss, bool update) {
  MVR_HIP(hipSetDevice(dev));
  UCHECK(batch >= 1 && P >= 4 && P % 4 == 0, "bad batch or patch size");
  if (ensure_scratch() || ensure_acts(train, batch, P, P, P, true)) return -1;
  const size_t pv = (size_t)P * P * P;
  for (int b = 0; b < batch; ++b) {
    UCHECK(volIdx[b] >= 0 && volIdx[b] < (int)vols.size(), "bad training volume index");
    for (int d = 0; d < 3; ++d)
      UCHECK(origins[3 * b + d] >= 0 && origins[3 * b + d] + P <= vols[volIdx[b]].N[d], "patch outside its volume");
  }
  for (int b0 = 0; b0 < batch; b0 += kPatches) {
    const int n = std::min(kPatches, batch - b0);
    PatchArgs pa{};
    for (int b = 0; b < n; ++b) {
      const TrainVolume& tv = vols[volIdx[b0 + b]];
      PatchArgs::Patch& p = pa.p[b];
      for (int v = 0; v < V; ++v) { p.img[v] = tv.img[v]; p.w[v] = tv.w[v]; }
      p.target = tv.target;
      for (int d = 0; d < 3; ++d) { p.N3[d] = tv.N[d]; p.o[d] = origins[3 * (b0 + b) + d]; }
      p.inv_scale = 1.f / tv.scale;
    }
    pa.V = V;
    pa.P = P;
    pa.out = train.x0 + pv * 16 * b0;
    pa.avg_out = train.avg + pv * b0;
    pa.target_out = train.target + pv * b0;
    launch_pack_patches(pa, n, stream);
  }
  if (forward(train, true, nullptr, nullptr, nullptr, 0.f)) return -1;
  if (backward(train)) return -1;
  if (update && adam_step(lr)) return -1;
  if (loss) return read_loss(train, loss);
  MVR_HIP(hipStreamSynchronize(stream));
  return 0;
}

// weighted mean intensity sum w_v img_v / sum w_v over voxels and views (FP64 device partials,
// summed on the host); 1 when no voxel has weight
int UNet::weighted_mean(const std::vector<float*>& img, const std::vector<float*>& w, size_t n, double* mean) {
  if (ensure_scratch()) return -1;
  InputArgs in{};
  for (int v = 0; v < V; ++v) { in.img[v] = img[v]; in.w[v] = w[v]; }
  in.V = V;
  double2* part = reinterpret_cast<double2*>(lossPart);
  const int nb = launch_wsum_partials(in, n, part, stream);
  MVR_HIP(hipGetLastError());
  std::vector<double2> h(nb);
  MVR_HIP(hipMemcpyAsync(h.data(), part, nb * sizeof(double2), hipMemcpyDeviceToHost, stream));
  MVR_HIP(hipStreamSynchronize(stream));
  double s = 0, sw = 0;
  for (const double2& x : h) { s += x.x; sw += x.y; }
  *mean = sw > 0 ? s / sw : 1.0;
  return 0;
}

int UNet::infer(const std::vector<float*>& img, const std::vector<float*>& w, const int N3[3], float minValue,
                float* psiDev) {
  MVR_HIP(hipSetDevice(dev));
  UCHECK((int)img.size() == V && (int)w.size() == V, "the network was built for a different number of views");
  const size_t n = (size_t)N3[0] * N3[1] * N3[2];
  double mean = 0;
  if (weighted_mean(img, w, n, &mean)) return -1;
  const float scale = (float)std::max(1e-6, mean);
  auto up4 = [](int v) { return (v + 3) / 4 * 4; };
  const int X = up4(N3[0]), Y = up4(N3[1]), Z = up4(N3[2]);
  const long long plane = (long long)X * Y;
  // The volume runs as one window when it fits the voxel budget, else as z slabs of `slab` planes, each
  // with kInferHalo planes of context on either side (clipped at the volume's faces).  Slab starts and
  // the halo are multiples of 4, so every window keeps the volume's pooling grid, and the halo exceeds
  // the network's receptive-field radius: the kept planes are the ones a single window computes.
  int slab = Z;
  if ((long long)Z * plane > inferWindow) {
    slab = (int)((inferWindow / plane - 2 * kInferHalo) / 4 * 4);
    UCHECK(slab >= 4, "inference window budget too small for one x-y plane plus its halo");
  }
  int maxDepth = 0;
  for (int zs = 0; zs < N3[2]; zs += slab)
    maxDepth = std::max(maxDepth, up4(std::min(N3[2], zs + slab + kInferHalo) - std::max(0, zs - kInferHalo)));
  if (ensure_acts(inf, 1, maxDepth, Y, X, false)) return -1;  // one allocation for every window
  for (int zs = 0; zs < N3[2]; zs += slab) {
    const int ze = std::min(N3[2], zs + slab);
    const int ws = std::max(0, zs - kInferHalo), we = std::min(N3[2], ze + kInferHalo);
    if (ensure_acts(inf, 1, up4(we - ws), Y, X, false)) return -1;
    const int o[3] = {0, 0, ws};
    pack(inf, img, w, N3, o, 1.f / scale);
    // psi planes [zs, ze) = window planes [zs - ws, ze - ws)
    const int od[4] = {N3[0], N3[1], ze - ws, zs - ws};
    if (forward(inf, false, &scale, psiDev + (size_t)ws * N3[1] * N3[0], od, minValue)) return -1;
  }
  MVR_HIP(hipStreamSynchronize(stream));
  return 0;
}

int UNet::clear_volumes() {
  MVR_HIP(hipSetDevice(dev));
  for (auto& tv : vols) {
    for (auto p : tv.img) (void)hipFree(p);
    for (auto p : tv.w) (void)hipFree(p);
    (void)hipFree(tv.target);
  }
  vols.clear();
  train.release();
  return 0;
}

void UNet::destroy() {
  (void)hipSetDevice(dev);
  if (stream) (void)hipStreamSynchronize(stream);
  for (Param& p : layer) {
    if (p.wbf) (void)hipFree(p.wbf);
    if (p.wt) (void)hipFree(p.wt);
    p = Param{};
  }
  if (params) (void)hipFree(params);
  params = nullptr;
  clear_volumes();
  inf.release();
  for (void* p : {(void*)wpart, (void*)bpart, (void*)lossPart})
    if (p) (void)hipFree(p);
  wpart = nullptr; bpart = nullptr; lossPart = nullptr;
  if (stream) (void)hipStreamDestroy(stream);
  stream = nullptr;
}

}  // namespace mvr
