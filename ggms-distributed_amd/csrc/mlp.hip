// Learned splitter network: a 65 -> 32 (ReLU) -> 1 (sigmoid) fp32 MLP.
//
// Inputs (built by the first-pass splitter from the sorted sample): a window
// of 64 consecutive sample keys around the target quantile, normalised to
// [0, 1] by the window's extremes, and the target's fractional position in the
// window.  Output: where between the two sample keys that bracket the target
// the true quantile lies.  Trained on exact k-th values produced by the plain
// method; the first pass builds its ranges from the predictions and the
// linear slope inside each range does the rest, so a poor prediction only
// costs work, never exactness.
//
// Parameter layout (row-major fp32): W1[32][65], b1[32], W2[32], b2.
//
// Kernels: batched forward; loss + gradient in two steps (per workgroup over
// its tiles of samples, then the sum of the workgroups' partials); an Adam step.
#include <hip/hip_runtime.h>

#include <algorithm>
#include <cstring>
#include <mutex>
#include <vector>

#include "ggms.h"

namespace ggms {

constexpr int MI = 65, MH = 32, MP = MH * MI + MH + MH + 1;

namespace {
std::mutex g_w_mu;
std::vector<float*> g_w;  // per device
}  // namespace

const float* learned_weights_device(int device) {
  std::lock_guard<std::mutex> lk(g_w_mu);
  if (device < 0 || device >= (int)g_w.size()) return nullptr;
  return g_w[device];
}

__device__ __forceinline__ float sigmoidf_(float o) { return 1.0f / (1.0f + __expf(-o)); }

// One 64-sample tile per step and workgroup, four waves.  The products run on
// the fp32 matrix cores (16x16x4): a sample's hidden layer is one row of
// X [64 x 68] * W1^T [68 x 32], column 65 of X being 1 and of W1 the bias.
constexpr uint32_t kTile = 64, kMlpThreads = 256;
// row strides in LDS: 68 = 4 mod 32 spreads the operands' 16 rows x 4 columns
// over every bank; 48 does the same for the 4 rows x 16 columns of dz
constexpr uint32_t kXStride = 68, kZStride = 48;
constexpr uint32_t kMaxGradWgs = 256;
constexpr uint32_t kPart = MP + 1;  // floats of one workgroup's partial: gradient, loss

using f32x4 = float __attribute__((ext_vector_type(4)));

struct MlpLds {
  float x[kTile * kXStride + 16];  // + 16: the last column tile reads past the last row (columns not used)
  float w1[MH * kXStride];
  float w2[MH + 1];
};

__device__ __forceinline__ void mlp_load_weights(MlpLds& L, const float* __restrict__ w) {
  for (uint32_t j = threadIdx.x; j < MH * kXStride; j += kMlpThreads) {
    const uint32_t h = j / kXStride, i = j % kXStride;
    L.w1[j] = i < (uint32_t)MI ? w[h * MI + i] : i == (uint32_t)MI ? w[MH * MI + h] : 0.0f;
  }
  if (threadIdx.x <= (uint32_t)MH) L.w2[threadIdx.x] = w[MH * MI + MH + threadIdx.x];
  if (threadIdx.x < 16) L.x[kTile * kXStride + threadIdx.x] = 0.0f;
}

// Rows past nb are zero (their samples take no part).
__device__ __forceinline__ void mlp_load_tile(MlpLds& L, const float* __restrict__ x, uint32_t b0, uint32_t nb) {
  const uint32_t rows = nb - b0 < kTile ? nb - b0 : kTile;
  const float* src = x + (size_t)b0 * MI;
  for (uint32_t j = threadIdx.x; j < kTile * MI; j += kMlpThreads)
    L.x[(j / MI) * kXStride + j % MI] = j < rows * MI ? src[j] : 0.0f;
  if (threadIdx.x < kTile) {
    float* r = L.x + threadIdx.x * kXStride + MI;
    r[0] = 1.0f;
    r[1] = 0.0f;
    r[2] = 0.0f;
  }
}

// The hidden layer of this wave's 16 samples: lane l holds, for hidden units
// l % 16 (z[0]) and 16 + l % 16 (z[1]), samples 4 * (l / 16) + r.  o[r] is the
// output before the sigmoid of those samples, in every lane of the group of 16.
__device__ __forceinline__ void mlp_tile_forward(const MlpLds& L, f32x4 (&z)[2], float (&o)[4]) {
  const uint32_t l = threadIdx.x & 63, wv = threadIdx.x >> 6;
  const float* xr = L.x + (wv * 16 + (l & 15)) * kXStride + (l >> 4);
  const float* wr = L.w1 + (l & 15) * kXStride + (l >> 4);
  z[0] = f32x4{0, 0, 0, 0};
  z[1] = f32x4{0, 0, 0, 0};
#pragma unroll
  for (uint32_t s = 0; s < kXStride / 4; ++s) {
    const float a = xr[4 * s];
    z[0] = __builtin_amdgcn_mfma_f32_16x16x4f32(a, wr[4 * s], z[0], 0, 0, 0);
    z[1] = __builtin_amdgcn_mfma_f32_16x16x4f32(a, wr[16 * kXStride + 4 * s], z[1], 0, 0, 0);
  }
  const float v0 = L.w2[l & 15], v1 = L.w2[16 + (l & 15)];
#pragma unroll
  for (int r = 0; r < 4; ++r) {
    float c = v0 * fmaxf(z[0][r], 0.0f) + v1 * fmaxf(z[1][r], 0.0f);
#pragma unroll
    for (int d = 8; d > 0; d >>= 1) c += __shfl_xor(c, d, 16);
    o[r] = c + L.w2[MH];
  }
}

__global__ void __launch_bounds__(kMlpThreads) k_mlp_forward(const float* __restrict__ w, const float* __restrict__ x,
                                                             uint32_t nb, float* __restrict__ out) {
  __shared__ MlpLds L;
  const uint32_t b0 = blockIdx.x * kTile;
  mlp_load_weights(L, w);
  mlp_load_tile(L, x, b0, nb);
  __syncthreads();
  f32x4 z[2];
  float o[4];
  mlp_tile_forward(L, z, o);
  const uint32_t l = threadIdx.x & 63, m = (threadIdx.x >> 6) * 16 + 4 * (l >> 4);
#pragma unroll
  for (uint32_t r = 0; r < 4; ++r)
    if ((l & 15) == r && b0 + m + r < nb) out[b0 + m + r] = sigmoidf_(o[r]);
}

// Loss and gradient of the tiles t = blockIdx.x, + gridDim.x, ...: the forward
// pass, dL/dz of the tile into LDS, then grad[W1 | b1] = dz^T [32 x 64] * X
// [64 x 66] as ten 16 x 16 products over the four waves (b1's column is X's
// column of ones); the last wave adds W2, b2 and the loss.  The sums stay in
// registers over the tiles and are written once: part[blockIdx.x], or the
// gradient itself when one workgroup does it all.  Bound by latency: at 4096
// samples 64 CUs hold one tile each (loads, two short chains of matrix
// products, four barriers), 11.6 us, and the sum of the partials 4.0 us.  A
// thread per sample and then a thread per parameter walking 1024 samples took
// 20.5 + 334 us, and its sums (one chain of 1024) were less exact.
__global__ void __launch_bounds__(kMlpThreads) k_mlp_grad(const float* __restrict__ w, const float* __restrict__ x,
                                                          const float* __restrict__ y, uint32_t nb,
                                                          float* __restrict__ part, float* __restrict__ grad,
                                                          float* __restrict__ loss) {
  __shared__ MlpLds L;
  __shared__ float dz[kTile * kZStride], act[kTile * kZStride], d_o[kTile], e2[kTile];
  const uint32_t l = threadIdx.x & 63, wv = threadIdx.x >> 6, c16 = l & 15, q = l >> 4;
  mlp_load_weights(L, w);
  // ten output tiles (two of hidden units x five of inputs): waves 0 and 1 take three, 2 and 3 two
  const uint32_t first = wv < 2 ? 3 * wv : 6 + 2 * (wv - 2), mine = wv < 2 ? 3u : 2u;
  f32x4 acc[3] = {f32x4{0, 0, 0, 0}, f32x4{0, 0, 0, 0}, f32x4{0, 0, 0, 0}};
  float g2 = 0.0f, gb = 0.0f, ls = 0.0f;  // the last wave's: W2 gradient (half the samples per lane), b2 gradient, loss
  const uint32_t tiles = (nb + kTile - 1) / kTile;
  for (uint32_t t = blockIdx.x; t < tiles; t += gridDim.x) {
    const uint32_t b0 = t * kTile;
    __syncthreads();  // the previous tile's rows are read
    mlp_load_tile(L, x, b0, nb);
    float yv[4];
#pragma unroll
    for (uint32_t r = 0; r < 4; ++r) {
      const uint32_t b = b0 + wv * 16 + 4 * q + r;
      yv[r] = b < nb ? y[b] : 0.0f;
    }
    __syncthreads();
    f32x4 z[2];
    float o[4];
    mlp_tile_forward(L, z, o);
    const float v0 = L.w2[c16], v1 = L.w2[16 + c16];
#pragma unroll
    for (uint32_t r = 0; r < 4; ++r) {
      const uint32_t m = wv * 16 + 4 * q + r;
      const float p = sigmoidf_(o[r]);
      const float e = p - yv[r];
      const bool in = b0 + m < nb;
      const float d = in ? e * p * (1.0f - p) / (float)nb : 0.0f;
      float* zr = dz + m * kZStride + c16;
      float* ar = act + m * kZStride + c16;
      zr[0] = z[0][r] > 0.0f ? d * v0 : 0.0f;
      zr[16] = z[1][r] > 0.0f ? d * v1 : 0.0f;
      ar[0] = fmaxf(z[0][r], 0.0f);
      ar[16] = fmaxf(z[1][r], 0.0f);
      if (c16 == r) {
        d_o[m] = d;
        e2[m] = in ? 0.5f * e * e / (float)nb : 0.0f;
      }
    }
    __syncthreads();
#pragma unroll
    for (uint32_t j = 0; j < 3; ++j) {
      if (j >= mine) break;
      const uint32_t ot = first + j;
      const float* zc = dz + q * kZStride + (ot / 5) * 16 + c16;
      const float* xc = L.x + q * kXStride + (ot % 5) * 16 + c16;
#pragma unroll
      for (uint32_t s = 0; s < kTile / 4; ++s)
        acc[j] = __builtin_amdgcn_mfma_f32_16x16x4f32(zc[4 * s * kZStride], xc[4 * s * kXStride], acc[j], 0, 0, 0);
    }
    if (wv == 3) {
      float a = 0.0f;
      const uint32_t h = l & 31, m0 = (l >> 5) * (kTile / 2);
#pragma unroll 8
      for (uint32_t m = m0; m < m0 + kTile / 2; ++m) a += d_o[m] * act[m * kZStride + h];
      g2 += a;
      gb += d_o[l];
      ls += e2[l];
    }
  }
  float* dst = gridDim.x == 1 ? grad : part + (size_t)blockIdx.x * kPart;
#pragma unroll
  for (uint32_t j = 0; j < 3; ++j) {
    if (j >= mine) break;
    const uint32_t ot = first + j, i = (ot % 5) * 16 + c16;
#pragma unroll
    for (uint32_t r = 0; r < 4; ++r) {
      const uint32_t h = (ot / 5) * 16 + 4 * q + r;
      if (i < (uint32_t)MI) dst[h * MI + i] = acc[j][r];
      else if (i == (uint32_t)MI) dst[MH * MI + h] = acc[j][r];
    }
  }
  if (wv == 3) {
    g2 += __shfl_xor(g2, 32, 64);
#pragma unroll
    for (int d = 32; d > 0; d >>= 1) {
      gb += __shfl_xor(gb, d, 64);
      ls += __shfl_xor(ls, d, 64);
    }
    if (l < (uint32_t)MH) dst[MH * MI + MH + l] = g2;
    if (l == 0) {
      dst[MP - 1] = gb;
      if (gridDim.x == 1) *loss = ls;
      else dst[MP] = ls;
    }
  }
}

// Sums the workgroups' partials in their order: 64 columns a workgroup, four
// waves taking every fourth partial, eight reads in flight.
__global__ void __launch_bounds__(256) k_mlp_sum(const float* __restrict__ part, uint32_t parts,
                                                 float* __restrict__ grad, float* __restrict__ loss) {
  __shared__ float s[4][64];
  const uint32_t l = threadIdx.x & 63, wv = threadIdx.x >> 6, c = blockIdx.x * 64 + l;
  float a = 0.0f;
  if (c < kPart) {
    uint32_t g = wv;
    for (; g + 28 < parts; g += 32) {
      float v[8];
#pragma unroll
      for (uint32_t u = 0; u < 8; ++u) v[u] = part[(size_t)(g + 4 * u) * kPart + c];
#pragma unroll
      for (uint32_t u = 0; u < 8; ++u) a += v[u];
    }
    for (; g < parts; g += 4) a += part[(size_t)g * kPart + c];
  }
  s[wv][l] = a;
  __syncthreads();
  if (wv == 0 && c < kPart) {
    const float t = (s[0][l] + s[1][l]) + (s[2][l] + s[3][l]);
    if (c < (uint32_t)MP) grad[c] = t;
    else *loss = t;
  }
}

__global__ void k_fill_f32(float* __restrict__ p, uint32_t n, float v) {
  uint32_t i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i < n) p[i] = v;
}

__global__ void k_adam(float* __restrict__ w, const float* __restrict__ g, float* __restrict__ m,
                       float* __restrict__ v, uint32_t n, float lr, float b1, float b2, float eps, float c1,
                       float c2) {
  uint32_t i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= n) return;
  float gi = g[i];
  float mi = b1 * m[i] + (1.0f - b1) * gi;
  float vi = b2 * v[i] + (1.0f - b2) * gi * gi;
  m[i] = mi;
  v[i] = vi;
  float mh = mi / c1, vh = vi / c2;
  w[i] -= lr * mh / (sqrtf(vh) + eps);
}

}  // namespace ggms

using namespace ggms;

extern "C" {

uint32_t ggms_mlp_param_count(void) { return (uint32_t)MP; }

ggms_status ggms_set_learned_weights(int device, const float* w_host, uint32_t n) {
  if (!w_host || n != (uint32_t)MP) return GGMS_EINVAL;
  int cur = 0;
  if (hipGetDevice(&cur) != hipSuccess) return GGMS_EDEVICE;
  std::lock_guard<std::mutex> lk(g_w_mu);
  if ((int)g_w.size() <= device) g_w.resize(device + 1, nullptr);
  if (hipSetDevice(device) != hipSuccess) return GGMS_EDEVICE;
  ggms_status s = GGMS_OK;
  if (!g_w[device] && hipMalloc(&g_w[device], sizeof(float) * MP) != hipSuccess) {
    g_w[device] = nullptr;
    s = GGMS_ENOMEM;
  }
  if (s == GGMS_OK && hipMemcpy(g_w[device], w_host, sizeof(float) * MP, hipMemcpyHostToDevice) != hipSuccess)
    s = GGMS_EDEVICE;
  (void)hipSetDevice(cur);
  return s;
}

ggms_status ggms_clear_learned_weights(int device) {
  std::lock_guard<std::mutex> lk(g_w_mu);
  if (device < 0 || device >= (int)g_w.size() || !g_w[device]) return GGMS_OK;
  int cur = 0;
  (void)hipGetDevice(&cur);
  (void)hipSetDevice(device);
  (void)hipFree(g_w[device]);
  g_w[device] = nullptr;
  (void)hipSetDevice(cur);
  return GGMS_OK;
}

ggms_status ggms_mlp_forward(const float* d_w, const float* d_x, uint32_t nb, float* d_out, void* stream) {
  if (!d_w || (!d_x && nb) || (!d_out && nb)) return GGMS_EINVAL;
  if (nb == 0) return GGMS_OK;
  k_mlp_forward<<<(nb - 1) / kTile + 1, kMlpThreads, 0, (hipStream_t)stream>>>(d_w, d_x, nb, d_out);
  return hipGetLastError() == hipSuccess ? GGMS_OK : GGMS_EDEVICE;
}

uint64_t ggms_mlp_workspace_floats(uint32_t nb) { return (uint64_t)nb * (2 * MH + 1); }

ggms_status ggms_mlp_loss_grad(const float* d_w, const float* d_x, const float* d_y, uint32_t nb, float* d_grad,
                               float* d_loss, float* d_work, void* stream) {
  if (!d_w || !d_grad || !d_loss || (nb && (!d_x || !d_y || !d_work))) return GGMS_EINVAL;
  hipStream_t st = (hipStream_t)stream;
  if (!nb) {
    k_fill_f32<<<(MP + 255) / 256, 256, 0, st>>>(d_grad, MP, 0.0f);
    k_fill_f32<<<1, 32, 0, st>>>(d_loss, 1, 0.0f);
  } else {
    // a workgroup per tile up to one per CU, and no more than the workspace
    // (2 MH + 1 floats a sample) holds partials of; a single one writes the result
    uint64_t wgs = std::min<uint64_t>((nb - 1) / kTile + 1, ggms_mlp_workspace_floats(nb) / kPart);
    wgs = std::max<uint64_t>(1, std::min<uint64_t>(wgs, kMaxGradWgs));
    k_mlp_grad<<<(uint32_t)wgs, kMlpThreads, 0, st>>>(d_w, d_x, d_y, nb, d_work, d_grad, d_loss);
    if (wgs > 1) k_mlp_sum<<<(kPart + 63) / 64, 256, 0, st>>>(d_work, (uint32_t)wgs, d_grad, d_loss);
  }
  return hipGetLastError() == hipSuccess ? GGMS_OK : GGMS_EDEVICE;
}

ggms_status ggms_mlp_adam_step(float* d_w, const float* d_grad, float* d_m, float* d_v, uint32_t step, float lr,
                               float beta1, float beta2, float eps, void* stream) {
  if (!d_w || !d_grad || !d_m || !d_v || step == 0) return GGMS_EINVAL;
  float c1 = 1.0f - powf(beta1, (float)step);
  float c2 = 1.0f - powf(beta2, (float)step);
  k_adam<<<(MP + 255) / 256, 256, 0, (hipStream_t)stream>>>(d_w, d_grad, d_m, d_v, MP, lr, beta1, beta2, eps, c1, c2);
  return hipGetLastError() == hipSuccess ? GGMS_OK : GGMS_EDEVICE;
}

}  // extern "C"
