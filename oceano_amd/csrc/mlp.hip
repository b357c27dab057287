// mlp.hip -- training and inference of the closure network (BF16 MFMA, FP32 accumulation).
//
// Training step = k_mlp_grad (forward of 16-sample tiles, MSE loss, backward; each wave
// accumulates its weight gradients in registers and writes one partial) + k_mlp_reduce (sum of
// the partials in a fixed order: deterministic) + k_mlp_adam (Adam in FP32 on the master
// parameters, then the BF16 copies the products read).
#include <hip/hip_runtime.h>

#include <cmath>
#include <random>
#include <string>
#include <vector>

#include "mlp_core.hpp"
#include "oceano_dg.h"
#include "oceano_mlp.h"

namespace oceano {
void set_error(const std::string &msg);
}

using namespace oceano::mlp;
using oceano::set_error;

struct oc_mlp
{
  int n_in = 0, n_out = 0;
  float *p = nullptr, *m = nullptr, *v = nullptr, *grad = nullptr, *norm = nullptr;
  float *partial = nullptr, *lossp = nullptr;
  bf16 *wt = nullptr, *wb = nullptr;
  int64_t step = 0;
  int gmax = 256;
};

namespace {

#define MLP_TRY(x)                                                   \
  do                                                                 \
    {                                                                \
      const hipError_t e_ = (x);                                     \
      if (e_ != hipSuccess)                                          \
        {                                                            \
          set_error(std::string("HIP error: ") + hipGetErrorString(e_)); \
          return OC_ERR_HIP;                                         \
        }                                                            \
    }                                                                \
  while (0)

// X rows base .. base + 15 as the A operand of a tile: row l % 16, inputs 8 (l / 16) .., normalised
// (mu, is: the lane's 8 means and inverse spreads), zero outside the n rows and n_in inputs
__device__ __forceinline__ bf16x8 load_inputs(const float *__restrict__ X, int64_t base, int64_t n,
                                              int n_in, const float (&mu)[8],
                                              const float (&is)[8])
{
  const int l = threadIdx.x & 63, k8 = (l >> 4) * 8;
  const int64_t row = base + (l & 15);
  float v[8];
#pragma unroll
  for (int j = 0; j < 8; ++j)
    v[j] = row < n && k8 + j < n_in ? X[row * n_in + k8 + j] : mu[j];
  bf16 h[8];
#pragma unroll
  for (int j = 0; j < 8; ++j)
    h[j] = to_bf16((v[j] - mu[j]) * is[j]);
  bf16x8 x;
  __builtin_memcpy(&x, h, sizeof(x));
  return x;
}

// Forward, loss and gradient of the rows of chunks blockIdx.x, blockIdx.x + gridDim.x, ... of 16
// samples; one wave per workgroup writes one partial gradient.
//
// The chain of one chunk (eight dependent products, three GELUs) bounds it, not its 150 MFMAs:
// at 4096 rows every wave has one chunk.  So nothing waits in it that need not: the weights of both
// directions and the weight gradients stay in registers (one wave per SIMD has 512, all used; 60
// more are spilled), and an
// accumulator's layout (sample 4 (l / 16) + j, unit 16 ct + l % 16) is already the operand
// layout of the 16-sample weight-gradient products, so only the row operands of the layer
// products cross LDS.  4096 rows: about 56 us with weights and gradients in LDS, 26.5 us.
__global__ __launch_bounds__(64, 1) void k_mlp_grad(const float *__restrict__ p,
                                                    const bf16 *__restrict__ wt,
                                                    const bf16 *__restrict__ wb,
                                                    const float *__restrict__ norm, int64_t n,
                                                    int n_in, int n_out,
                                                    const float *__restrict__ X,
                                                    const float *__restrict__ T, float gscale,
                                                    float *__restrict__ partial,
                                                    float *__restrict__ lossp)
{
  constexpr int HT = HID / 16, OT = OUT / 16, IT = IN / 16;
  __shared__ __attribute__((aligned(16))) bf16 s_h[2][16 * LDT];
  const int l = threadIdx.x, r = l & 15, g = l >> 4, kq = g * 4, k8 = g * 8;
  ForwardWeights W;
  W.load(wt, p);
  // B operands of the backward products dZ W^T: row-major W rows, 16 bytes each
  bf16x8 v2[2 * HT], v3[2 * HT], v4[HT];
#pragma unroll
  for (int ct = 0; ct < HT; ++ct)
    {
#pragma unroll
      for (int kk = 0; kk < 2; ++kk)
        {
          v2[2 * ct + kk] = load8(wb + W2 + (16 * ct + r) * HID + 32 * kk + k8);
          v3[2 * ct + kk] = load8(wb + W3 + (16 * ct + r) * HID + 32 * kk + k8);
        }
      v4[ct] = load8(wb + W4 + (16 * ct + r) * OUT + k8);
    }
  float mu[8], is[8];
#pragma unroll
  for (int j = 0; j < 8; ++j)
    {
      mu[j] = norm[k8 + j];
      is[j] = norm[IN + k8 + j];
    }
  float scale[OT], shift[OT], mut[IT], ist[IT];
#pragma unroll
  for (int ct = 0; ct < OT; ++ct)
    {
      scale[ct] = norm[2 * IN + 16 * ct + r];
      shift[ct] = norm[2 * IN + OUT + 16 * ct + r];
    }
#pragma unroll
  for (int rt = 0; rt < IT; ++rt)
    {
      mut[rt] = norm[16 * rt + r];
      ist[rt] = norm[IN + 16 * rt + r];
    }
  const f32x4 zero{0.f, 0.f, 0.f, 0.f};
  f32x4 g1[IT][HT], g2[HT][HT], g3[HT][HT], g4[HT][OT];
  float d1[HT], d2[HT], d3[HT], d4[OT];  // bias gradients, the lane's 4 samples of each chunk
#pragma unroll
  for (int ct = 0; ct < HT; ++ct)
    {
#pragma unroll
      for (int rt = 0; rt < IT; ++rt)
        g1[rt][ct] = zero;
#pragma unroll
      for (int rt = 0; rt < HT; ++rt)
        {
          g2[rt][ct] = zero;
          g3[rt][ct] = zero;
          if (ct < OT)
            g4[rt][ct] = zero;
        }
      d1[ct] = d2[ct] = d3[ct] = 0.f;
      if (ct < OT)
        d4[ct] = 0.f;
    }
  float lossacc = 0.f;
  const int64_t n_chunks = (n + 15) / 16;
  for (int64_t c = blockIdx.x; c < n_chunks; c += gridDim.x)
    {
      const int64_t base = c * 16;
      float t[OT][4], xt[IT][4];
#pragma unroll
      for (int j = 0; j < 4; ++j)
        {
          const int64_t row = base + kq + j;
#pragma unroll
          for (int ct = 0; ct < OT; ++ct)
            {
              const int o = 16 * ct + r;
              t[ct][j] = row < n && o < n_out ? T[row * n_out + o] : shift[ct];
            }
#pragma unroll
          for (int rt = 0; rt < IT; ++rt)
            {
              const int i = 16 * rt + r;
              xt[rt][j] = row < n && i < n_in ? X[row * n_in + i] : mut[rt];
            }
        }
      const bf16x8 x = load_inputs(X, base, n, n_in, mu, is);
      bf16x4 h[3][HT];
      f32x4 slope[3][HT], out[OT];
      forward_tile(x, W, s_h, out, h, slope);
      // dL/dy of the mean squared error over the n x n_out valid outputs
      bf16x4 dy[OT];
#pragma unroll
      for (int ct = 0; ct < OT; ++ct)
#pragma unroll
        for (int j = 0; j < 4; ++j)
          {
            const bool valid = base + kq + j < n && 16 * ct + r < n_out;
            const float d = valid ? out[ct][j] - (t[ct][j] - shift[ct]) / scale[ct] : 0.f;
            lossacc += d * d;
            const float gr = d * gscale;
            d4[ct] += gr;
            const bf16 b = to_bf16(gr);
            dy[ct][j] = (short)b;
            s_h[1][(kq + j) * LDT + 16 * ct + r] = b;
          }
      tile_fence();
      // output layer: dW4 = H3^T dY, dZ3 = (dY W4^T) gelu'
      f32x4 acc[HT];
      {
        const bf16x8 a = load8(s_h[1] + r * LDT + k8);
#pragma unroll
        for (int ct = 0; ct < HT; ++ct)
          acc[ct] = mfma32(a, v4[ct], zero);
      }
#pragma unroll
      for (int rt = 0; rt < HT; ++rt)
#pragma unroll
        for (int ct = 0; ct < OT; ++ct)
          g4[rt][ct] = mfma(h[2][rt], dy[ct], g4[rt][ct]);
      // hidden layers: dZ in operand form dz, its bias sums, and as rows in LDS
      bf16x4 dz[HT];
      auto scaled = [&](const f32x4(&sl)[HT], float(&db)[HT], bf16 *rows) {
#pragma unroll
        for (int ct = 0; ct < HT; ++ct)
#pragma unroll
          for (int j = 0; j < 4; ++j)
            {
              const float v = acc[ct][j] * sl[ct][j];
              db[ct] += v;
              const bf16 b = to_bf16(v);
              dz[ct][j] = (short)b;
              if (rows)
                rows[(kq + j) * LDT + 16 * ct + r] = b;
            }
      };
      scaled(slope[2], d3, s_h[0]);
      tile_fence();
      tile_product<HT>(s_h[0], v3, acc);
#pragma unroll
      for (int rt = 0; rt < HT; ++rt)
#pragma unroll
        for (int ct = 0; ct < HT; ++ct)
          g3[rt][ct] = mfma(h[1][rt], dz[ct], g3[rt][ct]);
      scaled(slope[1], d2, s_h[1]);
      tile_fence();
      tile_product<HT>(s_h[1], v2, acc);
#pragma unroll
      for (int rt = 0; rt < HT; ++rt)
#pragma unroll
        for (int ct = 0; ct < HT; ++ct)
          g2[rt][ct] = mfma(h[0][rt], dz[ct], g2[rt][ct]);
      scaled(slope[0], d1, nullptr);
      // first layer: dW1 = X^T dZ1
#pragma unroll
      for (int rt = 0; rt < IT; ++rt)
        {
          bf16x4 a;
#pragma unroll
          for (int j = 0; j < 4; ++j)
            a[j] = (short)to_bf16((xt[rt][j] - mut[rt]) * ist[rt]);
#pragma unroll
          for (int ct = 0; ct < HT; ++ct)
            g1[rt][ct] = mfma(a, dz[ct], g1[rt][ct]);
        }
      tile_fence();
    }
  float *out = partial + (size_t)blockIdx.x * NPARAM;
#pragma unroll
  for (int ct = 0; ct < HT; ++ct)
#pragma unroll
    for (int j = 0; j < 4; ++j)
      {
#pragma unroll
        for (int rt = 0; rt < IT; ++rt)
          out[W1 + (16 * rt + kq + j) * HID + 16 * ct + r] = g1[rt][ct][j];
#pragma unroll
        for (int rt = 0; rt < HT; ++rt)
          {
            out[W2 + (16 * rt + kq + j) * HID + 16 * ct + r] = g2[rt][ct][j];
            out[W3 + (16 * rt + kq + j) * HID + 16 * ct + r] = g3[rt][ct][j];
            if (ct < OT)
              out[W4 + (16 * rt + kq + j) * OUT + 16 * ct + r] = g4[rt][ct][j];
          }
      }
  auto over_samples = [](float v) {
    v += __shfl_xor(v, 16);
    return v + __shfl_xor(v, 32);
  };
#pragma unroll
  for (int ct = 0; ct < HT; ++ct)
    {
      const float s1 = over_samples(d1[ct]), s2 = over_samples(d2[ct]);
      const float s3 = over_samples(d3[ct]), s4 = ct < OT ? over_samples(d4[ct % OT]) : 0.f;
      if (g == 0)
        {
          out[B1 + 16 * ct + r] = s1;
          out[B2 + 16 * ct + r] = s2;
          out[B3 + 16 * ct + r] = s3;
          if (ct < OT)
            out[B4 + 16 * ct + r] = s4;
        }
    }
#pragma unroll
  for (int off = 32; off > 0; off >>= 1)
    lossacc += __shfl_xor(lossacc, off);
  if (l == 0)
    lossp[blockIdx.x] = lossacc;
}

// grad = sum of the G partials.  A workgroup takes 32 parameters: 8 threads share one parameter's
// partials (every eighth each, 8 loads in flight) and their sums are added in order, so the
// result does not depend on the launch.  G = 256: 54 us with one thread and one load at a time per
// parameter, 5.2 us.
constexpr int RED_PARAMS = 32, RED_LANES = 8;
__global__ __launch_bounds__(RED_PARAMS *RED_LANES) void k_mlp_reduce(
  const float *__restrict__ partial, int G, float *__restrict__ grad)
{
  __shared__ float part[RED_LANES][RED_PARAMS];
  const int q = threadIdx.x % RED_PARAMS, y = threadIdx.x / RED_PARAMS;
  const int i = blockIdx.x * RED_PARAMS + q;
  float s = 0.f;
  if (i < NPARAM)
    {
      int b = y;
      for (; b + 7 * RED_LANES < G; b += 8 * RED_LANES)
        {
          float v[8];
#pragma unroll
          for (int k = 0; k < 8; ++k)
            v[k] = partial[(size_t)(b + k * RED_LANES) * NPARAM + i];
#pragma unroll
          for (int k = 0; k < 8; ++k)
            s += v[k];
        }
      for (; b < G; b += RED_LANES)
        s += partial[(size_t)b * NPARAM + i];
    }
  part[y][q] = s;
  __syncthreads();
  if (y == 0 && i < NPARAM)
    {
#pragma unroll
      for (int k = 1; k < RED_LANES; ++k)
        s += part[k][q];
      grad[i] = s;
    }
}

__device__ inline int transposed_index(int i)
{
  if (i >= W1 && i < B1)
    return T1 + ((i - W1) % HID) * IN + (i - W1) / HID;
  if (i >= W2 && i < B2)
    return T2 + ((i - W2) % HID) * HID + (i - W2) / HID;
  if (i >= W3 && i < B3)
    return T3 + ((i - W3) % HID) * HID + (i - W3) / HID;
  if (i >= W4 && i < B4)
    return T4 + ((i - W4) % OUT) * HID + (i - W4) / OUT;
  return -1;
}

__global__ void k_mlp_adam(float *__restrict__ p, float *__restrict__ m, float *__restrict__ v,
                           const float *__restrict__ grad, bf16 *__restrict__ wt,
                           bf16 *__restrict__ wb, float lr_t, float beta1, float beta2,
                           float eps)
{
  const int i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= NPARAM)
    return;
  const float g = grad[i];
  const float mi = beta1 * m[i] + (1.f - beta1) * g;
  const float vi = beta2 * v[i] + (1.f - beta2) * g * g;
  m[i] = mi;
  v[i] = vi;
  const float w = p[i] - lr_t * mi / (sqrtf(vi) + eps);
  p[i] = w;
  wb[i] = to_bf16(w);
  const int t = transposed_index(i);
  if (t >= 0)
    wt[t] = to_bf16(w);
}

// rows of tiles blockIdx.x, blockIdx.x + gridDim.x, ... of 16; one wave, weights in registers
__global__ __launch_bounds__(64) void k_mlp_forward(const float *__restrict__ p,
                                                    const bf16 *__restrict__ wt,
                                                    const float *__restrict__ norm, int64_t n,
                                                    int n_in, int n_out,
                                                    const float *__restrict__ X,
                                                    float *__restrict__ Y)
{
  __shared__ __attribute__((aligned(16))) bf16 s_h[2][16 * LDT];
  const int l = threadIdx.x, r = l & 15, kq = (l >> 4) * 4, k8 = (l >> 4) * 8;
  ForwardWeights W;
  W.load(wt, p);
  float mu[8], is[8];
#pragma unroll
  for (int j = 0; j < 8; ++j)
    {
      mu[j] = norm[k8 + j];
      is[j] = norm[IN + k8 + j];
    }
  for (int64_t tile = blockIdx.x; tile * 16 < n; tile += gridDim.x)
    {
      const bf16x8 x = load_inputs(X, tile * 16, n, n_in, mu, is);
      f32x4 out[OUT / 16];
      forward_tile(x, W, s_h, out);
#pragma unroll
      for (int ct = 0; ct < OUT / 16; ++ct)
#pragma unroll
        for (int j = 0; j < 4; ++j)
          {
            const int64_t row = tile * 16 + kq + j;
            const int o = 16 * ct + r;
            if (row < n && o < n_out)
              Y[row * n_out + o] = output_value(out[ct][j], norm, o);
          }
      tile_fence();
    }
}

void host_copies(const std::vector<float> &p, std::vector<bf16> &wt, std::vector<bf16> &wb)
{
  wt.assign(NT, 0);
  wb.assign(NPARAM, 0);
  for (int i = 0; i < NPARAM; ++i)
    wb[i] = to_bf16(p[i]);
  auto put = [&](int W, int K, int N, int T) {
    for (int k = 0; k < K; ++k)
      for (int n = 0; n < N; ++n)
        wt[T + n * K + k] = to_bf16(p[W + k * N + n]);
  };
  put(W1, IN, HID, T1);
  put(W2, HID, HID, T2);
  put(W3, HID, HID, T3);
  put(W4, HID, OUT, T4);
}

int upload_params(oc_mlp *m, const std::vector<float> &p)
{
  std::vector<bf16> wt, wb;
  host_copies(p, wt, wb);
  MLP_TRY(hipMemcpy(m->p, p.data(), NPARAM * sizeof(float), hipMemcpyHostToDevice));
  MLP_TRY(hipMemcpy(m->wt, wt.data(), NT * sizeof(bf16), hipMemcpyHostToDevice));
  MLP_TRY(hipMemcpy(m->wb, wb.data(), NPARAM * sizeof(bf16), hipMemcpyHostToDevice));
  return OC_OK;
}

std::vector<float> default_norm()
{
  std::vector<float> nrm(NNORM, 0.f);
  for (int i = 0; i < IN; ++i)
    nrm[IN + i] = 1.f;
  for (int o = 0; o < OUT; ++o)
    {
      nrm[2 * IN + o] = 1.f;
      nrm[NLO + o] = -INFINITY;
      nrm[NHI + o] = INFINITY;
    }
  return nrm;
}

void release(oc_mlp *m)
{
  for (float *q : {m->p, m->m, m->v, m->grad, m->norm, m->partial, m->lossp})
    (void)hipFree(q);
  (void)hipFree(m->wt);
  (void)hipFree(m->wb);
}

int grad_launch(oc_mlp *m, int64_t n, const float *x, const float *t, hipStream_t s, int *G)
{
  const int64_t chunks = (n + 15) / 16;
  *G = (int)std::min<int64_t>(chunks, m->gmax);
  const float gscale = 2.0f / (float)((double)n * (double)m->n_out);
  hipLaunchKernelGGL(k_mlp_grad, dim3(*G), dim3(64), 0, s, m->p, m->wt, m->wb, m->norm, n,
                     m->n_in, m->n_out, x, t, gscale, m->partial, m->lossp);
  hipLaunchKernelGGL(k_mlp_reduce, dim3((NPARAM + RED_PARAMS - 1) / RED_PARAMS),
                     dim3(RED_PARAMS * RED_LANES), 0, s, m->partial, *G, m->grad);
  MLP_TRY(hipGetLastError());
  return OC_OK;
}

}  // namespace

extern "C" {

int oc_mlp_create(int32_t n_in, int32_t n_out, uint64_t seed, oc_mlp **out)
{
  if (!out || n_in < 1 || n_in > IN || n_out < 1 || n_out > OUT)
    {
      set_error("oc_mlp_create: n_in must be in 1..32, n_out in 1..32");
      return OC_ERR_ARGUMENT;
    }
  oc_mlp *m = new oc_mlp;
  m->n_in = n_in;
  m->n_out = n_out;
  bool ok = true;
  for (float **q : {&m->p, &m->m, &m->v, &m->grad})
    ok = ok && hipMalloc(q, NPARAM * sizeof(float)) == hipSuccess;
  ok = ok && hipMalloc(&m->norm, NNORM * sizeof(float)) == hipSuccess;
  ok = ok && hipMalloc(&m->partial, (size_t)m->gmax * NPARAM * sizeof(float)) == hipSuccess;
  ok = ok && hipMalloc(&m->lossp, m->gmax * sizeof(float)) == hipSuccess;
  ok = ok && hipMalloc(&m->wt, NT * sizeof(bf16)) == hipSuccess;
  ok = ok && hipMalloc(&m->wb, NPARAM * sizeof(bf16)) == hipSuccess;
  ok = ok && hipMemset(m->m, 0, NPARAM * sizeof(float)) == hipSuccess &&
       hipMemset(m->v, 0, NPARAM * sizeof(float)) == hipSuccess;
  if (!ok)
    {
      release(m);
      delete m;
      set_error("oc_mlp_create: device allocation failed");
      return OC_ERR_HIP;
    }
  // Glorot-uniform weights on the used block of each layer, zero pads and biases
  std::mt19937_64 eng(seed);
  auto u01 = [&]() { return double(eng() >> 11) * (1.0 / 9007199254740992.0); };
  std::vector<float> p(NPARAM, 0.f);
  auto fill = [&](int W, int K, int N, int k_used, int n_used) {
    const double lim = std::sqrt(6.0 / (k_used + n_used));
    for (int k = 0; k < k_used; ++k)
      for (int n = 0; n < n_used; ++n)
        p[W + k * N + n] = float((2.0 * u01() - 1.0) * lim);
  };
  fill(W1, IN, HID, n_in, HID);
  fill(W2, HID, HID, HID, HID);
  fill(W3, HID, HID, HID, HID);
  fill(W4, HID, OUT, HID, n_out);
  std::vector<float> nrm = default_norm();
  int rc = upload_params(m, p);
  if (!rc && hipMemcpy(m->norm, nrm.data(), NNORM * sizeof(float), hipMemcpyHostToDevice) !=
               hipSuccess)
    rc = OC_ERR_HIP;
  if (rc)
    {
      release(m);
      delete m;
      return rc;
    }
  *out = m;
  return OC_OK;
}

void oc_mlp_destroy(oc_mlp *m)
{
  if (!m)
    return;
  release(m);
  delete m;
}

int32_t oc_mlp_n_params(void) { return NPARAM; }

int oc_mlp_get_params(oc_mlp *m, float *params)
{
  if (!m || !params)
    return OC_ERR_ARGUMENT;
  MLP_TRY(hipMemcpy(params, m->p, NPARAM * sizeof(float), hipMemcpyDeviceToHost));
  return OC_OK;
}

int oc_mlp_set_params(oc_mlp *m, const float *params)
{
  if (!m || !params)
    {
      set_error("oc_mlp_set_params: null argument");
      return OC_ERR_ARGUMENT;
    }
  std::vector<float> p(params, params + NPARAM);
  // pads of the unused inputs / outputs stay zero
  for (int k = m->n_in; k < IN; ++k)
    for (int n = 0; n < HID; ++n)
      p[W1 + k * HID + n] = 0.f;
  for (int k = 0; k < HID; ++k)
    for (int o = m->n_out; o < OUT; ++o)
      p[W4 + k * OUT + o] = 0.f;
  for (int o = m->n_out; o < OUT; ++o)
    p[B4 + o] = 0.f;
  MLP_TRY(hipMemset(m->m, 0, NPARAM * sizeof(float)));
  MLP_TRY(hipMemset(m->v, 0, NPARAM * sizeof(float)));
  m->step = 0;
  return upload_params(m, p);
}

int oc_mlp_set_normalization(oc_mlp *m, const float *x_mean, const float *x_std,
                             const float *y_shift, const float *y_scale)
{
  if (!m || !x_mean || !x_std || !y_shift || !y_scale)
    {
      set_error("oc_mlp_set_normalization: null argument");
      return OC_ERR_ARGUMENT;
    }
  std::vector<float> nrm = default_norm();
  // keep the output range of an earlier oc_mlp_set_output_range
  MLP_TRY(hipMemcpy(nrm.data() + NLO, m->norm + NLO, 2 * OUT * sizeof(float),
                    hipMemcpyDeviceToHost));
  for (int i = 0; i < m->n_in; ++i)
    {
      if (!(x_std[i] > 0.f))
        {
          set_error("oc_mlp_set_normalization: x_std must be positive");
          return OC_ERR_ARGUMENT;
        }
      nrm[i] = x_mean[i];
      nrm[IN + i] = 1.f / x_std[i];
    }
  for (int o = 0; o < m->n_out; ++o)
    {
      if (!(y_scale[o] > 0.f))
        {
          set_error("oc_mlp_set_normalization: y_scale must be positive");
          return OC_ERR_ARGUMENT;
        }
      nrm[2 * IN + o] = y_scale[o];
      nrm[2 * IN + OUT + o] = y_shift[o];
    }
  MLP_TRY(hipMemcpy(m->norm, nrm.data(), NNORM * sizeof(float), hipMemcpyHostToDevice));
  return OC_OK;
}

int oc_mlp_set_output_range(oc_mlp *m, const float *lo, const float *hi)
{
  if (!m)
    {
      set_error("oc_mlp_set_output_range: null argument");
      return OC_ERR_ARGUMENT;
    }
  std::vector<float> r(2 * OUT);
  for (int o = 0; o < OUT; ++o)
    {
      r[o] = (lo && o < m->n_out) ? lo[o] : -INFINITY;
      r[OUT + o] = (hi && o < m->n_out) ? hi[o] : INFINITY;
      if (!(r[o] <= r[OUT + o]))
        {
          set_error("oc_mlp_set_output_range: lo > hi");
          return OC_ERR_ARGUMENT;
        }
    }
  MLP_TRY(hipMemcpy(m->norm + NLO, r.data(), 2 * OUT * sizeof(float), hipMemcpyHostToDevice));
  return OC_OK;
}

int oc_mlp_forward(oc_mlp *m, int64_t n, const float *x, float *y, void *stream)
{
  if (!m || n < 0 || (n > 0 && (!x || !y)))
    {
      set_error("oc_mlp_forward: null argument");
      return OC_ERR_ARGUMENT;
    }
  if (n == 0)
    return OC_OK;
  const int64_t tiles = (n + 15) / 16;
  hipLaunchKernelGGL(k_mlp_forward, dim3((unsigned)std::min<int64_t>(tiles, 4096)), dim3(64), 0,
                     (hipStream_t)stream, m->p, m->wt, m->norm, n, m->n_in, m->n_out, x, y);
  MLP_TRY(hipGetLastError());
  return OC_OK;
}

int oc_mlp_gradients(oc_mlp *m, int64_t n, const float *x, const float *t, float *grad,
                     double *loss, void *stream)
{
  if (!m || n < 1 || !x || !t)
    {
      set_error("oc_mlp_gradients: null argument or empty batch");
      return OC_ERR_ARGUMENT;
    }
  hipStream_t s = (hipStream_t)stream;
  int G = 0;
  int rc = grad_launch(m, n, x, t, s, &G);
  if (rc)
    return rc;
  if (grad)
    {
      MLP_TRY(hipMemcpyAsync(grad, m->grad, NPARAM * sizeof(float), hipMemcpyDeviceToHost, s));
    }
  if (loss)
    {
      std::vector<float> lp(G);
      MLP_TRY(hipMemcpyAsync(lp.data(), m->lossp, G * sizeof(float), hipMemcpyDeviceToHost, s));
      MLP_TRY(hipStreamSynchronize(s));
      double acc = 0.0;
      for (int b = 0; b < G; ++b)
        acc += lp[b];
      *loss = acc / ((double)n * m->n_out);
    }
  else if (grad)
    MLP_TRY(hipStreamSynchronize(s));
  return OC_OK;
}

int oc_mlp_adam(oc_mlp *m, float lr, float beta1, float beta2, float eps, void *stream)
{
  if (!m || !(lr >= 0.f))
    {
      set_error("oc_mlp_adam: null argument or negative learning rate");
      return OC_ERR_ARGUMENT;
    }
  m->step += 1;
  const double t = (double)m->step;
  const float lr_t =
    float(lr * std::sqrt(1.0 - std::pow((double)beta2, t)) / (1.0 - std::pow((double)beta1, t)));
  hipLaunchKernelGGL(k_mlp_adam, dim3((NPARAM + 255) / 256), dim3(256), 0, (hipStream_t)stream,
                     m->p, m->m, m->v, m->grad, m->wt, m->wb, lr_t, beta1, beta2, eps);
  MLP_TRY(hipGetLastError());
  return OC_OK;
}

int oc_mlp_train_step(oc_mlp *m, int64_t n, const float *x, const float *t, float lr,
                      double *loss, void *stream)
{
  int rc = oc_mlp_gradients(m, n, x, t, nullptr, loss, stream);
  if (rc)
    return rc;
  return oc_mlp_adam(m, lr, 0.9f, 0.999f, 1e-8f, stream);
}

int oc_mlp_dims(const oc_mlp *m, int32_t *n_in, int32_t *n_out)
{
  if (!m)
    return OC_ERR_ARGUMENT;
  if (n_in)
    *n_in = m->n_in;
  if (n_out)
    *n_out = m->n_out;
  return OC_OK;
}

// device pointers for the in-stage inference (library internal)
void oc_mlp_device_state(const oc_mlp *m, const float **p, const uint16_t **wt,
                         const float **norm)
{
  *p = m->p;
  *wt = m->wt;
  *norm = m->norm;
}

}  // extern "C"
