// Learned step-size proposer: training kernels of the network in
// kmt_mlp.hpp (8 -> 64 -> 64 -> 1, tanh, tanh, linear).  FP16 weights for the
// forward pass, FP32 master weights for the optimizer, FP32 accumulation
// everywhere.  No reference counterpart (an extension of the path).
//
// Loss: mean squared error (1/S) sum_s (out_s - y_s)^2.
//
//   mlp_fwd_bwd_kernel  one wave per sample, one lane per hidden unit: the
//                       forward pass the batched controller runs
//                       (mlp_wave_forward), output delta, back-propagated
//                       deltas; stores h1, h2, d1, d2 (S x 64) and d3 (S)
//   mlp_grad_kernel     one wave per row of parameters, fixed-order sum over
//                       the samples (deterministic); in training it also
//                       applies the Adam update of the FP32 master weights
//                       and writes the FP16 copy
#include <hip/hip_runtime.h>

#include <algorithm>
#include <cmath>
#include <cstring>
#include <type_traits>
#include <vector>

#include "../../include/kuramoto_amd.h"
#include "kmt_common.hpp"
#include "kmt_kernels.hpp"
#include "kmt_mlp.hpp"
#include "kmt_rng.h"

namespace kmt {

__global__ __launch_bounds__(kBlock) void mlp_fwd_bwd_kernel(const uint16_t *w, const float *X, const float *y, int S,
                                                             float *H1, float *H2, float *D1, float *D2, float *D3,
                                                             float *out, double *loss_part) {
  __shared__ double lsum[kBlock / kWave];
  const int wv = threadIdx.x / kWave, i = threadIdx.x % kWave;
  const int s = blockIdx.x * (kBlock / kWave) + wv;
  const bool valid = s < S;
  float xs[kIn];
#pragma unroll
  for (int j = 0; j < kIn; ++j) xs[j] = valid ? X[(size_t)s * kIn + j] : 0.f;
  float h1, h2;
  const float o = mlp_wave_forward(w, xs, h1, h2);
  const float ys = valid ? y[s] : 0.f;
  const float d3 = valid ? 2.f * (o - ys) / (float)S : 0.f;
  // back-propagation: d2_i = d3 W3_i (1 - h2_i^2), d1_i = (sum_k W2_ki d2_k) (1 - h1_i^2)
  const float d2 = d3 * hf(w[kOffW3 + i]) * (1.f - h2 * h2);
  float g = 0.f;
  for (int k = 0; k < kHid; ++k) g = fmaf(hf(w[kOffW2 + k * kHid + i]), __shfl(d2, k, kWave), g);
  const float d1 = g * (1.f - h1 * h1);
  if (valid) {
    H1[(size_t)s * kHid + i] = h1;
    H2[(size_t)s * kHid + i] = h2;
    D1[(size_t)s * kHid + i] = d1;
    D2[(size_t)s * kHid + i] = d2;
    if (i == 0) {
      D3[s] = d3;
      if (out) out[s] = o;
    }
  }
  if (i == 0) lsum[wv] = valid ? (double)(o - ys) * (double)(o - ys) : 0.0;
  __syncthreads();
  if (threadIdx.x == 0) {
    double t = 0;
    for (int q = 0; q < kBlock / kWave; ++q) t += lsum[q];
    loss_part[blockIdx.x] = t;
  }
}

// Adam's constants of one update (c1, c2: the bias corrections).
struct AdamArgs {
  float *w32, *m, *v;
  uint16_t *w16;
  float lr, b1, b2, eps, c1, c2;
};

// Every parameter's gradient is a sum over the samples of a product of two
// numbers per sample.  One wave owns up to 64 parameters that share one of
// them: the stream V (lane l reads V[s][l], a coalesced row per sample)
// times the factor U (one number per sample, the same for all lanes):
//   waves  0..63  dW2[i][l] = sum_s D2[s][i] H1[s][l]     V = H1, U = D2 column i
//   waves 64..71  dW1[l][j] = sum_s D1[s][l] X[s][j]      V = D1, U = X column j
//   waves 72..75  db1[l], db2[l] (V = D1, D2), dW3[l] (V = H2, U = D3), db3 (U = D3)
// The sum runs over s in order, one fma per sample, so that training gives
// the same bits whatever the shape of the launch; the chain itself would take
// 4 to 8 cycles per sample.  What bounds it are its operands, about 30 cycles
// per sample: a wave waits for a cache round trip per register set.  One
// thread per parameter with both loads inside the loop waited for memory
// once per few samples (227 us for 1024 samples).  Here V is loaded kMlpU
// samples at a time into one of two register sets while the other is summed
// (up to 64 loads in flight, all the counter holds), and U 64 samples per
// load, lane l fetching sample l's, broadcast through LDS four at a time (a
// lane read per sample costs three issue slots of the chain's one): 13 us for
// 1024 samples, and an epoch of 32768 samples in 32 minibatches 8.4 -> 0.76 ms.
constexpr int kMlpU = 32;
constexpr int kMlpGradWaves = kHid + kIn + 4;

// sum_s U[s SU] V[s kHid + lane], s ascending (SU = 0: U is 1; !HAS_V: V is
// 1).  The 64 samples of a step are addressed through buffer resources that
// start at the step's first sample: a sample's place is then a constant
// offset, and samples past the end (never summed) read zeros with no clamp.
template <int SU, bool HAS_V>
__device__ __forceinline__ float mlp_sample_sum(const float *V, const float *U, int S, int lane, float *us) {
  static_assert(2 * kMlpU == kWave, "one factor load covers both register sets");
  auto rsrc = [&](const float *p, long s0, int stride) {
    const long left = S > s0 ? S - s0 : 0;
    return __builtin_amdgcn_make_buffer_rsrc(const_cast<float *>(p + s0 * stride), (short)0,
                                             (int)((left < kWave ? left : kWave) * stride * (long)sizeof(float)), 0x00020000);
  };
  // samples s0 + base .. s0 + base + kMlpU - 1
  auto load = [&](long s0, int base, float (&v)[kMlpU]) {
    if constexpr (HAS_V) {
      const __amdgpu_buffer_rsrc_t r = rsrc(V, s0, kHid);
#pragma unroll
      for (int q = 0; q < kMlpU; ++q)
        v[q] = __builtin_bit_cast(float, __builtin_amdgcn_raw_buffer_load_b32(r, (base + q) * kHid * 4 + lane * 4, 0, 0));
    }
  };
  auto factor = [&](long s0) {
    if constexpr (SU > 0) {
      return __builtin_bit_cast(float, __builtin_amdgcn_raw_buffer_load_b32(rsrc(U, s0, SU), lane * SU * 4, 0, 0));
    } else {
      return 1.f;
    }
  };
  float acc = 0.f;
  // samples base .. base + kMlpU - 1 of the step; TAIL: only the first `left`
  auto sum = [&](auto tail, const float (&v)[kMlpU], int base, int left) {
#pragma unroll
    for (int c = 0; c < kMlpU; c += 4) {
      f32x4 uq = {1.f, 1.f, 1.f, 1.f};
      if constexpr (SU > 0) uq = *reinterpret_cast<const f32x4 *>(&us[base + c]);
      const float u4[4] = {uq.x, uq.y, uq.z, uq.w};
#pragma unroll
      for (int q = 0; q < 4; ++q) {
        const float t = fmaf(u4[q], HAS_V ? v[c + q] : 1.f, acc);
        acc = !decltype(tail)::value || base + c + q < left ? t : acc;
      }
    }
  };
  float v0[kMlpU], v1[kMlpU];
  float u = factor(0);
  load(0, 0, v0);
  long s0 = 0;
  for (; s0 + kWave <= S; s0 += kWave) {
    if constexpr (SU > 0) us[lane] = u;
    u = factor(s0 + kWave);
    load(s0, kMlpU, v1);
    __builtin_amdgcn_sched_barrier(0);
    sum(std::false_type{}, v0, 0, 0);
    __builtin_amdgcn_sched_barrier(0);
    load(s0 + kWave, 0, v0);
    __builtin_amdgcn_sched_barrier(0);
    sum(std::false_type{}, v1, kMlpU, 0);
    __builtin_amdgcn_sched_barrier(0);
  }
  if (s0 < S) {
    if constexpr (SU > 0) us[lane] = u;
    load(s0, kMlpU, v1);
    sum(std::true_type{}, v0, 0, (int)(S - s0));
    sum(std::true_type{}, v1, kMlpU, (int)(S - s0));
  }
  return acc;
}

template <bool UPDATE>
__global__ __launch_bounds__(kWave) void mlp_grad_kernel(const float *X, int S, const float *H1, const float *H2,
                                                         const float *D1, const float *D2, const float *D3, float *grad,
                                                         const AdamArgs ad) {
  __shared__ __align__(16) float us[kWave];  // this step's factors, read back by every lane (one wave: no barrier)
  const int t = blockIdx.x, lane = threadIdx.x;
  float acc;
  int p;
  if (t < kHid) {
    acc = mlp_sample_sum<kHid, true>(H1, D2 + t, S, lane, us), p = kOffW2 + t * kHid + lane;
  } else if (t < kHid + kIn) {
    acc = mlp_sample_sum<kIn, true>(D1, X + (t - kHid), S, lane, us), p = kOffW1 + lane * kIn + (t - kHid);
  } else if (t < kHid + kIn + 2) {
    const bool first = t == kHid + kIn;
    acc = mlp_sample_sum<0, true>(first ? D1 : D2, nullptr, S, lane, us), p = (first ? kOffB1 : kOffB2) + lane;
  } else if (t == kHid + kIn + 2) {
    acc = mlp_sample_sum<1, true>(H2, D3, S, lane, us), p = kOffW3 + lane;
  } else {
    acc = mlp_sample_sum<1, false>(nullptr, D3, S, lane, us), p = kOffB3;
    if (lane != 0) return;
  }
  if constexpr (!UPDATE) {
    grad[p] = acc;
  } else {
    const float mm = ad.b1 * ad.m[p] + (1.f - ad.b1) * acc;
    const float vv = ad.b2 * ad.v[p] + (1.f - ad.b2) * acc * acc;
    ad.m[p] = mm;
    ad.v[p] = vv;
    const float wn = ad.w32[p] - ad.lr * (mm / ad.c1) / (sqrtf(vv / ad.c2) + ad.eps);
    ad.w32[p] = wn;
    ad.w16[p] = __builtin_bit_cast(uint16_t, (_Float16)wn);
  }
}

}  // namespace kmt

using namespace kmt;

struct kmt_mlp {
  int device = 0;
  hipStream_t stream = nullptr;
  float *w32 = nullptr, *m = nullptr, *v = nullptr, *grad = nullptr;
  uint16_t *w16 = nullptr;
  float *X = nullptr, *y = nullptr, *H1 = nullptr, *H2 = nullptr, *D1 = nullptr, *D2 = nullptr, *D3 = nullptr,
        *out = nullptr;
  double *lpart = nullptr;
  int cap = 0;
  long step = 0;

  ~kmt_mlp() {
    if (stream) (void)hipStreamSynchronize(stream);
    void *p[] = {w32, m, v, grad, w16, X, y, H1, H2, D1, D2, D3, out, lpart};
    for (void *q : p)
      if (q) (void)hipFree(q);
    if (stream) (void)hipStreamDestroy(stream);
  }

  int init(int dev, const float *w_init, uint32_t seed) {
    device = dev;
    HIP_TRY(hipSetDevice(device));
    HIP_TRY(hipStreamCreateWithFlags(&stream, hipStreamNonBlocking));
    HIP_TRY(hipMalloc((void **)&w32, sizeof(float) * kNParams));
    HIP_TRY(hipMalloc((void **)&m, sizeof(float) * kNParams));
    HIP_TRY(hipMalloc((void **)&v, sizeof(float) * kNParams));
    HIP_TRY(hipMalloc((void **)&grad, sizeof(float) * kNParams));
    HIP_TRY(hipMalloc((void **)&w16, sizeof(uint16_t) * kNParams));
    std::vector<float> w(kNParams, 0.f);
    if (w_init) {
      std::memcpy(w.data(), w_init, sizeof(float) * kNParams);
    } else {
      // Glorot-uniform weights from the library's Philox stream; zero biases
      // and a zero output layer (the untrained proposer returns the standard
      // controller's step).
      std::vector<double> u((size_t)kHid * kIn + (size_t)kHid * kHid);
      kmt::gaussian_factor((long)u.size(), 1, seed, u.data());
      const double s1 = std::sqrt(2.0 / (kIn + kHid)), s2 = std::sqrt(2.0 / (kHid + kHid));
      for (int q = 0; q < kHid * kIn; ++q) w[kOffW1 + q] = (float)(s1 * u[q]);
      for (int q = 0; q < kHid * kHid; ++q) w[kOffW2 + q] = (float)(s2 * u[kHid * kIn + q]);
    }
    std::vector<uint16_t> h(kNParams);
    for (int q = 0; q < kNParams; ++q) h[q] = __builtin_bit_cast(uint16_t, (_Float16)w[q]);
    HIP_TRY(hipMemcpyAsync(w32, w.data(), sizeof(float) * kNParams, hipMemcpyHostToDevice, stream));
    HIP_TRY(hipMemcpyAsync(w16, h.data(), sizeof(uint16_t) * kNParams, hipMemcpyHostToDevice, stream));
    HIP_TRY(hipMemsetAsync(m, 0, sizeof(float) * kNParams, stream));
    HIP_TRY(hipMemsetAsync(v, 0, sizeof(float) * kNParams, stream));
    HIP_TRY(hipStreamSynchronize(stream));
    return KMT_OK;
  }

  int ensure(int n) {
    if (n <= cap) return KMT_OK;
    void *p[] = {X, y, H1, H2, D1, D2, D3, out, lpart};
    for (void *q : p)
      if (q) (void)hipFree(q);
    cap = n;
    HIP_TRY(hipMalloc((void **)&X, sizeof(float) * kIn * n));
    HIP_TRY(hipMalloc((void **)&y, sizeof(float) * n));
    HIP_TRY(hipMalloc((void **)&H1, sizeof(float) * kHid * n));
    HIP_TRY(hipMalloc((void **)&H2, sizeof(float) * kHid * n));
    HIP_TRY(hipMalloc((void **)&D1, sizeof(float) * kHid * n));
    HIP_TRY(hipMalloc((void **)&D2, sizeof(float) * kHid * n));
    HIP_TRY(hipMalloc((void **)&D3, sizeof(float) * n));
    HIP_TRY(hipMalloc((void **)&out, sizeof(float) * n));
    HIP_TRY(hipMalloc((void **)&lpart, sizeof(double) * n));  // at most one block per sample (minibatches of 1)
    return KMT_OK;
  }

  // forward + backward over samples [s0, s0 + S) of the uploaded set, the
  // per-block loss partials to lp; then the gradient (ad: nullptr), or the
  // gradient and the Adam update
  void fwd_bwd(int s0, int S, double *lp, const AdamArgs *ad) {
    const int blocks = (S + 3) / 4;
    mlp_fwd_bwd_kernel<<<blocks, kBlock, 0, stream>>>(w16, X + (size_t)s0 * kIn, y + s0, S, H1, H2, D1, D2, D3,
                                                      out + s0, lp);
    if (ad)
      mlp_grad_kernel<true><<<kMlpGradWaves, kWave, 0, stream>>>(X + (size_t)s0 * kIn, S, H1, H2, D1, D2, D3, grad, *ad);
    else
      mlp_grad_kernel<false><<<kMlpGradWaves, kWave, 0, stream>>>(X + (size_t)s0 * kIn, S, H1, H2, D1, D2, D3, grad,
                                                                  AdamArgs{});
  }

  int upload(const float *Xh, const float *yh, int n) {
    KMT_TRY(ensure(n));
    HIP_TRY(hipMemcpyAsync(X, Xh, sizeof(float) * kIn * n, hipMemcpyHostToDevice, stream));
    if (yh) HIP_TRY(hipMemcpyAsync(y, yh, sizeof(float) * n, hipMemcpyHostToDevice, stream));
    else HIP_TRY(hipMemsetAsync(y, 0, sizeof(float) * n, stream));
    return KMT_OK;
  }

  // sums of the per-block loss partials of every minibatch of S samples in
  // n (in block order), added up in minibatch order
  int loss_sum(int n, int S, double *out) {
    const size_t per = ((size_t)S + 3) / 4, nb = (n - 1) / S;  // whole minibatches before the last
    const size_t blocks = nb * per + ((size_t)n - nb * S + 3) / 4;
    std::vector<double> lp(blocks);
    HIP_TRY(hipMemcpyAsync(lp.data(), lpart, sizeof(double) * blocks, hipMemcpyDeviceToHost, stream));
    HIP_TRY(hipStreamSynchronize(stream));
    double tot = 0;
    for (size_t b0 = 0; b0 < blocks; b0 += per) {
      double t = 0;
      for (size_t q = b0; q < std::min(b0 + per, blocks); ++q) t += lp[q];
      tot += t;
    }
    *out = tot;
    return KMT_OK;
  }
};

extern "C" {

int kmt_mlp_create(kmt_mlp **out, int device, const float *w_init, uint32_t seed) {
  if (!out) return kmt_fail(KMT_ERR_ARG, "out is NULL");
  *out = nullptr;
  int ndev = 0;
  HIP_TRY(hipGetDeviceCount(&ndev));
  if (device < 0 || device >= ndev) return kmt_fail(KMT_ERR_ARG, "device %d not present", device);
  kmt_mlp *m = new kmt_mlp();
  int rc = m->init(device, w_init, seed);
  if (rc != KMT_OK) {
    delete m;
    return rc;
  }
  *out = m;
  return KMT_OK;
}

int kmt_mlp_destroy(kmt_mlp *m) {
  delete m;
  return KMT_OK;
}

int kmt_mlp_get_weights(kmt_mlp *m, float *w32, uint16_t *w16) {
  if (!m) return kmt_fail(KMT_ERR_ARG, "mlp is NULL");
  if (w32) HIP_TRY(hipMemcpyAsync(w32, m->w32, sizeof(float) * kNParams, hipMemcpyDeviceToHost, m->stream));
  if (w16) HIP_TRY(hipMemcpyAsync(w16, m->w16, sizeof(uint16_t) * kNParams, hipMemcpyDeviceToHost, m->stream));
  HIP_TRY(hipStreamSynchronize(m->stream));
  return KMT_OK;
}

int kmt_mlp_forward(kmt_mlp *m, const float *Xh, int n, float *outh) {
  if (!m || !Xh || !outh || n < 1) return kmt_fail(KMT_ERR_ARG, "bad forward arguments");
  KMT_TRY(m->upload(Xh, nullptr, n));
  m->fwd_bwd(0, n, m->lpart, nullptr);
  HIP_TRY(hipGetLastError());
  HIP_TRY(hipMemcpyAsync(outh, m->out, sizeof(float) * n, hipMemcpyDeviceToHost, m->stream));
  HIP_TRY(hipStreamSynchronize(m->stream));
  return KMT_OK;
}

int kmt_mlp_loss_grad(kmt_mlp *m, const float *Xh, const float *yh, int n, double *loss, float *gradh) {
  if (!m || !Xh || !yh || n < 1) return kmt_fail(KMT_ERR_ARG, "bad gradient arguments");
  KMT_TRY(m->upload(Xh, yh, n));
  m->fwd_bwd(0, n, m->lpart, nullptr);
  HIP_TRY(hipGetLastError());
  if (gradh) HIP_TRY(hipMemcpyAsync(gradh, m->grad, sizeof(float) * kNParams, hipMemcpyDeviceToHost, m->stream));
  HIP_TRY(hipStreamSynchronize(m->stream));
  if (loss) {
    double t = 0;
    KMT_TRY(m->loss_sum(n, n, &t));
    *loss = t / n;
  }
  return KMT_OK;
}

int kmt_mlp_train(kmt_mlp *m, const float *Xh, const float *yh, int n, int epochs, int batch, double lr,
                  double *loss_history) {
  if (!m || !Xh || !yh || n < 1 || epochs < 1 || batch < 1) return kmt_fail(KMT_ERR_ARG, "bad training arguments");
  KMT_TRY(m->upload(Xh, yh, n));
  const float b1 = 0.9f, b2 = 0.999f, eps = 1e-8f;
  // the launches of an epoch are queued back to back, each minibatch's loss
  // partials in their own place; the host waits once per epoch
  for (int ep = 0; ep < epochs; ++ep) {
    double *lp = m->lpart;
    for (int s0 = 0; s0 < n; s0 += std::min(batch, n - s0)) {
      const int S = std::min(batch, n - s0);
      ++m->step;
      const float c1 = 1.f - std::pow(b1, (float)m->step), c2 = 1.f - std::pow(b2, (float)m->step);
      const AdamArgs ad{m->w32, m->m, m->v, m->w16, (float)lr, b1, b2, eps, c1, c2};
      m->fwd_bwd(s0, S, lp, &ad);
      HIP_TRY(hipGetLastError());
      lp += (S + 3) / 4;
    }
    double tot = 0;
    KMT_TRY(m->loss_sum(n, std::min(batch, n), &tot));
    if (loss_history) loss_history[ep] = tot / n;
  }
  HIP_TRY(hipStreamSynchronize(m->stream));
  return KMT_OK;
}

}  // extern "C"
