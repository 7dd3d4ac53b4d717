// mlp.hip -- training and inference of the learned con2prim pressure guess
// (3 -> 64 -> 64 -> 1, ReLU, bf16 weights with FP32 masters and FP32
// accumulation, Adam) on gfx950.  No reference counterpart.
//
// Training step: one block per 64 samples (mlp_train_kernel) runs the forward
// pass, the MSE loss and the backward pass:
//   dW3, db2, db3: per-feature sums over the block's points (LDS);
//   dW2 = dZ2 . H1 and dH1^T = W2^T . dZ2 on the matrix cores (bf16 operands,
//   FP32 accumulate), the same 32x32x16 layout as the forward pass;
//   dW1, db1: per-unit sums over the block's points (LDS);
// and writes its partial gradient.  mlp_update_kernel sums the partials in a
// fixed order (deterministic), applies Adam to the FP32 masters and refreshes
// the bf16 working copies.
#include <algorithm>
#include <cmath>
#include <random>
#include <vector>

#include "bamhip_internal.h"
#include "mlp_device.h"

struct bamhip_mlp {
  float *p = nullptr;       // FP32 masters
  float *mom = nullptr;     // Adam first moment
  float *vel = nullptr;     // Adam second moment
  float *wq = nullptr;      // bf16-rounded W1, W3 as float (256)
  __bf16 *w2 = nullptr;     // [f][k]
  __bf16 *w2t = nullptr;    // [k][f]
  float norm[8] = {0, 0, 0, 1, 1, 1, 0, 1};  // xs[3], xk[3], ys, yk
  long step = 0;
  float *part = nullptr;    // per-wave partial gradients
  long part_blocks = 0;
  float *lossp = nullptr;   // per-wave loss partials
  float *grad = nullptr;    // reduced gradient (for bamhip_mlp_grad)
};

namespace bamhip {

MlpView mlp_view(const bamhip_mlp *m) {
  MlpView v;
  v.p = m->p;
  v.wq = m->wq;
  v.w2 = m->w2;
  v.w2t = m->w2t;
  for (int i = 0; i < 3; i++) {
    v.xs[i] = m->norm[i];
    v.xk[i] = m->norm[3 + i];
  }
  v.ys = m->norm[6];
  v.yk = m->norm[7];
  return v;
}

namespace {

constexpr int kWave = 64;

// Four wavefronts per 64 samples: the batch is small (4096 samples are 64
// blocks), so the kernel is one block's chain of latencies.  Each wavefront takes
// 16 units of layer 1, one 32x32 tile of every contraction and 16 samples of
// every per-feature sum; with one wavefront a block took all of them in turn
// (16.6 us for 4096 samples, now 8.0).
constexpr int kTrainWaves = 4;

__global__ void __launch_bounds__(kWave *kTrainWaves)
    mlp_train_kernel(MlpView M, const float *__restrict__ feat, const float *__restrict__ target, long n, long q0,
                     long batch, unsigned long long pa, unsigned long long pb, float *__restrict__ part,
                     float *__restrict__ lossp, float inv_batch) {
  __shared__ __attribute__((aligned(16))) __bf16 h1[kWave * kHStr];    // [pt][k]
  __shared__ __attribute__((aligned(16))) __bf16 h1t[kMlpH * kHStr];   // [k][pt]
  __shared__ __attribute__((aligned(16))) __bf16 dz2[kMlpH * kHStr];   // [f][pt]
  __shared__ __attribute__((aligned(16))) __bf16 dz2t[kWave * kHStr];  // [pt][f]
  __shared__ float h2[kMlpH * (kWave + 1)];                            // [f][pt]
  __shared__ float dz1[kMlpH * (kWave + 1)];                           // [k][pt]
  __shared__ float xsh[kWave * 3], ts[kWave], dys[kWave], ysum[2][kWave];
  __shared__ float red[kTrainWaves][7][kMlpH];  // per wave: dW3, db2, db3, dW1 (3), db1
  const int l = threadIdx.x % kWave, w = __builtin_amdgcn_readfirstlane(threadIdx.x / kWave);
  const int lr = l % 32, lh = l / 32, m = w / 2, n2 = w % 2;  // the wave's tile: rows 32m.., columns 32 n2..
  const long slot = (long)blockIdx.x * kWave + l;
  // ---- sample: a fixed affine permutation of [0, n) per epoch
  bool valid = slot < batch && q0 + slot < n;
  float x[3] = {0.f, 0.f, 0.f}, t = 0.f;
  if (valid) {
    const long idx = (long)((pa * (unsigned long long)(q0 + slot) + pb) % (unsigned long long)n);
    for (int j = 0; j < 3; j++) x[j] = (feat[3 * idx + j] - M.xs[j]) * M.xk[j];
    t = (target[idx] - M.ys) / M.yk;
    valid = isfinite(x[0]) && isfinite(x[1]) && isfinite(x[2]) && isfinite(t);
    if (!valid) x[0] = x[1] = x[2] = t = 0.f;
  }
  if (w == 0) {
    for (int j = 0; j < 3; j++) xsh[3 * l + j] = x[j];
    ts[l] = valid ? t : __builtin_nanf("");
  }
  // ---- forward: layer 1, units 16 w .. 16 w + 15 of every point
#pragma unroll
  for (int k0 = 0; k0 < 16; k0 += 8) {
    bf16x8 h;
#pragma unroll
    for (int e = 0; e < 8; e++) {
      const int k = 16 * w + k0 + e;
      h[e] = (__bf16)fmaxf(mlp_z1(M, k, x), 0.f);
      h1t[k * kHStr + l] = h[e];
    }
    *(bf16x8 *)(h1 + l * kHStr + 16 * w + k0) = h;
  }
  __syncthreads();
  // ---- layer 2: features 32m.., points 32 n2..; layer 3 summed over the features
  f32x16 c;
#pragma unroll
  for (int v = 0; v < 16; v++) c[v] = 0.f;
#pragma unroll
  for (int s = 0; s < 4; s++) {
    const bf16x8 b = *(const bf16x8 *)(h1 + (32 * n2 + lr) * kHStr + 16 * s + 8 * lh);
    const bf16x8 a = *(const bf16x8 *)(M.w2 + (32 * m + lr) * kMlpH + 16 * s + 8 * lh);
    c = __builtin_amdgcn_mfma_f32_32x32x16_bf16(a, b, c, 0, 0, 0);
  }
  float w3[16], yp = 0.f;
#pragma unroll
  for (int v = 0; v < 16; v++) {
    const int f = 32 * m + mfma_row(v, l);
    w3[v] = M.wq[192 + f];
    c[v] = fmaxf(c[v] + M.p[kOffB2 + f], 0.f);
    yp = fmaf(c[v], w3[v], yp);
  }
  yp += __shfl_xor(yp, 32);
  if (lh == 0) ysum[m][32 * n2 + lr] = yp;
  __syncthreads();
  const float y = ysum[0][l] + ysum[1][l] + M.p[kOffB3], tl = ts[l];
  const float r = isfinite(tl) ? y - tl : 0.f;
  const float dy = 2.f * r * inv_batch;
  if (w == 0) {
    float lsum = r * r;
    for (int o = 32; o > 0; o >>= 1) lsum += __shfl_xor(lsum, o);
    if (l == 0) lossp[blockIdx.x] = lsum;
    dys[l] = dy;
  }
  // ---- dZ2 = relu'(z2) * W3 * dy, kept as bf16 in both layouts; h2 kept in FP32
  {
    const int pt = 32 * n2 + lr;
    const float dyp = __shfl(dy, pt);
#pragma unroll
    for (int v = 0; v < 16; v++) {
      const int f = 32 * m + mfma_row(v, l);
      const float dz = c[v] > 0.f ? w3[v] * dyp : 0.f;
      h2[f * (kWave + 1) + pt] = c[v];
      dz2[f * kHStr + pt] = (__bf16)dz;
      dz2t[pt * kHStr + f] = (__bf16)dz;
    }
  }
  __syncthreads();
  float *g = part + (long)blockIdx.x * kMlpNParam;
  {
    // lane f, points 16 w ..: dW3[f], db2[f], db3
    const float w3f = M.wq[192 + l];
    float gw3 = 0.f, gb2 = 0.f, gb3 = 0.f;
#pragma unroll
    for (int e = 0; e < 16; e++) {
      const int pt = 16 * w + e;
      const float h = h2[l * (kWave + 1) + pt], d = dys[pt];
      gw3 = fmaf(h, d, gw3);
      gb2 += h > 0.f ? w3f * d : 0.f;
      gb3 += d;
    }
    red[w][0][l] = gw3;
    red[w][1][l] = gb2;
    red[w][2][l] = gb3;
  }
  f32x16 acc, acch;
#pragma unroll
  for (int v = 0; v < 16; v++) acc[v] = acch[v] = 0.f;
  // ---- dW2[f][k] = sum_pt dZ2[f][pt] H1[pt][k]   (A = dZ2, B = H1 with K = points)
  // ---- dH1^T[k][pt] = sum_f W2[f][k] dZ2[f][pt]   (A = W2^T, B = dZ2 with K = features)
#pragma unroll
  for (int s = 0; s < 4; s++) {
    const bf16x8 a = *(const bf16x8 *)(dz2 + (32 * m + lr) * kHStr + 16 * s + 8 * lh);
    const bf16x8 b = *(const bf16x8 *)(h1t + (32 * n2 + lr) * kHStr + 16 * s + 8 * lh);
    acc = __builtin_amdgcn_mfma_f32_32x32x16_bf16(a, b, acc, 0, 0, 0);
    const bf16x8 ah = *(const bf16x8 *)(M.w2t + (32 * m + lr) * kMlpH + 16 * s + 8 * lh);
    const bf16x8 bh = *(const bf16x8 *)(dz2t + (32 * n2 + lr) * kHStr + 16 * s + 8 * lh);
    acch = __builtin_amdgcn_mfma_f32_32x32x16_bf16(ah, bh, acch, 0, 0, 0);
  }
#pragma unroll
  for (int v = 0; v < 16; v++) {
    g[kOffW2 + (32 * m + mfma_row(v, l)) * kMlpH + 32 * n2 + lr] = acc[v];
    // dZ1 = relu'(z1) * dH1, with the forward pass's mask (h1 > 0)
    const int k = 32 * m + mfma_row(v, l), pt = 32 * n2 + lr;
    const bool on = (float)h1[pt * kHStr + k] > 0.f;
    dz1[k * (kWave + 1) + pt] = on ? acch[v] : 0.f;
  }
  __syncthreads();
  {
    // lane k, points 16 w ..: dW1[k][0..2], db1[k]
    float gw[3] = {0.f, 0.f, 0.f}, gb = 0.f;
#pragma unroll
    for (int e = 0; e < 16; e++) {
      const int pt = 16 * w + e;
      const float d = dz1[l * (kWave + 1) + pt];
      gb += d;
      for (int j = 0; j < 3; j++) gw[j] = fmaf(d, xsh[3 * pt + j], gw[j]);
    }
    for (int j = 0; j < 3; j++) red[w][3 + j][l] = gw[j];
    red[w][6][l] = gb;
  }
  __syncthreads();
  // the waves' sums, in wave order
  for (int i = threadIdx.x; i < 7 * kMlpH; i += kWave * kTrainWaves) {
    const int what = i / kMlpH, k = i % kMlpH;
    const float v = ((red[0][what][k] + red[1][what][k]) + red[2][what][k]) + red[3][what][k];
    if (what == 0) g[kOffW3 + k] = v;
    else if (what == 1) g[kOffB2 + k] = v;
    else if (what == 2) {
      if (k == 0) g[kOffB3] = v;
    } else if (what < 6) g[kOffW1 + 3 * k + (what - 3)] = v;
    else g[kOffB1 + k] = v;
  }
}

// Gradient reduction in a fixed order, Adam on the masters (skipped when lr ==
// 0), bf16 working copies.  A block takes kUpdP parameters and sums each one's
// block partials in kUpdS slices (partials s, s + kUpdS, ...), then the slices
// in order: with one thread per parameter, its 64 partials were a chain of
// loads in 18 blocks (16.3 us, now 4.4).
constexpr int kUpdP = 32, kUpdS = 16;
__global__ void __launch_bounds__(kUpdP *kUpdS)
    mlp_update_kernel(float *__restrict__ p, float *__restrict__ mom, float *__restrict__ vel, float *__restrict__ wq,
                      __bf16 *__restrict__ w2, __bf16 *__restrict__ w2t, const float *__restrict__ part, int nblk,
                      float *__restrict__ grad, float lr, float beta1, float beta2, float eps, float bc1, float bc2) {
  __shared__ float sums[kUpdS][kUpdP];
  const int i = blockIdx.x * kUpdP + threadIdx.x % kUpdP, sl = threadIdx.x / kUpdP;
  float gs = 0.f;
  if (i < kMlpNParam) {
#pragma unroll 4
    for (int b = sl; b < nblk; b += kUpdS) gs += part[(long)b * kMlpNParam + i];
  }
  sums[sl][threadIdx.x % kUpdP] = gs;
  __syncthreads();
  if (sl != 0 || i >= kMlpNParam) return;
  if (nblk > 0) {
#pragma unroll
    for (int s = 1; s < kUpdS; s++) gs += sums[s][threadIdx.x];
    if (grad) grad[i] = gs;
    if (lr > 0.f) {
      const float m1 = beta1 * mom[i] + (1.f - beta1) * gs;
      const float v1 = beta2 * vel[i] + (1.f - beta2) * gs * gs;
      mom[i] = m1;
      vel[i] = v1;
      p[i] -= lr * (m1 / bc1) / (sqrtf(v1 / bc2) + eps);
    }
  }
  const float w = p[i];
  if (i < kOffB1) wq[i] = (float)(__bf16)w;
  else if (i >= kOffW3 && i < kOffB3) wq[192 + (i - kOffW3)] = (float)(__bf16)w;
  else if (i >= kOffW2 && i < kOffB2) {
    const int f = (i - kOffW2) / kMlpH, k = (i - kOffW2) % kMlpH;
    w2[f * kMlpH + k] = (__bf16)w;
    w2t[k * kMlpH + f] = (__bf16)w;
  }
}

// network output (log(p / p_hi)) for n raw feature triples
__global__ void __launch_bounds__(256) mlp_predict_kernel(MlpView M, const float *__restrict__ feat, long n,
                                                          float *__restrict__ y) {
  __shared__ __attribute__((aligned(16))) __bf16 h1[4][kWave * kHStr];
  const int w = threadIdx.x / kWave, l = threadIdx.x % kWave;
  for (long base = (long)blockIdx.x * 256; base < n; base += (long)gridDim.x * 256) {
    const long q = base + threadIdx.x;
    float x[3] = {0.f, 0.f, 0.f};
    if (q < n)
      for (int j = 0; j < 3; j++) x[j] = (feat[3 * q + j] - M.xs[j]) * M.xk[j];
    mlp_layer1(M, x, h1[w] + l * kHStr);
    __syncthreads();
    f32x16 c[2][2];
    const float yn = mlp_layer23(M, h1[w], c, M.p + kOffB2, M.wq + 192);
    if (q < n) y[q] = M.ys + M.yk * yn;
    __syncthreads();
  }
}

int ensure_part(bamhip_mlp *m, long nblk) {
  if (nblk <= m->part_blocks) return BAMHIP_OK;
  if (m->part) (void)hipFree(m->part);
  if (m->lossp) (void)hipFree(m->lossp);
  m->part = nullptr;
  m->lossp = nullptr;
  m->part_blocks = 0;
  BH_HIP(hipMalloc(&m->part, sizeof(float) * kMlpNParam * nblk));
  BH_HIP(hipMalloc(&m->lossp, sizeof(float) * nblk));
  m->part_blocks = nblk;
  return BAMHIP_OK;
}

int refresh(bamhip_mlp *m) {
  mlp_update_kernel<<<(kMlpNParam + kUpdP - 1) / kUpdP, kUpdP * kUpdS, 0, stream()>>>(m->p, m->mom, m->vel, m->wq, m->w2, m->w2t,
                                                                    nullptr, 0, nullptr, 0.f, 0.f, 0.f, 0.f, 1.f,
                                                                    1.f);
  BH_HIP(hipGetLastError());
  return BAMHIP_OK;
}

// one optimisation step over `batch` samples starting at permuted position q0
int train_step(bamhip_mlp *m, const float *feat, const float *target, long n, long q0, long batch,
               unsigned long long pa, unsigned long long pb, float lr, float *grad_out) {
  const long nblk = (batch + kWave - 1) / kWave;
  if (int e = ensure_part(m, nblk)) return e;
  mlp_train_kernel<<<(unsigned)nblk, kWave * kTrainWaves, 0, stream()>>>(mlp_view(m), feat, target, n, q0, batch, pa, pb, m->part,
                                                           m->lossp, 1.f / (float)batch);
  BH_HIP(hipGetLastError());
  const float b1 = 0.9f, b2 = 0.999f;
  if (lr > 0.f) m->step++;
  const float bc1 = 1.f - powf(b1, (float)std::max<long>(m->step, 1));
  const float bc2 = 1.f - powf(b2, (float)std::max<long>(m->step, 1));
  mlp_update_kernel<<<(kMlpNParam + kUpdP - 1) / kUpdP, kUpdP * kUpdS, 0, stream()>>>(m->p, m->mom, m->vel, m->wq, m->w2, m->w2t,
                                                                    m->part, (int)nblk, grad_out, lr, b1, b2,
                                                                    1e-8f, bc1, bc2);
  BH_HIP(hipGetLastError());
  return BAMHIP_OK;
}

unsigned long long gcd64(unsigned long long a, unsigned long long b) {
  while (b) {
    const unsigned long long t = a % b;
    a = b;
    b = t;
  }
  return a;
}

}  // namespace
}  // namespace bamhip

using namespace bamhip;

extern "C" {

int bamhip_mlp_create(bamhip_mlp **out, unsigned long long seed) {
  if (!out) return set_error(BAMHIP_EINVAL, "bamhip_mlp_create: NULL");
  bamhip_mlp *m = new bamhip_mlp();
  const size_t np = sizeof(float) * kMlpNParam;
  if (hipMalloc(&m->p, np) != hipSuccess || hipMalloc(&m->mom, np) != hipSuccess ||
      hipMalloc(&m->vel, np) != hipSuccess || hipMalloc(&m->wq, sizeof(float) * 256) != hipSuccess ||
      hipMalloc(&m->w2, sizeof(__bf16) * kMlpH * kMlpH) != hipSuccess ||
      hipMalloc(&m->w2t, sizeof(__bf16) * kMlpH * kMlpH) != hipSuccess ||
      hipMalloc(&m->grad, np) != hipSuccess) {
    bamhip_mlp_free(m);
    return set_error(BAMHIP_ENOMEM, "bamhip_mlp_create: out of device memory");
  }
  // He-normal initialisation for the ReLU layers, small output layer, zero biases
  std::vector<float> h(kMlpNParam, 0.f);
  std::mt19937_64 rng(seed);
  std::normal_distribution<double> nd(0.0, 1.0);
  for (int i = 0; i < 192; i++) h[kOffW1 + i] = (float)(nd(rng) * std::sqrt(2.0 / 3.0));
  for (int i = 0; i < kMlpH * kMlpH; i++) h[kOffW2 + i] = (float)(nd(rng) * std::sqrt(2.0 / kMlpH));
  for (int i = 0; i < kMlpH; i++) h[kOffW3 + i] = (float)(nd(rng) * std::sqrt(1.0 / kMlpH));
  hipStream_t st = stream();
  if (hipMemcpyAsync(m->p, h.data(), np, hipMemcpyHostToDevice, st) != hipSuccess ||
      hipMemsetAsync(m->mom, 0, np, st) != hipSuccess || hipMemsetAsync(m->vel, 0, np, st) != hipSuccess ||
      hipStreamSynchronize(st) != hipSuccess) {
    bamhip_mlp_free(m);
    return set_error(BAMHIP_EDEVICE, "bamhip_mlp_create: initialisation failed");
  }
  if (int e = refresh(m)) {
    bamhip_mlp_free(m);
    return e;
  }
  *out = m;
  return BAMHIP_OK;
}

int bamhip_mlp_free(bamhip_mlp *m) {
  if (!m) return BAMHIP_OK;
  (void)hipStreamSynchronize(stream());
  for (void *p : {(void *)m->p, (void *)m->mom, (void *)m->vel, (void *)m->wq, (void *)m->w2, (void *)m->w2t,
                  (void *)m->part, (void *)m->lossp, (void *)m->grad})
    if (p) (void)hipFree(p);
  delete m;
  return BAMHIP_OK;
}

int bamhip_mlp_get_params(const bamhip_mlp *m, float *params, float *norm) {
  if (!m) return set_error(BAMHIP_EINVAL, "bamhip_mlp_get_params: NULL model");
  if (params) {
    BH_HIP(hipMemcpyAsync(params, m->p, sizeof(float) * kMlpNParam, hipMemcpyDeviceToHost, stream()));
    BH_HIP(hipStreamSynchronize(stream()));
  }
  if (norm) std::copy(m->norm, m->norm + 8, norm);
  return BAMHIP_OK;
}

int bamhip_mlp_set_params(bamhip_mlp *m, const float *params, const float *norm) {
  if (!m) return set_error(BAMHIP_EINVAL, "bamhip_mlp_set_params: NULL model");
  if (norm) {
    for (int i = 3; i < 6; i++)
      if (!(norm[i] != 0.f) || !std::isfinite(norm[i]))
        return set_error(BAMHIP_EINVAL, "bamhip_mlp_set_params: input scale %d is %g", i - 3, (double)norm[i]);
    if (!(norm[7] != 0.f)) return set_error(BAMHIP_EINVAL, "bamhip_mlp_set_params: output scale is 0");
    std::copy(norm, norm + 8, m->norm);
  }
  if (params) {
    const size_t np = sizeof(float) * kMlpNParam;
    BH_HIP(hipMemcpyAsync(m->p, params, np, hipMemcpyHostToDevice, stream()));
    BH_HIP(hipMemsetAsync(m->mom, 0, np, stream()));
    BH_HIP(hipMemsetAsync(m->vel, 0, np, stream()));
    BH_HIP(hipStreamSynchronize(stream()));
    m->step = 0;
    if (int e = refresh(m)) return e;
  }
  return BAMHIP_OK;
}

int bamhip_mlp_grad(bamhip_mlp *m, long n, const float *feat, const float *target, float *grad, float *loss) {
  if (!m || !feat || !target || n < 1) return set_error(BAMHIP_EINVAL, "bamhip_mlp_grad: bad arguments");
  if (int e = train_step(m, feat, target, n, 0, n, 1ULL, 0ULL, 0.f, m->grad)) return e;
  const long nblk = (n + kWave - 1) / kWave;
  std::vector<float> lp(nblk);
  if (grad) BH_HIP(hipMemcpyAsync(grad, m->grad, sizeof(float) * kMlpNParam, hipMemcpyDeviceToHost, stream()));
  BH_HIP(hipMemcpyAsync(lp.data(), m->lossp, sizeof(float) * nblk, hipMemcpyDeviceToHost, stream()));
  BH_HIP(hipStreamSynchronize(stream()));
  if (loss) {
    double s = 0;
    for (float v : lp) s += v;
    *loss = (float)(s / n);
  }
  return BAMHIP_OK;
}

int bamhip_mlp_train(bamhip_mlp *m, long n, const float *feat, const float *target, int epochs, long batch,
                     float lr, unsigned long long seed, float *epoch_loss) {
  if (!m || !feat || !target || n < 1 || epochs < 1 || batch < kWave || lr <= 0.f)
    return set_error(BAMHIP_EINVAL, "bamhip_mlp_train: bad arguments");
  std::mt19937_64 rng(seed);
  const long steps_per_epoch = (n + batch - 1) / batch;
  const long total = steps_per_epoch * epochs;
  const long nblk = (batch + kWave - 1) / kWave;
  long t = 0;
  std::vector<float> lp(nblk);
  TimerScope ts("mlp_train");
  for (int ep = 0; ep < epochs; ep++) {
    // affine permutation q -> (a q + b) mod n with gcd(a, n) = 1
    unsigned long long a;
    do {
      a = (rng() % (unsigned long long)n) | 1ULL;
    } while (gcd64(a, (unsigned long long)n) != 1ULL);
    const unsigned long long b = rng() % (unsigned long long)n;
    double lsum = 0;
    for (long s = 0; s < steps_per_epoch; s++, t++) {
      const long q0 = s * batch;
      const long bs = std::min(batch, n - q0);
      const float lrt = lr * (0.02f + 0.98f * 0.5f * (1.f + cosf(3.14159265f * (float)t / (float)total)));
      if (int e = train_step(m, feat, target, n, q0, bs, a, b, lrt, nullptr)) return e;
      if (epoch_loss && s == steps_per_epoch - 1) {
        const long nb = (bs + kWave - 1) / kWave;
        BH_HIP(hipMemcpyAsync(lp.data(), m->lossp, sizeof(float) * nb, hipMemcpyDeviceToHost, stream()));
        BH_HIP(hipStreamSynchronize(stream()));
        for (long i = 0; i < nb; i++) lsum += lp[i];
        epoch_loss[ep] = (float)(lsum / bs);
      }
    }
  }
  return BAMHIP_OK;
}

int bamhip_mlp_predict(const bamhip_mlp *m, long n, const float *feat, float *y) {
  if (!m || !feat || !y || n < 0) return set_error(BAMHIP_EINVAL, "bamhip_mlp_predict: bad arguments");
  if (n == 0) return BAMHIP_OK;
  long blocks = std::min<long>((n + 255) / 256, 4096);
  TimerScope ts("mlp");
  mlp_predict_kernel<<<(unsigned)blocks, 256, 0, stream()>>>(mlp_view(m), feat, n, y);
  BH_HIP(hipGetLastError());
  return BAMHIP_OK;
}

}  // extern "C"
