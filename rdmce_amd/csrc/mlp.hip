// Learned root-cost model: per-root features and a small FP32 MLP
// (8 -> 32 -> 32 -> 1, ReLU) trained with Adam, all in HIP.
//
// The model predicts log(1 + cost) of an edge root from cheap structural
// features; the scheduler orders roots by predicted cost and splits the
// heaviest before launch.  It never changes results, only the order and
// the eager-split flags (see mce_kernel.hip).
//
// Backward is deterministic: each block writes its partial gradient for a
// fixed slice of the minibatch, and a second kernel sums the partials in
// block order.
#include <hip/hip_runtime.h>

#include <cstdint>

#include "mlp.hpp"

namespace rdmce {
namespace {

__device__ __forceinline__ uint64_t lower_bound_u32(const uint32_t *a, uint64_t lo, uint64_t hi, uint32_t key) {
  while (lo < hi) {
    uint64_t mid = (lo + hi) >> 1;
    if (a[mid] < key) lo = mid + 1;
    else hi = mid;
  }
  return lo;
}

// Features of edge root (v0, v1), v0 < v1:
//   log1p(deg v0), log1p(deg v1), core v0 / degeneracy, core v1 / degeneracy,
//   log1p(outdeg v0), log1p(outdeg v1), log1p(t), log1p(t)^2
// where t = |N+(v1) ^ N(v0)| counts the triangles (v0, v1, w) with w above
// v1 - the size of the root's candidate set P.  One thread per root.
__global__ __launch_bounds__(256) void features_kernel(const uint64_t *rowoff, const uint32_t *col,
                                                       const uint32_t *core, float inv_degen, const uint64_t *roots,
                                                       uint64_t n_roots, float *out) {
  uint64_t r = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (r >= n_roots) return;
  uint32_t v0 = (uint32_t)(roots[r] >> 32), v1 = (uint32_t)roots[r];
  uint64_t b0 = rowoff[v0], e0 = rowoff[v0 + 1], b1 = rowoff[v1], e1 = rowoff[v1 + 1];
  uint64_t f0 = lower_bound_u32(col, b0, e0, v0 + 1), f1 = lower_bound_u32(col, b1, e1, v1 + 1);
  // t: entries of N+(v1) found in N(v0) above v1
  uint64_t lo = lower_bound_u32(col, b0, e0, v1 + 1);
  uint32_t t = 0;
  for (uint64_t i = f1; i < e1 && lo < e0; ++i) {
    lo = lower_bound_u32(col, lo, e0, col[i]);
    if (lo < e0 && col[lo] == col[i]) ++t;
  }
  float lt = log1pf((float)t);
  float *o = out + r * kFeat;
  o[0] = log1pf((float)(e0 - b0));
  o[1] = log1pf((float)(e1 - b1));
  o[2] = (float)core[v0] * inv_degen;
  o[3] = (float)core[v1] * inv_degen;
  o[4] = log1pf((float)(e0 - f0));
  o[5] = log1pf((float)(e1 - f1));
  o[6] = lt;
  o[7] = lt * lt;
}

// Parameter layout (floats): W1[kFeat][kH1] b1[kH1] W2[kH1][kH2] b2[kH2]
// W3[kH2] b3, plus per-feature normalisation mean[kFeat] inv_std[kFeat]
// (not trained).
struct Params {
  const float *W1, *b1, *W2, *b2, *W3, *b3, *mean, *istd;
};
__device__ __forceinline__ Params params_at(const float *p) {
  Params q;
  q.W1 = p;
  q.b1 = q.W1 + kFeat * kH1;
  q.W2 = q.b1 + kH1;
  q.b2 = q.W2 + kH1 * kH2;
  q.W3 = q.b2 + kH2;
  q.b3 = q.W3 + kH2;
  q.mean = q.b3 + 1;
  q.istd = q.mean + kFeat;
  return q;
}

// Forward for one sample; keeps activations for backward.
__device__ __forceinline__ float forward_one(const Params &q, const float *x, float *xn, float *h1, float *h2) {
  // Fully unrolled: the activation arrays stay in registers, indexed by
  // constants only.
#pragma unroll
  for (int i = 0; i < kFeat; ++i) xn[i] = (x[i] - q.mean[i]) * q.istd[i];
#pragma unroll
  for (int j = 0; j < kH1; ++j) {
    float s = q.b1[j];
#pragma unroll
    for (int i = 0; i < kFeat; ++i) s = fmaf(xn[i], q.W1[i * kH1 + j], s);
    h1[j] = s > 0.f ? s : 0.f;
  }
#pragma unroll
  for (int j = 0; j < kH2; ++j) {
    float s = q.b2[j];
#pragma unroll
    for (int i = 0; i < kH1; ++i) s = fmaf(h1[i], q.W2[i * kH2 + j], s);
    h2[j] = s > 0.f ? s : 0.f;
  }
  float y = q.b3[0];
  for (int i = 0; i < kH2; ++i) y = fmaf(h2[i], q.W3[i], y);
  return y;
}

__global__ __launch_bounds__(256) void forward_kernel(const float *params, const float *X, uint64_t n, float *out) {
  __shared__ float sp[kParamFloats];
  for (int i = threadIdx.x; i < kParamFloats; i += blockDim.x) sp[i] = params[i];
  __syncthreads();
  uint64_t r = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (r >= n) return;
  Params q = params_at(sp);
  float xn[kFeat], h1[kH1], h2[kH2];
  out[r] = forward_one(q, X + r * kFeat, xn, h1, h2);
}

// One training step's gradient, and before it, when `apply` names one, the
// reduction and Adam update of the previous step.
//
// Gradient of the mean squared error over samples idx[0 .. count) (scaled by
// 1/count): block b takes samples [b*kRows, (b+1)*kRows).  Wave w computes
// hidden units 2w and 2w+1 of every sample (lane = sample, weights broadcast),
// the activations and back-propagated errors are staged in LDS, and each
// gradient entry is a dot product over the block's samples by one thread,
// summed in sample order; the blocks' partial gradients are summed in block
// order (deterministic, no atomics).  Every sum runs in the order it had when
// one thread computed a whole sample, so the results are the same bits.
//
// Update: each block sums the previous step's partials and updates its own
// copy of the weights in LDS (the same arithmetic in each), block 0 stores
// them; read and written state alternate between two buffers.  That leaves
// one launch a step instead of three.
//
// What bounds it: latency - a step of 1,024 samples is 8 MFLOP in 16 blocks.
// One wave per block (64 threads, a sample each, then 21 entries of 64 terms
// each) took 55 us + 5.6 us reduction + 5.1 us Adam a step; this form takes
// 11.8 us in all.
constexpr int kRows = 64;
constexpr int kStep = 1024;            // threads: 16 waves, two hidden units each
constexpr int kPad = kRows + 4;        // LDS row of one unit over the samples: 16-byte reads without bank conflicts
static_assert(kH1 == 32 && kH2 == 32 && kFeat == 8, "the thread mapping below");
constexpr int oW1 = 0, ob1 = oW1 + kFeat * kH1, oW2 = ob1 + kH1, ob2 = oW2 + kH1 * kH2, oW3 = ob2 + kH2, ob3 = oW3 + kH2;

// Adam (Kingma & Ba 2015) for one parameter.
__device__ __forceinline__ void adam_one(float &p, float g, float &m, float &v, const AdamStep &a) {
  m = a.b1 * m + (1.f - a.b1) * g;
  v = a.b2 * v + (1.f - a.b2) * g * g;
  p -= a.lr * (m / a.bc1) / (sqrtf(v / a.bc2) + a.eps);
}

// Sum over s of x[s] * y[s], s ascending.
__device__ __forceinline__ float dot_rows(const float *x, const float *y) {
  float acc = 0.f;
#pragma unroll
  for (int s = 0; s < kRows; s += 4) {
    const float4 a = *(const float4 *)(x + s), b = *(const float4 *)(y + s);
    acc = fmaf(a.x, b.x, acc);
    acc = fmaf(a.y, b.y, acc);
    acc = fmaf(a.z, b.z, acc);
    acc = fmaf(a.w, b.w, acc);
  }
  return acc;
}
__device__ __forceinline__ float sum_rows(const float *x) {
  float acc = 0.f;
#pragma unroll
  for (int s = 0; s < kRows; s += 4) {
    const float4 a = *(const float4 *)(x + s);
    acc += a.x;
    acc += a.y;
    acc += a.z;
    acc += a.w;
  }
  return acc;
}

__global__ __launch_bounds__(kStep) void step_kernel(const float *params, const float *X, const float *Y,
                                                     const uint32_t *idx, uint64_t count, float scale, float *partial,
                                                     float *loss_partial, AdamStep ap) {
  __shared__ float sp[kParamFloats];
  __shared__ __align__(16) float s_xn[kFeat * kPad], s_h1[kH1 * kPad], s_h2[kH2 * kPad], s_d1[kH1 * kPad],
      s_d2[kH2 * kPad], s_dy[kPad], s_loss[kPad];
  const int t = threadIdx.x, l = t & 63, wv = t >> 6;
  for (int i = t; i < kParamFloats; i += kStep) {
    float p = params[i];
    if (ap.blocks && i < kTrainFloats) {
      float g = 0.f;
#pragma unroll 8
      for (uint32_t b = 0; b < ap.blocks; ++b) g += ap.partial[(uint64_t)b * kTrainFloats + i];
      float m = ap.m_in[i], v = ap.v_in[i];
      adam_one(p, g, m, v, ap);
      if (blockIdx.x == 0) {
        ap.m_out[i] = m;
        ap.v_out[i] = v;
      }
    }
    sp[i] = p;
    if (ap.blocks && blockIdx.x == 0) ap.p_out[i] = p;
  }
  if (ap.blocks && blockIdx.x == 0 && t == kStep - 1) {
    float sum = 0.f;
    for (uint32_t b = 0; b < ap.blocks; ++b) sum += ap.loss_partial[b];
    *ap.loss = sum;
  }
  const uint64_t si = (uint64_t)blockIdx.x * kRows + l;
  const bool live = si < count;
  const uint64_t r = live ? (idx ? idx[si] : si) : 0;
  const float target = live ? Y[r] : 0.f;
  __syncthreads();
  const Params q = params_at(sp);
  if (wv < kFeat) s_xn[wv * kPad + l] = live ? (X[r * kFeat + wv] - q.mean[wv]) * q.istd[wv] : 0.f;
  __syncthreads();
  const int u0 = 2 * wv, u1 = u0 + 1;
  {
    float a0 = q.b1[u0], a1 = q.b1[u1];
#pragma unroll
    for (int i = 0; i < kFeat; ++i) {
      const float x = s_xn[i * kPad + l];
      a0 = fmaf(x, q.W1[i * kH1 + u0], a0);
      a1 = fmaf(x, q.W1[i * kH1 + u1], a1);
    }
    s_h1[u0 * kPad + l] = live && a0 > 0.f ? a0 : 0.f;
    s_h1[u1 * kPad + l] = live && a1 > 0.f ? a1 : 0.f;
  }
  __syncthreads();
  {
    float a0 = q.b2[u0], a1 = q.b2[u1];
#pragma unroll
    for (int i = 0; i < kH1; ++i) {
      const float x = s_h1[i * kPad + l];
      a0 = fmaf(x, q.W2[i * kH2 + u0], a0);
      a1 = fmaf(x, q.W2[i * kH2 + u1], a1);
    }
    s_h2[u0 * kPad + l] = live && a0 > 0.f ? a0 : 0.f;
    s_h2[u1 * kPad + l] = live && a1 > 0.f ? a1 : 0.f;
  }
  __syncthreads();
  float y = q.b3[0];  // every wave: the errors need no exchange
#pragma unroll
  for (int i = 0; i < kH2; ++i) y = fmaf(s_h2[i * kPad + l], q.W3[i], y);
  const float d = live ? y - target : 0.f;
  const float dy = live ? 2.f * d * scale : 0.f;
  s_d2[u0 * kPad + l] = s_h2[u0 * kPad + l] > 0.f ? dy * q.W3[u0] : 0.f;
  s_d2[u1 * kPad + l] = s_h2[u1 * kPad + l] > 0.f ? dy * q.W3[u1] : 0.f;
  if (wv == 0) {
    s_dy[l] = dy;
    s_loss[l] = d * d;
  }
  __syncthreads();
  {
    float a0 = 0.f, a1 = 0.f;
#pragma unroll
    for (int j = 0; j < kH2; ++j) {
      const float e = s_d2[j * kPad + l];
      a0 = fmaf(q.W2[u0 * kH2 + j], e, a0);
      a1 = fmaf(q.W2[u1 * kH2 + j], e, a1);
    }
    s_d1[u0 * kPad + l] = s_h1[u0 * kPad + l] > 0.f ? a0 : 0.f;
    s_d1[u1 * kPad + l] = s_h1[u1 * kPad + l] > 0.f ? a1 : 0.f;
  }
  __syncthreads();
  float *out = partial + (uint64_t)blockIdx.x * kTrainFloats;
  out[oW2 + t] = dot_rows(s_h1 + (t / kH2) * kPad, s_d2 + (t % kH2) * kPad);  // kStep entries
  if (t < kFeat * kH1)
    out[oW1 + t] = dot_rows(s_xn + (t / kH1) * kPad, s_d1 + (t % kH1) * kPad);
  else if (t < kFeat * kH1 + kH1)
    out[ob1 + t - kFeat * kH1] = sum_rows(s_d1 + (t - kFeat * kH1) * kPad);
  else if (t < kFeat * kH1 + kH1 + kH2)
    out[ob2 + t - kFeat * kH1 - kH1] = sum_rows(s_d2 + (t - kFeat * kH1 - kH1) * kPad);
  else if (t < kFeat * kH1 + kH1 + 2 * kH2)
    out[oW3 + t - kFeat * kH1 - kH1 - kH2] = dot_rows(s_dy, s_h2 + (t - kFeat * kH1 - kH1 - kH2) * kPad);
  else if (t == kStep - 64)
    out[ob3] = sum_rows(s_dy);
  else if (t == kStep - 128)
    loss_partial[blockIdx.x] = sum_rows(s_loss);
}
static_assert(kH1 * kH2 == kStep, "one W2 entry per thread");

// grad[i] = sum over blocks (in order) of partial[b][i].
__global__ __launch_bounds__(64) void reduce_partials_kernel(const float *partial, uint32_t blocks, float *grad,
                                                             const float *loss_partial, float *loss) {
  int i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i < kTrainFloats) {
    float s = 0.f;
#pragma unroll 8
    for (uint32_t b = 0; b < blocks; ++b) s += partial[(uint64_t)b * kTrainFloats + i];
    grad[i] = s;
  }
  if (i == kTrainFloats) {
    float s = 0.f;
    for (uint32_t b = 0; b < blocks; ++b) s += loss_partial[b];
    *loss = s;
  }
}

// The reduction and update of a step whose next one does not do it.
__global__ __launch_bounds__(64) void adam_kernel(const float *params, AdamStep ap) {
  int i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i < kTrainFloats) {
    float g = 0.f;
#pragma unroll 8
    for (uint32_t b = 0; b < ap.blocks; ++b) g += ap.partial[(uint64_t)b * kTrainFloats + i];
    float p = params[i], m = ap.m_in[i], v = ap.v_in[i];
    adam_one(p, g, m, v, ap);
    ap.m_out[i] = m;
    ap.v_out[i] = v;
    ap.p_out[i] = p;
  } else if (i < kParamFloats) {
    ap.p_out[i] = params[i];
  } else if (i == kParamFloats) {
    float s = 0.f;
    for (uint32_t b = 0; b < ap.blocks; ++b) s += ap.loss_partial[b];
    *ap.loss = s;
  }
}

}  // namespace

hipError_t launch_features(const uint64_t *rowoff, const uint32_t *col, const uint32_t *core, float inv_degen,
                           const uint64_t *roots, uint64_t n_roots, float *out, hipStream_t s) {
  if (!n_roots) return hipSuccess;
  hipLaunchKernelGGL(features_kernel, dim3((uint32_t)((n_roots + 255) / 256)), dim3(256), 0, s, rowoff, col, core,
                     inv_degen, roots, n_roots, out);
  return hipGetLastError();
}

hipError_t launch_forward(const float *params, const float *X, uint64_t n, float *out, hipStream_t s) {
  if (!n) return hipSuccess;
  hipLaunchKernelGGL(forward_kernel, dim3((uint32_t)((n + 255) / 256)), dim3(256), 0, s, params, X, n, out);
  return hipGetLastError();
}

uint32_t backward_blocks(uint64_t count) { return (uint32_t)((count + kRows - 1) / kRows); }

hipError_t launch_step(const float *params, const float *X, const float *Y, const uint32_t *idx, uint64_t count,
                       float *partial, float *loss_partial, const AdamStep &apply, hipStream_t s) {
  uint32_t blocks = backward_blocks(count);
  if (!blocks) return hipSuccess;
  hipLaunchKernelGGL(step_kernel, dim3(blocks), dim3(kStep), 0, s, params, X, Y, idx, count, 1.0f / (float)count,
                     partial, loss_partial, apply);
  return hipGetLastError();
}

hipError_t launch_reduce(const float *partial, uint32_t blocks, float *grad, const float *loss_partial, float *loss,
                         hipStream_t s) {
  hipLaunchKernelGGL(reduce_partials_kernel, dim3(kTrainFloats / 64 + 1), dim3(64), 0, s, partial, blocks, grad,
                     loss_partial, loss);
  return hipGetLastError();
}

AdamStep adam_step(float lr, int step) {
  AdamStep a{};
  a.lr = lr;
  a.b1 = 0.9f;
  a.b2 = 0.999f;
  a.eps = 1e-8f;
  a.bc1 = 1.f - powf(a.b1, (float)step);
  a.bc2 = 1.f - powf(a.b2, (float)step);
  return a;
}

hipError_t launch_adam(const float *params, const AdamStep &apply, hipStream_t s) {
  hipLaunchKernelGGL(adam_kernel, dim3(kParamFloats / 64 + 1), dim3(64), 0, s, params, apply);
  return hipGetLastError();
}

}  // namespace rdmce
