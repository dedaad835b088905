// AdamW step with the masked decay folded in, for gfx950: one pass over parameter, gradient, both
// moments and the mask instead of a masked_add_ pass over (grad, p, mask) followed by the optimizer's
// passes.  Per element, float32, every product and sum rounded separately (no fused multiply-add),
// in the order of the reference's optimizer (sparse/adamw.py:70-113) preceded by its decay
// (sparse/decay.py:27-37, applied in README.md:205-213 before optimizer.step()):
//     g  = grad (+ alpha * p where mask == 0)
//     p  = p * (1 - lr * weight_decay)
//     m  = m * beta1 + (1 - beta1) * g
//     v  = v * beta2 + ((1 - beta2) * g) * g
//     p  = p + (-(lr / bc1)) * (m / (sqrt(v) / sqrt(bc2) + eps))
// The gradient is only read.  One launch updates a whole list of tensors: a block owns kBlockElems consecutive
// elements of one of them and finds it by a binary search of the list, which travels in the kernel arguments
// (every step of the search is a scalar load).  Lane owns 4 consecutive elements (16-byte accesses of the float32
// operands).
#include "tf24_common.hpp"

namespace tf24 {
namespace {

constexpr int kThreads = 256;

struct AdamArgs {
  float decay_mul;        // 1 - lr * weight_decay
  float beta1, one_m_beta1, beta2, one_m_beta2;
  float sqrt_bc2;         // sqrt(v) is divided by it
  float eps, neg_step_size, alpha;
};

// The hyper-parameters as the caller gave them.  The per-step scalars are formed in double like the Python of the
// reference and rounded once to float32 where a tensor meets them -- on the host when the step count is a host
// number, by the first lane of every block when it lives in device memory (a recorded graph replays with the
// count of the replay, not of the recording).
struct AdamHyper {
  double lr, beta1, beta2, eps, weight_decay, alpha;
};

__host__ __device__ inline AdamArgs adam_args(const AdamHyper& h, int64_t step) {
  const double bc1 = 1.0 - pow(h.beta1, (double)step), bc2 = 1.0 - pow(h.beta2, (double)step);
  AdamArgs a;
  a.decay_mul = (float)(1.0 - h.lr * h.weight_decay);
  a.beta1 = (float)h.beta1; a.one_m_beta1 = (float)(1.0 - h.beta1);
  a.beta2 = (float)h.beta2; a.one_m_beta2 = (float)(1.0 - h.beta2);
  a.sqrt_bc2 = (float)sqrt(bc2);
  a.eps = (float)h.eps;
  a.neg_step_size = (float)(-(h.lr / bc1));
  a.alpha = (float)h.alpha;
  return a;
}

__device__ __forceinline__ void adam_element(float& p, float g, float& m, float& v, bool decay, const AdamArgs& a) {
  if (decay) g = g + p * a.alpha;
  p = p * a.decay_mul;
  m = m * a.beta1 + a.one_m_beta1 * g;
  v = v * a.beta2 + (a.one_m_beta2 * g) * g;
  const float denom = __builtin_sqrtf(v) / a.sqrt_bc2 + a.eps;
  p = p + a.neg_step_size * (m / denom);
}

constexpr int kBlockElems = kThreads * 4;
constexpr int kMaxTensors = 56;         // 64 bytes each: the list and the scalars stay below the 4 KB of a launch's arguments

struct AdamTensor {
  float *p, *m, *v;
  const void *grad, *mask;              // mask == nullptr: no decay
  const int64_t* step;                  // step count in device memory, or nullptr: the launch's scalars hold
  int64_t n;
  uint32_t first_block;                 // blocks of the launch before this tensor's
  uint32_t vec;                         // 16-byte accesses: every pointer is aligned for them
};
struct AdamList {
  AdamTensor t[kMaxTensors];
  int count;
};

// Bound by memory: 29 bytes per element (float32 gradient, byte mask).  24 weights of 3072 x 768 and their 24 biases,
// 56.6 M elements: 254 us = 6.47 TB/s in one launch, against 16 us per weight (4.3 TB/s: too short to fill the memory
// pipeline and drain it again) and 3.8 us per bias, 442 us in all, with a launch per tensor.  The moments and the
// parameter are loaded AND stored with the streaming forms: ordinary accesses 295 us, streaming stores alone 295 us.
// Two rounds of 1024 elements per block are slower (262 us).
template <typename G, typename M>
__global__ void __launch_bounds__(kThreads)
adamw_list(const AdamList list, const AdamArgs a_host, const AdamHyper h) {
  int lo = 0, hi = list.count;          // the last tensor whose first_block is not behind this block
  while (hi - lo > 1) {
    const int mid = (lo + hi) >> 1;
    if (list.t[mid].first_block <= blockIdx.x) lo = mid; else hi = mid;
  }
  const AdamTensor& t = list.t[lo];
  AdamArgs a = a_host;
  if (t.step) {                         // (uniform over the block)
    __shared__ AdamArgs shared;
    if (threadIdx.x == 0) shared = adam_args(h, *t.step);
    __syncthreads();
    a = shared;
  }
  const int64_t base = (int64_t)(blockIdx.x - t.first_block) * kBlockElems;
  float* const p = t.p + base;
  float* const m = t.m + base;
  float* const v = t.v + base;
  const G* const grad = (const G*)t.grad + base;
  const M* const mask = t.mask ? (const M*)t.mask + base : nullptr;
  const int64_t left = t.n - base;
  if (t.vec && left >= kBlockElems) {
    const int u = threadIdx.x * 4;
    Pack<float, 4> pv, mv, vv;
    Pack<G, 4> gv;
    Pack<M, 4> mk;
    pv.load_stream(p + u); mv.load_stream(m + u); vv.load_stream(v + u); gv.load_stream(grad + u);
    if (mask) mk.load_stream(mask + u);
#pragma unroll
    for (int i = 0; i < 4; i++) adam_element(pv.v[i], to_float(gv.v[i]), mv.v[i], vv.v[i], mask && to_float(mk.v[i]) == 0.0f, a);
    pv.store_stream(p + u); mv.store_stream(m + u); vv.store_stream(v + u);
  } else {                              // the last block of a tensor, or unaligned pointers
    const int n = (int)(left < kBlockElems ? left : kBlockElems);
    for (int i = threadIdx.x; i < n; i += kThreads) {
      float pi = p[i], mi = m[i], vi = v[i];
      adam_element(pi, to_float(grad[i]), mi, vi, mask && to_float(mask[i]) == 0.0f, a);
      p[i] = pi; m[i] = mi; v[i] = vi;
    }
  }
}

template <typename G, typename M>
int launch(const char* fn, AdamList& list, const AdamArgs& a, const AdamHyper& h, hipStream_t s) {
  int64_t blocks = 0;
  for (int i = 0; i < list.count; i++) {
    AdamTensor& t = list.t[i];
    t.first_block = (uint32_t)blocks;
    t.vec = (uintptr_t)t.p % 16 == 0 && (uintptr_t)t.m % 16 == 0 && (uintptr_t)t.v % 16 == 0 &&
            (uintptr_t)t.grad % (4 * sizeof(G)) == 0 && (uintptr_t)t.mask % (4 * sizeof(M)) == 0;
    blocks += (t.n + kBlockElems - 1) / kBlockElems;
  }
  if (blocks > 0x7fffffff) return fail(TF24_ERR_SHAPE, "%s: too many elements for one launch", fn);
  hipLaunchKernelGGL((adamw_list<G, M>), dim3((unsigned)blocks), dim3(kThreads), 0, s, list, a, h);
  return check_launch(fn);
}

template <typename G>
int dispatch_mask(const char* fn, int mask_dtype, AdamList& list, const AdamArgs& a, const AdamHyper& h, hipStream_t s) {
  switch (mask_dtype) {
    case TF24_U8: return launch<G, uint8_t>(fn, list, a, h, s);
    case TF24_F32: return launch<G, float>(fn, list, a, h, s);
    case TF24_F16: return launch<G, f16_t>(fn, list, a, h, s);
    case TF24_BF16: return launch<G, bf16_t>(fn, list, a, h, s);
  }
  return fail(TF24_ERR_DTYPE, "%s: unsupported mask dtype %d", fn, mask_dtype);
}

}  // namespace
}  // namespace tf24

// Every tensor with its own step count in device memory (step_host 0), or all of them at step_host >= 1.
static int adamw_masked_decay(const char* fn, const tf24_adamw_tensor* tensors, int count, int grad_dtype, int mask_dtype, double lr,
                              double beta1, double beta2, double eps, double weight_decay, double decay_alpha, int64_t step_host,
                              void* stream) {
  using namespace tf24;
  if (count < 0 || (count > 0 && !tensors)) return fail(TF24_ERR_ARG, "%s: bad tensor list", fn);
  if (!(lr >= 0.0) || !(eps >= 0.0) || !(beta1 >= 0.0 && beta1 < 1.0) || !(beta2 >= 0.0 && beta2 < 1.0))
    return fail(TF24_ERR_ARG, "%s: invalid hyper-parameter (lr %g, eps %g, betas %g %g)", fn, lr, eps, beta1, beta2);
  if (grad_dtype != TF24_F32 && grad_dtype != TF24_F16 && grad_dtype != TF24_BF16)
    return fail(TF24_ERR_DTYPE, "%s: unsupported gradient dtype %d", fn, grad_dtype);
  for (int i = 0; i < count; i++) {            // the whole list is checked before anything is launched
    const tf24_adamw_tensor& t = tensors[i];
    if (t.n < 0) return fail(TF24_ERR_SHAPE, "%s: negative element count", fn);
    if (t.n == 0) continue;
    if (!t.p || !t.grad || !t.exp_avg || !t.exp_avg_sq) return fail(TF24_ERR_ARG, "%s: null pointer", fn);
    if (!t.step && step_host < 1) return fail(TF24_ERR_ARG, "%s: step %lld must be >= 1", fn, (long long)step_host);
    if (t.step && (uintptr_t)t.step % 8 != 0) return fail(TF24_ERR_STRIDE, "%s: the step count must be 8-byte aligned", fn);
  }
  const AdamHyper h{lr, beta1, beta2, eps, weight_decay, decay_alpha};
  const AdamArgs a = adam_args(h, step_host < 1 ? 1 : step_host);
  hipStream_t s = (hipStream_t)stream;
  AdamList list;
  for (int i = 0; i < count;) {
    list.count = 0;
    for (; i < count && list.count < kMaxTensors; i++) {
      const tf24_adamw_tensor& t = tensors[i];
      if (t.n > 0) list.t[list.count++] = AdamTensor{t.p, t.exp_avg, t.exp_avg_sq, t.grad, t.mask, t.step, t.n, 0, 0};
    }
    if (!list.count) break;
    int rc;
    switch (grad_dtype) {
      case TF24_F32: rc = dispatch_mask<float>(fn, mask_dtype, list, a, h, s); break;
      case TF24_F16: rc = dispatch_mask<f16_t>(fn, mask_dtype, list, a, h, s); break;
      default: rc = dispatch_mask<bf16_t>(fn, mask_dtype, list, a, h, s); break;
    }
    if (rc) return rc;
  }
  return TF24_OK;
}

extern "C" int tf24_adamw_masked_decay_list(const tf24_adamw_tensor* tensors, int count, int grad_dtype, int mask_dtype, double lr,
                                            double beta1, double beta2, double eps, double weight_decay, double decay_alpha,
                                            int64_t step, void* stream) {
  return adamw_masked_decay("tf24_adamw_masked_decay_list", tensors, count, grad_dtype, mask_dtype, lr, beta1, beta2, eps, weight_decay,
                            decay_alpha, step, stream);
}

extern "C" int tf24_adamw_masked_decay(float* p, const void* grad, int grad_dtype, float* exp_avg, float* exp_avg_sq,
                                       const void* mask, int mask_dtype, int64_t n, double lr, double beta1, double beta2,
                                       double eps, double weight_decay, double decay_alpha, int64_t step, void* stream) {
  if (n == 0) return TF24_OK;
  const tf24_adamw_tensor t{p, grad, exp_avg, exp_avg_sq, mask, nullptr, n};
  return adamw_masked_decay("tf24_adamw_masked_decay", &t, 1, grad_dtype, mask ? mask_dtype : TF24_U8, lr, beta1, beta2, eps,
                            weight_decay, decay_alpha, step, stream);
}

extern "C" int tf24_adamw_masked_decay_device_step(float* p, const void* grad, int grad_dtype, float* exp_avg, float* exp_avg_sq,
                                                   const void* mask, int mask_dtype, int64_t n, double lr, double beta1,
                                                   double beta2, double eps, double weight_decay, double decay_alpha,
                                                   const int64_t* step, void* stream) {
  if (!step) return tf24::fail(TF24_ERR_ARG, "tf24_adamw_masked_decay_device_step: null step pointer");
  if (n == 0) return TF24_OK;
  const tf24_adamw_tensor t{p, grad, exp_avg, exp_avg_sq, mask, step, n};
  return adamw_masked_decay("tf24_adamw_masked_decay_device_step", &t, 1, grad_dtype, mask ? mask_dtype : TF24_U8, lr, beta1, beta2, eps,
                            weight_decay, decay_alpha, 0, stream);
}
