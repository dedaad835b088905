// Masked decay for gfx950: grad[i] += alpha * p[i] where mask[i] == 0, in place, one pass.
// Lane owns 16 consecutive bytes of the widest operand (4 float32 or 8 half-precision elements); float32 arithmetic
// as a rounded product followed by a rounded sum (no fused multiply-add).
// Bound by memory.  At 8 float32 elements per lane (two 16-byte accesses, 32 bytes from lane to lane) every wave
// instruction touched half lines: 8192 x 8192 float32 with a byte mask 147 us = 5.9 TB/s, streaming accesses of the
// gradient 154 us.  With one 16-byte access per lane and streaming accesses of everything, the gradient included:
// 134.7 us = 6.5 TB/s (11008 x 4096: 101 -> 88 us, 3072 x 768: 7.0 -> 6.2 us).
#include "tf24_common.hpp"

namespace tf24 {
namespace {

constexpr int kThreads = 256;

template <typename G, typename P> constexpr int lane_elems() { return sizeof(G) == 4 || sizeof(P) == 4 ? 4 : 8; }

template <typename G, typename P, typename M>
__global__ void __launch_bounds__(kThreads)
masked_add_vec(G* __restrict__ grad, const P* __restrict__ p, const M* __restrict__ mask, int64_t units, float alpha) {
  constexpr int E = lane_elems<G, P>();
  const int64_t u = (int64_t)blockIdx.x * kThreads + threadIdx.x;
  if (u >= units) return;
  Pack<G, E> g;
  Pack<P, E> pv;
  Pack<M, E> mk;
  g.load_stream(grad + u * E);
  pv.load_stream(p + u * E);
  mk.load_stream(mask + u * E);
#pragma unroll
  for (int i = 0; i < E; i++) {
    const float prod = to_float(pv.v[i]) * alpha;
    const float sum = to_float(g.v[i]) + prod;
    if (to_float(mk.v[i]) == 0.0f) g.v[i] = from_float<G>(sum);
  }
  g.store_stream(grad + u * E);
}

template <typename G, typename P, typename M>
__global__ void __launch_bounds__(kThreads)
masked_add_scalar(G* __restrict__ grad, const P* __restrict__ p, const M* __restrict__ mask, int64_t begin, int64_t n, float alpha) {
  const int64_t i = begin + (int64_t)blockIdx.x * kThreads + threadIdx.x;
  if (i >= n) return;
  if (to_float(mask[i]) == 0.0f) {
    const float prod = to_float(p[i]) * alpha;
    grad[i] = from_float<G>(to_float(grad[i]) + prod);
  }
}

template <typename G, typename P, typename M>
int launch(void* grad, const void* p, const void* mask, int64_t n, float alpha, hipStream_t s) {
  const bool aligned = ((uintptr_t)grad % 16 == 0) && ((uintptr_t)p % 16 == 0) && ((uintptr_t)mask % 8 == 0);
  constexpr int E = lane_elems<G, P>();
  const int64_t units = aligned ? n / E : 0;
  if (units > 0) {
    dim3 grid((unsigned)((units + kThreads - 1) / kThreads));
    hipLaunchKernelGGL((masked_add_vec<G, P, M>), grid, dim3(kThreads), 0, s, (G*)grad, (const P*)p, (const M*)mask, units, alpha);
  }
  const int64_t begin = units * E;
  if (begin < n) {
    dim3 grid((unsigned)((n - begin + kThreads - 1) / kThreads));
    hipLaunchKernelGGL((masked_add_scalar<G, P, M>), grid, dim3(kThreads), 0, s, (G*)grad, (const P*)p, (const M*)mask, begin, n, alpha);
  }
  return check_launch("tf24_masked_add");
}

template <typename G, typename P>
int dispatch_mask(int mask_dtype, void* grad, const void* p, const void* mask, int64_t n, float alpha, hipStream_t s) {
  switch (mask_dtype) {
    case TF24_U8: return launch<G, P, uint8_t>(grad, p, mask, n, alpha, s);
    case TF24_F32: return launch<G, P, float>(grad, p, mask, n, alpha, s);
    case TF24_F16: return launch<G, P, f16_t>(grad, p, mask, n, alpha, s);
    case TF24_BF16: return launch<G, P, bf16_t>(grad, p, mask, n, alpha, s);
  }
  return fail(TF24_ERR_DTYPE, "tf24_masked_add: unsupported mask dtype %d", mask_dtype);
}

template <typename G>
int dispatch_p(int p_dtype, int mask_dtype, void* grad, const void* p, const void* mask, int64_t n, float alpha, hipStream_t s) {
  switch (p_dtype) {
    case TF24_F32: return dispatch_mask<G, float>(mask_dtype, grad, p, mask, n, alpha, s);
    case TF24_F16: return dispatch_mask<G, f16_t>(mask_dtype, grad, p, mask, n, alpha, s);
    case TF24_BF16: return dispatch_mask<G, bf16_t>(mask_dtype, grad, p, mask, n, alpha, s);
  }
  return fail(TF24_ERR_DTYPE, "tf24_masked_add: unsupported parameter dtype %d", p_dtype);
}

}  // namespace
}  // namespace tf24

extern "C" int tf24_masked_add(void* grad, int grad_dtype, const void* p, int p_dtype, const void* mask, int mask_dtype,
                               int64_t n, float alpha, void* stream) {
  using namespace tf24;
  if (n < 0) return fail(TF24_ERR_SHAPE, "tf24_masked_add: negative element count");
  if (n == 0) return TF24_OK;
  if (!grad || !p || !mask) return fail(TF24_ERR_ARG, "tf24_masked_add: null pointer");
  hipStream_t s = (hipStream_t)stream;
  switch (grad_dtype) {
    case TF24_F32: return dispatch_p<float>(p_dtype, mask_dtype, grad, p, mask, n, alpha, s);
    case TF24_F16: return dispatch_p<f16_t>(p_dtype, mask_dtype, grad, p, mask, n, alpha, s);
    case TF24_BF16: return dispatch_p<bf16_t>(p_dtype, mask_dtype, grad, p, mask, n, alpha, s);
  }
  return fail(TF24_ERR_DTYPE, "tf24_masked_add: unsupported gradient dtype %d", grad_dtype);
}
