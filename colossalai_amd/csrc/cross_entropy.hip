// Cross entropy over rows of bf16 logits for gfx950: the passes between the GEMMs of the chunked fused linear +
// cross entropy (ops/fused_ce.py).
//
// Memory-bound: the forward reads a row once (online maximum and sum of exponentials), the backward reads it
// once and writes the gradient, over it unless the forward's logits are kept. As library passes (to float32, logsumexp; to float32, subtract, exp,
// scatter, scale, to bf16) a chunk of 4096 x 32000 took 0.74 ms forward and 0.81 ms backward; it takes 0.05 and 0.11 ms,
// 262 and 524 MB at 5 TB/s. A vocabulary that is no multiple of 8 has rows that no wider load fits: 4096 x 50257 took 1.11 and
// 1.26 ms and takes 0.24 and 0.31 (50304 columns 0.07 and 0.17), bound by its two-byte accesses and, forward, three
// exponentials a logit. All arithmetic is float32; a gradient is rounded to bf16 once, as before.
//
// One block a row: 32000 columns are 125 a thread, and a step has thousands of rows.

#include <torch/extension.h>
#include <ATen/hip/HIPContext.h>

#include "common.h"

namespace cai {

constexpr int CE_BLOCK = 256;
constexpr float CE_LOG2E = 1.44269504f;

// A row's running state: maximum m and s = sum exp(x - ref(m)), where an infinite maximum is no reference (a row with a
// logit of +inf has a log-sum-exp of +inf, one of nothing but -inf has -inf). A NaN is in s; fmaxf leaves it out of m, so
// with a maximum of -inf s is 0 or NaN and stays as it is.
DEV_INLINE float ce_ref(float m) { return fabsf(m) == INFINITY ? 0.0f : m; }

DEV_INLINE float ce_moved(float m, float s, float ref) {
  return m == -INFINITY ? s : s * __builtin_amdgcn_exp2f((ce_ref(m) - ref) * CE_LOG2E);
}

DEV_INLINE void ce_merge(float& m, float& s, float om, float os) {
  const float top = fmaxf(m, om), ref = ce_ref(top);
  s = ce_moved(m, s, ref) + ce_moved(om, os, ref);
  m = top;
}

// lse [rows] and nll [rows] = lse - logits[label] (0 lse for an ignored row: what is not finite there shows, as it does in
// the general form; NaN for a label outside the row).
// VEC: rows of a multiple of 8 columns, 16-byte loads.
template <bool VEC>
__global__ __launch_bounds__(CE_BLOCK) void ce_fwd_kernel(float* __restrict__ lse, float* __restrict__ nll,
                                                          const unsigned short* __restrict__ logits,
                                                          const long* __restrict__ labels, long ignore_index, long rows, int V) {
  __shared__ float sm[CE_BLOCK / WAVE], ss[CE_BLOCK / WAVE];
  const long row = (long)blockIdx.y * gridDim.x + blockIdx.x;
  if (row >= rows) return;
  const unsigned short* x = logits + row * V;
  float m = -INFINITY, s = 0.0f;
  if (VEC) {
    const int nvec = V / 8;
#pragma unroll 4
    for (int i = threadIdx.x; i < nvec; i += CE_BLOCK) {
      const short8 v = *reinterpret_cast<const short8*>(x + i * 8);
      float f[8], top = m;
#pragma unroll
      for (int k = 0; k < 8; ++k) {
        f[k] = bf2f((unsigned short)v[k]);
        top = fmaxf(top, f[k]);
      }
      const float ref = ce_ref(top);
      s = ce_moved(m, s, ref);
      m = top;
#pragma unroll
      for (int k = 0; k < 8; ++k) s += __builtin_amdgcn_exp2f((f[k] - ref) * CE_LOG2E);
    }
  } else {
    for (int i = threadIdx.x; i < V; i += CE_BLOCK) {
      const float f = bf2f(x[i]);
      ce_merge(m, s, f, __builtin_amdgcn_exp2f((f - ce_ref(f)) * CE_LOG2E));
    }
  }
#pragma unroll
  for (int off = 32; off > 0; off >>= 1) ce_merge(m, s, __shfl_xor(m, off), __shfl_xor(s, off));
  if ((threadIdx.x & 63) == 0) {
    sm[threadIdx.x >> 6] = m;
    ss[threadIdx.x >> 6] = s;
  }
  __syncthreads();
  if (threadIdx.x == 0) {
#pragma unroll
    for (int w = 1; w < CE_BLOCK / WAVE; ++w) ce_merge(m, s, sm[w], ss[w]);
    const float ls = logf(s);
    const long label = labels[row];
    lse[row] = ce_ref(m) + ls;
    // the difference of two logits first: it is exact or nearly so, and the sum is rounded once
    nll[row] = label == ignore_index ? 0.0f * (ce_ref(m) + ls) : label >= 0 && label < V ? (ce_ref(m) - bf2f(x[label])) + ls : NAN;
  }
}

// logits -> their gradient (softmax - onehot) * valid * grad / n_valid (NaN for a label outside the row), in place or, where
// the logits are kept, elsewhere: a thread writes what it has read.
template <bool VEC>
__global__ __launch_bounds__(CE_BLOCK) void ce_bwd_kernel(unsigned short* out, const unsigned short* logits, const float* __restrict__ lse,
                                                          const long* __restrict__ labels, const float* __restrict__ grad,
                                                          const float* __restrict__ loss, long ignore_index, long rows,
                                                          int V) {
  const long row = (long)blockIdx.y * gridDim.x + blockIdx.x;
  if (row >= rows) return;
  const unsigned short* x = logits + row * V;
  unsigned short* y = out + row * V;
  const long label = labels[row];
  const float scale = (label == ignore_index ? 0.0f : label >= 0 && label < V ? 1.0f : NAN) * (grad[0] / loss[1]);
  const float l = lse[row];
  auto one = [&](unsigned short raw, int col) {
    float p = __builtin_amdgcn_exp2f((bf2f(raw) - l) * CE_LOG2E);
    if (col == label) p -= 1.0f;
    return f2bf(p * scale);
  };
  if (VEC) {
    const int nvec = V / 8;
#pragma unroll 4
    for (int i = threadIdx.x; i < nvec; i += CE_BLOCK) {
      short8 v = *reinterpret_cast<const short8*>(x + i * 8);
#pragma unroll
      for (int k = 0; k < 8; ++k) v[k] = (short)one((unsigned short)v[k], i * 8 + k);
      *reinterpret_cast<short8*>(y + i * 8) = v;
    }
  } else {
    for (int i = threadIdx.x; i < V; i += CE_BLOCK) y[i] = one(x[i], i);
  }
}

// loss[0] = sum(nll) / n, loss[1] = n = rows that are not ignored (at least 1). One block: a float a row. The sum is a
// double: in float32 its roundings were most of the loss's error (7.8e-7 at 4096 rows of 32000 columns, now
// 3.4e-7; the library passes over float32 logits are 4.9e-7 off).
__global__ __launch_bounds__(1024) void ce_loss_kernel(float* __restrict__ loss, const float* __restrict__ nll,
                                                       const long* __restrict__ labels, long ignore_index, long rows) {
  __shared__ double sm[1024 / WAVE];
  __shared__ float sn[1024 / WAVE];
  double sum = 0.0;
  float n = 0.0f;  // counts are exact up to 2^24 rows
#pragma unroll 4
  for (long i = threadIdx.x; i < rows; i += 1024) {
    sum += nll[i];
    n += labels[i] == ignore_index ? 0.0f : 1.0f;
  }
#pragma unroll
  for (int off = 32; off > 0; off >>= 1) sum += __shfl_xor(sum, off);
  n = wave_reduce_sum(n);
  if ((threadIdx.x & 63) == 0) {
    sm[threadIdx.x >> 6] = sum;
    sn[threadIdx.x >> 6] = n;
  }
  __syncthreads();
  if (threadIdx.x == 0) {
    for (int w = 1; w < 1024 / WAVE; ++w) {
      sum += sm[w];
      n += sn[w];
    }
    n = fmaxf(n, 1.0f);
    loss[0] = (float)(sum / n);
    loss[1] = n;
  }
}

// =============================================================== host side

static void check_ce(const at::Tensor& logits, const at::Tensor& labels, const at::Tensor& lse) {
  TORCH_CHECK(logits.is_cuda() && logits.dim() == 2 && logits.is_contiguous() && logits.scalar_type() == at::kBFloat16,
              "cross_entropy: logits must be contiguous bf16 [rows, vocab]");
  TORCH_CHECK(labels.is_cuda() && labels.is_contiguous() && labels.scalar_type() == at::kLong &&
              labels.numel() == logits.size(0), "cross_entropy: labels must be contiguous int64 [rows]");
  TORCH_CHECK(lse.is_cuda() && lse.is_contiguous() && lse.scalar_type() == at::kFloat && lse.numel() == logits.size(0),
              "cross_entropy: row statistics must be contiguous float32 [rows]");
}

static bool ce_vec(const at::Tensor& logits) {
  return logits.size(1) % 8 == 0 && reinterpret_cast<uintptr_t>(logits.data_ptr()) % 16 == 0;
}

// A block a row. A grid dimension of 2^32 threads or more is cut short without an error: from 2^20 rows on it is two.
static dim3 ce_grid(long rows) {
  const long width = rows < (1L << 20) ? rows : 1L << 20;
  return dim3((unsigned)width, (unsigned)((rows + width - 1) / width));
}

void ce_fwd(at::Tensor logits, at::Tensor labels, int64_t ignore_index, at::Tensor lse, at::Tensor nll) {
  check_ce(logits, labels, lse);
  check_ce(logits, labels, nll);
  const long rows = logits.size(0);
  if (rows == 0) return;
  auto stream = at::hip::getCurrentHIPStream();
  auto kernel = ce_vec(logits) ? ce_fwd_kernel<true> : ce_fwd_kernel<false>;
  hipLaunchKernelGGL(kernel, ce_grid(rows), dim3(CE_BLOCK), 0, stream.stream(), lse.data_ptr<float>(),
                     nll.data_ptr<float>(), (const unsigned short*)logits.data_ptr(), (const long*)labels.data_ptr(),
                     (long)ignore_index, rows, (int)logits.size(1));
  HIP_CHECK_LAST();
}

void ce_bwd(at::Tensor logits, at::Tensor labels, int64_t ignore_index, at::Tensor lse, at::Tensor grad, at::Tensor loss,
            c10::optional<at::Tensor> into) {
  check_ce(logits, labels, lse);
  const at::Tensor out = into ? *into : logits;
  check_ce(out, labels, lse);
  TORCH_CHECK(out.sizes() == logits.sizes(), "cross_entropy: the gradient has the logits' shape");
  TORCH_CHECK(grad.is_cuda() && grad.numel() == 1 && grad.scalar_type() == at::kFloat && loss.is_cuda() && loss.numel() == 2 &&
              loss.is_contiguous() && loss.scalar_type() == at::kFloat, "cross_entropy: grad is one float32, loss two");
  const long rows = logits.size(0);
  if (rows == 0) return;
  auto stream = at::hip::getCurrentHIPStream();
  auto kernel = ce_vec(logits) && ce_vec(out) ? ce_bwd_kernel<true> : ce_bwd_kernel<false>;
  hipLaunchKernelGGL(kernel, ce_grid(rows), dim3(CE_BLOCK), 0, stream.stream(), (unsigned short*)out.data_ptr(), (const unsigned short*)logits.data_ptr(),
                     lse.data_ptr<float>(), (const long*)labels.data_ptr(), grad.data_ptr<float>(), loss.data_ptr<float>(),
                     (long)ignore_index, rows, (int)logits.size(1));
  HIP_CHECK_LAST();
}

at::Tensor ce_loss(at::Tensor nll, at::Tensor labels, int64_t ignore_index) {
  TORCH_CHECK(nll.is_cuda() && nll.is_contiguous() && nll.scalar_type() == at::kFloat && labels.is_cuda() &&
              labels.is_contiguous() && labels.scalar_type() == at::kLong && labels.numel() == nll.numel(),
              "cross_entropy: nll must be float32 and labels int64, one a row");
  auto loss = at::empty({2}, nll.options());
  auto stream = at::hip::getCurrentHIPStream();
  hipLaunchKernelGGL(ce_loss_kernel, dim3(1), dim3(1024), 0, stream.stream(), loss.data_ptr<float>(), nll.data_ptr<float>(),
                     (const long*)labels.data_ptr(), (long)ignore_index, (long)nll.numel());
  HIP_CHECK_LAST();
  return loss;
}

}  // namespace cai
