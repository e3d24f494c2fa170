// Fused RMSNorm forward/backward for gfx950 (bf16 in/out, fp32 accumulate).
//
// MI355X design notes:
//  - memory-bound: all bf16 traffic is vectorized short8 (16 B/lane).
//  - a row is one wave's up to 2048 channels (four rows a block, no barrier) and one block's of 256
//    threads up to 8192; a thread's slice is V groups of 8 channels in registers.
//  - forward saves inv_rms (fp32 per row) so backward skips the re-reduce.
//  - fused residual-add variant: h = x + residual is computed once and
//    written as the new residual stream (pre-norm transformer block),
//    saving one full read+write per layer vs separate add.
//  - backward: a thread owns its channels over all rows of its block, so dweight sums stay in
//    registers; each block writes one partial row and a second kernel adds those. (Every block
//    adding its row with atomics met on H addresses: 60.6 us for 8192 x 768, of which 12 are memory.)
//    The gradient that flows past the norm on the residual stream is added in the same pass.
//
// 8192 x 768: backward 60.6 -> 13 us; 16384 x 4096: 123 -> 90 us (400 MB, 4.5 TB/s).
//
// Equivalent reference op: extensions/csrc/kernel/cuda/rms_layernorm_kernel.cu
// (re-designed; warp-size-32 assumptions do not carry to CDNA4).

#include <torch/extension.h>
#include <ATen/hip/HIPContext.h>

#include "common.h"

namespace cai {

constexpr int RMS_BLOCK = 256;
constexpr int RMS_MAX_H = 8192;

// Sum over the TPR threads of a row: a wave, or the whole block.
template <int TPR>
DEV_INLINE float row_sum(float v, float* smem) {
  return TPR == WAVE ? wave_reduce_sum(v) : block_reduce_sum(v, smem);
}

template <int TPR, int V, bool FUSED_ADD>
__global__ __launch_bounds__(RMS_BLOCK) void rmsnorm_fwd_kernel(
    unsigned short* __restrict__ out,          // [rows, H] bf16
    unsigned short* res_out,                   // [rows, H] bf16 (FUSED_ADD), may be residual itself
    const unsigned short* residual,            // [rows, H] bf16 (FUSED_ADD)
    const unsigned short* __restrict__ input,  // [rows, H] bf16
    const unsigned short* __restrict__ weight, // [H] bf16
    float* __restrict__ inv_rms_out,           // [rows] fp32
    float eps,
    long rows,
    int H) {
  __shared__ float red_smem[RMS_BLOCK / WAVE];
  const int nvec = H / 8;  // H % 8 == 0 enforced on host
  const int t = threadIdx.x % TPR;
  constexpr int RPB = RMS_BLOCK / TPR;  // rows per block

  for (long row = (long)blockIdx.x * RPB + threadIdx.x / TPR; row < rows; row += (long)gridDim.x * RPB) {
    short8 xv[V], rv[V];
#pragma unroll
    for (int v = 0; v < V; ++v) {
      const int i = t + v * TPR;
      if (i < nvec) {
        xv[v] = *reinterpret_cast<const short8*>(input + row * H + i * 8);
        if (FUSED_ADD) rv[v] = *reinterpret_cast<const short8*>(residual + row * H + i * 8);
      }
    }
    float vals[V][8];
    float ssq = 0.0f;
#pragma unroll
    for (int v = 0; v < V; ++v) {
      const int i = t + v * TPR;
      if (i >= nvec) continue;
#pragma unroll
      for (int k = 0; k < 8; ++k) {
        float f = bf2f((unsigned short)xv[v][k]);
        if (FUSED_ADD) f += bf2f((unsigned short)rv[v][k]);
        vals[v][k] = f;
        ssq += f * f;
      }
      if (FUSED_ADD) {
        short8 hv;
#pragma unroll
        for (int k = 0; k < 8; ++k) hv[k] = (short)f2bf(vals[v][k]);
        *reinterpret_cast<short8*>(res_out + row * H + i * 8) = hv;
      }
    }
    ssq = row_sum<TPR>(ssq, red_smem);
    const float inv_rms = rsqrtf(ssq / (float)H + eps);
    if (t == 0 && inv_rms_out != nullptr) inv_rms_out[row] = inv_rms;
#pragma unroll
    for (int v = 0; v < V; ++v) {
      const int i = t + v * TPR;
      if (i >= nvec) continue;
      const short8 wv = *reinterpret_cast<const short8*>(weight + i * 8);
      short8 yv;
#pragma unroll
      for (int k = 0; k < 8; ++k) yv[k] = (short)f2bf(vals[v][k] * inv_rms * bf2f((unsigned short)wv[k]));
      *reinterpret_cast<short8*>(out + row * H + i * 8) = yv;
    }
  }
}

// backward: x here is the NORMALIZATION INPUT (post residual-add when fused).
//   dx_i = inv_rms * (w_i*dy_i - x_i * inv_rms^2/H * sum_j(w_j*dy_j*x_j)) [+ dres_i]
//   dw_j += dy_j * x_j * inv_rms        (accumulated over the block's rows, one partial row per block)
template <int TPR, int V>
__global__ __launch_bounds__(RMS_BLOCK) void rmsnorm_bwd_kernel(
    unsigned short* __restrict__ dx,            // [rows, H] bf16 out
    float* __restrict__ dw_part,                // [gridDim.x, H] fp32 out
    const unsigned short* __restrict__ dy,      // [rows, H] bf16
    const unsigned short* __restrict__ dres,    // [rows, H] bf16 or null
    const unsigned short* __restrict__ x,       // [rows, H] bf16
    const unsigned short* __restrict__ weight,  // [H] bf16
    const float* __restrict__ inv_rms,          // [rows]
    long rows,
    int H) {
  __shared__ float red_smem[RMS_BLOCK / WAVE];
  __shared__ float dw_lds[TPR == WAVE ? RMS_BLOCK / WAVE : 1][TPR == WAVE ? WAVE * V * 8 : 1];
  const int nvec = H / 8;
  const int t = threadIdx.x % TPR, sub = threadIdx.x / TPR;
  constexpr int RPB = RMS_BLOCK / TPR;

  float dw[V][8];
#pragma unroll
  for (int v = 0; v < V; ++v)
#pragma unroll
    for (int k = 0; k < 8; ++k) dw[v][k] = 0.0f;

  // (a block whose rows end early still meets the others in the block-wide sum: all its threads share the row)
  for (long row = (long)blockIdx.x * RPB + sub; row < rows; row += (long)gridDim.x * RPB) {
    const float r = inv_rms[row];
    short8 xv[V], dv[V], av[V];
#pragma unroll
    for (int v = 0; v < V; ++v) {
      const int i = t + v * TPR;
      if (i < nvec) {
        xv[v] = *reinterpret_cast<const short8*>(x + row * H + i * 8);
        dv[v] = *reinterpret_cast<const short8*>(dy + row * H + i * 8);
        if (dres != nullptr) av[v] = *reinterpret_cast<const short8*>(dres + row * H + i * 8);
      }
    }
    float xf[V][8], dyw[V][8];
    float dot = 0.0f;
#pragma unroll
    for (int v = 0; v < V; ++v) {
      const int i = t + v * TPR;
      if (i >= nvec) continue;
      const short8 wv = *reinterpret_cast<const short8*>(weight + i * 8);
#pragma unroll
      for (int k = 0; k < 8; ++k) {
        xf[v][k] = bf2f((unsigned short)xv[v][k]);
        const float df = bf2f((unsigned short)dv[v][k]);
        dyw[v][k] = df * bf2f((unsigned short)wv[k]);
        dot += dyw[v][k] * xf[v][k];
        dw[v][k] += df * xf[v][k] * r;
      }
    }
    dot = row_sum<TPR>(dot, red_smem);
    const float c = dot * r * r / (float)H;
#pragma unroll
    for (int v = 0; v < V; ++v) {
      const int i = t + v * TPR;
      if (i >= nvec) continue;
      short8 ov;
#pragma unroll
      for (int k = 0; k < 8; ++k) {
        float g = r * (dyw[v][k] - xf[v][k] * c);
        if (dres != nullptr) g += bf2f((unsigned short)av[v][k]);
        ov[k] = (short)f2bf(g);
      }
      *reinterpret_cast<short8*>(dx + row * H + i * 8) = ov;
    }
  }
  float* mine = dw_part + (long)blockIdx.x * H;
  if (TPR == WAVE) {  // the block's four waves meet in LDS
#pragma unroll
    for (int v = 0; v < V; ++v)
#pragma unroll
      for (int k = 0; k < 8; ++k) dw_lds[sub][(t + v * TPR) * 8 + k] = dw[v][k];
    __syncthreads();
    for (int j = threadIdx.x; j < H; j += RMS_BLOCK) {
      float sum = 0.0f;
#pragma unroll
      for (int w = 0; w < RPB; ++w) sum += dw_lds[w][j];
      mine[j] = sum;
    }
  } else {
#pragma unroll
    for (int v = 0; v < V; ++v) {
      const int i = t + v * TPR;
      if (i >= nvec) continue;
#pragma unroll
      for (int k = 0; k < 8; k += 4)
        *reinterpret_cast<float4v*>(mine + i * 8 + k) = float4v{dw[v][k], dw[v][k + 1], dw[v][k + 2], dw[v][k + 3]};
    }
  }
}

// dweight = sum of the partial rows: 32 columns x 32 row groups a block.
template <typename T>
__global__ __launch_bounds__(1024) void rmsnorm_dw_kernel(T* __restrict__ dweight, const float* __restrict__ part, int parts, int H) {
  __shared__ float lds[32][33];
  const int c = threadIdx.x & 31, g = threadIdx.x >> 5;
  const int col = blockIdx.x * 32 + c;
  float sum = 0.0f;
  if (col < H) {
#pragma unroll 8
    for (int p = g; p < parts; p += 32) sum += part[(long)p * H + col];
  }
  lds[g][c] = sum;
  __syncthreads();
  if (g == 0 && col < H) {
    float total = 0.0f;
#pragma unroll
    for (int k = 0; k < 32; ++k) total += lds[k][c];
    if constexpr (sizeof(T) == 2) dweight[col] = f2bf(total);
    else dweight[col] = total;
  }
}

// =============================================================== host side

static void check_rms_args(const at::Tensor& t, int H) {
  TORCH_CHECK(t.is_contiguous(), "rmsnorm: tensors must be contiguous");
  TORCH_CHECK(t.scalar_type() == at::kBFloat16, "rmsnorm: bf16 only");
  TORCH_CHECK(H % 8 == 0 && H <= RMS_MAX_H, "rmsnorm: hidden must be %8==0 and <= 8192");
}

// Threads of a row and groups of 8 channels a thread holds.
#define RMS_DISPATCH(H, ...)                                                         \
  do {                                                                               \
    const int nv_ = (H) / 8;                                                         \
    if (nv_ <= 4 * WAVE) {                                                           \
      constexpr int TPR = WAVE;                                                      \
      if (nv_ <= WAVE) { constexpr int V = 1; __VA_ARGS__; }                         \
      else if (nv_ <= 2 * WAVE) { constexpr int V = 2; __VA_ARGS__; }                \
      else { constexpr int V = 4; __VA_ARGS__; }                                     \
    } else {                                                                         \
      constexpr int TPR = RMS_BLOCK;                                                 \
      if (nv_ <= 2 * RMS_BLOCK) { constexpr int V = 2; __VA_ARGS__; }                \
      else { constexpr int V = 4; __VA_ARGS__; }                                     \
    }                                                                                \
  } while (0)

static std::vector<at::Tensor> rmsnorm_forward(const at::Tensor& input, const at::Tensor* residual, const at::Tensor* res_out,
                                               const at::Tensor& weight, double eps, bool save_inv_rms) {
  const int H = (int)input.size(-1);
  const long rows = input.numel() / H;
  check_rms_args(input, H);
  auto out = at::empty_like(input);
  auto inv_rms = save_inv_rms ? at::empty({rows}, input.options().dtype(at::kFloat)) : at::Tensor();
  auto stream = at::hip::getCurrentHIPStream();
#define RMS_FWD(ADD)                                                                                                  \
  hipLaunchKernelGGL((rmsnorm_fwd_kernel<TPR, V, ADD>), dim3(capped_grid((rows + RMS_BLOCK / TPR - 1) / (RMS_BLOCK / TPR), 8192)), \
                     dim3(RMS_BLOCK), 0, stream.stream(), (unsigned short*)out.data_ptr(),                             \
                     ADD ? (unsigned short*)res_out->data_ptr() : nullptr,                                            \
                     ADD ? (const unsigned short*)residual->data_ptr() : nullptr, (const unsigned short*)input.data_ptr(), \
                     (const unsigned short*)weight.data_ptr(), save_inv_rms ? inv_rms.data_ptr<float>() : nullptr,    \
                     (float)eps, rows, H)
  RMS_DISPATCH(H, if (residual != nullptr) RMS_FWD(true); else RMS_FWD(false));
#undef RMS_FWD
  HIP_CHECK_LAST();
  return {out, inv_rms};
}

std::vector<at::Tensor> rmsnorm_fwd(at::Tensor input, at::Tensor weight, double eps, bool save_inv_rms) {
  return rmsnorm_forward(input, nullptr, nullptr, weight, eps, save_inv_rms);
}

// h = input + residual (written into res_out, or into residual without one); out = rmsnorm(h)
std::vector<at::Tensor> rmsnorm_fused_add_fwd(at::Tensor input, at::Tensor residual, at::Tensor weight,
                                              double eps, bool save_inv_rms, c10::optional<at::Tensor> res_out) {
  at::Tensor to = res_out.has_value() ? *res_out : residual;
  TORCH_CHECK(residual.numel() == input.numel() && to.numel() == input.numel(), "rmsnorm: input and residual must match");
  if (res_out.has_value())
    TORCH_CHECK(residual.is_contiguous() && to.is_contiguous() && residual.scalar_type() == at::kBFloat16 &&
                to.scalar_type() == at::kBFloat16, "rmsnorm: residuals must be contiguous bf16");
  return rmsnorm_forward(input, &residual, &to, weight, eps, save_inv_rms);
}

// dres: gradient of the residual stream, added to dx. dweight is float32, or of the weight's type with cast_dw.
std::vector<at::Tensor> rmsnorm_bwd(at::Tensor dy, at::Tensor x, at::Tensor weight, at::Tensor inv_rms,
                                    c10::optional<at::Tensor> dres, bool cast_dw) {
  const int H = (int)x.size(-1);
  const long rows = x.numel() / H;
  check_rms_args(x, H);
  if (dres.has_value())
    TORCH_CHECK(dres->is_contiguous() && dres->scalar_type() == at::kBFloat16 && dres->numel() == x.numel(),
                "rmsnorm: dres must be contiguous bf16 of x's size");
  auto dx = at::empty_like(x);
  const bool narrow = cast_dw && weight.scalar_type() == at::kBFloat16;
  auto dweight = at::empty({H}, x.options().dtype(narrow ? at::kBFloat16 : at::kFloat));
  auto stream = at::hip::getCurrentHIPStream();
  at::Tensor part;
  int grid = 0;
  // 1024 blocks are 16 waves a CU, all at once where a thread holds one or two groups (67 to 114 registers) and in two turns
  // where it holds four (190 and 199: 8 waves a CU); their partial rows are 4 KB per 1024 channels each, which a block of a row's
  // width makes up for with at least four rows
  RMS_DISPATCH(H, {
    constexpr int RPB = RMS_BLOCK / TPR;
    const long most = TPR == WAVE ? (rows + RPB - 1) / RPB : (rows + 3) / 4;
    grid = capped_grid(most, 1024);
    part = at::empty({(long)grid * H}, x.options().dtype(at::kFloat));
    hipLaunchKernelGGL((rmsnorm_bwd_kernel<TPR, V>), dim3(grid), dim3(RMS_BLOCK), 0, stream.stream(),
                       (unsigned short*)dx.data_ptr(), part.data_ptr<float>(), (const unsigned short*)dy.data_ptr(),
                       dres.has_value() ? (const unsigned short*)dres->data_ptr() : nullptr,
                       (const unsigned short*)x.data_ptr(), (const unsigned short*)weight.data_ptr(),
                       inv_rms.data_ptr<float>(), rows, H);
  });
  HIP_CHECK_LAST();
  if (narrow)
    hipLaunchKernelGGL((rmsnorm_dw_kernel<unsigned short>), dim3((H + 31) / 32), dim3(1024), 0, stream.stream(),
                       (unsigned short*)dweight.data_ptr(), part.data_ptr<float>(), grid, H);
  else
    hipLaunchKernelGGL((rmsnorm_dw_kernel<float>), dim3((H + 31) / 32), dim3(1024), 0, stream.stream(),
                       dweight.data_ptr<float>(), part.data_ptr<float>(), grid, H);
  HIP_CHECK_LAST();
  return {dx, dweight};
}

}  // namespace cai
