// Parallel residual streams ("hyper-connections"): instead of one residual row a token carries S rows
// x_1 .. x_S (float32). A sublayer reads u = sum_s in[s] x_s and, from its output y,
// x_t <- sum_s mix[s, t] x_s + out[t] y for all t at once from the old rows.
//   streams_start  : the (scaled) embedding row becomes every stream, and the first sublayer's input
//                    rms_norm(u) * w is formed in the same launch;
//   streams_update : the write of one sublayer, in place, and the read + norm of the next one
//                    (or of the output, with in = 1 everywhere) in one pass over the streams;
//   streams_pass   : either what an update would read and norm, without the write, or the writes of two sublayers, the second formed
//                    over the first in registers, with the read and norm after them.
// A layer of two sublayers then reads the streams twice and writes them once with the last two, where two updates write them twice: 4096 tokens, four
// streams of 2048, 47 + 47 -> 30 + 51 us. Ahead of the first write every stream is the token's embedding row, which streams_pass reads in the
// place of them (`table`, `tokens`), so that they need not be written at the start (37 -> 15 us). It serves up to 4 streams of a
// width that is a multiple of 4 up to 4096; others are updated one sublayer at a time.
#include "serving_common.h"

namespace cai {
namespace serving {

DEV_INLINE void load4(const float* p, float* o) {
  const float4v a = *reinterpret_cast<const float4v*>(p);
  o[0] = a[0]; o[1] = a[1]; o[2] = a[2]; o[3] = a[3];
}
DEV_INLINE void load4(const bf16s* p, float* o) {
  const short4v a = *reinterpret_cast<const short4v*>(p);
#pragma unroll
  for (int e = 0; e < 4; ++e) o[e] = bf2f((bf16s)a[e]);
}
DEV_INLINE void store4(float* p, const float* v) { *reinterpret_cast<float4v*>(p) = float4v{v[0], v[1], v[2], v[3]}; }
DEV_INLINE void store4(bf16s* p, const float* v) {
  short4v a;
#pragma unroll
  for (int e = 0; e < 4; ++e) a[e] = (short)f2bf(v[e]);
  *reinterpret_cast<short4v*>(p) = a;
}

constexpr int STREAMS_MAX = 8;  // streams the register form is built for; more take the general form

// A sublayer's write: mix [S, S], out [S] and its output's rows. Multiplications are fused as written, so that every form rounds alike.
template <int S>
struct Write {
  float mix[S][S], out[S];
  DEV_INLINE Write(const float* m, const float* o) {
#pragma unroll
    for (int s = 0; s < S; ++s) {
      out[s] = o[s];
#pragma unroll
      for (int t = 0; t < S; ++t) mix[s][t] = m[s * S + t];
    }
  }
  DEV_INLINE void apply(const float (&old)[S][4], const float (&y)[4], float (&nv)[S][4]) const {
#pragma unroll
    for (int t = 0; t < S; ++t) {
#pragma unroll
      for (int e = 0; e < 4; ++e) {
#pragma clang fp contract(off)
        nv[t][e] = out[t] * y[e];
      }
#pragma unroll
      for (int s = 0; s < S; ++s)
#pragma unroll
        for (int e = 0; e < 4; ++e) nv[t][e] = fmaf(mix[s][t], old[s][e], nv[t][e]);
    }
  }
};

// One block per token; a thread owns the same four neighbouring channels of all S streams, CH times 1024 channels
// apart. Every stream element is read once and written once (STORE); u stays in registers over the block's reduction. TWO: y1 with mix1 and
// out1 is written ahead of y. ROW: the old streams are all the token's row of `table`.
template <typename TY, typename TO, int S, int CH, bool STORE, bool TWO, bool ROW>
__global__ __launch_bounds__(256) void streams_update_rows_kernel(
    TO* __restrict__ h, float* __restrict__ x, const TY* __restrict__ y, const float* __restrict__ mix,
    const float* __restrict__ w_out, const float* __restrict__ w_in, const float* __restrict__ w, int W, float eps,
    const TY* __restrict__ y1, const float* __restrict__ mix1, const float* __restrict__ out1, const TY* __restrict__ table,
    const long* __restrict__ tokens) {
  __shared__ float red[8];
  const long row = blockIdx.x;
  const Write<S> last(mix, w_out), first(TWO ? mix1 : mix, TWO ? out1 : w_out);
  float wi[S];
#pragma unroll
  for (int s = 0; s < S; ++s) wi[s] = w_in != nullptr ? w_in[s] : 1.0f;
  float* xr = x + row * S * (long)W;
  const TY* er = ROW ? table + tokens[row] * (long)W : nullptr;
  float u[CH][4];
  float ssq = 0.0f;
#pragma unroll
  for (int c = 0; c < CH; ++c) {
    const int i = (threadIdx.x + 256 * c) * 4;
    if (i < W) {
      float old[S][4], yv[4], nv[S][4];
#pragma unroll
      for (int s = 0; s < S; ++s) {
        if (!ROW) load4(xr + (long)s * W + i, old[s]);
        else if (s == 0) load4(er + i, old[0]);
        else
#pragma unroll
          for (int e = 0; e < 4; ++e) old[s][e] = old[0][e];
      }
      if (TWO) {
        float y1v[4], mid[S][4];
        load4(y1 + row * (long)W + i, y1v);
        first.apply(old, y1v, mid);
#pragma unroll
        for (int s = 0; s < S; ++s)
#pragma unroll
          for (int e = 0; e < 4; ++e) old[s][e] = mid[s][e];
      }
      load4(y + row * (long)W + i, yv);
      last.apply(old, yv, nv);
#pragma unroll
      for (int e = 0; e < 4; ++e) u[c][e] = 0.0f;
#pragma unroll
      for (int t = 0; t < S; ++t) {
        if (STORE) store4(xr + (long)t * W + i, nv[t]);
#pragma unroll
        for (int e = 0; e < 4; ++e) u[c][e] = fmaf(wi[t], nv[t][e], u[c][e]);
      }
#pragma unroll
      for (int e = 0; e < 4; ++e) ssq = fmaf(u[c][e], u[c][e], ssq);
    }
  }
  if (h == nullptr) return;
  ssq = block_reduce_sum(ssq, red);
  const float inv = 1.0f / sqrtf(ssq / (float)W + eps);
#pragma unroll
  for (int c = 0; c < CH; ++c) {
    const int i = (threadIdx.x + 256 * c) * 4;
    if (i < W) {
      float wv[4];
      load4(w + i, wv);
#pragma unroll
      for (int e = 0; e < 4; ++e) wv[e] *= u[c][e] * inv;
      store4(h + row * (long)W + i, wv);
    }
  }
}

// Any width and up to 32 streams: a thread owns single channels (all streams of them), u is formed again from the
// rows it has written.
template <typename TY, typename TO>
__global__ __launch_bounds__(256) void streams_update_kernel(
    TO* __restrict__ h, float* __restrict__ x, const TY* __restrict__ y, const float* __restrict__ mix,
    const float* __restrict__ w_out, const float* __restrict__ w_in, const float* __restrict__ w, int W, int S, float eps) {
  __shared__ float red[8];
  const long row = blockIdx.x;
  float* xr = x + row * S * (long)W;
  float old[32];
  float ssq = 0.0f;
  for (int i = threadIdx.x; i < W; i += blockDim.x) {
    for (int s = 0; s < S; ++s) old[s] = xr[(long)s * W + i];
    const float yv = ldf(y + row * (long)W + i);
    float u = 0.0f;
    for (int t = 0; t < S; ++t) {
      float nv = w_out[t] * yv;
      for (int s = 0; s < S; ++s) nv += mix[s * S + t] * old[s];
      xr[(long)t * W + i] = nv;
      u += (w_in != nullptr ? w_in[t] : 1.0f) * nv;
    }
    ssq += u * u;
  }
  if (h == nullptr) return;
  ssq = block_reduce_sum(ssq, red);
  const float inv = 1.0f / sqrtf(ssq / (float)W + eps);
  for (int i = threadIdx.x; i < W; i += blockDim.x) {
    float u = 0.0f;
    for (int t = 0; t < S; ++t) u += (w_in != nullptr ? w_in[t] : 1.0f) * xr[(long)t * W + i];
    stf(h + row * (long)W + i, u * inv * w[i]);
  }
}

c10::optional<at::Tensor> streams_update(at::Tensor x, at::Tensor y, at::Tensor mix, at::Tensor w_out,
                                         c10::optional<at::Tensor> w_in, c10::optional<at::Tensor> weight, double eps,
                                         at::ScalarType out_dtype) {
  check_act(y, "y");
  TORCH_CHECK(x.is_cuda() && is_f32(x) && x.dim() == 3 && x.is_contiguous(), "streams must be contiguous float32 [N, S, W]");
  const long N = x.size(0);
  const int S = (int)x.size(1), W = (int)x.size(2);
  TORCH_CHECK(S >= 1 && S <= 32, "between 1 and 32 streams");
  TORCH_CHECK(y.is_contiguous() && y.dim() == 2 && y.size(0) == N && y.size(1) == W, "y must be contiguous [N, W]");
  TORCH_CHECK(out_dtype == at::kFloat || out_dtype == at::kBFloat16);
  at::Tensor mx = f32c(mix), wo = f32c(w_out), wi, w, h;
  TORCH_CHECK(mx.is_cuda() && mx.dim() == 2 && mx.size(0) == S && mx.size(1) == S && wo.is_cuda() && wo.numel() == S,
              "mix must be [S, S], out [S]");
  const float* wip = nullptr;
  const float* wp = nullptr;
  if (w_in.has_value()) {
    wi = f32c(*w_in);
    TORCH_CHECK(wi.is_cuda() && wi.numel() == S, "in must be [S]");
    wip = wi.data_ptr<float>();
  }
  if (weight.has_value()) {
    w = f32c(*weight);
    TORCH_CHECK(w.is_cuda() && w.numel() == W, "the norm's weight must be [W]");
    wp = w.data_ptr<float>();
    h = at::empty({N, W}, y.options().dtype(out_dtype));
  }
  if (N > 0) {
    const at::Tensor& like = weight.has_value() ? h : y;  // without a norm nothing is written through h
    auto al16 = [](const void* p) { return p == nullptr || reinterpret_cast<uintptr_t>(p) % 16 == 0; };
    const bool rows = S <= STREAMS_MAX && W % 4 == 0 && W <= 8192 && al16(x.data_ptr()) && al16(y.data_ptr()) && al16(wp);
#define STREAMS_ROWS(S_, CH_)                                                                                      \
  hipLaunchKernelGGL((streams_update_rows_kernel<TY, TO, S_, CH_, true, false, false>), dim3((unsigned)N), dim3(256), 0, stream(), hp,  \
                     x.data_ptr<float>(), ptr<TY>(y), mx.data_ptr<float>(), wo.data_ptr<float>(), wip, wp, W, (float)eps,   \
                     (const TY*)nullptr, (const float*)nullptr, (const float*)nullptr, (const TY*)nullptr, (const long*)nullptr)
#define STREAMS_CASE(S_)                    \
  case S_:                                  \
    if (W <= 1024) STREAMS_ROWS(S_, 1);     \
    else if (W <= 2048) STREAMS_ROWS(S_, 2); \
    else if (W <= 4096) STREAMS_ROWS(S_, 4); \
    else STREAMS_ROWS(S_, 8);               \
    break
    SERVING_DISPATCH_ACT(y, TY, {
      SERVING_DISPATCH_ACT(like, TO, {
        TO* hp = weight.has_value() ? ptr<TO>(h) : (TO*)nullptr;
        if (rows) {
          switch (S) {
            STREAMS_CASE(1); STREAMS_CASE(2); STREAMS_CASE(3); STREAMS_CASE(4);
            STREAMS_CASE(5); STREAMS_CASE(6); STREAMS_CASE(7); STREAMS_CASE(8);
          }
        } else {
          hipLaunchKernelGGL((streams_update_kernel<TY, TO>), dim3((unsigned)N), dim3(256), 0, stream(), hp,
                             x.data_ptr<float>(), ptr<TY>(y), mx.data_ptr<float>(), wo.data_ptr<float>(), wip, wp, W, S,
                             (float)eps);
        }
      });
    });
#undef STREAMS_CASE
#undef STREAMS_ROWS
    HIP_CHECK_LAST();
  }
  if (!weight.has_value()) return c10::nullopt;
  return h;
}

// Without y1 nothing is written; with it both sublayers' writes go to x [N, S, W], with `table` to be filled. The old streams are x or, with `table`
// [vocab, W] of y's type and `tokens` [N], S times the token's row. For up to 4 streams of a width that is a multiple of 4 up to
// 4096, everything at addresses of 16 bytes (streams_pairs says so); returns nothing otherwise, having done nothing.
bool streams_pairs(int64_t S, int64_t W) { return S >= 1 && S <= 4 && W % 4 == 0 && W <= 4096; }

c10::optional<at::Tensor> streams_pass(c10::optional<at::Tensor> x, c10::optional<at::Tensor> table, c10::optional<at::Tensor> tokens,
                                       c10::optional<at::Tensor> y1, c10::optional<at::Tensor> mix1, c10::optional<at::Tensor> out1, at::Tensor y,
                                       at::Tensor mix, at::Tensor w_out, c10::optional<at::Tensor> w_in, at::Tensor weight, double eps,
                                       at::ScalarType out_dtype) {
  check_act(y, "y");
  const bool two = y1.has_value(), row = table.has_value();
  const long N = y.size(0);
  const int S = (int)w_out.numel(), W = (int)y.size(1);
  TORCH_CHECK(y.dim() == 2 && y.is_contiguous() && streams_pairs(S, W), "streams_pass: up to 4 streams of a multiple of 4 channels up to 4096");
  TORCH_CHECK(row == tokens.has_value() && two == mix1.has_value() && two == out1.has_value() && (two || row || x.has_value()) &&
              (x.has_value() || (row && !two)), "streams_pass: which streams?");
  if (x.has_value())
    TORCH_CHECK(x->is_cuda() && is_f32(*x) && x->is_contiguous() && x->dim() == 3 && x->size(0) == N && x->size(1) == S && x->size(2) == W,
                "streams must be contiguous float32 [N, S, W]");
  if (row)
    TORCH_CHECK(table->is_cuda() && table->scalar_type() == y.scalar_type() && table->is_contiguous() && table->dim() == 2 && table->size(1) == W &&
                tokens->is_cuda() && tokens->scalar_type() == at::kLong && tokens->is_contiguous() && tokens->numel() == N,
                "table must be contiguous [vocab, W] of y's type, tokens int64 [N]");
  if (two)
    TORCH_CHECK(y1->is_cuda() && y1->scalar_type() == y.scalar_type() && y1->is_contiguous() && y1->sizes() == y.sizes(), "y1 must be like y");
  TORCH_CHECK(out_dtype == at::kFloat || out_dtype == at::kBFloat16);
  const at::Tensor mx = f32c(mix), wo = f32c(w_out), wt = f32c(weight), wi = w_in.has_value() ? f32c(*w_in) : at::Tensor();
  const at::Tensor mx1 = two ? f32c(*mix1) : at::Tensor(), wo1 = two ? f32c(*out1) : at::Tensor();
  TORCH_CHECK(mx.is_cuda() && mx.numel() == S * S && wo.is_cuda() && wt.is_cuda() && wt.numel() == W && (!wi.defined() || (wi.is_cuda() && wi.numel() == S)) &&
              (!two || (mx1.is_cuda() && mx1.numel() == S * S && wo1.is_cuda() && wo1.numel() == S)), "streams_pass: mix [S, S], out and in [S], weight [W]");
  const at::Tensor h = at::empty({N, W}, y.options().dtype(out_dtype));
  auto al16 = [](const at::Tensor& t) { return reinterpret_cast<uintptr_t>(t.data_ptr()) % 16 == 0; };
  if (!al16(y) || !al16(wt) || (x.has_value() && !al16(*x)) || (row && !al16(*table)) || (two && !al16(*y1))) return c10::nullopt;
  if (N == 0) return h;
#define STREAMS_PASS(S_, CH_, TWO_, ROW_)                                                                                             \
  hipLaunchKernelGGL((streams_update_rows_kernel<TY, TO, S_, CH_, TWO_, TWO_, ROW_>), dim3((unsigned)N), dim3(256), 0, stream(), ptr<TO>(h), \
                     x.has_value() ? x->data_ptr<float>() : (float*)nullptr, ptr<TY>(y), mx.data_ptr<float>(), wo.data_ptr<float>(),   \
                     wi.defined() ? wi.data_ptr<float>() : (const float*)nullptr, wt.data_ptr<float>(), W, (float)eps,                 \
                     TWO_ ? ptr<TY>(*y1) : (const TY*)nullptr, TWO_ ? mx1.data_ptr<float>() : (const float*)nullptr,                    \
                     TWO_ ? wo1.data_ptr<float>() : (const float*)nullptr, ROW_ ? ptr<TY>(*table) : (const TY*)nullptr,                 \
                     ROW_ ? (const long*)tokens->data_ptr<int64_t>() : (const long*)nullptr)
#define STREAMS_FORM(S_, CH_)                       \
  do {                                              \
    if (two && row) STREAMS_PASS(S_, CH_, true, true);   \
    else if (two) STREAMS_PASS(S_, CH_, true, false);    \
    else if (row) STREAMS_PASS(S_, CH_, false, true);    \
    else STREAMS_PASS(S_, CH_, false, false);            \
  } while (0)
#define STREAMS_OF(S_)                         \
  case S_:                                     \
    if (W <= 1024) STREAMS_FORM(S_, 1);        \
    else if (W <= 2048) STREAMS_FORM(S_, 2);   \
    else STREAMS_FORM(S_, 4);                  \
    break
  SERVING_DISPATCH_ACT(y, TY, {
    SERVING_DISPATCH_ACT(h, TO, {
      switch (S) {
        STREAMS_OF(1); STREAMS_OF(2); STREAMS_OF(3); STREAMS_OF(4);
      }
    });
  });
#undef STREAMS_OF
#undef STREAMS_FORM
#undef STREAMS_PASS
  HIP_CHECK_LAST();
  return h;
}

// One block per token: table row tokens[n] -> all S streams, and rms_norm((sum_s in[s]) * row) * w. V channels per
// thread and step (4: the width is a multiple of 4 and every row 16-byte aligned); the row is read again for the norm.
template <typename TE, int V>
__global__ __launch_bounds__(256) void streams_start_kernel(TE* __restrict__ h, float* __restrict__ x,
                                                            const TE* __restrict__ table, const long* __restrict__ tokens,
                                                            const float* __restrict__ w_in, const float* __restrict__ w,
                                                            int W, int S, float eps, float scale) {
  __shared__ float red[8];
  const long row = blockIdx.x;
  const TE* er = table + tokens[row] * (long)W;
  float* xr = x + row * S * (long)W;
  float ssq = 0.0f, total = 0.0f;
  for (int s = 0; s < S; ++s) total += w_in[s];
#pragma unroll 2
  for (int i = threadIdx.x * V; i < W; i += blockDim.x * V) {
    float e[V];
    if constexpr (V == 4) load4(er + i, e);
    else e[0] = ldf(er + i);
#pragma unroll
    for (int k = 0; k < V; ++k) {
      e[k] *= scale;
      ssq += (total * e[k]) * (total * e[k]);
    }
    for (int s = 0; s < S; ++s) {
      if (x == nullptr) break;
      if constexpr (V == 4) store4(xr + (long)s * W + i, e);
      else xr[(long)s * W + i] = e[0];
    }
  }
  ssq = block_reduce_sum(ssq, red);
  const float inv = total / sqrtf(ssq / (float)W + eps);
#pragma unroll 2
  for (int i = threadIdx.x * V; i < W; i += blockDim.x * V) {
    float e[V], wv[V];
    if constexpr (V == 4) {
      load4(er + i, e);
      load4(w + i, wv);
#pragma unroll
      for (int k = 0; k < V; ++k) e[k] = e[k] * scale * inv * wv[k];
      store4(h + row * (long)W + i, e);
    } else {
      stf(h + row * (long)W + i, ldf(er + i) * scale * inv * w[i]);
    }
  }
}

// without `fill` only the normed input is formed, and the streams are left to streams_pass
std::vector<at::Tensor> streams_start(at::Tensor table, at::Tensor tokens, int64_t streams, at::Tensor w_in,
                                      at::Tensor weight, double eps, double scale, bool fill) {
  check_act(table, "table");
  TORCH_CHECK(table.dim() == 2 && table.is_contiguous(), "table must be contiguous [vocab, W]");
  TORCH_CHECK(tokens.is_cuda() && tokens.scalar_type() == at::kLong && tokens.dim() == 1 && tokens.is_contiguous(),
              "tokens must be contiguous int64 [N]");
  const long N = tokens.size(0);
  const int W = (int)table.size(1), S = (int)streams;
  at::Tensor wi = f32c(w_in), w = f32c(weight);
  TORCH_CHECK(S >= 1 && S <= 32 && wi.is_cuda() && wi.numel() == S && w.is_cuda() && w.numel() == W);
  at::Tensor x = at::empty({fill ? N : 0, S, W}, table.options().dtype(at::kFloat));
  float* xp = fill ? x.data_ptr<float>() : nullptr;
  at::Tensor h = at::empty({N, W}, table.options());
  auto al16 = [](const at::Tensor& t) { return reinterpret_cast<uintptr_t>(t.data_ptr()) % 16 == 0; };
  const bool vec = W % 4 == 0 && al16(table) && al16(w) && (!fill || al16(x)) && al16(h);
  if (N > 0) {
    SERVING_DISPATCH_ACT(table, TE, {
      if (vec)
        hipLaunchKernelGGL((streams_start_kernel<TE, 4>), dim3((unsigned)N), dim3(256), 0, stream(), ptr<TE>(h),
                           xp, ptr<TE>(table), (const long*)tokens.data_ptr<int64_t>(),
                           wi.data_ptr<float>(), w.data_ptr<float>(), W, S, (float)eps, (float)scale);
      else
        hipLaunchKernelGGL((streams_start_kernel<TE, 1>), dim3((unsigned)N), dim3(256), 0, stream(), ptr<TE>(h),
                           xp, ptr<TE>(table), (const long*)tokens.data_ptr<int64_t>(),
                           wi.data_ptr<float>(), w.data_ptr<float>(), W, S, (float)eps, (float)scale);
    });
    HIP_CHECK_LAST();
  }
  return {x, h};
}

}  // namespace serving
}  // namespace cai
