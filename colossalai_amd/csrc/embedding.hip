// The gradient of an embedding table in bfloat16: row v is the sum, in float32 and in the order of the tokens, of the rows of dY whose token is v.
//
// Two launches. The first lists the tokens of every row: a block has 128 rows, its 16 waves a part of the tokens each. They count those below the block's rows
// (where its lists begin) and those in each row, and go through their tokens once more to put each behind the equal ones ahead of it. No block
// needs another's result, and what a block reads of the tokens (131 KB of 16384) comes from L2. The second writes the table: a wave has 512
// channels of a row; rows of many tokens are divided among the four waves of a block, whose sums meet in order.
//
// What bounds it: the bytes of the second launch, the table once (most of its rows are zeros) and dY once. us, with the library's sort -> here:
//   tokens 16384, rows 32000 of 4096   601 -> 124 (tokens by frequency 431 -> 181, all alike 731 -> 628)     8192, 32000 of 768   111 -> 41 (107 -> 57, 302 -> 231)
//   512, 32000 of 4096   68 -> 41     4096, 8000 of 2048   104 -> 41     16384, 128000 of 4096   769 -> 386     65536, 32000 of 2048   729 -> 140
// of which about 40 are the host's around a lone gradient; below, as at 512 tokens and 1024 rows of 512, both are bound by it.
#include <torch/extension.h>
#include <ATen/hip/HIPContext.h>
#include <c10/hip/HIPGuard.h>

#include <type_traits>

#include "common.h"
#include "plain.h"

namespace cai {

namespace emb {

constexpr int ROWS = 128, WAVES = 16;   // of a block that lists

// lists [T]: positions of the tokens, row by row, in their order; from [V + 1]: where a row's begin
__global__ __launch_bounds__(64 * WAVES) void list_kernel(const long* __restrict__ tokens, int T, int V, int* __restrict__ lists, int* __restrict__ from) {
  __shared__ int place[WAVES][ROWS];
  __shared__ int below[WAVES], sums[2];
  const int lane = threadIdx.x & 63, w = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const long v0 = (long)blockIdx.x * ROWS;
  const int rows = (int)min((long)ROWS, V - v0);
  const int part = ((T + WAVES - 1) / WAVES + 63) / 64 * 64, t0 = min(T, w * part), t1 = min(T, t0 + part);
  for (int i = threadIdx.x; i < WAVES * ROWS; i += 64 * WAVES) place[i / ROWS][i % ROWS] = 0;
  __syncthreads();
  int before = 0;
  for (int t = t0; t < t1; t += 256) {
    long v[4];
#pragma unroll
    for (int i = 0; i < 4; ++i) v[i] = (t + 64 * i + lane < t1 ? tokens[t + 64 * i + lane] : (long)V) - v0;
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      before += __builtin_popcountll(__ballot(v[i] < 0));
      if (v[i] >= 0 && v[i] < rows) atomicAdd(&place[w][(int)v[i]], 1);
    }
  }
  if (lane == 0) below[w] = before;
  __syncthreads();
  // a row's tokens in all parts, then the rows' beginnings: two waves of 64 rows
  int mine = 0, upto = 0;
  if (w < 2) {
    for (int i = 0; i < WAVES; ++i) mine += place[i][threadIdx.x];
    upto = mine;
#pragma unroll
    for (int o = 1; o < 64; o <<= 1) {
      const int other = __shfl_up(upto, o);
      upto += lane >= o ? other : 0;
    }
    if (lane == 63) sums[w] = upto;
  }
  __syncthreads();
  if (w < 2) {
    int at = upto - mine + (w ? sums[0] : 0);
    for (int i = 0; i < WAVES; ++i) at += below[i];
    if ((int)threadIdx.x < rows) from[v0 + threadIdx.x] = at;
    if (v0 + threadIdx.x + 1 == V) from[V] = at + mine;
    for (int i = 0; i < WAVES; ++i) {
      const int n = place[i][threadIdx.x];
      place[i][threadIdx.x] = at;
      at += n;
    }
  }
  __syncthreads();
  for (int t = t0; t < t1; t += 256) {
    long v[4];
#pragma unroll
    for (int i = 0; i < 4; ++i) v[i] = (t + 64 * i + lane < t1 ? tokens[t + 64 * i + lane] : (long)V) - v0;
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      unsigned long long left = __ballot(v[i] >= 0 && v[i] < rows);
      while (left != 0) {   // each row's tokens of these 64 together
        const int row = __builtin_amdgcn_readlane((int)v[i], __builtin_ctzll(left));
        const unsigned long long same = __ballot(v[i] == row) & left;
        const int at = place[w][row];
        if (same >> lane & 1) lists[at + __builtin_popcountll(same & ((1ull << lane) - 1))] = t + 64 * i + lane;
        if (lane == 0) place[w][row] = at + __builtin_popcountll(same);
        __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");   // the other lanes read it for the next of these 64
        left &= ~same;
      }
    }
  }
}

constexpr int MANY = 64;   // tokens of a row beyond which the block's waves share it

// DEEP: rows of a long list that are on their way together
template <int DEEP>
__global__ __launch_bounds__(256) void sum_kernel(const unsigned short* __restrict__ dy, const int* __restrict__ lists, const int* __restrict__ from,
                                                  int V, int W, int chunks, unsigned short* __restrict__ dw) {
  __shared__ float4v part[4][2][64];
  const int lane = threadIdx.x & 63, w = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int ch = (int)(blockIdx.x % chunks) * 512 + lane * 8;
  // Four rows, 64 apart: a table's frequent rows are often neighbours. Lane r has what row r's list is.
  const long group = blockIdx.x / chunks, r0 = group / 64 * 256 + group % 64, of_lane = r0 + (lane & 3) * 64;
  const int begin = of_lane < V ? from[of_lane] : 0, count = of_lane < V ? from[of_lane + 1] - begin : 0;
  const bool in = ch < W;
  float sum[8];
#pragma unroll
  for (int e = 0; e < 8; ++e) sum[e] = 0.0f;
  // tokens lo .. hi, `deep` (a constant) at a time on their way; past the end the last one again, which is not added
  auto add = [&](int lo, int hi, auto deep) {
    constexpr int N = decltype(deep)::value;
    for (int j = lo; j < hi; j += 64) {
      const int own = lists[min(j + lane, hi - 1)], n = min(64, hi - j);
      for (int k = 0; k < n; k += N) {
        short8 x[N];
#pragma unroll
        for (int i = 0; i < N; ++i)
          x[i] = *reinterpret_cast<const short8*>(dy + (long)__builtin_amdgcn_readlane(own, k + i) * W + (in ? ch : 0));
#pragma unroll
        for (int i = 0; i < N; ++i)
          if (k + i < n)
#pragma unroll
            for (int e = 0; e < 8; ++e) sum[e] += bf2f((unsigned short)x[i][e]);
      }
    }
  };
  auto store = [&](long row) {
    short8 o;
#pragma unroll
    for (int e = 0; e < 8; ++e) o[e] = (short)f2bf(sum[e]);
    if (in) *reinterpret_cast<short8*>(dw + row * W + ch) = o;
  };
  const long row = r0 + w * 64;
  const int lo = __builtin_amdgcn_readlane(begin, w), n = __builtin_amdgcn_readlane(count, w);
  if (row < V && n <= MANY) {
    if (n <= 2) add(lo, lo + n, std::integral_constant<int, 2>());
    else add(lo, lo + n, std::integral_constant<int, 8>());
    store(row);
  }
  unsigned many = (unsigned)__ballot(count > MANY) & 15;   // the same for all waves
  for (; many != 0; many &= many - 1) {
    const int r = __builtin_ctz(many), first = __builtin_amdgcn_readlane(begin, r), all = __builtin_amdgcn_readlane(count, r);
    const int share = (all + 3) / 4;
#pragma unroll
    for (int e = 0; e < 8; ++e) sum[e] = 0.0f;
    add(first + min(all, w * share), first + min(all, (w + 1) * share), std::integral_constant<int, DEEP>());
    part[w][0][lane] = float4v{sum[0], sum[1], sum[2], sum[3]};
    part[w][1][lane] = float4v{sum[4], sum[5], sum[6], sum[7]};
    __syncthreads();
    if (w == 0) {
      const float4v a = part[0][0][lane] + part[1][0][lane] + part[2][0][lane] + part[3][0][lane];
      const float4v b = part[0][1][lane] + part[1][1][lane] + part[2][1][lane] + part[3][1][lane];
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        sum[e] = a[e];
        sum[e + 4] = b[e];
      }
      store(r0 + r * 64);
    }
    __syncthreads();
  }
}

// What the kernels take; everything else is the library's. One row's tokens are summed by one block for each 512 channels, the library's segments by many: over
// many tokens, of which the frequent rows have their share (a row's number is log-uniform below), narrow tables and tables of few rows wait for the most frequent.
// us, here and there, 16384, 32768 and 131072 tokens: 8192 rows of 128 97 and 101, 191 and 148, 767 and 391; 2048 of 512 116 and 112, 229 and 182, 877 and 504; 32000 of
// 768 103 and 132, 185 and 206, 705 and 583; 8192 of 1024 105 and 133, 205 and 205, 834 and 667, 32000 of 1024 104 and 144, 185 and 226, 773 and 781; 512 of 2048
// 139 and 156, 267 and 259, 1147 and 1207; 32000 of 2048 107 and 214, 195 and 406, 828 and 1119. All tokens alike: 131072 in 32000 rows of 1024 3600 and 3960, in 256 of
// 4096 3400 and 6000. Every listing block goes through all tokens: up to 2^26 of them in all that is no more than the library's sort takes (1048576 tokens, 8192 rows).
bool serves(const at::Tensor& dy, const at::Tensor& tokens, int64_t V) {
  const long T = tokens.numel(), W = dy.size(-1);
  if (T > 16384 && W < 2048 && (W < 1024 || V < 32000)) return false;
  return plain(dy) && plain(tokens) && dy.is_cuda() && tokens.device() == dy.device() && dy.scalar_type() == at::kBFloat16 && tokens.scalar_type() == at::kLong
      && W > 0 && W % 8 == 0 && T > 0 && V > 0 && (V + 255) / 256 * 64 * ((W + 511) / 512) < (1L << 23) && (V + ROWS - 1) / ROWS * T <= (1L << 26);
}

at::Tensor grad(const at::Tensor& dy_in, const at::Tensor& tokens_in, int64_t V) {
  const c10::hip::HIPGuard guard(dy_in.device().index());
  at::Tensor dy = dy_in.contiguous();
  if (reinterpret_cast<uintptr_t>(dy.data_ptr()) % 16 != 0) dy = dy.clone();
  const at::Tensor tokens = tokens_in.contiguous();
  const int T = (int)tokens.numel(), W = (int)dy.size(-1), chunks = (W + 511) / 512;
  const at::Tensor ws = at::empty({T + V + 1}, tokens.options().dtype(at::kInt));
  at::Tensor dw = at::empty({V, W}, dy.options());
  int *lists = ws.data_ptr<int>(), *from = lists + T;
  const auto stream = at::hip::getCurrentHIPStream();
  list_kernel<<<(unsigned)((V + ROWS - 1) / ROWS), 64 * WAVES, 0, stream>>>(tokens.data_ptr<long>(), T, (int)V, lists, from);
  HIP_CHECK_LAST();
  // 16 rows on their way take registers that halve the waves in flight: only where rows have several tokens each (65536 tokens in 32000 rows of 2048, spread
  // evenly, by frequency and all alike 140, 429 and 1830 us, with eight 125, 456 and 2322; 16384 in rows of 4096 161, 191 and 509, with eight 124, 176 and 627)
  const auto kernel = T > V ? sum_kernel<16> : sum_kernel<8>;
  kernel<<<(unsigned)((V + 255) / 256 * 64 * chunks), 256, 0, stream>>>(reinterpret_cast<const unsigned short*>(dy.data_ptr()), lists, from, (int)V, W, chunks,
                                                                        reinterpret_cast<unsigned short*>(dw.data_ptr()));
  HIP_CHECK_LAST();
  return dw;
}

struct Embedding : torch::autograd::Function<Embedding> {
  static at::Tensor forward(torch::autograd::AutogradContext* ctx, const at::Tensor& tokens, const at::Tensor& weight) {
    ctx->save_for_backward({tokens});
    ctx->saved_data["rows"] = weight.size(0);
    return at::embedding(weight, tokens);
  }
  static torch::autograd::variable_list backward(torch::autograd::AutogradContext* ctx, torch::autograd::variable_list grads) {
    const at::Tensor tokens = ctx->get_saved_variables()[0], &dy = grads[0];
    const int64_t rows = ctx->saved_data["rows"].toInt();
    if (!dy.defined()) return {at::Tensor(), at::Tensor()};
    // a backward that is part of a graph itself (create_graph), or that something watches, takes an operation it can see
    if (!at::GradMode::is_enabled() && serves(dy, tokens, rows)) return {at::Tensor(), grad(dy, tokens, rows)};
    return {at::Tensor(), at::embedding_dense_backward(dy, tokens, rows, -1, false)};
  }
};

}  // namespace emb

// rows of `weight` [V, W] by `tokens`, as the built-in operation; its gradient as above
at::Tensor embedding(const at::Tensor& tokens, const at::Tensor& weight) {
  if (!plain(tokens) || !plain(weight) || has_tangent(weight)) return at::embedding(weight, tokens);
  return emb::Embedding::apply(tokens, weight);
}

}  // namespace cai
