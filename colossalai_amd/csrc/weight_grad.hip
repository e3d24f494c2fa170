// Weight gradients of linear layers: dW[M, N] = dY[K, M]^T X[K, N] in bfloat16, summed in float32, K tokens.
//
// Both operands lie token by token, so that the contracted index is the slow one of both: transposing LDS reads
// (ds_read_b64_tr_b16, see flash_attn.hip) give the columns that the matrix unit takes. Four waves hold a tile's sums in registers, one
// quarter each: 256 x 256 where there is enough of them, which is the least LDS and memory traffic a product has here (a
// wave's 128 x 128 sums are 256 registers, one wave a SIMD), else 128 x 128 with two blocks a CU. Four steps of 32 tokens lie in
// LDS: while one is multiplied the next is there and two are on their way, so that a step waits for loads that are two steps old
// (s_waitcnt vmcnt, never 0) and for one barrier. A wave reads the fragments of the next 16 tokens and issues its loads one by
// one between the products of the 16 before.
//
// What bounds it: a step of the large tile takes 1203 cycles of which the products are 1024; the clock falls to 1.4 to 1.6
// GHz under it (M 4096 and 12288, N 4096, K 16384). The small tile takes 725 cycles for two blocks, 512 of them products.
//
// M, N, K; us with the library's product -> here:
//   22016, 4096, 16384   2785 -> 2214     4096, 11008, 16384   1536 -> 1132     4096, 4096, 16384   470 -> 404
//   32000, 4096, 4096     952 -> 859      32000, 768, 4096      223 -> 191      4096, 768, 8192      84 -> 65
//   768, 2048, 8192        65 -> 40       768, 768, 8192         49 -> 22       2048, 512, 512       21 -> 10
#include <torch/extension.h>
#include <ATen/hip/HIPContext.h>
#include <c10/hip/HIPGuard.h>

#include <algorithm>

#include "lds_tiles.h"

namespace cai {

namespace wg {

constexpr int KT = 32;       // tokens of a step
constexpr int STEPS = 4;     // steps in LDS: one in use, one arrived, two on their way

// A step of one operand in LDS: pieces of 8 tokens of 64 columns, 1024 bytes each, the four pieces of 64 columns one after the
// other. A piece is one load of a wave straight into LDS, 16 bytes a lane, 128 neighbouring bytes of a token.
// A token's 16-byte unit u lies at place u ^ 4 * (token / 2 % 2), so that the four tokens of 32
// columns that half a wave's transposing read takes spread over all banks.
template <int COLS>
__host__ __device__ constexpr int step_bytes() { return COLS * KT * 2; }

// One operand's way from memory into LDS. The descriptor of a step ends with the last token: tokens past
// it come as zeros; columns past the last one bring what follows, into results that are not stored.
struct StepLoad {
  const unsigned short* base;   // first column of the tile
  long stride;
  int cols, end;                // columns left from there, tokens
  unsigned off;

  DEV_INLINE StepLoad(const unsigned short* base, long stride, int cols, int end) : base(base), stride(stride), cols(cols), end(end) {
    const int lane = threadIdx.x & 63, row = lane >> 3;
    off = (unsigned)(row * stride) * 2u + (((lane & 7) ^ ((row >> 1 & 1) << 2)) * 16);
  }
  DEV_INLINE __amdgpu_buffer_rsrc_t step(int row0) const {
    const int left = min(end - row0, KT);
    const unsigned bytes = ((unsigned)(left - 1) * (unsigned)stride + (unsigned)cols) * 2u;
    return __builtin_amdgcn_make_buffer_rsrc(const_cast<unsigned short*>(base + row0 * stride), 0, left > 0 ? (int)bytes : 0, 0x00027000);
  }
  // the piece of tokens 8 w .. 8 w + 7 and columns 64 cg .. 64 cg + 63
  DEV_INLINE void piece(__amdgpu_buffer_rsrc_t t, char* __restrict__ lds, int w, int cg) const {
    __builtin_amdgcn_raw_ptr_buffer_load_lds(t, (lds_ptr)(lds + (cg * 4 + w) * 1024), 16, (int)off, (int)(unsigned)((w * 8 * stride + cg * 64) * 2), 0, 0);
  }
};

struct At {
  int even, odd;   // of a group of 32 columns
  DEV_INLINE explicit At(int lane) {
    const int m = lane & 15;
    even = (lane >> 5) * 1024 + (m >> 2) * 128 + (m >> 3 & 1) * 64 + (lane >> 4 & 1) * 32 + (m & 3) * 8;
    odd = even ^ 64;
  }
};
// fragment of 16 tokens (16 ks ..) of 32 columns (32 cb ..)
DEV_INLINE bf16x8_v frag(const char* __restrict__ lds, const At& at, int ks, int cb) {
  const int o = (cb & 1 ? at.odd : at.even) + (cb >> 1) * 4096 + ks * 2048;
  const bf16x4_v lo = ld_tr16(lds, o), hi = ld_tr16(lds, o + 512);
  return __builtin_shufflevector(lo, hi, 0, 1, 2, 3, 4, 5, 6, 7);
}

template <int N>
DEV_INLINE void arrived_but() { asm volatile("s_waitcnt vmcnt(%0)\n\ts_barrier" ::"n"(N) : "memory"); }

struct Args {
  const unsigned short *dy, *x;
  long ldy, ldx;
  int M, N, K;
  int tiles_m, tiles_n, full;   // tiles written at once; the rest are cut in parts
  int parts, part_k;
  const float* add;             // what the product is added to, or null
  float* sum;                   // float32 result, or null: out
  unsigned short* out;
  float* ws;                    // of the parts
};

DEV_INLINE void where(const Args& a, int t, int& tm, int& tn) {
  constexpr int G = 4;
  const int per = G * a.tiles_n, g = t / per, rows = min(G, a.tiles_m - g * G), i = t - g * per;
  tm = g * G + i % rows;
  tn = i / rows;
}

DEV_INLINE int xcd_chunk(int f, int n) {
  const int q = n >> 3, r = n & 7, xcd = f & 7;
  return (xcd < r ? xcd * (q + 1) : r * (q + 1) + (xcd - r) * q) + (f >> 3);
}

// four neighbouring sums of a fragment
DEV_INLINE float4v sums(const f32x16& c, int jj) { return float4v{c[jj * 4], c[jj * 4 + 1], c[jj * 4 + 2], c[jj * 4 + 3]}; }

DEV_INLINE void put(const Args& a, long at, float4v v) {
  if (a.sum) {
    *reinterpret_cast<float4v*>(a.sum + at) = v;
    return;
  }
  short4v pk;
#pragma unroll
  for (int e = 0; e < 4; ++e) pk[e] = (short)f2bf(v[e]);
  *reinterpret_cast<short4v*>(a.out + at) = pk;
}

template <int TM, int TN>
__global__ __launch_bounds__(256, TM == 256 ? 1 : 2) void weight_grad_kernel(const Args a) {
  extern __shared__ char smem[];
  constexpr int FA = TN / 64, FB = TM / 64;
  constexpr int YB = step_bytes<TM>(), SB = YB + step_bytes<TN>();
  constexpr int PER = FA + FB;
  const int lane = threadIdx.x & 63, half = lane >> 5, ln = lane & 31;
  const int w = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int wm = w & 1, wn = w >> 1;

  int f = blockIdx.x, tile, part = -1, k0 = 0, k1 = a.K;
  if (f < a.full) {
    tile = xcd_chunk(f, a.full);
  } else {
    f = xcd_chunk(f - a.full, (int)gridDim.x - a.full);
    const int rest = a.tiles_m * a.tiles_n - a.full;
    part = f / rest;
    tile = a.full + f % rest;
    k0 = part * a.part_k;
    k1 = min(a.K, k0 + a.part_k);
  }
  int tm, tn;
  where(a, tile, tm, tn);
  const int m0 = tm * TM, n0 = tn * TN;
  const StepLoad yl(a.dy + m0, a.ldy, a.M - m0, k1), xl(a.x + n0, a.ldx, a.N - n0, k1);

  f32x16 acc[FA][FB];
#pragma unroll
  for (int i = 0; i < FA; ++i)
#pragma unroll
    for (int j = 0; j < FB; ++j)
#pragma unroll
      for (int e = 0; e < 16; ++e) acc[i][j][e] = 0.0f;

  const int steps = (k1 - k0 + KT - 1) / KT;
  auto bring = [&](int s, char* __restrict__ to, int i, __amdgpu_buffer_rsrc_t yt, __amdgpu_buffer_rsrc_t xt) __attribute__((always_inline)) {
    if (i < FB) yl.piece(yt, to, w, i);
    else xl.piece(xt, to + YB, w, i - FB);
  };
#pragma unroll
  for (int s = 0; s < STEPS - 1; ++s) {
    const auto yt = yl.step(k0 + s * KT), xt = xl.step(k0 + s * KT);
#pragma unroll
    for (int i = 0; i < PER; ++i) bring(s, smem + s * SB, i, yt, xt);
  }
  const At at(lane);
  bf16x8_v fx[2][FA], fy[2][FB];
  // fragments in the order of their use
  auto read = [&](const char* __restrict__ st, int ks, int r, bf16x8_v (&px)[FA], bf16x8_v (&py)[FB]) __attribute__((always_inline)) {
    if (r == 0) px[0] = frag(st + YB, at, ks, wn * FA);
    else if (r <= FB) py[r - 1] = frag(st, at, ks, wm * FB + r - 1);
    else px[r - FB] = frag(st + YB, at, ks, wn * FA + r - FB);
  };
  arrived_but<2 * PER>();
#pragma unroll
  for (int r = 0; r < PER; ++r) read(smem, 0, r, fx[0], fy[0]);

  constexpr int NM = FA * FB;
  auto step = [&](int s, const char* __restrict__ cur, const char* __restrict__ nxt, char* __restrict__ to) __attribute__((always_inline)) {
    __amdgpu_buffer_rsrc_t yt, xt;
    const int row = k0 + (s + STEPS - 1) * KT;
#pragma unroll
    for (int i = 0; i < NM; ++i) {
#pragma unroll
      for (int r = i * PER / NM; r < (i + 1) * PER / NM; ++r) read(cur, 1, r, fx[1], fy[1]);
      if (i == NM / 2 - 1) yt = yl.step(row);
      if (i == NM / 2) xt = xl.step(row);
      acc[i / FB][i % FB] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(fx[0][i / FB], fy[0][i % FB], acc[i / FB][i % FB], 0, 0, 0);
      __builtin_amdgcn_sched_barrier(0);
    }
    arrived_but<PER>();
#pragma unroll
    for (int i = 0; i < NM; ++i) {
#pragma unroll
      for (int r = i * PER / NM; r < (i + 1) * PER / NM; ++r) {
        read(nxt, 0, r, fx[0], fy[0]);
        bring(s, to, r, yt, xt);
      }
      acc[i / FB][i % FB] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(fx[1][i / FB], fy[1][i % FB], acc[i / FB][i % FB], 0, 0, 0);
      __builtin_amdgcn_sched_barrier(0);
    }
  };
  for (int s = 0; s < steps; ++s)
    step(s, smem + (s % STEPS) * SB, smem + ((s + 1) % STEPS) * SB, smem + ((s + STEPS - 1) % STEPS) * SB);

  loads_done();   // what is still on its way has no bytes
#pragma unroll
  for (int ib = 0; ib < FB; ++ib) {
    const int ml = (wm * FB + ib) * 32 + ln, m = m0 + ml;
    const int nl = wn * FA * 32 + 4 * half;
    if (part >= 0) {
      float* p = a.ws + ((long)(tile - a.full) * a.parts + part) * TM * TN + ml * TN + nl;
#pragma unroll
      for (int i = 0; i < FA * 4; ++i) *reinterpret_cast<float4v*>(p + i * 8) = sums(acc[i / 4][ib], i % 4);
      continue;
    }
    if (m >= a.M) continue;
    const long at_out = (long)m * a.N + n0 + nl;
    const int left = a.N - n0 - nl;
    float4v add[FA * 4];   // read together: the result may lie in the same place
#pragma unroll
    for (int i = 0; i < FA * 4; ++i) add[i] = a.add && i * 8 < left ? *reinterpret_cast<const float4v*>(a.add + at_out + i * 8) : float4v{0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll
    for (int i = 0; i < FA * 4; ++i)
      if (i * 8 < left) put(a, at_out + i * 8, sums(acc[i / 4][ib], i % 4) + add[i]);
  }
}

// sums the parts of the tiles that were cut
template <int TM, int TN>
__global__ __launch_bounds__(256) void weight_grad_sum_kernel(const Args a) {
  constexpr int PER_TILE = TM * TN / 1024;   // blocks a tile
  const int t = blockIdx.x / PER_TILE, e = ((blockIdx.x % PER_TILE) * 256 + threadIdx.x) * 4;
  int tm, tn;
  where(a, a.full + t, tm, tn);
  const int m = tm * TM + e / TN, n = tn * TN + e % TN;
  if (m >= a.M || n >= a.N) return;
  const float* p = a.ws + (long)t * a.parts * TM * TN + e;
  float4v v = *reinterpret_cast<const float4v*>(p);
  for (int s = 1; s < a.parts; ++s) v += *reinterpret_cast<const float4v*>(p + (long)s * TM * TN);
  const long at_out = (long)m * a.N + n;
  if (a.add) v += *reinterpret_cast<const float4v*>(a.add + at_out);
  put(a, at_out, v);
}

template <int T>
void launch(const Args& a, hipStream_t stream) {
  constexpr int LDS = 2 * step_bytes<T>() * STEPS;
  static const hipError_t ok = hipFuncSetAttribute((const void*)weight_grad_kernel<T, T>, hipFuncAttributeMaxDynamicSharedMemorySize, LDS);
  TORCH_CHECK(ok == hipSuccess, "weight_grad: no ", LDS, " bytes of LDS");
  const int rest = a.tiles_m * a.tiles_n - a.full;
  weight_grad_kernel<T, T><<<a.full + rest * a.parts, 256, LDS, stream>>>(a);
  if (rest) weight_grad_sum_kernel<T, T><<<rest * (T * T / 1024), 256, 0, stream>>>(a);
}

struct Plan {
  int tile, full, parts;
};

// Tile size and parts by the time that they should take. A round of blocks over the 256 CUs takes a step in 0.79 us with large tiles
// (1.36 PFLOP/s) and in 0.25 us with small ones (1.07; two blocks share a CU, each then at half the speed), 5 us
// around its steps; what is left after whole rounds of tiles may be cut into parts of at least 256 tokens, whose sums travel
// at about 5 TB/s both ways and take another launch. A cut has to promise 2 %. Measured, large tiles whole / cut, small
// ones whole / cut, us: 22016 x 4096 x 16384: 2370 / 2214; 4096 x 11008 x 16384: 1132 / 1181, 1927 / 1656;
// 4096 x 768 x 8192: 140 / 65, 69 / 68; 768 x 768 x 8192: 138 / 31, 62 / 22; 512 x 512 x 512: 19 / 18, 8.3 / 10.5.
Plan plan(long M, long N, long K) {
  Plan best{0, 0, 1};
  double least = 0;
  for (int t = 256; t >= 128; t -= 128) {
    const long tiles = ((M + t - 1) / t) * ((N + t - 1) / t), steps = (K + KT - 1) / KT, slots = t == 256 ? 256 : 512;
    const double c = t == 256 ? 0.79 : 0.25;
    auto take = [&](long full, long parts, double us) {
      if (best.tile && us > 0.98 * least) return;
      best = Plan{t, (int)full, (int)parts};
      least = us;
    };
    auto round = [&](long blocks, long n) { return (double)((blocks + 255) / 256) * (n * c + 5.0); };
    take(tiles, 1, round(tiles, steps));
    const long full = tiles / slots * slots, rest = tiles - full;
    for (long p = 2; rest && p * rest <= 512 && p * 8 <= steps; ++p)
      take(full, p, round(full, steps) + round(rest * p, (steps + p - 1) / p) + 3.0 + rest * p * t * t * 8 / 5e6);
  }
  return best;
}

// one operand as the loads take it: columns together, tokens at most 2^24 elements apart, all at addresses of 16 bytes
at::Tensor rows(const at::Tensor& t) {
  const bool as_is = t.stride(1) == 1 && t.stride(0) % 8 == 0 && t.stride(0) >= t.size(1) && t.stride(0) <= (1L << 24)
      && reinterpret_cast<uintptr_t>(t.data_ptr()) % 16 == 0;
  return as_is ? t : t.clone(at::MemoryFormat::Contiguous);
}

}  // namespace wg

// what the kernel multiplies; everything else takes the library's product
bool weight_grad_serves(const at::Tensor& dy, const at::Tensor& x) {
  const long most = 1L << 24;
  return dy.is_cuda() && x.device() == dy.device() && dy.scalar_type() == at::kBFloat16 && x.scalar_type() == at::kBFloat16
      && dy.dim() == 2 && x.dim() == 2 && dy.size(0) == x.size(0) && dy.size(0) > 0 && dy.size(0) < (1L << 30)
      && dy.size(1) > 0 && x.size(1) > 0 && dy.size(1) <= most && x.size(1) <= most && dy.size(1) % 8 == 0 && x.size(1) % 8 == 0
      && ((dy.size(1) + 127) / 128) * ((x.size(1) + 127) / 128) < (1L << 20);
}

// dy [K, M], x [K, N] -> dy^T x (+ add, float32 [M, N]) in bfloat16, or in float32 with `keep`: then in `add` if that is given.
at::Tensor weight_grad(const at::Tensor& dy_in, const at::Tensor& x_in, const c10::optional<at::Tensor>& add, bool keep) {
  if (add)
    TORCH_CHECK(add->device() == dy_in.device() && add->scalar_type() == at::kFloat && add->is_contiguous() && add->dim() == 2
                && add->size(0) == dy_in.size(1) && add->size(1) == x_in.size(1), "weight_grad: add is not a float32 [M, N] matrix");
  if (!weight_grad_serves(dy_in, x_in)) {
    at::Tensor r = at::mm(dy_in.t(), x_in);
    if (add) r = keep ? add->add_(r) : at::add(*add, r);
    return r.to(keep ? at::kFloat : dy_in.scalar_type());
  }
  const c10::hip::HIPGuard guard(dy_in.device().index());
  const at::Tensor dy = wg::rows(dy_in), x = wg::rows(x_in);
  wg::Args a{};
  a.dy = reinterpret_cast<const unsigned short*>(dy.data_ptr());
  a.x = reinterpret_cast<const unsigned short*>(x.data_ptr());
  a.ldy = dy.stride(0);
  a.ldx = x.stride(0);
  a.K = (int)dy.size(0);
  a.M = (int)dy.size(1);
  a.N = (int)x.size(1);
  const wg::Plan plan = wg::plan(a.M, a.N, a.K);
  a.tiles_m = (a.M + plan.tile - 1) / plan.tile;
  a.tiles_n = (a.N + plan.tile - 1) / plan.tile;
  a.full = plan.full;
  a.part_k = ((a.K + plan.parts - 1) / plan.parts + wg::KT - 1) / wg::KT * wg::KT;
  a.parts = (a.K + a.part_k - 1) / a.part_k;
  if (add) a.add = add->data_ptr<float>();
  at::Tensor out = keep && add ? *add : at::empty({a.M, a.N}, dy.options().dtype(keep ? at::kFloat : at::kBFloat16));
  if (keep) a.sum = out.data_ptr<float>();
  else a.out = reinterpret_cast<unsigned short*>(out.data_ptr());
  at::Tensor ws;
  const long rest = (long)a.tiles_m * a.tiles_n - a.full;
  if (rest) {
    ws = at::empty({rest * a.parts * plan.tile * plan.tile}, dy.options().dtype(at::kFloat));
    a.ws = ws.data_ptr<float>();
  }
  const auto stream = at::hip::getCurrentHIPStream();
  if (plan.tile == 256) wg::launch<256>(a, stream);
  else wg::launch<128>(a, stream);
  TORCH_CHECK(hipGetLastError() == hipSuccess, "weight_grad: launch");
  return out;
}

}  // namespace cai
