// The products of linear layers in bfloat16, summed in float32, that are written here and not left to the library:
// weight gradients dW[M, N] = dY[K, M]^T X[K, N] over K tokens, and small X[M, K] W[N, K]^T and dY[M, K] W[K, N].
//
// Operands lie as they come: with the contracted index fast, fragments are plain LDS reads, with it slow (both of a weight
// gradient) transposing ones (ds_read_b64_tr_b16, see flash_attn.hip). Four waves hold a tile's sums in registers, one
// quarter each: 256 x 256 where there is enough of them, which is the least LDS and memory traffic a product has here (a
// wave's 128 x 128 sums are 256 registers, one wave a SIMD), else 256 x 128, also one block a CU (96 KB of LDS), or 128 x 128 with
// two. Four steps of 32
// contracted indices lie in LDS: while one is multiplied the next is there and two are on their way, so that a step waits for
// loads that are two steps old (s_waitcnt vmcnt, never 0) and for one barrier. A wave reads the fragments of the next 16
// indices and issues its loads one by one between the products of the 16 before.
//
// What bounds it: a step of the large tile takes 1203 cycles of which the products are 1024; the clock falls to 1.4 to 1.6
// GHz under it (M 4096 and 12288, N 4096, K 16384). The small tile takes 725 cycles for two blocks, 512 of them products.
//
// Weight gradients M, N, K; us with the library's product -> here:
//   22016, 4096, 16384   2785 -> 2214     4096, 11008, 16384   1536 -> 1132     4096, 4096, 16384   470 -> 404
//   32000, 4096, 4096     952 -> 859      32000, 768, 4096      223 -> 191      4096, 768, 8192      84 -> 61
//   768, 2048, 8192        65 -> 38       768, 768, 8192         49 -> 22       2048, 512, 512       21 -> 10
// Small others, back to back (the library's call takes the host 19 to 20 us, its kernels 5 to 11):
//   x W^T: 512, 1536, 512   19.2 -> 9.0   512, 512, 1024   19.7 -> 11.4     dy W: 512, 512, 2048   19.2 -> 13.9
// Large ones stay with the library: 16384, 12288, 4096   1080 us there, 1468 here; dy W 16384, 4096, 12288   1224, 1377.
#include <torch/extension.h>
#include <ATen/hip/HIPContext.h>
#include <c10/hip/HIPGuard.h>

#include <algorithm>

#include "lds_tiles.h"
#include "plain.h"

namespace cai {

namespace pr {

constexpr int KT = 32;       // contracted indices of a step

// One operand of a product: how a step of it comes into LDS and how the matrix unit's fragments are read from there. A step is pieces
// of 1024 bytes, each brought by one load of a wave straight into LDS, 16 bytes a lane; 32 free indices are
// 2048 bytes. Either form spreads every access over the 64 banks, and both hand out the contracted indices in the same order.
//
// COLS: the free index is the fast one ([K, free] in memory). Pieces of 8 contracted by 64 free indices, the four pieces of 64 free
// indices one after the other, 128 neighbouring bytes a row. A row's 16-byte unit u lies at place u ^ 4 * (row / 2 % 2),
// so that the four rows of 32 columns that half a wave's transposing read takes are in different banks. The descriptor of a
// step ends with the last row: rows past it come as zeros; columns past the last one bring what follows, into results
// that are not stored.
// Rows otherwise ([free, K] in memory). Pieces of 16 free by 32 contracted indices as in lds_tiles.h; free indices past the last
// one come as zeros, and the contracted ones must be a multiple of 32.
template <bool COLS, int T>
struct Operand {
  static constexpr int PER = T / 64, BYTES = T * KT * 2;   // pieces of a wave, bytes of a step
  const unsigned short* base;
  long stride;
  int left, end;                // free indices left from the tile's first one, contracted ones
  unsigned off;
  int even, odd;                // where a lane reads: free indices 0-31 and 32-63 of 64, or contracted ones 0-15 and 16-31

  DEV_INLINE Operand(const unsigned short* p, long stride, int first, int all, int end) : stride(stride), left(all - first), end(end) {
    const int lane = threadIdx.x & 63, half = lane >> 5;
    if (COLS) {
      base = p + first;
      const int row = lane >> 3, m = lane & 15;
      off = (unsigned)(row * stride) * 2u + (((lane & 7) ^ ((row >> 1 & 1) << 2)) * 16);
      even = half * 1024 + (m >> 2) * 128 + (m >> 3 & 1) * 64 + (lane >> 4 & 1) * 32 + (m & 3) * 8;
      odd = even ^ 64;
    } else {
      base = p + (long)first * stride;
      const int row = lane >> 2;
      off = (unsigned)(row * stride) * 2u + (((lane & 3) ^ (row >> 2 & 3)) * 16);
      const RowAt at(lane & 31, half);
      even = at.even;
      odd = at.odd;
    }
  }
  DEV_INLINE __amdgpu_buffer_rsrc_t step(int k) const {
    const int rows = COLS ? min(end - k, KT) : min(left, T);
    const unsigned bytes = ((unsigned)(rows - 1) * (unsigned)stride + (unsigned)(COLS ? left : end - k)) * 2u;
    return __builtin_amdgcn_make_buffer_rsrc(const_cast<unsigned short*>(base + (COLS ? k * stride : (long)k)), 0, k < end ? (int)bytes : 0, 0x00027000);
  }
  // piece i of wave w
  DEV_INLINE void piece(__amdgpu_buffer_rsrc_t t, char* __restrict__ lds, int w, int i) const {
    const int c = i * 4 + w;
    const unsigned at = COLS ? (unsigned)(w * 8 * stride + i * 64) * 2u : (unsigned)(c * 16 * stride) * 2u;
    __builtin_amdgcn_raw_ptr_buffer_load_lds(t, (lds_ptr)(lds + c * 1024), 16, (int)off, (int)at, 0, 0);
  }
  // contracted indices 16 ks .. of free ones 32 b ..
  DEV_INLINE bf16x8_v frag(const char* __restrict__ lds, int ks, int b) const {
    if (!COLS) return *reinterpret_cast<const bf16x8_v*>(lds + (ks ? odd : even) + b * 2048);
    const int o = (b & 1 ? odd : even) + (b >> 1) * 4096 + ks * 2048;
    const bf16x4_v lo = ld_tr16(lds, o), hi = ld_tr16(lds, o + 512);
    return __builtin_shufflevector(lo, hi, 0, 1, 2, 3, 4, 5, 6, 7);
  }
};

template <int N>
DEV_INLINE void arrived_but() { asm volatile("s_waitcnt vmcnt(%0)\n\ts_barrier" ::"n"(N) : "memory"); }

struct Args {
  const unsigned short *p, *q;  // C[m, n] = sum over k of P(m, k) Q(n, k)
  long ldp, ldq;
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

// STEPS steps lie in LDS: one in use, one arrived, the others on their way.
template <bool PC, bool QC, int TM, int TN, int STEPS>
__global__ __launch_bounds__(256, TM == 256 ? 1 : 2) void product_kernel(const Args a) {
  extern __shared__ char smem[];
  constexpr int FA = TN / 64, FB = TM / 64;
  constexpr int YB = Operand<PC, TM>::BYTES, SB = YB + Operand<QC, TN>::BYTES;
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
  const Operand<PC, TM> P(a.p, a.ldp, m0, a.M, k1);
  const Operand<QC, TN> Q(a.q, a.ldq, n0, a.N, k1);

  f32x16 acc[FA][FB];
#pragma unroll
  for (int i = 0; i < FA; ++i)
#pragma unroll
    for (int j = 0; j < FB; ++j)
#pragma unroll
      for (int e = 0; e < 16; ++e) acc[i][j][e] = 0.0f;

  const int steps = (k1 - k0 + KT - 1) / KT;
  auto bring = [&](int s, char* __restrict__ to, int i, __amdgpu_buffer_rsrc_t yt, __amdgpu_buffer_rsrc_t xt) __attribute__((always_inline)) {
    if (i < FB) P.piece(yt, to, w, i);
    else Q.piece(xt, to + YB, w, i - FB);
  };
#pragma unroll
  for (int s = 0; s < STEPS - 1; ++s) {
    const auto yt = P.step(k0 + s * KT), xt = Q.step(k0 + s * KT);
#pragma unroll
    for (int i = 0; i < PER; ++i) bring(s, smem + s * SB, i, yt, xt);
  }
  bf16x8_v fx[2][FA], fy[2][FB];
  // fragments in the order of their use
  auto read = [&](const char* __restrict__ st, int ks, int r, bf16x8_v (&px)[FA], bf16x8_v (&py)[FB]) __attribute__((always_inline)) {
    if (r == 0) px[0] = Q.frag(st + YB, ks, wn * FA);
    else if (r <= FB) py[r - 1] = P.frag(st, ks, wm * FB + r - 1);
    else px[r - FB] = Q.frag(st + YB, ks, wn * FA + r - FB);
  };
  arrived_but<(STEPS - 2) * PER>();
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
      if (i == NM / 2 - 1) yt = P.step(row);
      if (i == NM / 2) xt = Q.step(row);
      acc[i / FB][i % FB] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(fx[0][i / FB], fy[0][i % FB], acc[i / FB][i % FB], 0, 0, 0);
      __builtin_amdgcn_sched_barrier(0);
    }
    arrived_but<(STEPS - 3) * PER>();
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
  int at = 0;   // the step's place in the ring
  for (int s = 0; s < steps; ++s) {
    const int next = at + SB == STEPS * SB ? 0 : at + SB, last = at == 0 ? (STEPS - 1) * SB : at - SB;
    step(s, smem + at, smem + next, smem + last);
    at = next;
  }

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
__global__ __launch_bounds__(256) void product_sum_kernel(const Args a) {
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

template <bool PC, bool QC, int TM, int TN, int STEPS>
void launch(const Args& a, hipStream_t stream) {
  constexpr int LDS = (TM + TN) * KT * 2 * STEPS;
  const auto kernel = product_kernel<PC, QC, TM, TN, STEPS>;
  if (LDS > 65536) (void)hipFuncSetAttribute((const void*)kernel, hipFuncAttributeMaxDynamicSharedMemorySize, LDS);   // of the current device
  const int rest = a.tiles_m * a.tiles_n - a.full;
  kernel<<<a.full + rest * a.parts, 256, LDS, stream>>>(a);
  if (rest) product_sum_kernel<TM, TN><<<rest * (TM * TN / 1024), 256, 0, stream>>>(a);
}

struct Plan {
  int tm, tn, full, parts;
  double us;
};

// Tile size and parts by the time that they should take. A round of blocks over the 256 CUs takes a step in 0.76 us with 256 x 256 tiles
// (1.41 PFLOP/s) and in 0.25 us with 128 x 128 ones (1.07; two blocks share a CU, each then at half the speed), 14 and 5 us
// around its steps (the first loads, the stores); what is left after whole rounds of tiles may be cut into parts of at least 256
// contracted indices, whose sums travel at about 5 TB/s both ways and take another launch. Tiles of 256 x 128 take 0.36 us and 9 around them as long as one round
// is all; over several the clock falls, and they are no better than 128 x 128. A change has to promise 2 %. Measured, weight
// gradients, 256 x 256 whole / cut, 256 x 128 cut, 128 x 128 whole / cut, us: 22016 x 4096 x 16384: 2370 / 2214, 2731, -;
// 4096 x 11008 x 16384: 1132 / 1181, -, 1927 / 1656; 4096 x 768 x 8192: 140 / 63, 61, 69 / 66; 768 x 2048 x 8192: 146 / 44, 38, 68 / 39;
// 768 x 768 x 8192: 138 / 31, 25, 62 / 22; 512 x 512 x 512: 19 / 18, 14, 8.3 / 10.5.
Plan plan(long M, long N, long K, bool small_only) {
  struct { int tm, tn; double step, around; long slots; bool one_round; } forms[] = {
      {256, 256, 0.76, 14.0, 256, false}, {256, 128, 0.36, 9.0, 256, true}, {128, 128, 0.25, 5.0, 512, false}};
  Plan best{0, 0, 0, 1, 0.0};
  for (const auto& form : forms) {
    if (small_only && form.tm != 128) continue;
    const long tiles = ((M + form.tm - 1) / form.tm) * ((N + form.tn - 1) / form.tn), steps = (K + KT - 1) / KT;
    if (form.one_round && tiles > 256) continue;
    auto take = [&](long full, long parts, double us) {
      if (best.tm == 0 || us < 0.98 * best.us) best = Plan{form.tm, form.tn, (int)full, (int)parts, us};
    };
    auto round = [&](long blocks, long n) { return (double)((blocks + 255) / 256) * (n * form.step + form.around); };
    take(tiles, 1, round(tiles, steps));
    const long full = tiles / form.slots * form.slots, rest = tiles - full;
    for (long p = 2; rest && p * rest <= (form.one_round ? 256 : 512) && p * 8 <= steps; ++p)
      take(full, p, round(full, steps) + round(rest * p, (steps + p - 1) / p) + 3.0 + rest * p * form.tm * form.tn * 8 / 5e6);
  }
  return best;
}

// an operand as the loads take it: the fast index together, the slow one's elements at most 2^22 apart, all at addresses of 16 bytes
bool loadable(const at::Tensor& t) {
  return t.stride(1) == 1 && t.stride(0) % 8 == 0 && t.stride(0) >= t.size(1) && t.stride(0) <= (1L << 22)
      && reinterpret_cast<uintptr_t>(t.data_ptr()) % 16 == 0;
}

template <bool PC, bool QC>
at::Tensor run(const at::Tensor& p, const at::Tensor& q, Plan plan, const c10::optional<at::Tensor>& add, bool keep) {
  const c10::hip::HIPGuard guard(p.device().index());
  Args a{};
  a.p = reinterpret_cast<const unsigned short*>(p.data_ptr());
  a.q = reinterpret_cast<const unsigned short*>(q.data_ptr());
  a.ldp = p.stride(0);
  a.ldq = q.stride(0);
  a.K = (int)p.size(PC ? 0 : 1);
  a.M = (int)p.size(PC ? 1 : 0);
  a.N = (int)q.size(QC ? 1 : 0);
  a.tiles_m = (a.M + plan.tm - 1) / plan.tm;
  a.tiles_n = (a.N + plan.tn - 1) / plan.tn;
  a.full = plan.full;
  a.part_k = ((a.K + plan.parts - 1) / plan.parts + KT - 1) / KT * KT;
  a.parts = (a.K + a.part_k - 1) / a.part_k;
  if (add) a.add = add->data_ptr<float>();
  at::Tensor out = keep && add ? *add : at::empty({a.M, a.N}, p.options().dtype(keep ? at::kFloat : at::kBFloat16));
  if (keep) a.sum = out.data_ptr<float>();
  else a.out = reinterpret_cast<unsigned short*>(out.data_ptr());
  at::Tensor ws;
  const long rest = (long)a.tiles_m * a.tiles_n - a.full;
  if (rest) {
    ws = at::empty({rest * a.parts * plan.tm * plan.tn}, p.options().dtype(at::kFloat));
    a.ws = ws.data_ptr<float>();
  }
  const auto stream = at::hip::getCurrentHIPStream();
  if constexpr (PC) {
    if (plan.tn == 256) launch<PC, QC, 256, 256, 4>(a, stream);
    else if (plan.tm == 256) launch<PC, QC, 256, 128, 4>(a, stream);
    else launch<PC, QC, 128, 128, 4>(a, stream);
  } else {
    launch<PC, QC, 128, 128, 4>(a, stream);
  }
  HIP_CHECK_LAST();
  return out;
}

// bfloat16 matrices on one device that nothing watches: a mode that counts or rewrites operations is to see the library's products
bool bf16_pair(const at::Tensor& p, const at::Tensor& q) {
  return plain(p) && plain(q) && p.is_cuda() && q.device() == p.device() && p.scalar_type() == at::kBFloat16 && q.scalar_type() == at::kBFloat16
      && p.dim() == 2 && q.dim() == 2 && p.size(0) < (1L << 30) && p.numel() > 0 && q.numel() > 0;
}

}  // namespace pr

// what the kernel can multiply; everything else takes the library's product
bool weight_grad_serves(const at::Tensor& dy, const at::Tensor& x) {
  const long most = 1L << 22;
  return pr::bf16_pair(dy, x) && dy.size(0) == x.size(0) && dy.size(1) <= most && x.size(1) <= most && dy.size(1) % 8 == 0
      && x.size(1) % 8 == 0 && ((dy.size(1) + 127) / 128) * ((x.size(1) + 127) / 128) < (1L << 20);
}

// dy [K, M], x [K, N] -> dy^T x (+ add, float32 [M, N]) in bfloat16, or in float32 with `keep`: then in `add` if that is given.
at::Tensor weight_grad(const at::Tensor& dy, const at::Tensor& x, const c10::optional<at::Tensor>& add, bool keep) {
  if (add)
    TORCH_CHECK(add->device() == dy.device() && add->scalar_type() == at::kFloat && add->is_contiguous() && add->dim() == 2
                && add->size(0) == dy.size(1) && add->size(1) == x.size(1), "weight_grad: add is not a float32 [M, N] matrix");
  // the kernels read and write sums 16 bytes at a time
  if (add && reinterpret_cast<uintptr_t>(add->data_ptr()) % 16 != 0) {
    const at::Tensor r = weight_grad(dy, x, c10::nullopt, true);
    return keep ? add->add_(r) : at::add(*add, r).to(dy.scalar_type());
  }
  const bool serves = weight_grad_serves(dy, x);
  const pr::Plan plan = serves ? pr::plan(dy.size(1), x.size(1), dy.size(0), false) : pr::Plan{};
  // Over few tokens storing a large result is most of the work, which the library does faster. Its time and the kernel's, us: 22016 x 4096 over
  // 64, 256, 512, 1024 and 2048 tokens 63, 103, 126, 213, 404 and 112, 143, 176, 241, 373; 4096 x 4096 12, 18, 26, 40, 71 and 23, 27,
  // 33, 45, 70. Over results of 9 to 131 million elements the kernel takes 1.5 times the library's at 100 tokens, 1.2 at 500, 1.06 from 1000 to
  // 1500 (1.2 at 1536) and 1 at 1700 to 2000; below 2^23 elements it is ahead or, up to 10 us, bound by the host (see multiply). A
  // float32 result the library does not have.
  if (!serves || (!add && !keep && dy.size(0) < 1600 && dy.size(1) * x.size(1) > (1L << 23))) {
    at::Tensor r = at::mm(dy.t(), x);
    if (add) r = keep ? add->add_(r) : at::add(*add, r);
    return r.to(keep ? at::kFloat : dy.scalar_type());
  }
  return pr::run<true, true>(pr::loadable(dy) ? dy : dy.clone(at::MemoryFormat::Contiguous),
                             pr::loadable(x) ? x : x.clone(at::MemoryFormat::Contiguous), plan, add, keep);
}

// x [M, K] times w [N, K]^T, or with `slow` times w [K, N]. Products that should take at most 14 us are formed here, because the host
// takes 19 to 20 us for the library's call and 9 for this one, and a chain of such products waits for it. On the device they
// are no faster, 6 to 13 us where the library's kernels take 4 to 11. Steps of two layers, us, library and here: width 512, 512 tokens 1320
// and 1050 (kernels 490 and 525); 1024, 512 tokens 1130 and 900; where the device is the bound nothing shows: 512, 4096 tokens 1316 and
// 1301, 1024, 2048 tokens 1343 and 1347.
at::Tensor multiply(const at::Tensor& x, const at::Tensor& w, bool slow) {
  if (pr::bf16_pair(x, w) && x.size(1) == w.size(slow ? 0 : 1) && x.size(1) % pr::KT == 0 && w.size(slow ? 1 : 0) % 8 == 0
      && pr::loadable(x) && pr::loadable(w)) {
    const long M = x.size(0), N = w.size(slow ? 1 : 0), K = x.size(1);
    if (((M + 127) / 128) * ((N + 127) / 128) <= 256) {
      const pr::Plan plan = pr::plan(M, N, K, true);
      if (plan.us <= 14.0) return slow ? pr::run<false, true>(x, w, plan, c10::nullopt, false) : pr::run<false, false>(x, w, plan, c10::nullopt, false);
    }
  }
  return slow ? at::mm(x, w) : at::mm(x, w.t());
}

}  // namespace cai
