// The products of linear layers in bfloat16, summed in float32, that are written here and not left to the library:
// weight gradients dW[M, N] = dY[K, M]^T X[K, N] over K tokens, and small X[M, K] W[N, K]^T and dY[M, K] W[K, N].
//
// Operands lie as they come: with the contracted index fast, fragments are plain LDS reads, with it slow (both of a weight
// gradient) transposing ones (ds_read_b64_tr_b16, see flash_attn.hip). Four waves hold a tile's sums in registers, one
// quarter each: 256 x 256 where there is enough of them, which is the least LDS and memory traffic a product has here (a
// wave's 128 x 128 sums are 256 registers, one wave a SIMD), else 256 x 128, also one block a CU (96 KB of LDS), or 128 x 128 with
// two. Four steps of 32 contracted indices lie in LDS. A wave reads each fragment again, from the next step, as soon as its last product of this
// one is done; loads go to a step's place half a step after all of its fragments are read, so that they are two and a half to three
// steps old when they are waited for (s_waitcnt vmcnt, never 0), at one barrier a step.
//
// What bounds it: power, and the issue of one wave a SIMD. Matrix instructions of 16 x 16 x 32 instead of 32 x 32 x 16 touch the sums half as
// often: a loop of nothing else runs at 2060 TFLOP/s on the full chip for 1775. They leave room for two to three other instructions
// each (a third one costs 4 cycles of 16), so that reads and loads stand one by one between them, nothing else is computed in the loop, and the ring
// is unrolled. M 12288, N 4096, K 16384: 32 x 32 x 16 74 % of the cycles are products, at 1.44 GHz; 16 x 16 x 32 in the same order 61 %, 1.71 GHz; as
// it is now 78 %, 1.50 GHz.
//
// Weight gradients M, N, K; us with the library's product -> 32 x 32 x 16 -> here:
//   22016, 4096, 16384   2800 -> 2270 -> 2060     4096, 11008, 16384   1540 -> 1140 -> 1040     4096, 4096, 16384   460 -> 403 -> 375
//   32000, 4096, 4096     940 -> 893 -> 806       32000, 768, 8192     462 -> 347 -> 320        4096, 768, 8192      77 -> 59 -> 56
//   768, 2048, 8192        62 -> 36 -> 34         768, 768, 8192        48 -> 21 -> 19          3072, 1024, 2048     24 -> 22 -> 19
// Small others, back to back (the library's call takes the host 19 to 20 us, its kernels 5 to 11), with the products of 32 x 32 x 16:
//   x W^T: 512, 1536, 512   19.2 -> 9.0   512, 512, 1024   19.7 -> 11.4     dy W: 512, 512, 2048   19.2 -> 13.9 (with the weight gradient: linear_grads)
// Large ones stay with the library: 16384, 12288, 4096   1048 us there, 1490 here (its rows are read 64 bytes at a time); dy W 16384, 4096, 12288   1181 there, 1255
// here with the present products, 16384, 4096, 22016   2122, 2130, 16384, 11008, 4096   1192, 1144, 8192, 768, 4096   59, 59.
#include <torch/extension.h>
#include <ATen/hip/HIPContext.h>
#include <c10/hip/HIPGuard.h>

#include <algorithm>

#include "lds_tiles.h"
#include "plain.h"

namespace cai {

namespace pr {

constexpr int KT = 32;       // contracted indices of a step

// One operand of a product: how a step of it comes into LDS and how the matrix unit's fragments (16 free by 32 contracted indices, eight of the
// contracted ones a lane) are read from there. A step is pieces of 1024 bytes, each brought by one load of a wave straight into LDS, 16 bytes a lane.
// Either form spreads every access over the 64 banks, and both hand out the contracted indices in the same order.
//
// COLS: the free index is the fast one ([K, free] in memory). Pieces of 8 contracted by 64 free indices, the four pieces of 64 free
// indices one after the other, 128 neighbouring bytes a row. A row's 16-byte unit u lies at place u ^ 4 * (row / 2 % 2) ^ 2 * (piece % 2),
// so that the eight rows of 16 columns that half a wave's transposing read takes, four of either piece, are in different banks. The descriptor of a
// step ends with the last row: rows past it come as zeros; columns past the last one bring what follows, into results
// that are not stored.
// Rows otherwise ([free, K] in memory). Pieces of 16 free by 32 contracted indices as in lds_tiles.h; free indices past the last
// one come as zeros, and the contracted ones must be a multiple of 32.
template <bool COLS, int T>
struct Operand {
  static constexpr int PER = T / 64, BYTES = T * KT * 2;   // pieces of a wave, bytes of a step
  const unsigned short* base;   // of the next step to be brought
  long stride;
  int whole, last;              // bytes of a step, of the last one
  unsigned off;
  int at[COLS ? 4 : 1];         // where a lane reads, by which 16 of 64 free indices

  // the operand's free indices from `first` on, of `all`, contracted ones from k0 up to k1
  DEV_INLINE Operand(const unsigned short* p, long stride, int first, int all, int k0, int k1, int w) : stride(stride) {
    const int lane = threadIdx.x & 63, m = lane & 15, g = lane >> 4, left = all - first;
    if (COLS) {
      base = p + first + k0 * stride;
      whole = (int)(((unsigned)(KT - 1) * (unsigned)stride + (unsigned)left) * 2u);
      last = (int)(((unsigned)((k1 - k0 - 1) % KT) * (unsigned)stride + (unsigned)left) * 2u);
      const int row = lane >> 3;
      off = (unsigned)(row * stride) * 2u + (((lane & 7) ^ ((row >> 1 & 1) << 2) ^ ((w & 1) << 1)) * 16);
#pragma unroll
      for (int b = 0; b < 4; ++b)
        at[COLS ? b : 0] = g * 1024 + (m >> 2) * 128 + ((b * 2) ^ (m >> 1 & 1) ^ ((m >> 3 & 1) << 2) ^ ((g & 1) << 1)) * 16 + (m & 1) * 8;
    } else {
      base = p + (long)first * stride + k0;
      whole = last = (int)(((unsigned)(min(left, T) - 1) * (unsigned)stride + KT) * 2u);
      const int row = lane >> 2;
      off = (unsigned)(row * stride) * 2u + (((lane & 3) ^ (row >> 2 & 3)) * 16);
      at[0] = m * 64 + (g ^ (m >> 2)) * 16;
    }
  }
  // the next step, `left` of them with it
  DEV_INLINE __amdgpu_buffer_rsrc_t step(int left) {
    const auto t = __builtin_amdgcn_make_buffer_rsrc(const_cast<unsigned short*>(base), 0, left > 1 ? whole : left == 1 ? last : 0, 0x00027000);
    base += COLS ? KT * stride : (long)KT;
    return t;
  }
  // piece i of wave w
  DEV_INLINE void piece(__amdgpu_buffer_rsrc_t t, char* __restrict__ lds, int w, int i) const {
    const int c = i * 4 + w;
    const unsigned from = COLS ? (unsigned)(w * 8 * stride + i * 64) * 2u : (unsigned)(c * 16 * stride) * 2u;
    __builtin_amdgcn_raw_ptr_buffer_load_lds(t, (lds_ptr)(lds + c * 1024), 16, (int)off, (int)from, 0, 0);
  }
  // A step's contracted indices of free ones 16 b ..: lane l has those from 8 * (l / 16) on of free index l % 16. Read r of READS.
  static constexpr int READS = COLS ? 2 : 1;
  struct Frag {
    bf16x4_v lo, hi;
    bf16x8_v row;
    DEV_INLINE bf16x8_v all() const { return COLS ? __builtin_shufflevector(lo, hi, 0, 1, 2, 3, 4, 5, 6, 7) : row; }
  };
  DEV_INLINE void read(const char* __restrict__ lds, int b, int r, Frag& f) const {
    if constexpr (COLS) (r ? f.hi : f.lo) = ld_tr16(lds, at[b & 3] + (b >> 2) * 4096 + r * 512);
    else f.row = *reinterpret_cast<const bf16x8_v*>(lds + at[0] + b * 1024);
  }
};

// every wave's loads but the last N have arrived, and what it has read from LDS too
template <int N>
DEV_INLINE void arrived_but() { asm volatile("s_waitcnt vmcnt(%0) lgkmcnt(0)\n\ts_barrier" ::"n"(N) : "memory"); }

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

// c += x y. The compiler copies sums that are loop-carried in accumulation registers to other ones and back around each product of this size (128 moves and 50
// waits in a loop of 32 products), so it is told the register. What the compiler would otherwise look after: settled() stands between these products and
// any other use of the sums, ahead of them and behind them. check_products.py looks for these distances in what each build has made of it.
template <bool ACC>
DEV_INLINE void mac(float4v& c, bf16x8_v x, bf16x8_v y) {
  if constexpr (ACC) asm volatile("v_mfma_f32_16x16x32_bf16 %0, %1, %2, %0" : "+a"(c) : "v"(x), "v"(y));
  else c = __builtin_amdgcn_mfma_f32_16x16x32_bf16(x, y, c, 0, 0, 0);
}
// A product's result may be read 7 cycles of issue after it, and a product may read what another instruction wrote 2 after that.
template <int FA, int FB>
DEV_INLINE void settled(float4v (&c)[FA][FB]) {
  auto each = [&]() __attribute__((always_inline)) {
#pragma unroll
    for (int i = 0; i < FA; ++i)
#pragma unroll
      for (int j = 0; j < FB; ++j) asm volatile("" : "+a"(c[i][j]));
  };
  each();
  asm volatile("s_nop 15");
  each();
}

// Behind which of a half step's N products its reads and loads stand: of `reads` those from `at` on are each not before a product of their own
// (`each` reads every `every` products), loads where no read is, as long as there is room.
template <int N, int READS, int LOADS>
struct Places {
  int read[READS] = {}, load[LOADS] = {};
  constexpr Places(int at, int each, int every) {
    constexpr int MOST = (READS + LOADS + N - 1) / N;   // between two products
    int used[N] = {};
    for (int r = 0, n = 0; r < READS; ++r) {
      const int first = r < at ? 0 : ((r - at) / each + 1) * every;
      if (n < first) n = first;
      while (n < N - 1 && used[n] >= MOST) ++n;
      read[r] = n;
      ++used[n];
    }
    for (int l = 0, n = 0; l < LOADS; ++l) {
      const int even = (2 * l + 1) * N / (2 * LOADS);
      if (n < even) n = even;
      while (n < N - 1 && used[n] >= MOST) ++n;
      if (used[n] >= MOST) n = even;
      load[l] = n;
      ++used[n];
    }
  }
};

// Block f of `blocks`. STEPS steps lie in LDS: one in use, one arrived, the others on their way.
template <bool PC, bool QC, int TM, int TN, int STEPS>
DEV_INLINE void product_block(const Args& a, char* smem, int f, int blocks) {
  constexpr int FA = TN / 32, FB = TM / 32;      // fragments of a wave
  constexpr int YB = Operand<PC, TM>::BYTES, SB = YB + Operand<QC, TN>::BYTES;
  constexpr int PY = Operand<PC, TM>::PER, PER = PY + Operand<QC, TN>::PER;
  const int lane = threadIdx.x & 63, quarter = lane >> 4, ln = lane & 15;
  const int w = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int wm = w & 1, wn = w >> 1;

  int tile, part = -1, k0 = 0, k1 = a.K;
  if (f < a.full) {
    tile = xcd_chunk(f, a.full);
  } else {
    f = xcd_chunk(f - a.full, blocks - a.full);
    const int rest = a.tiles_m * a.tiles_n - a.full;
    part = f / rest;
    tile = a.full + f % rest;
    k0 = part * a.part_k;
    k1 = min(a.K, k0 + a.part_k);
  }
  int tm, tn;
  where(a, tile, tm, tn);
  const int m0 = tm * TM, n0 = tn * TN;
  Operand<PC, TM> P(a.p, a.ldp, m0, a.M, k0, k1, w);
  Operand<QC, TN> Q(a.q, a.ldq, n0, a.N, k0, k1, w);

  float4v acc[FA][FB];
#pragma unroll
  for (int i = 0; i < FA; ++i)
#pragma unroll
    for (int j = 0; j < FB; ++j) acc[i][j] = float4v{0.0f, 0.0f, 0.0f, 0.0f};

  const int steps = (k1 - k0 + KT - 1) / KT;
  auto bring = [&](char* __restrict__ to, int i, __amdgpu_buffer_rsrc_t yt, __amdgpu_buffer_rsrc_t xt) __attribute__((always_inline)) {
    if (i < PY) P.piece(yt, to, w, i);
    else Q.piece(xt, to + YB, w, i - PY);
  };
#pragma unroll
  for (int s = 0; s < STEPS - 1; ++s) {
    const auto yt = P.step(steps - s), xt = Q.step(steps - s);
#pragma unroll
    for (int i = 0; i < PER; ++i) bring(smem + s * SB, i, yt, xt);
  }
  // A step multiplies the first half of P's fragments with all of Q's, then the second half. Each fragment is read again as soon as its last product
  // is done, in the same registers: Q's and the first half of P's in a step's second half, from the next step, the others in the first half. Between the
  // halves every wave has read all of the step, and the step that is STEPS ahead goes to its place: half of its loads in this second half, half in
  // the next first one. One read or load stands between two products, where there is time for three instructions.
  constexpr int H = FB / 2, NM = FA * H, LH = PER / 2;
  constexpr bool ACC = TM == 256;
  typename Operand<PC, TM>::Frag fy[FB];
  typename Operand<QC, TN>::Frag fx[FA];
  constexpr int RP = Operand<PC, TM>::READS, RQ = Operand<QC, TN>::READS;
  auto read_x = [&](const char* __restrict__ st, int i, int r) __attribute__((always_inline)) { Q.read(st + YB, wn * FA + i, r, fx[i]); };
  auto read_y = [&](const char* __restrict__ st, int j, int r) __attribute__((always_inline)) { P.read(st, wm * FB + j, r, fy[j]); };
  __amdgpu_buffer_rsrc_t yt = P.step(steps - (STEPS - 1)), xt = Q.step(steps - (STEPS - 1));
#pragma unroll
  for (int i = 0; i < LH; ++i) bring(smem + (STEPS - 1) * SB, i, yt, xt);
  arrived_but<(STEPS - 2) * PER + LH>();
#pragma unroll
  for (int j = 0; j < H * RP; ++j) read_y(smem, j / RP, j % RP);
#pragma unroll
  for (int i = 0; i < (FA - 1) * RQ; ++i) read_x(smem, i / RQ, i % RQ);

  constexpr Places<NM, RQ + H * RP, LH> one(RQ + H * RP, 1, 1);
  constexpr Places<NM, H * RP + (FA - 1) * RQ, LH> two(H * RP, RQ, H);
  auto step = [&](int left, const char* __restrict__ cur, const char* __restrict__ nxt, char* __restrict__ before) __attribute__((always_inline)) {
#pragma unroll
    for (int n = 0; n < NM; ++n) {
      mac<ACC>(acc[n / H][n % H], fx[n / H].all(), fy[n % H].all());
#pragma unroll
      for (int r = 0; r < RQ + H * RP; ++r)
        if (one.read[r] == n) {
          if (r < RQ) read_x(cur, FA - 1, r);
          else read_y(cur, H + (r - RQ) / RP, (r - RQ) % RP);
        }
#pragma unroll
      for (int l = 0; l < LH; ++l)
        if (one.load[l] == n) bring(before, LH + l, yt, xt);
      if (n == (one.load[LH - 1] > NM - 2 ? one.load[LH - 1] : NM - 2)) yt = P.step(left - STEPS);   // behind the last load that takes it
      __builtin_amdgcn_sched_barrier(0);
    }
    arrived_but<(STEPS - 2) * PER>();
#pragma unroll
    for (int n = 0; n < NM; ++n) {
      mac<ACC>(acc[n / H][H + n % H], fx[n / H].all(), fy[H + n % H].all());
#pragma unroll
      for (int r = 0; r < H * RP + (FA - 1) * RQ; ++r)
        if (two.read[r] == n) {
          if (r < H * RP) read_y(nxt, r / RP, r % RP);
          else read_x(nxt, (r - H * RP) / RQ, (r - H * RP) % RQ);
        }
#pragma unroll
      for (int l = 0; l < LH; ++l)
        if (two.load[l] == n) bring(const_cast<char*>(cur), l, yt, xt);
      if (n == NM - 2) xt = Q.step(left - STEPS);
      __builtin_amdgcn_sched_barrier(0);
    }
  };
  if (ACC) settled(acc);
  auto turn = [&](int left, int at) __attribute__((always_inline)) {
    step(left, smem + at * SB, smem + (at + 1) % STEPS * SB, smem + (at + STEPS - 1) % STEPS * SB);
  };
  for (int left = steps; left > 0;) {   // around the ring
#pragma unroll
    for (int at = 0; at < STEPS; ++at) {
      turn(left, at);
      if (--left == 0) break;
    }
  }
  if (ACC) settled(acc);

  loads_done();   // what is still on its way has no bytes
#pragma unroll
  for (int j = 0; j < FB; ++j) {
    const int ml = (wm * FB + j) * 16 + ln, m = m0 + ml;
    const int nl = wn * FA * 16 + 4 * quarter;
    if (part >= 0) {
      float* p = a.ws + ((long)(tile - a.full) * a.parts + part) * TM * TN + ml * TN + nl;
#pragma unroll
      for (int i = 0; i < FA; ++i) *reinterpret_cast<float4v*>(p + i * 16) = acc[i][j];
      continue;
    }
    if (m >= a.M) continue;
    const long at_out = (long)m * a.N + n0 + nl;
    const int left = a.N - n0 - nl;
    float4v add[FA];   // read together: the result may lie in the same place
#pragma unroll
    for (int i = 0; i < FA; ++i) add[i] = a.add && i * 16 < left ? *reinterpret_cast<const float4v*>(a.add + at_out + i * 16) : float4v{0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll
    for (int i = 0; i < FA; ++i)
      if (i * 16 < left) put(a, at_out + i * 16, acc[i][j] + add[i]);
  }
}

template <bool PC, bool QC, int TM, int TN, int STEPS>
__global__ __launch_bounds__(256, TM == 256 ? 1 : 2) void product_kernel(const Args a) {
  extern __shared__ char smem[];
  product_block<PC, QC, TM, TN, STEPS>(a, smem, blockIdx.x, gridDim.x);
}

// dY W (n blocks) and a weight gradient (the others) together
__global__ __launch_bounds__(256, 2) void product_pair_kernel(const Args dx, const Args dw, int n) {
  extern __shared__ char smem[];
  const int f = blockIdx.x;
  if (f < n) product_block<false, true, 128, 128, 4>(dx, smem, f, n);
  else product_block<true, true, 128, 128, 4>(dw, smem, f - n, (int)gridDim.x - n);
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

// Tile size and parts by the time that they should take. A round of blocks over the 256 CUs takes a step in 0.705 us with 256 x 256 tiles
// (1.52 PFLOP/s), in 0.40 us with 256 x 128 and in 0.27 us with 128 x 128 ones (0.21 where the operands come from near; two blocks share a CU, each
// then at half the speed), and 16, 11 and 6 us around its steps (the first loads, the stores); what is left after whole rounds of tiles may be cut into
// parts of at least 256 contracted indices, whose sums travel at about 10 TB/s both ways and take another launch. Tiles of 256 x 128 pay as long as
// one round is all; over several they are no better than 128 x 128. A change has to promise 2 %. Measured, weight gradients, 256 x 256 whole / cut,
// 256 x 128 cut, 128 x 128 whole / cut, us, operands from memory: 4096 x 768 x 8192: 174 / 66, 84, 91 / 86; 2304 x 768 x 8192: 167 / 52, 50, 84 / 56;
// 768 x 2048 x 8192: 161 / 46, 43, 83 / 50; 768 x 768 x 8192: 161 / 35, 28, 78 / 26; 32000 x 768 x 8184: 377 / 342, 410 (whole), 498; 3072 x 1024 x
// 2048: 60 / 37, 32, 28 / 33; 6144 x 2048 x 4096: 106 / 127, 130 (whole), 121 / 133; and the same product over and over: 22016 x 4096 x 16384:
// 2174 / 2056, 2746, 3237; 4096 x 11008 x 16384: 1050 / 1105, 1217 (whole), 1969 / 1708.
// Many parts of few tiles are summed by few blocks, one part after the other: 0.15 us for each part of 128 x 128 tiles. us by parts, operands from memory: 168 x 352 x 9685:
// 34 22.6, 22 19.9; 1328 x 72 x 5463: 19 19.8, 9 17.7; 208 x 480 x 14360: 30 26.6, 18 24.6; 368 x 1304 x 2893: 7 20.4, 4 19.5; 952 x 408 x 970: 3 13.1, whole 17.4.
// Small products (`small`) have 128 x 128 tiles, operands from near, 0.25 us a step and 5 around, and sums that a launch behind them waits for, 5 TB/s.
Plan plan(long M, long N, long K, bool small) {
  struct { int tm, tn; double step, around; long slots; bool one_round; } forms[] = {
      {256, 256, 0.705, 16.0, 256, false}, {256, 128, 0.40, 11.0, 256, true}, {128, 128, small ? 0.25 : 0.27, small ? 5.0 : 6.0, 512, false}};
  Plan best{0, 0, 0, 1, 0.0};
  for (const auto& form : forms) {
    if (small && form.tm != 128) continue;
    const long tiles = ((M + form.tm - 1) / form.tm) * ((N + form.tn - 1) / form.tn), steps = (K + KT - 1) / KT;
    if (form.one_round && tiles > 256) continue;
    auto take = [&](long full, long parts, double us) {
      if (best.tm == 0 || us < 0.98 * best.us) best = Plan{form.tm, form.tn, (int)full, (int)parts, us};
    };
    auto round = [&](long blocks, long n) { return (double)((blocks + 255) / 256) * (n * form.step + form.around); };
    take(tiles, 1, round(tiles, steps));
    const long full = tiles / form.slots * form.slots, rest = tiles - full;
    for (long p = 2; rest && p * rest <= (form.one_round ? 256 : 512) && p * 8 <= steps; ++p)
      take(full, p, round(full, steps) + round(rest * p, (steps + p - 1) / p) + 3.0 + rest * p * form.tm * form.tn * 8 / (small ? 5e6 : 10e6)
                    + (form.tm == 128 && !small ? 0.15 * p : 0.0));
  }
  return best;
}

// an operand as the loads take it: the fast index together, the slow one's elements at most 2^22 apart, all at addresses of 16 bytes
bool loadable(const at::Tensor& t) {
  return t.stride(1) == 1 && t.stride(0) % 8 == 0 && t.stride(0) >= t.size(1) && t.stride(0) <= (1L << 22)
      && reinterpret_cast<uintptr_t>(t.data_ptr()) % 16 == 0;
}

// what a launch takes, with its result and the sums' place
struct Call {
  Args a{};
  at::Tensor out, ws;
  int rest;
  int blocks() const { return a.full + rest * a.parts; }
};

template <bool PC, bool QC>
Call call(const at::Tensor& p, const at::Tensor& q, const Plan& plan, const c10::optional<at::Tensor>& add, bool keep) {
  Call c;
  Args& a = c.a;
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
  c.out = keep && add ? *add : at::empty({a.M, a.N}, p.options().dtype(keep ? at::kFloat : at::kBFloat16));
  if (keep) a.sum = c.out.data_ptr<float>();
  else a.out = reinterpret_cast<unsigned short*>(c.out.data_ptr());
  c.rest = a.tiles_m * a.tiles_n - a.full;
  if (c.rest) {
    c.ws = at::empty({(long)c.rest * a.parts * plan.tm * plan.tn}, p.options().dtype(at::kFloat));
    a.ws = c.ws.data_ptr<float>();
  }
  return c;
}

template <bool PC, bool QC>
at::Tensor run(const at::Tensor& p, const at::Tensor& q, Plan plan, const c10::optional<at::Tensor>& add, bool keep) {
  const c10::hip::HIPGuard guard(p.device().index());
  const Call c = call<PC, QC>(p, q, plan, add, keep);
  const Args& a = c.a;
  const auto stream = at::hip::getCurrentHIPStream();
  if constexpr (PC) {
    if (plan.tn == 256) launch<PC, QC, 256, 256, 4>(a, stream);
    else if (plan.tm == 256) launch<PC, QC, 256, 128, 4>(a, stream);
    else launch<PC, QC, 128, 128, 4>(a, stream);
  } else {
    launch<PC, QC, 128, 128, 4>(a, stream);
  }
  HIP_CHECK_LAST();
  return c.out;
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

// Over few tokens storing a large result is most of the work, which the library does faster. Its time and the kernel's, us: 22016 x 4096 over
// 64, 256, 512, 1024 and 2048 tokens 63, 103, 126, 213, 404 and 112, 143, 176, 241, 373; 4096 x 4096 12, 18, 26, 40, 71 and 23, 27,
// 33, 45, 70. Over results of 9 to 131 million elements the kernel takes 1.5 times the library's at 100 tokens, 1.2 at 500, 1.06 from 1000 to
// 1500 (1.2 at 1536) and 1 at 1700 to 2000; below 2^23 elements it is ahead or, up to 10 us, bound by the host (see multiply).
static bool mostly_stores(const at::Tensor& dy, const at::Tensor& x) { return dy.size(0) < 1600 && dy.size(1) * x.size(1) > (1L << 23); }

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
  // a float32 result the library does not have
  if (!serves || (!add && !keep && mostly_stores(dy, x))) {
    at::Tensor r = at::mm(dy.t(), x);
    if (add) r = keep ? add->add_(r) : at::add(*add, r);
    return r.to(keep ? at::kFloat : dy.scalar_type());
  }
  return pr::run<true, true>(pr::loadable(dy) ? dy : dy.clone(at::MemoryFormat::Contiguous),
                             pr::loadable(x) ? x : x.clone(at::MemoryFormat::Contiguous), plan, add, keep);
}

// x [M, K] times w [N, K]^T, or with `slow` times w [K, N]. Products that should take at most 14 us by the plan are formed here, because the host
// takes 19 to 20 us for the library's call and 9 for this one, and a chain of such products waits for it. On the device they
// are no faster, 6 to 13 us where the library's kernels take 4 to 11. Where the line lies, us in a chain and from a graph, here and there: 512, 3072, 1152
// (whole; here) 12.9 and 13.7, 18.7 and 11.2; 512, 1024, 2048 (cut; there) 14.8 and 15.0, 18.9 and 9.6; 256, 3072, 1536 (there) 15.7 and 16.0, 19.0 and 9.4.
// Steps of two layers, us, library and here: width 512, 512 tokens 1320
// and 1050 (kernels 490 and 525); 1024, 512 tokens 1130 and 900; where the device is the bound nothing shows: 512, 4096 tokens 1316 and
// 1301, 1024, 2048 tokens 1343 and 1347.
static bool small_product(const at::Tensor& x, const at::Tensor& w, bool slow, pr::Plan& plan) {
  if (pr::bf16_pair(x, w) && x.size(1) == w.size(slow ? 0 : 1) && x.size(1) % pr::KT == 0 && w.size(slow ? 1 : 0) % 8 == 0
      && pr::loadable(x) && pr::loadable(w)) {
    const long M = x.size(0), N = w.size(slow ? 1 : 0), K = x.size(1);
    if (((M + 127) / 128) * ((N + 127) / 128) <= 256) {
      plan = pr::plan(M, N, K, true);
      return plan.us <= 14.0;
    }
  }
  return false;
}

at::Tensor multiply(const at::Tensor& x, const at::Tensor& w, bool slow) {
  pr::Plan plan;
  if (small_product(x, w, slow, plan)) return slow ? pr::run<false, true>(x, w, plan, c10::nullopt, false) : pr::run<false, false>(x, w, plan, c10::nullopt, false);
  return slow ? at::mm(x, w) : at::mm(x, w.t());
}

// Both gradients of a small linear layer, dy [K, M] times w [M, N] and dy^T x with x [K, N], by one launch; empty where one of them is not small. Neither
// fills the chip, and the host takes some 4 us for a launch, of which a step of two layers has eight less. A weight gradient of 128 x 128 tiles beside a small
// product takes at most 27 us by the plan, over all sizes. Kernels of both, us, one after the other and together, tokens, M, N: 512, 512, 512 18.5, 9.9;
// 3000, 512, 512 24.3, 17.4; 512, 1024, 2048 22.6, 13.9; 1500, 1024, 2048 30.9, 24.4; 2000, 1024, 2048 33.6, 28.4; 12000, 256, 256 32.9, 26.1; 16000, 128, 256 33.1, 29.1.
std::vector<at::Tensor> linear_grads(const at::Tensor& dy, const at::Tensor& w, const at::Tensor& x) {
  pr::Plan dx_plan;
  if (!small_product(dy, w, true, dx_plan) || !weight_grad_serves(dy, x) || !pr::loadable(x) || mostly_stores(dy, x)) return {};
  const pr::Plan dw_plan = pr::plan(dy.size(1), x.size(1), dy.size(0), false);
  if (dw_plan.tm != 128) return {};
  const c10::hip::HIPGuard guard(dy.device().index());
  const pr::Call dx = pr::call<false, true>(dy, w, dx_plan, c10::nullopt, false), dw = pr::call<true, true>(dy, x, dw_plan, c10::nullopt, false);
  const auto stream = at::hip::getCurrentHIPStream();
  constexpr int LDS = (128 + 128) * pr::KT * 2 * 4;
  pr::product_pair_kernel<<<dx.blocks() + dw.blocks(), 256, LDS, stream>>>(dx.a, dw.a, dx.blocks());
  if (dx.rest) pr::product_sum_kernel<128, 128><<<dx.rest * 16, 256, 0, stream>>>(dx.a);
  if (dw.rest) pr::product_sum_kernel<128, 128><<<dw.rest * 16, 256, 0, stream>>>(dw.a);
  HIP_CHECK_LAST();
  return {dx.out, dw.out};
}

}  // namespace cai
