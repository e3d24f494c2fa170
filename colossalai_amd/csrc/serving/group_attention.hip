// Attention of decode tokens on the matrix cores (bfloat16, head sizes 64 and 128): one block per (token, kv head, part of the
// token's keys) with the kv head's whole group of query heads, so that every cached row is read once.
//
// A wave takes a tile of 32 keys by itself: its keys and values come straight into LDS of its own (lds_tiles.h), no
// barrier until the end. As in the prompt portions' kernel the products are formed transposed,
//   S^T = K Q^T (A = key rows, B = query rows in registers: column = head), O^T = V^T P^T (the float32 weights in the C
//   layout they were born in, each as three bfloat16 pieces, which hold all of its 24 bits; A = values by transposing reads),
// so a head is a lane and its half-wave twin. Of the 32 columns the group fills 1 to 16; the products cost a tenth of the time that
// the tile's 16 KB take to arrive. Up to 10 heads stand three times in the columns, once for each piece of their weights: one
// product then does for three (16 x 1024 keys with a cap and a sink, 16 heads on 4 of 128: 17.5 us with three, 16.6 with one). The
// pieces' sums meet at the end; where the first one's is infinite it is the result, as the rests of a weight, 0 or negative, times infinity
// are not its part. The next tile's keys are on their way from the moment the scores are formed, its values from the end of the
// products.
// What bounds it: memory beyond about 8 us of dependent loads (position, page table, rows), launch and the end. The form with a
// row in the registers of a few lanes (row_attention.hip) and this one, us, replayed from a graph: 16 heads on 4 of 128: 16 x 1024 keys with a
// cap and a sink 15.6, 11.7, 4 x 16384 38.6, 28.1 (4.8 TB/s), 16 x 8192 56.2, 47.0 (5.7 TB/s); 8 on 2 of 128, 7 x 5000 20.2, 13.0; 16
// on 8 of 64, 16 x 3000 25.6, 23.0; one head a key head, 16 x 2000 45.7, 43.5; 16 on 1 of 128, 16 x 2000 21.0, 14.8.
// The eight waves' states meet in LDS at the end; few tokens have their keys cut into parts, whose states the block that ends last puts
// together (a launch for that took 4 to 6 us, and the host as long as the first one's). Which one that is needs no memory that somebody has cleared: a part
// leaves its states, then a mark that belongs to this launch alone, then looks at all marks of its token and key head. The last
// one to look finds them all; if two do, both write the same. What passes between the blocks goes around the L2 caches, which
// the XCDs do not share, word by word: fences at the scope of the device, which write back and empty these caches, took up to 100 us of a launch.
// 16 x 1024 keys with a cap and a sink 20.2 -> 16.0 us, 1 x 8192 16.6 -> 13.4, 4 x 16384 39.2 -> 36.5 (other keys and values in every
// call). Beside prompt portions the kernel may serve just the sequences that bring one token.
#include "paged_attention.h"
#include "../lds_tiles.h"

#include <algorithm>
#include <atomic>
#include <cmath>
#include <random>
#include <type_traits>

namespace cai {
namespace serving {

namespace {

constexpr int GROUP_WAVES = 8;
constexpr size_t GROUP_LDS = 160 * 1024;   // of a CU
constexpr int GROUP_HEADS = 16;     // most query heads of a kv head: their states must fit into a wave's tile
constexpr int PIECE_HEADS = 10;     // that stand three times in 32 columns
typedef __bf16 bf16x2_v __attribute__((ext_vector_type(2)));

DEV_INLINE float rounded_product(float a, float b) {
#pragma clang fp contract(off)
  return a * b;
}

__device__ __align__(16) const bf16s no_values[128] = {};   // a key's past the end

// A part's state, for a block on any XCD to read: every access is one of its own at the scope of the device, past the L2 caches.
DEV_INLINE void put_state(float* p, float v) { __hip_atomic_store(p, v, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT); }
DEV_INLINE float get_state(float* p) { return __hip_atomic_load(p, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT); }
// this wave's stores and atomics have been performed where every XCD sees them
DEV_INLINE void stores_done() { asm volatile("s_waitcnt vmcnt(0) lgkmcnt(0)" ::: "memory"); }
// floats of a part's states of a group of R heads, in cache lines of its own
__host__ __device__ constexpr long part_floats(int R, int Dv) { return (R * (2 + Dv) + 63L) / 64 * 64; }

template <int DS, int VT, bool COLS>
__global__ __launch_bounds__(64 * GROUP_WAVES, 2) void group_attention_kernel(
    bf16s* __restrict__ out, const bf16s* __restrict__ q, long q_stride, const bf16s* __restrict__ kpool,
    const bf16s* __restrict__ vpool, const int* __restrict__ block_tables, int bt_stride, const int* __restrict__ tok_seq,
    const int* __restrict__ positions, const float* __restrict__ slopes, const bf16s* __restrict__ gate, long gate_stride,
    const float* __restrict__ sink_logits, int H, int G, int page_shift, float scale, int window, int keep_first, int chunk,
    float softcap, int sink, int vrep, long vrow, long vhead, int splits, float* __restrict__ ws, const int* __restrict__ cu,
    unsigned long long* __restrict__ marks, unsigned long long mark, int seqs, int width) {
  constexpr int D = DS * 16, Dv = VT * 32, KQ = D / 32, KT = D * 64, VTT = Dv * 64;   // bytes of a tile's keys, values
  constexpr float LOG2E = 1.4426950408889634f;
  extern __shared__ __align__(16) char tiles[];   // [waves][KT + VTT], later the waves' states; then the pages
  int* pages = reinterpret_cast<int*>(tiles + GROUP_WAVES * (KT + VTT));
  const int wid = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), lane = threadIdx.x & 63;
  const int col = lane & 31, hf = lane >> 5;
  const int split = (int)(blockIdx.x % splits);
  const long unit = blockIdx.x / splits / G;   // a token, or with `cu` a sequence
  long n = unit;
  if (cu != nullptr) {
    if (cu[unit + 1] - cu[unit] != 1) return;
    n = cu[unit];
  }
  const int g = (int)(blockIdx.x / splits % G);
  const int R = H / G, h0 = g * R;
  // A page table of few pages (width > 0) is read whole, into registers, beside the token's position and sequence and not after them: on the guess that
  // token n is of sequence n, as in a step of decode tokens alone it is.
  const int guess = width > 0 ? block_tables[min(unit, seqs - 1L) * bt_stride + min((int)threadIdx.x, width - 1)] : 0;
  const int pos = positions[n], seq = tok_seq[n];
  const int* bt = block_tables + (long)seq * bt_stride;
  const int page_mask = (1 << page_shift) - 1;
  const int piece = COLS ? col / PIECE_HEADS : 0, hcol = col - piece * PIECE_HEADS;   // of the weights, head of the group
  const bool head = hcol < R;
  bf16x8_v qf[DS];
#pragma unroll
  for (int s = 0; s < DS; ++s) qf[s] = ld_g16b(q + n * q_stride + (long)(h0 + min(hcol, R - 1)) * D + 16 * s + hf * 8);
  const bool sloped = slopes != nullptr;
  float sl2 = sloped ? slopes[h0 + min(hcol, R - 1)] : 0.0f;

  // The token's keys: kept first ones, then those from `lo` to its own position
  const int lo = first_visible(pos, window, chunk);
  const int n_keep = window > 0 ? min(keep_first, lo) : 0;
  const int total = n_keep + (pos - lo + 1);
  const int all = (total + 31) >> 5, per = (all + splits - 1) / splits;
  const int last = min(all, (split + 1) * per);
  const int lkey = lane >> 2, lch = ((lane & 3) ^ (lane >> 4 & 3)) * 8;   // of a load: this lane's key of 16, channel of 32
  // Page numbers of this block's keys in LDS: looked up in memory tile by tile, they would stand between the keys' and
  // values' loads, and waiting for one would be waiting for all of these.
  const int i0 = split * per * 32, i1 = min(last * 32, total);      // the block's keys, counted from the first kept one
  const int w0 = i0 < n_keep ? lo : lo + (i0 - n_keep);             // the first one beyond the kept ones
  const int keep_pages = i0 < n_keep ? (n_keep + page_mask) >> page_shift : 0;
  const int num_pages = i0 < i1 ? keep_pages + ((lo + (i1 - 1 - n_keep)) >> page_shift) - (w0 >> page_shift) + 1 : 0;
  const int skip = width > 0 ? 0 : keep_pages - (w0 >> page_shift);   // from a page's number in the table to its place in LDS, beyond the kept ones
  if (width > 0) {
    if ((int)threadIdx.x < width) pages[threadIdx.x] = seq == unit ? guess : bt[threadIdx.x];
  } else {
    for (int i = threadIdx.x; i < num_pages; i += 64 * GROUP_WAVES) pages[i] = bt[i < keep_pages ? i : i - skip];
  }
  __syncthreads();
  struct Rows {
    int at[2];
    bool past[2];
  };
  auto lookup = [&](int t) {
    Rows r;
#pragma unroll
    for (int i = 0; i < 2; ++i) {
      const int key = t * 32 + i * 16 + lkey, idx = min(key, total - 1);   // past the end: the token's own row
      r.past[i] = key >= total;
      const int j = idx < n_keep ? idx : lo + (idx - n_keep);
      const int p = (j >> page_shift) + (idx < n_keep ? 0 : skip);
      r.at[i] = (pages[p] << page_shift) + (j & page_mask);
    }
    return r;
  };
  const char* kbase = reinterpret_cast<const char*>(kpool + (long)g * D + lch);
  const char* vbase = reinterpret_cast<const char*>(vpool + (long)(g / vrep) * vhead + lch);
  const char* none = reinterpret_cast<const char*>(no_values + lch);
  const unsigned krs = (unsigned)(G * D) * 2u, vrs = (unsigned)vrow * 2u;   // bytes between neighbouring keys' rows
  auto load_keys = [&](const Rows& r, char* __restrict__ dst) __attribute__((always_inline)) {
#pragma unroll
    for (int i = 0; i < 2; ++i)
#pragma unroll
      for (int c = 0; c < KQ; ++c)
        __builtin_amdgcn_global_load_lds((global_ptr)(kbase + (unsigned long)(unsigned)r.at[i] * krs + c * 64), (lds_ptr)(dst + (c * 2 + i) * 1024), 16, 0, 0);
  };
  auto load_values = [&](const Rows& r, char* __restrict__ dst) __attribute__((always_inline)) {
#pragma unroll
    for (int i = 0; i < 2; ++i) {
      const char* at = r.past[i] ? none : vbase + (unsigned long)(unsigned)r.at[i] * vrs;   // a weight of 0 times a value that may be infinite
#pragma unroll
      for (int c = 0; c < VT; ++c)
        __builtin_amdgcn_global_load_lds((global_ptr)(at + c * 64), (lds_ptr)(dst + (c * 2 + i) * 1024), 16, 0, 0);
    }
  };

  const int t0 = split * per + wid;
  int t = t0;
  Rows first;
  if (t < last) {
    first = lookup(t);
    load_keys(first, tiles + wid * (KT + VTT));
    load_values(first, tiles + wid * (KT + VTT) + KT);
  }
  sl2 *= LOG2E;
  if (scale < 0.0f) {   // exact: the largest product of a head is then its largest score
#pragma unroll
    for (int s = 0; s < DS; ++s) qf[s] = -qf[s];
    scale = -scale;
  }
  // Scores in the base-2 domain; the reference m is raised only where a tile's sum shows that it must be, as in the prompt
  // portions' kernel, and in the wave's first tile, which has a key that counts.
  const float c1 = scale * LOG2E < 1e-30f ? 1e-30f : scale * LOG2E;   // NaN stays
  const bool capped = softcap > 0.0f;
  const float inv_cap = capped ? scale / softcap : 0.0f, cap2 = softcap * LOG2E, t2 = capped ? 2.0f * LOG2E * scale / softcap : 0.0f;
  float m = -INFINITY, m_ref = -3.0e38f, l = 0.0f;
  f32x16 oacc[VT], orest[COLS ? 1 : VT];   // the first pieces' sums apart from the others', or with COLS a piece a column
#pragma unroll
  for (int t = 0; t < VT; ++t)
#pragma unroll
    for (int i = 0; i < 16; ++i) {
      oacc[t][i] = 0.0f;
      if (!COLS) orest[t][i] = 0.0f;
    }
  const float sel[2] = {piece >= 1 ? -1.0f : 0.0f, piece >= 2 ? -1.0f : 0.0f};
  const RowAt row_at(col, hf);
  const ColAt col_at(lane);
  char* keys = tiles + wid * (KT + VTT);

  auto tile = [&](int t, auto more, const Rows& next, char* __restrict__ K_, char* __restrict__ V_) __attribute__((always_inline)) {
    f32x16 x;
#pragma unroll
    for (int i = 0; i < 16; ++i) x[i] = 0.0f;
    constexpr int AHEAD = 4;
    bf16x8_v kf[DS];
#pragma unroll
    for (int s = 0; s < AHEAD; ++s) kf[s] = frag_row<32>(K_, row_at, 0, s);
#pragma unroll
    for (int s = 0; s < DS; ++s) {
      if (s + AHEAD < DS) kf[s + AHEAD] = frag_row<32>(K_, row_at, 0, s + AHEAD);
      x = __builtin_amdgcn_mfma_f32_32x32x16_bf16(kf[s], qf[s], x, 0, 0, 0);
    }
    __builtin_amdgcn_sched_barrier(0);
    if (more) load_keys(next, K_);   // the key fragments are in registers
    if (capped) {
      float far = 0.0f;
#pragma unroll
      for (int i = 0; i < 16; ++i) far = fmaxf(far, fabsf(x[i]));
      // tanh(y) = y P(y^2) for |y| <= 1/2, P a polynomial through the Chebyshev nodes (1.3e-8 off); beyond, the exponential
      // form, for the scores that are large themselves
      if (__all(far * inv_cap <= 0.5f)) {
#pragma unroll
        for (int i = 0; i < 16; ++i) {
          const float y = x[i] * inv_cap, z = y * y;
          x[i] = cap2 * y * fmaf(z, fmaf(z, fmaf(z, fmaf(z, 0.017131345f, -0.052984238f), 0.13324751f), -0.33333069f), 1.0f);
        }
        asm volatile("" ::: "memory");
      } else {
#pragma unroll
        for (int i = 0; i < 16; ++i) {
          const float y = x[i] * inv_cap, z = y * y;
          const float small = cap2 * y * fmaf(z, fmaf(z, fmaf(z, fmaf(z, 0.017131345f, -0.052984238f), 0.13324751f), -0.33333069f), 1.0f);
          const float large = cap2 - 2.0f * cap2 * __builtin_amdgcn_rcpf(__builtin_amdgcn_exp2f(fabsf(x[i]) * t2) + 1.0f);
          x[i] = fabsf(y) <= 0.5f ? small : copysignf(large, y);
        }
      }
    }
    // rounded once for the weights and the largest of them: fused into the difference below, a score of 4e9 would miss itself by 2^8
    if (!capped) {
#pragma unroll
      for (int i = 0; i < 16; ++i) x[i] = rounded_product(x[i], c1);
    }
    if (sloped) {
#pragma unroll
      for (int i = 0; i < 16; ++i) {
        const int idx = t * 32 + (i & 3) + 8 * (i >> 2) + 4 * hf;
        const int j = idx < n_keep ? idx : lo + (idx - n_keep);
        x[i] = x[i] - sl2 * (float)(pos - j);
      }
    }
    if (t * 32 + 32 > total) {
#pragma unroll
      for (int i = 0; i < 16; ++i) x[i] = t * 32 + (i & 3) + 8 * (i >> 2) + 4 * hf < total ? x[i] : -INFINITY;
    }
    bf16x8_v pw[COLS ? 1 : 3][2];
    float psum;
    for (bool raised = false;; raised = true) {
      psum = 0.0f;
#pragma unroll
      for (int i = 0; i < 16; i += 2) {
        const float p0 = __builtin_amdgcn_exp2f(x[i] - m_ref), p1 = __builtin_amdgcn_exp2f(x[i + 1] - m_ref);
        psum += p0 + p1;
        float2v rest = {p0, p1};
#pragma unroll
        for (int k = 0; k < 3; ++k) {   // one conversion packs two pieces; what it leaves is exact
          const bf16x2_v two = __builtin_convertvector(rest, bf16x2_v);
          const unsigned bits = __builtin_bit_cast(unsigned, two);
          if (!COLS || k == 2) {
            pw[COLS ? 0 : k][i >> 3][i & 7] = two[0];
            pw[COLS ? 0 : k][i >> 3][(i & 7) + 1] = two[1];
          }
          if (k < 2) {
            rest[0] = fmaf(__builtin_bit_cast(float, bits << 16), COLS ? sel[k] : -1.0f, rest[0]);
            rest[1] = fmaf(__builtin_bit_cast(float, bits & 0xffff0000u), COLS ? sel[k] : -1.0f, rest[1]);
          }
        }
      }
      if (raised || (t != t0 && __all(!head || psum <= 4096.0f))) break;
      float top = x[0];
#pragma unroll
      for (int i = 1; i < 16; ++i) top = fmaxf(top, x[i]);
      top = fmaxf(top, __shfl_xor(top, 32));
      const float m_new = fmaxf(m, top);
      const float corr = m == -INFINITY ? 1.0f : __builtin_amdgcn_exp2f(m - m_new);   // nothing accumulated: nothing to rescale
      l *= corr;
#pragma unroll
      for (int c = 0; c < VT; ++c)
#pragma unroll
        for (int i = 0; i < 16; ++i) {
          oacc[c][i] *= corr;
          if (!COLS) orest[c][i] *= corr;
        }
      m = m_new;
      m_ref = m_new == -INFINITY ? -3.0e38f : m_new;
    }
    l += psum;
    if (more) loads_left<2 * KQ>();   // younger than this tile's values: the next keys
    else loads_left<0>();
#pragma unroll
    for (int s2 = 0; s2 < 2; ++s2)
#pragma unroll
      for (int c = 0; c < VT; ++c) {
        const bf16x8_v va = frag_born<32>(V_, col_at, 16 * s2, 32 * c);
        oacc[c] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(va, pw[0][s2], oacc[c], 0, 0, 0);
        if constexpr (!COLS) {
          orest[c] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(va, pw[1][s2], orest[c], 0, 0, 0);
          orest[c] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(va, pw[2][s2], orest[c], 0, 0, 0);
        }
      }
    __builtin_amdgcn_sched_barrier(0);
    if (more) load_values(next, V_);
  };

  if (t < last) {
    for (; t + GROUP_WAVES < last; t += GROUP_WAVES) {
      const Rows next = lookup(t + GROUP_WAVES);
      loads_left<2 * VT>();          // younger than this tile's keys: its values
      tile(t, std::true_type(), next, keys, keys + KT);
    }
    loads_left<2 * VT>();
    tile(t, std::false_type(), first, keys, keys + KT);
  }
  // The waves' states: [head][2 + Dv] in the wave's own tiles, with COLS [piece][head][2 + Dv]
  constexpr int PS = 2 + Dv;
  auto whole = [](float first, float rest) { return fabsf(first) < INFINITY ? first + rest : first; };
  l += __shfl_xor(l, 32);
  float* mine = reinterpret_cast<float*>(keys) + (piece * R + hcol) * PS;
  if (head && piece < 3) {
    if (hf == 0) {
      mine[0] = m;
      mine[1] = l;
    }
#pragma unroll
    for (int c = 0; c < VT; ++c)
#pragma unroll
      for (int i = 0; i < 16; ++i) mine[2 + c * 32 + (i & 3) + 8 * (i >> 2) + 4 * hf] = COLS ? oacc[c][i] : whole(oacc[c][i], orest[c][i]);
  }
  __syncthreads();
  constexpr int WS = (KT + VTT) / 4;   // floats between the waves' states
  const float* states = reinterpret_cast<const float*>(tiles);
  for (int i = threadIdx.x; i < R * Dv; i += 64 * GROUP_WAVES) {
    const int r = i / Dv, dv = i % Dv;
    float top = -INFINITY;
#pragma unroll
    for (int w = 0; w < GROUP_WAVES; ++w) top = fmaxf(top, states[w * WS + r * PS]);
    if (splits == 1 && sink_logits != nullptr) top = fmaxf(top, sink_logits[h0 + r] * LOG2E);
    float ll = 0.0f, o = 0.0f;
#pragma unroll
    for (int w = 0; w < GROUP_WAVES; ++w) {
      const float mw = states[w * WS + r * PS];
      const float f = mw == -INFINITY ? 0.0f : __builtin_amdgcn_exp2f(mw - top);
      ll += states[w * WS + r * PS + 1] * f;     // a wave without keys: 0 * 0
      const float* sums = states + w * WS + r * PS + 2 + dv;
      o += (COLS ? whole(sums[0], sums[R * PS] + sums[2 * R * PS]) : sums[0]) * f;
    }
    if (splits > 1) {   // a part without keys has a maximum of -inf
      float* state = ws + ((unit * G + g) * splits + split) * part_floats(R, Dv) + r * PS;
      put_state(state + 2 + dv, o);
      if (dv == 0) {
        put_state(state, top);
        put_state(state + 1, ll);
      }
    } else {
      if (sink_logits != nullptr) ll += __builtin_amdgcn_exp2f(sink_logits[h0 + r] * LOG2E - top);
      else if (sink) ll += __builtin_amdgcn_exp2f(-top);   // the sink's score is 0
      float c = 1.0f / ll;
      if (gate != nullptr) c *= sigmoidf_(ldf(gate + n * gate_stride + h0 + r));
      stf(out + (n * H + h0 + r) * (long)Dv + dv, o * c);
    }
  }
  if (splits == 1) return;

  // The part that finds all marks of its token and kv head set puts the states together.
  int* all_there = pages;   // the page numbers are done with
  stores_done();
  __syncthreads();
  marks += (unit * G + g) * splits;
  if (wid == 0) {
    if (lane == split) (void)__hip_atomic_exchange(marks + lane, mark, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    stores_done();                   // own mark first: of two parts that look at the same time one sees the other's
    unsigned long long none = 0;
    asm volatile("" : "+v"(none));   // an addition to where the marks are ordered, not a load
    const int there = __all(lane >= splits || __hip_atomic_fetch_add(marks + lane, none, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) == mark);
    if (lane == 0) *all_there = there;
  }
  __syncthreads();
  if (!*all_there) return;
  float* coef = reinterpret_cast<float*>(tiles);   // [R][WAVE]
  const long step = part_floats(R, Dv);
  float* parts = ws + (unit * G + g) * splits * step;
  constexpr int AHEAD = 8;
  float v[AHEAD];
  auto fetch = [&](int i, int p0) {
    float* sums = parts + i / Dv * PS + 2 + i % Dv;
#pragma unroll
    for (int e = 0; e < AHEAD; ++e) v[e] = get_state(sums + min(p0 + e, splits - 1) * step);
  };
  if ((int)threadIdx.x < R * Dv) fetch(threadIdx.x, 0);
  for (int r = wid; r < R; r += GROUP_WAVES) {
    float* state = parts + min(lane, splits - 1) * step + r * PS;
    const float m_at = get_state(state), l_at = get_state(state + 1);
    const float mp = lane < splits ? m_at : -INFINITY, lp = lane < splits ? l_at : 0.0f;
    float top = wave_reduce_max(mp);
    if (sink_logits != nullptr) top = fmaxf(top, sink_logits[h0 + r] * LOG2E);
    const float f = mp == -INFINITY ? 0.0f : __builtin_amdgcn_exp2f(mp - top);
    float ll = wave_reduce_sum(lp * f);
    if (sink_logits != nullptr) ll += __builtin_amdgcn_exp2f(sink_logits[h0 + r] * LOG2E - top);
    else if (sink) ll += __builtin_amdgcn_exp2f(-top);   // the sink's score is 0
    float c = f / ll;
    if (gate != nullptr) c *= sigmoidf_(ldf(gate + n * gate_stride + h0 + r));
    coef[r * WAVE + lane] = c;
  }
  __syncthreads();
  for (int i = threadIdx.x; i < R * Dv; i += 64 * GROUP_WAVES) {
    const float* c = coef + i / Dv * WAVE;
    float o = 0.0f;
    for (int p0 = 0; p0 < splits; p0 += AHEAD) {
      if (i != (int)threadIdx.x || p0 > 0) fetch(i, p0);
#pragma unroll
      for (int e = 0; e < AHEAD; ++e)
        if (p0 + e < splits) o += c[p0 + e] * v[e];
    }
    stf(out + (n * H + h0 + i / Dv) * (long)Dv + i % Dv, o);
  }
  // a launch that a graph repeats has the same mark each time (whoever looks now finds too little, and is not needed)
  if (wid == 0 && lane < splits) __hip_atomic_store(marks + lane, 0ull, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}

// A number that no launch of this process had before and that memory does not hold by chance.
unsigned long long new_mark() {
  static const unsigned long long seed = [] {
    std::random_device r;
    return (unsigned long long)r() << 32 | r();
  }();
  static std::atomic<unsigned long long> count{0};
  unsigned long long z = seed + ++count * 0x9e3779b97f4a7c15ull;   // splitmix64, one to one
  z = (z ^ z >> 30) * 0xbf58476d1ce4e5b9ull;
  z = (z ^ z >> 27) * 0x94d049bb133111ebull;
  return z ^ z >> 31;
}

}  // namespace

bool launch_group_attention(at::Tensor& out, const at::Tensor& q, const at::Tensor& kpool, const at::Tensor& vpool,
                            const at::Tensor& block_tables, const at::Tensor& tok_seq, const at::Tensor& positions,
                            const float* slopes, const c10::optional<at::Tensor>& gate, long gate_stride, double scale,
                            int64_t window, int64_t keep_first, double softcap, bool sink, int page_shift, long vrow,
                            long vhead, const ScalarExtras& x, const SingleTokens& only) {
  const bool some = only.cu != nullptr;
  const long N = some ? only.count : q.size(0), units = some ? only.seqs : N;   // tokens, and what takes their place
  const int H = (int)q.size(1), D = (int)q.size(2), G = (int)kpool.size(2), Dv = (int)vpool.size(3), R = H / G;
  if (!is_bf16(q) || x.dist_bias != nullptr || x.ksum != nullptr || x.cross_out != nullptr || x.key_fac != nullptr ||
      x.out32 != nullptr || (D != 64 && D != 128) || (Dv != 64 && Dv != 128) || R > GROUP_HEADS)
    return false;
  auto al16 = [](const at::Tensor& t) { return reinterpret_cast<uintptr_t>(t.data_ptr()) % 16 == 0; };
  if (!al16(q) || !al16(kpool) || !al16(vpool) || q.stride(0) % 8 != 0 || vrow % 8 != 0 || vrow >= (1L << 30) ||
      vhead % 8 != 0)
    return false;
  long keys = block_tables.size(1) << page_shift;           // most that a token can see
  if (window > 0) keys = std::min<long>(keys, window + keep_first);
  if (x.chunk > 0) keys = std::min<long>(keys, x.chunk);
  // Values that are the keys stay in the other form, which reads each row once.
  if (vpool.data_ptr() == kpool.data_ptr()) return false;
  const long blocks = N * G;
  // Up to a tile a wave: few tokens with many heads a key head go to the other form, whose end is shorter (that form and this, us: 8 x 200 keys,
  // 8 heads on 1 of 128: 7.1, 7.8; 16 on 1 7.3, 8.9; but 48 x 200 14.1, 9.0; 16 on 4, 1 x 200 7.1, 6.6, 128 x 200 43.0, 20.8; 64 channels 8 x 200
  // 7.2, 5.0), and so do tokens beside prompt portions, which then ride with these.
  if (keys <= 32 * GROUP_WAVES && (some || (D + Dv > 128 && R > 4 && blocks < 48))) return false;
  // every piece's sums of a head must fit into a wave's tile as well
  const bool cols = R <= PIECE_HEADS && 3 * R * (2 + Dv) * 4 <= (D + Dv) * 64;
  // Little work goes to the other form too, where a wave's own chain is longer here than the row's: with three products a tile (16 heads on 1
  // of 128, that form and this: 1 x 512 11.7, 13.2, 4 x 2048 16.4, 17.5, 16 x 600 12.3, 14.4, but 16 x 1300 17.9, 17.5, 1 x 8192 26.5,
  // 18.9 us), and over 257 to 512 keys with a distance penalty (4 x 300, 16 heads on 4 of 128: 9.1, 9.4; 16 x 400 11.0, 12.0; 64 x 512: 32, 17.5).
  if (keys > 32 * GROUP_WAVES) {
    if (!cols && blocks < 32 && keys < 8192 && blocks * keys < 20000) return false;
    if (slopes != nullptr && blocks <= 64 && keys <= 512) return false;
  }
  // Parts of the keys while there are fewer blocks than CUs. A tile of 32 keys takes a wave 1.75 us at 128 channels, and eight waves run
  // side by side; parts cost 2.4 us (64 channels) to 3.6 for a store and three round trips to memory, and each of them
  // 0.08 and more for the reading of its states, which one block does for all heads of the group, eight parts at a time. Whole and in
  // parts, other keys and values in every call, us: 16 heads on 4 of 128, 16 x 1000 14.5, 2: 13.8, 4: 13.4; 4 x 600 8.6, 2: 9.9, 8: 9.2; 1 x 2000 18.3,
  // 4: 11.0, 8: 10.5, 16: 9.8; 1 x 8000 64, 8: 16.9, 24: 13.2, 64: 16.0; 4 x 16000 223, 8: 40.9, 16: 33.2; 16 on 1 of 128, 16 x 2000 23.7, 4: 17.2, 8: 15.9,
  // 12: 18.0; 8 x 16000 132, 8: 31.0, 16: 26.1, 24: 27.9, 32: 29.8; 8 on 8 of 128, 16 x 800 13.9, 2: 16.6; 8 on 4 of 64, 8 x 1000 9.4, 4: 8.7,
  // 8: 8.2. Over 1219 such sizes the rule's choice takes 0.6 % more than the best one on average.
  const double whole = (double)((keys + 31) / 32) * 0.22 * (D + Dv) / 256, each = std::max(0.08, 0.02 * R * Dv / 128);
  const long most = std::max<long>(1, std::min<long>(256 / blocks, WAVE));
  long parts = std::min(most, std::lround(std::sqrt(whole / each)));
  if (parts >= 6) parts = std::min(most, (parts + 4) / 8 * 8);
  if (parts > 8) parts = parts / 8 * 8;
  const int splits = parts < 2 || whole <= whole / parts + 1.2 + 2.4 * (D + Dv) / 256 + each * parts ? 1 : (int)parts;
  // page numbers of a part: of its keys, rounded up to whole tiles, of a page more for where they begin, and of the kept ones
  const long part_keys = ((keys + 31) / 32 + splits - 1) / splits * 32;
  const long table = block_tables.size(1);
  const int width = table <= 64 * GROUP_WAVES ? (int)table : 0;   // a page a thread
  const size_t lds = (size_t)GROUP_WAVES * (D + Dv) * 64 +
                     (size_t)(width > 0 ? width : (part_keys >> page_shift) + (keep_first >> page_shift) + 4) * sizeof(int);
  if (lds > GROUP_LDS) return false;
  at::Tensor ws;
  unsigned long long* marks = nullptr;
  if (splits > 1) {   // states, then marks
    const long states = units * G * splits * part_floats(R, Dv);
    ws = at::empty({states + units * G * splits * 2}, q.options().dtype(at::kFloat));
    marks = reinterpret_cast<unsigned long long*>(ws.data_ptr<float>() + states);
  }
#define GROUP_LAUNCH(DS_, VT_)                                                                                       \
  do {                                                                                                             \
    auto kernel = cols ? group_attention_kernel<DS_, VT_, true> : group_attention_kernel<DS_, VT_, false>;          \
    if (lds > 65536) (void)hipFuncSetAttribute((const void*)kernel, hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds); \
    hipLaunchKernelGGL(kernel, dim3((unsigned)(units * G * splits)), dim3(64 * GROUP_WAVES), lds, stream(), ptr<bf16s>(out), \
                       ptr<bf16s>(q), (long)q.stride(0), ptr<bf16s>(kpool), ptr<bf16s>(vpool), block_tables.data_ptr<int>(), \
                       (int)block_tables.stride(0), tok_seq.data_ptr<int>(), positions.data_ptr<int>(), slopes,    \
                       gate.has_value() ? ptr<bf16s>(*gate) : (const bf16s*)nullptr, gate_stride, x.sink_logits, H, G, page_shift, \
                       (float)scale, (int)window, (int)keep_first, x.chunk, (float)softcap, sink ? 1 : 0, x.vrep, vrow, vhead, \
                       splits, splits > 1 ? ws.data_ptr<float>() : (float*)nullptr, only.cu, marks, splits > 1 ? new_mark() : 0ull, \
                       (int)block_tables.size(0), width);                            \
  } while (0)
  if (D == 128) { if (Dv == 128) GROUP_LAUNCH(8, 4); else GROUP_LAUNCH(8, 2); }
  else { if (Dv == 128) GROUP_LAUNCH(4, 4); else GROUP_LAUNCH(4, 2); }
#undef GROUP_LAUNCH
  HIP_CHECK_LAST();
  return true;
}

}  // namespace serving
}  // namespace cai
