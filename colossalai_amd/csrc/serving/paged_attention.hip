// Attention of a ragged batch over paged keys/values with a sliding window,
// kept first tokens, a linear distance penalty, a per-head output gate, a tanh
// soft cap on the scaled score and an optional sink (one more place of score 0
// in the softmax denominator that carries no value; with sink logits its score is learned per
// head), an additive per-distance table, block summaries (one mean key/value per block of
// positions that lies wholly before the window, kept in a small pool of their own), for
// talking heads every query head's weights applied to every key/value head's values, visibility
// inside fixed blocks of positions instead of a window, a float32 factor per cached key (keys that
// are normed when they are read), value heads shared by several key heads, and float32 output.
//
// One wave per (token, query head). The visible keys of a token are two
// position ranges: the kept prefix [0, min(keep_first, lo)) and the window
// [lo, pos] with lo = max(0, pos - window + 1) (lo = 0 without a window); the
// wave walks their concatenation 64 keys at a time. Phase 1: lane = key, each
// lane takes the full dot product of its key with the query (query in LDS,
// key row read with its own page lookup). Online softmax in float32 across
// the 64-key blocks. Phase 2: lane = value channel, the block's weights and
// pool rows are broadcast from LDS. A prompt portion and a decode token can run
// the same code. The other forms sum the same float32 terms in an order that depends on the call as well
// (decode: on the number of tokens and the width of the page table, which choose heads a block and parts
// of the keys), so that a position's results agree to rounding and not bit for bit.
// Calls without a distance table, block summaries or cross values run the form in row_attention.hip
// where the row sizes fit it; bfloat16 prompt portions run the matrix-core kernel.
#include <algorithm>
#include <type_traits>

#include "../lds_tiles.h"
#include "paged_attention.h"

namespace cai {
namespace serving {

constexpr int ATT_WAVES = 16;  // most waves of a block: they split the key blocks of one (token, kv head)
constexpr int RC_MAX = 4;      // most query heads of a kv head's group that one block handles together
typedef __bf16 bf16x2_v __attribute__((ext_vector_type(2)));

constexpr int MFMA_TILES_PER_STEP = 2;  // 32-key tiles the matrix-core kernel stages and multiplies between two barriers

// sum over the 8 adjacent lanes that share a key (quad xor 1, quad xor 2, half-row mirror)
DEV_INLINE float reduce8(float v) { return dpp_add<0x141>(dpp_add<0x4E>(dpp_add<0xB1>(v))); }

// Scalar kernel (decode tokens, float32 serving, shapes the MFMA kernel does not take).
// One block per (token, kv head, group of up to RC query heads of that kv head): keys and
// values are read once for the whole group. The block's nw waves (16, or 8 when the partial
// states of 16 would not fit in LDS) take every nw-th block of 64 keys and merge their partial
// softmax states through LDS at the end. The eight key steps of a block are unrolled so that
// their page lookups and key loads are all in flight before the first product.
// Scores: 8 adjacent lanes share a key, each takes a contiguous slice of the head size
// (16-byte loads, few cache lines per instruction) and the slices are summed on the DPP path.
// Values: lane = a pair of value channels, the block's weights and pool rows come from LDS.
// RC = query heads per block: 4 shares each key/value read between the most heads; 2 or 1 are
// chosen when a decode step would otherwise leave most CUs without a block (the re-reads hit L2).
// V8 (value head sizes that are multiples of 8 up to 512): a lane takes 8 consecutive value channels of a key with
// one 16/32-byte load, vl = Dv / 8 rounded up to a power of two lanes cover a key's row and the 64 / vl lane groups
// take different keys of the block, so a block of 64 keys is read by vl load instructions instead of 64; the groups' sums meet in a butterfly of
// shuffles after the last block.
template <typename T, int RC, bool V8>
__global__ __launch_bounds__(64 * ATT_WAVES) void paged_attention_kernel(
    T* __restrict__ out, const T* __restrict__ q, long q_stride, const T* __restrict__ kpool,
    const T* __restrict__ vpool, const int* __restrict__ block_tables, int bt_stride, const int* __restrict__ tok_seq,
    const int* __restrict__ positions, const float* __restrict__ slopes, const T* __restrict__ gate, long gate_stride,
    int H, int G, int D, int Dv, int page_shift, float scale, int window, int keep_first, int kvec, int vvec,
    float softcap, int sink, long vrow, long vhead, const float* __restrict__ sink_logits,
    const float* __restrict__ dist_bias, int dist_rows, const T* __restrict__ ksum, const T* __restrict__ vsum,
    int sum_shift, int sum_block, float* __restrict__ cross_out, int chunk, const float* __restrict__ key_fac, int vrep,
    float* __restrict__ out32) {
  // sink_logits [H]: the sink's score per head instead of 0. dist_bias [dist_rows, H]: added to the score of a key at
  // distance d (row min(d, dist_rows - 1)). ksum / vsum: block summaries, rows [pages << sum_shift]; a query at
  // `pos` sees the first max(0, (pos - window + 1) / sum_block) of its sequence's, ahead of its other keys and
  // without distance terms. cross_out [N, H, G, Dv] float32: the grid then has G blocks per (token, kv head, chunk),
  // block c applies the heads' weights to the values of kv head c. chunk > 0: a query sees its own block of `chunk`
  // positions only (counted from position 0). key_fac [pool rows, G]: the cached key's score is multiplied by it. vrep:
  // key heads per value head (the value pool has G / vrep heads). out32 [N, H, Dv]: float32 output instead of `out`.
  // vrow / vhead: elements between the value rows of neighbouring pool rows / kv heads (G * Dv and Dv for a
  // pool of its own; a value pool that is a view into wider rows, e.g. the leading channels of the keys, has others)
  extern __shared__ __align__(16) float lds[];
  const int wid = threadIdx.x >> 6, lane = threadIdx.x & 63, nw = blockDim.x >> 6;
  const int Dp = (D + 7) & ~7;
  const int R = H / G, chunks = (R + RC - 1) / RC;
  float* qs = lds;                                        // [RC][Dp] queries
  float* pw = lds + RC * Dp + wid * (RC * 64 + 64);       // [RC][64] scores, then weights, of this wave's key block
  int* prow = reinterpret_cast<int*>(pw + RC * 64);       // [64] pool rows of the block
  float* part = lds + RC * Dp + nw * (RC * 64 + 64);      // [waves][RC][2 + Dv] partial states
  const int VC = cross_out != nullptr ? G : 1;
  const long bx = blockIdx.x / VC;
  const long n = bx / (G * chunks);
  const int g = (int)(bx / chunks) % G;
  const int vg = cross_out != nullptr ? (int)(blockIdx.x % VC) : g / vrep;  // kv head whose values this block reads
  const int h0 = g * R + (int)(bx % chunks) * RC;  // first query head of this block
  const int nh = min(RC, g * R + R - h0);
  const int b = tok_seq[n];
  const int pos = positions[n];
  const int* bt = block_tables + (long)b * bt_stride;
  const int page_mask = (1 << page_shift) - 1;

  for (int i = threadIdx.x; i < RC * Dp; i += blockDim.x) {
    const int r = i / Dp, d = i % Dp;
    qs[i] = (r < nh && d < D) ? ldf(q + n * q_stride + (long)(h0 + r) * D + d) : 0.0f;
  }
  __syncthreads();
  float slope[RC];
#pragma unroll
  for (int r = 0; r < RC; ++r) slope[r] = (slopes != nullptr && r < nh) ? slopes[h0 + r] : 0.0f;

  const int lo = first_visible(pos, window, chunk);
  const int n_sum = (ksum != nullptr && window > 0) ? max(0, (pos - window + 1) / sum_block) : 0;
  const int sum_mask = (1 << sum_shift) - 1;
  const int n_keep = (window > 0 ? min(keep_first, lo) : 0) + n_sum;  // summaries, then kept first tokens
  const int total = n_keep + (pos - lo + 1);
  const float inv_cap = softcap > 0.0f ? 1.0f / softcap : 0.0f;
  const int part8 = lane & 7, ksub = lane >> 3;
  const int DS = (((D + 7) >> 3) + 7) & ~7;  // slice of the head size per lane, a multiple of 8
  const int d_lo = part8 * DS, d_hi = min(D, d_lo + DS);

  constexpr int NA = V8 ? 8 : 4;  // value channels a lane accumulates
  float m[RC], l[RC], acc[RC][NA];
#pragma unroll
  for (int r = 0; r < RC; ++r) {
    m[r] = -INFINITY;
    l[r] = 0.0f;
#pragma unroll
    for (int i = 0; i < NA; ++i) acc[r][i] = 0.0f;
  }
  int vl = 1;                                 // V8: lanes per key row: the power of two that holds Dv / 8 ...
  while (vl * 8 < Dv) vl <<= 1;               // (lanes of a row beyond Dv / 8 idle when Dv / 8 is no power of two)
  const int vks = V8 ? 64 / vl : 1;           // ... keys per load instruction ...
  const int vsub = V8 ? lane / vl : 0;        // ... this lane's key group ...
  const int vch = V8 ? (lane % vl) * 8 : 0;   // ... and its first value channel
  const bool vlive = vch < Dv;

  for (int base = wid * 64; base < total; base += 64 * nw) {
    const int cnt = min(64, total - base);
    auto score_step = [&](int sub) {
      const int idx = base + sub * 8 + ksub;
      const bool valid = idx < total;
      const bool summary = valid && idx < n_sum;
      const int j = valid ? (idx < n_keep ? idx - n_sum : lo + (idx - n_keep)) : pos;
      const int row = summary ? (bt[idx >> sum_shift] << sum_shift) + (idx & sum_mask)
                              : (bt[j >> page_shift] << page_shift) + (j & page_mask);
      float dots[RC];
#pragma unroll
      for (int r = 0; r < RC; ++r) dots[r] = 0.0f;
      const T* kr = (summary ? ksum : kpool) + ((long)row * G + g) * D;
      if (kvec) {
        for (int d = d_lo; d < d_hi; d += 8) {
          float kv[8];
          load8(kr + d, kv);
#pragma unroll
          for (int r = 0; r < RC; ++r) {
            const float4v qa = *reinterpret_cast<const float4v*>(qs + r * Dp + d);
            const float4v qb = *reinterpret_cast<const float4v*>(qs + r * Dp + d + 4);
            dots[r] += kv[0] * qa[0] + kv[1] * qa[1] + kv[2] * qa[2] + kv[3] * qa[3] + kv[4] * qb[0] + kv[5] * qb[1] +
                       kv[6] * qb[2] + kv[7] * qb[3];
          }
        }
      } else {
        for (int d = d_lo; d < d_hi; ++d) {
          const float kv = ldf(kr + d);
#pragma unroll
          for (int r = 0; r < RC; ++r) dots[r] += kv * qs[r * Dp + d];
        }
      }
#pragma unroll
      for (int r = 0; r < RC; ++r) dots[r] = reduce8(dots[r]);
      if (part8 == 0) {
#pragma unroll
        for (int r = 0; r < RC; ++r) {
          float sc = dots[r] * scale;
          if (key_fac != nullptr && !summary) sc *= key_fac[(long)row * G + g];
          if (softcap > 0.0f) sc = softcap * tanhf(sc * inv_cap);
          if (!summary) {
            sc -= slope[r] * (float)(pos - j);
            if (dist_bias != nullptr && r < nh) sc += dist_bias[(long)min(pos - j, dist_rows - 1) * H + h0 + r];
          }
          pw[r * 64 + sub * 8 + ksub] = valid ? sc : -INFINITY;
        }
        prow[sub * 8 + ksub] = summary ? -1 - row : row;  // a summary row is marked by its sign
      }
    };
    if (cnt == 64) {  // straight-line: all eight steps' lookups and key loads issue before the first product
#pragma unroll
      for (int sub = 0; sub < 8; ++sub) score_step(sub);
    } else {          // the last block of a key range: only the steps that hold keys
      for (int sub = 0; sub * 8 < cnt; ++sub) score_step(sub);
    }
    // the wave is its own producer and consumer of pw/prow: wait for its LDS writes
    __builtin_amdgcn_s_waitcnt(0xc07f);  // lgkmcnt(0)
    float corr[RC];
#pragma unroll
    for (int r = 0; r < RC; ++r) {
      const float s = lane < cnt ? pw[r * 64 + lane] : -INFINITY;
      const float m_new = fmaxf(m[r], wave_reduce_max(s));  // a block holds at least one visible key
      const float w = expf(s - m_new);                      // exp(-inf) = 0 for the block's empty places
      corr[r] = expf(m[r] - m_new);                         // m = -inf before the first block: 0
      l[r] = l[r] * corr[r] + wave_reduce_sum(w);
      m[r] = m_new;
      pw[r * 64 + lane] = w;
    }
    __builtin_amdgcn_s_waitcnt(0xc07f);
#pragma unroll
    for (int r = 0; r < RC; ++r)
#pragma unroll
      for (int i = 0; i < NA; ++i) acc[r][i] *= corr[r];
    if constexpr (V8) {
#pragma unroll 4
      for (int jj = vsub; jj < cnt; jj += vks) {
        float v[8];
        if (vlive) {
          const int pr = prow[jj];
          load8((pr < 0 ? vsum : vpool) + (long)(pr < 0 ? -1 - pr : pr) * vrow + (long)vg * vhead + vch, v);
        } else {
#pragma unroll
          for (int e = 0; e < 8; ++e) v[e] = 0.0f;
        }
#pragma unroll
        for (int r = 0; r < RC; ++r) {
          const float w = pw[r * 64 + jj];
#pragma unroll
          for (int e = 0; e < 8; ++e) acc[r][e] += w * v[e];
        }
      }
    } else {
    const int dva = 2 * lane, dvb = 128 + 2 * lane;
#pragma unroll 8
    for (int jj = 0; jj < cnt; ++jj) {
      const int pr = prow[jj];
      const T* vr = (pr < 0 ? vsum : vpool) + (long)(pr < 0 ? -1 - pr : pr) * vrow + (long)vg * vhead;
      float v0 = 0.0f, v1 = 0.0f, v2 = 0.0f, v3 = 0.0f;
      if (vvec) {
        if (dva < Dv) load2(vr + dva, v0, v1);
        if (dvb < Dv) load2(vr + dvb, v2, v3);
      } else {
        if (dva < Dv) v0 = ldf(vr + dva);
        if (dva + 1 < Dv) v1 = ldf(vr + dva + 1);
        if (dvb < Dv) v2 = ldf(vr + dvb);
        if (dvb + 1 < Dv) v3 = ldf(vr + dvb + 1);
      }
#pragma unroll
      for (int r = 0; r < RC; ++r) {
        const float w = pw[r * 64 + jj];
        acc[r][0] += w * v0; acc[r][1] += w * v1; acc[r][2] += w * v2; acc[r][3] += w * v3;
      }
    }
    }
    __builtin_amdgcn_s_waitcnt(0xc07f);
  }
  const int PS = 2 + Dv;
  float* mine = part + (long)wid * RC * PS;
#pragma unroll
  for (int r = 0; r < RC; ++r) {
    if (lane == 0) { mine[r * PS] = m[r]; mine[r * PS + 1] = l[r]; }
    if constexpr (V8) {
#pragma unroll
      for (int e = 0; e < 8; ++e) {
        float v = acc[r][e];
        for (int off = vl; off < 64; off <<= 1) v += __shfl_xor(v, off);  // the key groups' sums of this channel
        if (vsub == 0 && vlive) mine[r * PS + 2 + vch + e] = v;
      }
    } else {
      const int dva = 2 * lane, dvb = 128 + 2 * lane;
      if (dva < Dv) mine[r * PS + 2 + dva] = acc[r][0];
      if (dva + 1 < Dv) mine[r * PS + 2 + dva + 1] = acc[r][1];
      if (dvb < Dv) mine[r * PS + 2 + dvb] = acc[r][2];
      if (dvb + 1 < Dv) mine[r * PS + 2 + dvb + 1] = acc[r][3];
    }
  }
  __syncthreads();
  for (int i = threadIdx.x; i < nh * Dv; i += blockDim.x) {
    const int r = i / Dv, dv = i % Dv;
    float mm = -INFINITY;
    for (int w = 0; w < nw; ++w) mm = fmaxf(mm, part[(w * RC + r) * PS]);
    float ll = 0.0f, o = 0.0f;
    for (int w = 0; w < nw; ++w) {
      const float mw = part[(w * RC + r) * PS];
      if (mw != -INFINITY) {
        const float f = expf(mw - mm);
        ll += part[(w * RC + r) * PS + 1] * f;
        o += part[(w * RC + r) * PS + 2 + dv] * f;
      }
    }
    if (sink_logits != nullptr) {  // a learned score: it may be the largest of the row
      const float sk = sink_logits[h0 + r], m2 = fmaxf(mm, sk), f2 = expf(mm - m2);
      ll = ll * f2 + expf(sk - m2);
      o *= f2;
    } else if (sink) {
      ll += expf(-mm);  // the sink's score is 0
    }
    float scale_out = 1.0f / ll;
    if (gate != nullptr) scale_out *= sigmoidf_(ldf(gate + n * gate_stride + h0 + r));
    if (cross_out != nullptr) cross_out[((n * H + h0 + r) * G + vg) * (long)Dv + dv] = o * scale_out;
    else if (out32 != nullptr) out32[(n * H + h0 + r) * (long)Dv + dv] = o * scale_out;
    else stf(out + (n * H + h0 + r) * (long)Dv + dv, o * scale_out);
  }
}

// MFMA kernel (bfloat16 prompt portions). One block per (32-token tile of one sequence, kv head,
// pass); its waves are query heads of that kv head's group, so a key/value tile is fetched once
// for all of them: 16-byte loads through the page table into LDS, double-buffered (the next
// tile's loads are in flight while this tile is multiplied). All per-token quantities are
// lane-local because the products are formed transposed:
//   S^T = K Q^T   (A = key rows from LDS, B = query rows kept in registers)
//   O^T = V^T P^T (B = the float32 weights in the C layout they were born in, split into a
//                  high and a low bfloat16 half, 16 to 17 of a weight's 24 bits, twice what
//                  the matrix unit takes at once; A = values, read from LDS with the transposing
//                  64-bit read in the same key order)
// so column = token = lane & 31 everywhere: running max, running sum, rescaling and the gate
// never cross lanes except for one exchange between the two half-waves.
// The tiles are DS * 16 key channels by VT * 32 value channels; a head whose sizes Dr / Dvr are
// smaller (multiples of 8) is padded with zeros on its way into registers and LDS, and only its
// own channels are stored.
// What bounds it: the vector unit's issue. A product occupies the matrix unit for 32 cycles and the issue for 11, another instruction the issue for 4
// to 5 (an exponential 8), for a SIMD's waves together; the halves of the weights, a cap and a penalty make 5 to 9 of these a product. In
// phases (scores, weights, values) a wave's times for both add up, and two waves that meet at a barrier each step have the same phase; so
// a wave's instructions alternate between the products of two tiles and the weights of a third (`turn`). 256 registers at 128 channels, a few spilled
// around the loop; with the branches of several forms in one loop it was 60.
// One 4096-token prompt, 16 heads on 4 of 128, page 64, us, in phases -> now: 131 -> 122, a cap and a sink 140 -> 127; 2000 tokens 64 -> 48, with a
// cap 71 -> 54 (lanes past a sequence's last token repeat it, and its tiles need no masks for them); 3 x 200 after 1500 54 -> 42; 14
// decode tokens beside portions of 1000 and 963, window 1024: 58 -> 53. A lone prompt of 40 or 100 tokens has one turn more in its chain, 11.1 -> 11.3
// to 11.9. Weights' low halves by dot products with (-1, 0) instead of a shift, a mask and two differences: the same or slower.
// A page number is left as it comes until its row is needed, a step later: formed behind the lookup the row waited for it in every step. With that, and
// fewer scalar instructions about masks (18 % of what a SIMD issued), us: 4096 tokens 121.5 -> 116.5, a cap and a sink 125 -> 121; 2000 49.0 -> 47.3,
// with a cap 54.5 -> 52.2; 3 x 200 after 1500 44.8 -> 42.9; 8 x 512 after 512, window 512 42.9 -> 41.1. While its waves run, 87 % of the cycles issue.
__device__ __align__(16) const bf16s zero_channels[8] = {0, 0, 0, 0, 0, 0, 0, 0};

template <int DS, int VT, int NG, int FORM>
__global__ __launch_bounds__(256 * NG, 2) void paged_attention_mfma_kernel(
    bf16s* __restrict__ out, const bf16s* __restrict__ q, long q_stride, const bf16s* __restrict__ kpool,
    const bf16s* __restrict__ vpool, const int* __restrict__ block_tables, int bt_stride, const int* __restrict__ cu,
    const int* __restrict__ start, const float* __restrict__ slopes, const bf16s* __restrict__ gate, long gate_stride,
    int H, int G, int Dr, int Dvr, int page_shift, float scale, int window, int keep_first, float softcap, int sink,
    int tile_waves, const float* __restrict__ sink2, const float* __restrict__ dist2, int dist_rows,
    const bf16s* __restrict__ ksum, const bf16s* __restrict__ vsum, int sum_shift, int sum_block,
    float* __restrict__ cross_out, int chunk, const float* __restrict__ key_fac, int vrep, float* __restrict__ out32,
    int num_tiles, int fewest, int seqs, int sorted) {
  // The optional extras of the split-key kernel, in the base-2 domain: sink2 [H] = learned sink scores * log2e;
  // dist2 [H, dist_rows] = the per-distance bias * log2e, one row per head; ksum / vsum = block summaries, staged as
  // the first tiles of a block (summary idx of a sequence is seen by a token at pos when idx < (pos - window + 1) /
  // sum_block); cross_out [N, H, G, Dv] float32: a row is then also the kv head whose values a block
  // multiplies the weights with; chunk, key_fac [pool rows, G], vrep and out32 as in the split-key kernel (the factors of
  // a key tile are staged with it).
  // tile_waves (log2; kv heads with one or two query heads): the four waves of a block are four consecutive 32-token tiles of
  // the one head, or two tiles of the two heads, instead of four heads; a block covers 128 or 64 tokens then, which is what `num_tiles`
  // counts, and the staged key/value tiles are still shared by all computing waves. The block stages the key range of all
  // its tokens; a wave skips the tiles that lie wholly after its own tokens.
  // FORM 0: no block summaries, no distance table; with their branches in it the common form has no registers left. 1: all there is. 2: capped
  // scores and a sink, against the fixed reference (see below), and nothing else on the scores
  constexpr bool MORE = FORM == 1, CAPPED = FORM == 2;
  if constexpr (!MORE) ksum = vsum = nullptr, dist2 = nullptr;
  constexpr int D = DS * 16, Dv = VT * 32;
  bf16x8_v zero8;
#pragma unroll
  for (int e = 0; e < 8; ++e) zero8[e] = (__bf16)0.0f;
  // A staged tile: 32 keys, pieces of 16 keys of 32 channels (lds_tiles.h), keys and values alike. 48 channels end in half a piece.
  constexpr int KQ = (D + 31) / 32, VQ = VT;            // pieces side by side
  constexpr int KT = KQ * 2048, VTT = VQ * 2048;        // bytes of one staged tile
  constexpr int TP = MFMA_TILES_PER_STEP, TS = NG * TP;   // tiles of a step: a group's, the block's
  extern __shared__ __align__(16) char tiles[];  // [NG][2][TP] key tiles and [2][TP] value tiles, then [3][TS][32] key factors (float)
  float* facs = reinterpret_cast<float*>(tiles + 2 * TS * (KT + VTT));
  constexpr int nthreads = 256;  // of a group, always four waves: those beyond the kv head's group of heads only help staging
  const int tid = threadIdx.x & 255, grp = NG > 1 ? __builtin_amdgcn_readfirstlane(threadIdx.x >> 8) : 0;
  const int wid = __builtin_amdgcn_readfirstlane(tid >> 6), lane = tid & 63;
  const int rep = H / G, heads = 4 >> tile_waves;   // heads of a block
  const int VC = cross_out != nullptr ? G : 1;
  // Which (tile, row of kv head x pass) this block is. Block f runs on XCD f % 8: with rows that divide 8 or are a
  // multiple of it a row's keys and values stay in as few L2s as possible (4 kv heads: two XCDs a head, every second
  // tile each). Under a causal mask a late tile of a long prompt has many more key tiles than an early one: late ones
  // start first, and where all blocks of an XCD (32 CUs, two blocks each) run at once, the second 32 go the other way, so
  // that a CU's two blocks are a long and a short one.
  const int f = blockIdx.x, rows = G * ((rep + heads - 1) / heads) * VC;
  int row, tile, b = 0;
  if (rows <= 8 && 8 % rows == 0) {
    const int sub = 8 / rows, xcd = f & 7, i = f >> 3, per = (num_tiles + sub - 1) / sub;   // tiles of a row on this XCD
    const int k = NG == 1 && per <= 64 && i >= 32 ? i - 32 : per - 1 - i;
    row = xcd % rows;
    tile = k * sub + xcd / rows;
    if (tile >= num_tiles) return;
  } else {  // a row's tiles all go one way, every second row's the other way where all blocks run at once
    const bool by8 = rows % 8 == 0;
    const int at = by8 ? f >> 3 : f, turn = at / num_tiles, i = at - turn * num_tiles;
    row = by8 ? (f & 7) + 8 * turn : turn;
    tile = NG == 1 && num_tiles * rows <= 512 && (turn & 1) ? i : num_tiles - 1 - i;
  }
  const int g = row % G, zrow = row / G;
  const int vg = cross_out != nullptr ? zrow % VC : g / vrep;   // kv head of the values
  const int Gv = G / vrep;
  const int hl = (zrow / VC) * heads + (wid >> tile_waves);  // head inside the group
  const int h = g * rep + (hl < rep ? hl : 0);
  const int bshift = 5 + tile_waves;                  // log2 of the tokens a block covers
  // The block's sequence, 64 a time: there are exactly sum_b ceil(count_b / tokens per block) tiles, of the sequences of `fewest` tokens or more.
  // (One by one a step of 16 sequences took 4700 cycles here.)
  int first, cnt, s0;   // its first token, number of tokens, of tokens before them
  for (int b0 = 0;; b0 += 64) {
    const int at = min(b0 + lane, seqs - 1), from = cu[at], count = cu[at + 1] - from, held = start[at];
    const int own = b0 + lane >= seqs || count < fewest ? 0 : (count + (1 << bshift) - 1) >> bshift;
    // over the lanes up to this one: inside rows of 16, then over the rows
    auto summed = [](int v) {
      v += __builtin_amdgcn_update_dpp(0, v, 0x111, 0xf, 0xf, false);
      v += __builtin_amdgcn_update_dpp(0, v, 0x112, 0xf, 0xf, false);
      v += __builtin_amdgcn_update_dpp(0, v, 0x114, 0xf, 0xf, false);
      v += __builtin_amdgcn_update_dpp(0, v, 0x118, 0xf, 0xf, false);
      v += __builtin_amdgcn_update_dpp(0, v, 0x142, 0xa, 0xf, false);
      v += __builtin_amdgcn_update_dpp(0, v, 0x143, 0xc, 0xf, false);
      return v;
    };
    if (sorted) {
      // The tiles of up to 64 sequences by the position they end at (in tiles): those that end after `past`, found by halving, go ahead of this
      // one. In the sequences' order the long tiles of the last one would start when half of the time is over (4 x 1000 tokens, two groups of waves: 53 us).
      const int before = held >> bshift, rank = num_tiles - 1 - tile;
      auto ending = [&](int end) {   // tiles that end there or later
        return __builtin_amdgcn_readlane(summed(max(0, min(before + own - end + 1, own))), 63); };
      int lo = 1, hi = (int)wave_reduce_max((float)(before + own)) + 1, ahead = 0;
      lo = __builtin_amdgcn_readfirstlane(lo);
      hi = __builtin_amdgcn_readfirstlane(hi);
      while (hi - lo > 1) {   // ending(lo) > rank >= ending(hi) = ahead
        const int mid = (lo + hi) >> 1, n = ending(mid);
        if (n > rank) {
          lo = mid;
        } else {
          hi = mid;
          ahead = n;
        }
      }
      unsigned long long same = __ballot(lo > before && lo <= before + own);
      for (int skip = rank - ahead; skip > 0; --skip) same &= same - 1;
      const int at_lane = same != 0 ? __builtin_ctzll(same) : 0;
      b = at_lane;
      first = __builtin_amdgcn_readlane(from, at_lane);
      cnt = __builtin_amdgcn_readlane(count, at_lane);
      s0 = __builtin_amdgcn_readlane(held, at_lane);
      tile = lo - 1 - __builtin_amdgcn_readlane(before, at_lane);
      break;
    }
    const int upto = summed(own);
    const unsigned long long past = __ballot(tile < upto);
    if (past != 0 || b0 + 64 >= seqs) {
      const int at_lane = past != 0 ? __builtin_ctzll(past) : 63;
      b = b0 + at_lane;
      first = __builtin_amdgcn_readlane(from, at_lane);
      cnt = __builtin_amdgcn_readlane(count, at_lane);
      s0 = __builtin_amdgcn_readlane(held, at_lane);
      tile -= __builtin_amdgcn_readlane(upto - own, at_lane);
      break;
    }
    tile -= __builtin_amdgcn_readlane(upto, 63);
  }
  const int col = lane & 31, hf = lane >> 5;
  const int bt_off = tile << bshift;                          // first token of the block
  const int t_off = bt_off + (wid & ((1 << tile_waves) - 1)) * 32;  // first token of this wave
  const bool head_ok = hl < rep && t_off < cnt;               // this wave computes
  const bool tok_ok = t_off + col < cnt;
  const int my_i = tok_ok ? t_off + col : cnt - 1;
  const long n = first + my_i;
  const int pos = s0 + my_i;
  const int p0 = s0 + t_off, p1 = s0 + min(t_off + 31, cnt - 1);              // this wave's positions
  const int bp0 = s0 + bt_off, bp1 = s0 + min(bt_off + (1 << bshift) - 1, cnt - 1);  // the block's
  const int* bt = block_tables + (long)b * bt_stride;
  const int page_mask = (1 << page_shift) - 1;
  const float slope = slopes != nullptr ? slopes[h] : 0.0f;

  bf16x8_v qf[DS];
#pragma unroll
  for (int s = 0; s < DS; ++s)
    qf[s] = 16 * s + hf * 8 < Dr ? ld_g16b(q + n * q_stride + (long)h * Dr + 16 * s + hf * 8) : zero8;
  if (scale < 0.0f) {  // exact: the largest product of a row is then its largest score
#pragma unroll
    for (int s = 0; s < DS; ++s) qf[s] = -qf[s];
    scale = -scale;
  }

  const int lo_min = first_visible(bp0, window, chunk);   // the staged key range is the block's
  const int lo = first_visible(pos, window, chunk);       // this token's first key
  const int lo_p0 = first_visible(p0, window, chunk), lo_p1 = first_visible(p1, window, chunk);  // the wave's
  const int wstart = lo_min & ~31;
  const int n_sink = window > 0 ? min(keep_first, wstart) : 0;  // kept keys below the window's first tile
  const int n_sum = (MORE && ksum != nullptr && window > 0) ? max(0, (bp1 - window + 1) / sum_block) : 0;  // the block's last token's
  const int sum_tiles = (n_sum + 31) >> 5;
  const int sum_mask = (1 << sum_shift) - 1;
  const int sink_tiles = sum_tiles + ((n_sink + 31) >> 5);   // summary tiles, then kept-prefix tiles, then the window's
  const int tiles_n = sink_tiles + ((bp1 - wstart) >> 5) + 1;
  const int my_sum = (MORE && ksum != nullptr && window > 0) ? max(0, (pos - window + 1) / sum_block) : 0;  // this token's
  const float* db = MORE && dist2 != nullptr ? dist2 + (long)h * dist_rows : nullptr;

  // Staging: a wave brings every second piece of its 16 keys of a tile (wave & 1) straight into LDS, piece n the channels
  // (wave / 2 + 2 n) * 32 of them: a lane looks up one key of a tile, for keys and values alike. A lane whose channels are
  // beyond the head's brings zeros.
  constexpr int KR = (KQ + 1) / 2, VR = (VQ + 1) / 2;      // pieces per wave and tile
  const int row_group = wid & 1, quad0 = wid >> 1;
  const int lkey = 16 * row_group + (lane >> 2);           // this lane's key of the tile
  const int lch = ((lane & 3) ^ (lane >> 4 & 3)) * 8;      // and channel of the piece's 32
  // TP key tiles are staged, and multiplied, between two barriers: their loads go out one by one between the products
  // of the TP tiles before them (issued together, they held a wave up for 1600 of the 9200 cycles that a step took, and
  // their stores for 590)
  auto tile_base = [&](int it) {
    if (MORE && it < sum_tiles) return it * 32;
    return it < sink_tiles ? (it - sum_tiles) * 32 : wstart + (it - sink_tiles) * 32;
  };
  // The key of the sequence, or the summary, that a lane brings. Keys past the sequence's end are masked, those of a step past the last (below 0) not
  // used: the block's last token stands for them, whose page exists.
  auto pool_key = [&](int j) { return (int)min((unsigned)j, (unsigned)bp1); };
  auto sum_key = [&](int idx) { return min(idx, n_sum - 1); };   // a summary tile exists only when n_sum > 0
  // The page-table lookups of a tile run one step ahead of its key/value loads (two ahead of its use), so that a
  // load's address never waits for a lookup issued in the same step.
  const unsigned krs = (unsigned)(G * Dr) * 2u, vrs = (unsigned)(Gv * Dvr) * 2u;   // bytes between neighbouring keys' rows
  // Page numbers stay as they come until their rows are needed: what they go through would be waited for right behind the lookup, in every step.
  struct Pages {
    int key[TP], fac[TP];
  };
  auto summed_tile = [&](int it) { return MORE && it >= 0 && it < sum_tiles; };
  // Steps go from the nearest keys to the farthest. The other way round the scores of a head with a steep distance penalty rise by
  // more than 30 from step to step, so that many steps raise the reference and take their weights twice (with 12: 4000 tokens, window 1024:
  // 83 us, 75 this way; 14 decode tokens beside portions of 1000 and 963: 72, 65). Without a penalty it is all the same (4096
  // tokens 125 and 125 us), but a way that depends on the call costs 2 to 3 %.
  const int steps_n = (tiles_n + TS - 1) / TS;
  constexpr int way = -TS;
  const int first_tile = (steps_n - 1) * TS;
  auto lookup = [&](int tile0) {   // of the step whose first tile this is
    Pages r;
#pragma unroll
    for (int u = 0; u < TP; ++u) {
      const int it = tile0 + grp * TP + u, kbase = tile_base(it);  // a tile past the last one reads rows that exist and is not used
      r.key[u] = bt[summed_tile(it) ? sum_key(kbase + lkey) >> sum_shift : pool_key(kbase + lkey) >> page_shift];
      if (key_fac != nullptr && tid < 32) r.fac[u] = bt[pool_key(kbase + tid) >> page_shift];
    }
    return r;
  };
  struct Rows {
    int key[TP];
  };
  auto rows_of = [&](const Pages& p, int tile0) {
    Rows r;
#pragma unroll
    for (int u = 0; u < TP; ++u) {
      const int it = tile0 + grp * TP + u, kbase = tile_base(it);
      r.key[u] = summed_tile(it) ? (p.key[u] << sum_shift) + (sum_key(kbase + lkey) & sum_mask)
                                 : (p.key[u] << page_shift) + (pool_key(kbase + lkey) & page_mask);
    }
    return r;
  };
  const char* zeros = reinterpret_cast<const char*>(zero_channels);
  // Pieces of a step's keys (to the step's place among the two of them) and values, n of the wave's TP * KR and TP * VR. Head sizes that fill the
  // tiles, as nearly all do, need no look at the channel.
  auto piece = [&](const char* row, int n, int channels, int fewest_channels, char* __restrict__ dst) __attribute__((always_inline)) {
    const int quad = quad0 + 2 * (n / TP);
    const char* at = row + (n / TP) * 128;
    if (64 * (n / TP + 1) > fewest_channels && channels % 64 != 0 && quad * 32 + lch >= channels) at = zeros;
    __builtin_amdgcn_global_load_lds((global_ptr)at, (lds_ptr)(dst + (quad * 2 + row_group) * 1024), 16, 0, 0);
  };
  auto key_row = [&](const Rows& r, int tile0, int u) {
    return reinterpret_cast<const char*>((summed_tile(tile0 + grp * TP + u) ? ksum : kpool) + (long)g * Dr + quad0 * 32 + lch) + (unsigned long)(unsigned)r.key[u] * krs;
  };
  auto value_row = [&](const Rows& r, int tile0, int u) {
    return reinterpret_cast<const char*>((summed_tile(tile0 + grp * TP + u) ? vsum : vpool) + (long)vg * Dvr + quad0 * 32 + lch) + (unsigned long)(unsigned)r.key[u] * vrs;
  };
  auto key_piece = [&](const char* const (&row)[TP], char* __restrict__ dst, int n) __attribute__((always_inline)) {
    if (KQ % 2 != 0 && quad0 + 2 * (n / TP) >= KQ) return;
    piece(row[n % TP], n, Dr, DS == 8 ? 97 : DS == 6 ? 65 : D - 15, dst + n % TP * KT);
  };
  auto value_piece = [&](const char* const (&row)[TP], char* __restrict__ dst, int n) __attribute__((always_inline)) {
    if (VQ % 2 != 0 && quad0 + 2 * (n / TP) >= VQ) return;
    piece(row[n % TP], n, Dvr, Dv - 31, dst + n % TP * VTT);
  };
  float rf[TP];
  auto fetch_factors = [&](const Pages& p, int tile0) {
#pragma unroll
    for (int u = 0; u < TP; ++u)
      if (key_fac != nullptr && tid < 32)
        rf[u] = key_fac[(long)((p.fac[u] << page_shift) + (pool_key(tile_base(tile0 + grp * TP + u) + tid) & page_mask)) * G + g];
  };
  // of a step among three: a step's last tile is weighted in the next one, when the factors of the one after that arrive
  auto stash_factors = [&](int at) {
#pragma unroll
    for (int u = 0; u < TP; ++u)
      if (key_fac != nullptr && tid < 32) facs[(at * TS + grp * TP + u) * 32 + tid] = rf[u];
  };

  // With a sink and a soft cap the scores live in [-cap2, cap2] (a distance penalty only lowers them) and the
  // denominator holds the sink's exp2(0) = 1: the weights can be taken against the fixed reference 0 instead of a
  // running maximum. exp2(cap2) cannot overflow for cap2 <= 96, and a weight that underflows is nothing beside the
  // sink's 1. No maximum to track, no accumulator to rescale.
  const bool fixed_ref = CAPPED || (sink != 0 && softcap > 0.0f && softcap * 1.4426950408889634f <= 96.0f);
  // Without one, m is a maximum the token has had, not always its newest: weights are taken against it as it stands, and
  // only where the sum of a tile's weights shows that some passed 2^12 (a token's first visible score gives inf; NaN counts
  // too) is the maximum formed, m raised and the weights taken again. A weight of 2^12 has the mantissa of one of 1, and its
  // products with values of up to 2^100 are finite in any number.
  float m = fixed_ref ? 0.0f : -INFINITY, l = 0.0f;  // m in the base-2 domain
  float m_ref = fixed_ref ? 0.0f : -3.0e38f;         // m, and below every finite score until there is one
  f32x16 oacc[VT];
#pragma unroll
  for (int t = 0; t < VT; ++t)
#pragma unroll
    for (int i = 0; i < 16; ++i) oacc[t][i] = 0.0f;
  constexpr float LOG2E = 1.4426950408889634f;
  // a scale of 0 must not meet -inf in a product, one of NaN stays (fmaxf drops it)
  const float c1 = scale * LOG2E < 1e-30f ? 1e-30f : scale * LOG2E, sl2 = slope * LOG2E;
  // soft cap in the base-2 domain: cap log2e tanh(x scale / cap), tanh(y) = 1 - 2 / (exp2(2 log2e y) + 1)
  const bool capped = CAPPED || softcap > 0.0f;
  const float inv_cap = capped ? scale / softcap : 0.0f;
  const float cap2 = softcap * LOG2E, t2 = capped ? 2.0f * LOG2E * scale / softcap : 0.0f;
  // of the polynomial of tanh(y) / y in y^2; with CAPPED in the raw product's square, for which the host bounds the ratio of scale and cap, whose
  // eighth power is one of its factors
  struct Poly {
    float c0, c1, c2, c3, c4;
  };
  const float ic = CAPPED ? inv_cap : 1.0f, ic2 = ic * ic, ic4 = ic2 * ic2, cx = cap2 * ic;
  const Poly cap_poly{cx, cx * ic2 * -0.33333069f, cx * ic4 * 0.13324751f, cx * ic4 * ic2 * -0.052984238f, cx * ic4 * ic4 * 0.017131345f};
  auto cap_base2 = [&](float dot) {
    const float e = __builtin_amdgcn_exp2f(dot * t2);  // +inf: the quotient is 0; a NaN stays one
    return cap2 - 2.0f * cap2 * __builtin_amdgcn_rcpf(e + 1.0f);
  };
  const bool sloped = !CAPPED && slopes != nullptr;
  // Without a cap, a penalty or a table the scores stay raw products and their factor enters with the fma that
  // subtracts the reference (a negative factor has moved into the query); otherwise they are formed in the base-2 domain.
  const bool raw = !capped && !sloped && db == nullptr;
  const float k1 = raw ? c1 : 1.0f;

  const RowAt row_at(col, hf);
  const ColAt col_at(lane);
  Pages next = lookup(first_tile);
  // this group's place: [2] steps' keys, [2] steps' values
  constexpr int KS = TP * KT, VS = TP * VTT;
  char* keys = tiles + grp * (2 * KS + 2 * VS);
  char* values = keys + 2 * KS;
  const char *krow[TP], *vrow[TP];
  Rows of_values = rows_of(next, first_tile);
#pragma unroll
  for (int u = 0; u < TP; ++u) krow[u] = key_row(of_values, first_tile, u);
#pragma unroll
  for (int n = 0; n < TP * KR; ++n) key_piece(krow, keys, n);
  fetch_factors(next, first_tile);
#pragma unroll
  for (int u = 0; u < TP; ++u) vrow[u] = value_row(of_values, first_tile, u);
  if (steps_n > 1) next = lookup(first_tile + way);
  stash_factors(0);
  __builtin_amdgcn_sched_barrier(0);
  // the first step's values behind its keys: they are not waited for yet
#pragma unroll
  for (int n = 0; n < TP * VR; ++n) value_piece(vrow, values, n);
  if (quad0 == 0) loads_left<TP * VR>();
  else loads_left<TP * (VQ / 2)>();
  __syncthreads();

  // What a tile's scores go through before they are weights: factors, the cap, a penalty or a table, masks. `it` is the tile, `fc` its keys' factors.
  struct Tile {
    int it, kbase;
    bool summ, inner;
  };
  // inner: every key is visible to every token of the wave (lanes past the last one repeat it), no masks to evaluate: the tiles of the window from
  // in_lo on, inner_n of them
  const int in_lo = sink_tiles + ((lo_p1 - wstart + 31) >> 5);
  const unsigned inner_n = head_ok ? (unsigned)max(0, sink_tiles + ((p0 - 31 - wstart) >> 5) - in_lo + 1) : 0u;
  auto tile_of = [&](int it) {
    Tile t;
    t.it = it;
    t.kbase = tile_base(it);
    t.summ = MORE && it < sum_tiles;
    t.inner = (unsigned)(it - in_lo) < inner_n;
    return t;
  };
  // (several token tiles) a tile wholly after this wave's tokens, or wholly before what they see, is not live
  auto live = [&](const Tile& t) {
    return t.inner || (head_ok && t.it < tiles_n && (t.it < sink_tiles || !(t.kbase > p1 || (t.kbase + 31 < lo_p0 && t.kbase >= keep_first))));
  };
  auto factors = [&](f32x16& x, int place) __attribute__((always_inline)) {
    if (key_fac != nullptr) {
      const float* fc = facs + place * 32 + 4 * hf;
#pragma unroll
      for (int a = 0; a < 4; ++a) {
        const float4v f4 = *reinterpret_cast<const float4v*>(fc + 8 * a);
#pragma unroll
        for (int c = 0; c < 4; ++c) x[4 * a + c] *= f4[c];
      }
    }
  };
  // tanh(y) = y P(y^2) for |y| <= 1/2, P a polynomial through the Chebyshev nodes (1.3e-8 off): fused
  // multiplications where the general form takes an exponential and a reciprocal
  auto near = [&](const f32x16& x) __attribute__((always_inline)) {
    // A NaN is the largest, and takes the general form. One instruction for two scores, which the compiler knows to read a product's result: as
    // inline assembly it could stand behind the product without the wait that this takes.
    float far = 0.0f;
#pragma unroll
    for (int i = 0; i < 16; i += 2) far = __builtin_elementwise_maximum(__builtin_elementwise_maximum(far, fabsf(x[i])), fabsf(x[i + 1]));
    return __all(far * fabsf(inv_cap) <= 0.5f);
  };
  auto near_cap = [&](f32x16& x) __attribute__((always_inline)) {
#pragma unroll
    for (int i = 0; i < 16; ++i) {
      const float y = CAPPED ? x[i] : x[i] * inv_cap, z = y * y;
      x[i] = y * fmaf(z, fmaf(z, fmaf(z, fmaf(z, cap_poly.c4, cap_poly.c3), cap_poly.c2), cap_poly.c1), cap_poly.c0);
    }
  };
  auto prepare = [&](const Tile& t, f32x16& x) __attribute__((always_inline)) {
    if (capped) {
      if (near(x)) {
        near_cap(x);
      } else {
#pragma unroll
        for (int i = 0; i < 16; ++i) x[i] = cap_base2(x[i]);
      }
    }
    if (!raw) {
      if (sloped && !t.summ) {
        // a key's share of the distance penalty, its offset inside the tile (row of the C layout); the tile's own comes with the reference
#pragma unroll
        for (int i = 0; i < 16; ++i) x[i] = fmaf(sl2, (float)((i & 3) + 8 * (i >> 2)), capped ? x[i] : x[i] * c1);
      } else if (!capped) {
#pragma unroll
        for (int i = 0; i < 16; ++i) x[i] *= c1;
      }
      if (db != nullptr && !t.summ) {
#pragma unroll
        for (int i = 0; i < 16; ++i) {
          const int j = t.kbase + (i & 3) + 8 * (i >> 2) + 4 * hf;
          x[i] += db[min(max(pos - j, 0), dist_rows - 1)];
        }
      }
    }
    if (!t.inner) {
      const bool ahead = t.it < sink_tiles;  // a tile ahead of the window's: summaries or kept first tokens
      // the tile's keys that this token sees: those up to `last`, from `first` on or below `keep` (offsets in the tile)
      const int last = !live(t) ? -1 : t.summ ? my_sum - 1 - t.kbase : (ahead ? min(n_sink - 1, pos) : min(p1, pos)) - t.kbase;
      const int first = t.summ ? 0 : lo - t.kbase, keep = t.summ ? 0 : keep_first - t.kbase;
#pragma unroll
      for (int i = 0; i < 16; ++i) {
        const int j = (i & 3) + 8 * (i >> 2) + 4 * hf;
        x[i] = (j <= last) & ((j >= first) | (j < keep)) ? x[i] : CAPPED ? -1e18f : -INFINITY;   // finite where its square meets 0
      }
      asm volatile("" ::: "memory");   // a body of its own: merged into the common one, every tile would pay for it
    }
  };
  constexpr std::true_type yes{};
  constexpr std::false_type no{};
  struct Weights {
    bf16x8_v hi[2], lo[2];
  };
  // Two weights in stages: (0) with CAPPED, where the near form of the cap is a part of them, and (1) the exponentials, (2) sum and high halves, (3)
  // low halves; one conversion packs two. A tile that has been through `prepare` takes the polynomial 1.
  struct Pair {
    float a, b, za, zb;
    unsigned bits;
  };
  auto stage = [&](int k, const Poly& c, const f32x16& x, float base, int i, Pair& s, float& psum, Weights& p) __attribute__((always_inline)) {
    if (k == 0) {
      s.za = x[i] * x[i];
      s.zb = x[i + 1] * x[i + 1];
      s.a = fmaf(s.za, c.c4, c.c3);
      s.b = fmaf(s.zb, c.c4, c.c3);
      s.a = fmaf(s.za, s.a, c.c2);
      s.b = fmaf(s.zb, s.b, c.c2);
    } else if (k == 1) {
      if (CAPPED) {
        s.a = fmaf(s.za, fmaf(s.za, s.a, c.c1), c.c0);
        s.b = fmaf(s.zb, fmaf(s.zb, s.b, c.c1), c.c0);
        s.a = __builtin_amdgcn_exp2f(x[i] * s.a);
        s.b = __builtin_amdgcn_exp2f(x[i + 1] * s.b);
      } else {
        s.a = __builtin_amdgcn_exp2f(fmaf(x[i], k1, base));
        s.b = __builtin_amdgcn_exp2f(fmaf(x[i + 1], k1, base));
      }
    } else if (k == 2) {
      psum += s.a;
      psum += s.b;
      const bf16x2_v hi = __builtin_convertvector(float2v{s.a, s.b}, bf16x2_v);
      s.bits = __builtin_bit_cast(unsigned, hi);
      p.hi[i >> 3][i & 7] = hi[0];
      p.hi[i >> 3][(i & 7) + 1] = hi[1];
    } else {
      const bf16x2_v lo = __builtin_convertvector(float2v{s.a - __builtin_bit_cast(float, s.bits << 16),
                                                          s.b - __builtin_bit_cast(float, s.bits & 0xffff0000u)}, bf16x2_v);
      p.lo[i >> 3][i & 7] = lo[0];
      p.lo[i >> 3][(i & 7) + 1] = lo[1];
    }
  };
  // where the sum of a tile's weights shows that some passed 2^12: the maximum, and the weights again
  auto raise = [&](const f32x16& x, float off, float psum, Weights& p) __attribute__((always_inline)) {
    if (!fixed_ref && __builtin_expect(!__all(psum <= 4096.0f), 0)) {
      Pair again;
      float top = x[0];
#pragma unroll
      for (int i = 1; i < 16; ++i) top = fmaxf(top, x[i]);
      float tmax = top == -INFINITY ? -INFINITY : fmaf(top, k1, off);
      tmax = fmaxf(tmax, __shfl_xor(tmax, 32));
      const float m_new = fmaxf(m, tmax);
      const float corr = (m == -INFINITY) ? 1.0f : __builtin_amdgcn_exp2f(m - m_new);  // nothing accumulated: nothing to rescale
      l *= corr;
#pragma unroll
      for (int t = 0; t < VT; ++t)
#pragma unroll
        for (int i = 0; i < 16; ++i) oacc[t][i] *= corr;
      m = m_new;
      m_ref = (m_new == -INFINITY) ? -3.0e38f : m_new;  // nothing visible yet: every weight is exp2(-inf) = 0
      psum = 0.0f;
#pragma unroll
      for (int i = 0; i < 16; i += 2)
#pragma unroll
        for (int k = 1; k < 4; ++k) stage(k, cap_poly, x, off - m_ref, i, again, psum, p);
    }
    l += psum;
  };
  auto offset = [&](const Tile& t) { return sloped && !t.summ ? -sl2 * (float)(pos - t.kbase - 4 * hf) : 0.0f; };

  // One tile's turn: the scores of the tile after it (keys at `K_`) into `xn`, the weights of this one's scores `x` into `p`, and what the tile
  // before it adds, its weights `pp` times the values at `V_`, none of which waits for another. A wave's instructions alternate between them, so that
  // the matrix unit has work while the exponentials are formed.
  // O^T += V^T P^T: slot hf * 8 + e of half s2 holds key 16 s2 + 8 (e >> 2) + 4 hf + (e & 3)
  constexpr int GROUPS = DS > 2 * VT ? DS : 2 * VT, AHEAD = 2;
  auto turn = [&](auto with_scores, auto with_weights, auto with_values, const Poly& poly, const char* __restrict__ K_, const char* __restrict__ V_,
                  f32x16& xn, const f32x16& x, float off, Weights& p, const Weights& pp, auto load) __attribute__((always_inline)) {
    bf16x8_v kf[DS], vf[2 * VT];
    const float base = off - m_ref;
    float psum = 0.0f;
    Pair s[8];
    auto read = [&](int i) __attribute__((always_inline)) {
      if (with_scores && i < DS) kf[i] = frag_row<32>(K_, row_at, 0, i);
      if (with_values && i < 2 * VT) vf[i] = frag_born<32>(V_, col_at, 16 * (i / VT), 32 * (i % VT));
    };
    // after product n of all: its share of the weights' stages. One product's time is that of eight other instructions, of which a wave issues
    // none while its next product waits for the unit: they have to stand between the products.
    constexpr int PRODUCTS = (decltype(with_scores)::value ? DS : 0) + (decltype(with_values)::value ? 4 * VT : 0);
    auto weigh = [&](int n) __attribute__((always_inline)) {
      constexpr int FROM = CAPPED ? 0 : 1, STAGES = 4 - FROM;
      if (with_weights) {
#pragma unroll
        for (int k = n * 8 * STAGES / PRODUCTS; k < (n + 1) * 8 * STAGES / PRODUCTS; ++k)
          stage(FROM + k % STAGES, poly, x, base, k / STAGES * 2, s[k / STAGES], psum, p);
      }
      __builtin_amdgcn_sched_barrier(0);
    };
    if (with_scores) {
#pragma unroll
      for (int i = 0; i < 16; ++i) xn[i] = 0.0f;
    }
#pragma unroll
    for (int i = 0; i < AHEAD; ++i) read(i);
    __builtin_amdgcn_sched_barrier(0);
    int n = 0;
#pragma unroll
    for (int i = 0; i < GROUPS; ++i) {
      read(i + AHEAD);
      if (with_scores && i < DS) {
        xn = __builtin_amdgcn_mfma_f32_32x32x16_bf16(kf[i], qf[i], xn, 0, 0, 0);
        weigh(n++);
      }
      if (with_values && i < 2 * VT) {
        oacc[i % VT] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(vf[i], pp.hi[i / VT], oacc[i % VT], 0, 0, 0);
        weigh(n++);
        oacc[i % VT] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(vf[i], pp.lo[i / VT], oacc[i % VT], 0, 0, 0);
        weigh(n++);
      }
      load(i);
      __builtin_amdgcn_sched_barrier(0);
    }
    if (with_weights) {
      // formed here: the compiler moves them to where they are used, behind the products
#pragma unroll
      for (int e = 0; e < 2; ++e) asm volatile("" : "+v"(p.hi[e]), "+v"(p.lo[e]));
      raise(x, off, psum, p);
    }
  };
  // the weights' turn of a tile, by what its scores need ahead of it
  auto weights_turn = [&](auto with_scores, auto with_values, const Tile& t, int place, const char* __restrict__ K_, const char* __restrict__ V_,
                          f32x16& xn, f32x16& x, Weights& p, const Weights& pp, auto load) __attribute__((always_inline)) {
    factors(x, place);
    Poly poly = cap_poly;
    if (!CAPPED || !t.inner || !near(x)) {
      prepare(t, x);
      poly = Poly{1.0f, 0.0f, 0.0f, 0.0f, 0.0f};
    }
    turn(with_scores, yes, with_values, poly, K_, V_, xn, x, offset(t), p, pp, load);
  };
  // Keys are a step ahead of values. In step s a wave forms the scores of the step's two tiles, the weights of the tile before them and
  // of the first one, and adds what the two tiles of the step before are worth; the next step's keys and this step's values are on their way.
  // Steps in which a wave sees nothing (several token tiles) only load, and nothing they hold meets a weight of 0; a wave without tokens or a head
  // does no other.
  int tile0 = first_tile, step = 0, third = 0;   // third: the step's place among three
  auto begin = [&]() __attribute__((always_inline)) {   // the next step's keys and this step's values; past the last step the loads repeat rows
    const Pages now = next;
    const Rows rows = rows_of(now, tile0 + way);
#pragma unroll
    for (int u = 0; u < TP; ++u) {
      krow[u] = key_row(rows, tile0 + way, u);
      vrow[u] = value_row(of_values, tile0, u);
    }
    of_values = rows;
    next = lookup(tile0 + 2 * way);
    if (step + 1 < steps_n) fetch_factors(now, tile0 + way);
  };
  auto end = [&]() __attribute__((always_inline)) {
    third = third == 2 ? 0 : third + 1;
    if (step + 1 < steps_n) stash_factors(third);
    loads_done();
    __syncthreads();
    ++step;
    tile0 += way;
  };
  // all of them in the first of a step's two turns: those that go out last have to arrive before the step ends
  auto load_keys = [&](int i) __attribute__((always_inline)) {
#pragma unroll
    for (int n = i * (TP * KR) / GROUPS; n < (i + 1) * (TP * KR) / GROUPS; ++n) key_piece(krow, keys + (~step & 1) * KS, n);
  };
  auto load_values = [&](int i) __attribute__((always_inline)) {
#pragma unroll
    for (int n = i * (TP * VR) / GROUPS; n < (i + 1) * (TP * VR) / GROUPS; ++n) value_piece(vrow, values + (step & 1) * VS, n);
  };
  auto load = [&](int i) __attribute__((always_inline)) {
    load_keys(i);
    load_values(i);
  };
  auto load_first = [&](int i) __attribute__((always_inline)) {   // the values of step 0 are on their way; a lone step waits for nothing more
    if (step + 1 < steps_n) load_keys(i);
    if (step > 0) load_values(i);
  };
  auto nothing = [](int) {};
  auto idle = [&]() __attribute__((always_inline)) {
    begin();
#pragma unroll
    for (int i = 0; i < GROUPS; ++i) load_first(i);
    end();
  };
  // A wave that has begun goes on up to `stop`, the first step with nothing of its window, and where kept first keys or summaries lie apart, from `again` on:
  // numbers, as a look at each step's tiles in the loop cost up to 470 spilled registers. A loop around both parts is slower too (decode tokens two
  // by two, 16 heads on 8, 1000 keys 27.9 us for 26.9).
  const int mine0 = first_tile + grp * TP;      // the group's first tile of step 0
  const int w_lo = keep_first > wstart ? sink_tiles : sink_tiles + (max(0, lo_p0 - wstart) >> 5);   // lowest tile of the wave's window
  const int again = head_ok ? (max(0, mine0 - sink_tiles + 1) + TS - 1) / TS : steps_n;
  int stop = (mine0 + 1 - w_lo + TS) / TS;
  if (again <= stop) stop = steps_n;
  auto mine_of = [&](int u) { return tile_of(tile0 + grp * TP + u); };
  while (step < steps_n && !live(mine_of(0)) && !live(mine_of(1))) idle();
  if (step < steps_n) {
    f32x16 xe, xo;            // scores of an even and an odd tile of the wave's
    Weights pe, po;
    {
      begin();
      const char* K_ = keys + (step & 1) * KS;
      turn(yes, no, no, cap_poly, K_, K_, xe, xo, 0.0f, po, pe, load_first);
      weights_turn(yes, no, mine_of(0), third * TS + grp * TP, K_ + KT, K_, xo, xe, pe, po, nothing);
      end();
    }
    while (step < stop) {
      const Tile odd = tile_of(tile0 - way + grp * TP + 1), even = mine_of(0);
      begin();
      const char* K_ = keys + (step & 1) * KS;
      const char* V_ = values + (~step & 1) * VS;
      weights_turn(yes, yes, odd, (third == 0 ? 2 : third - 1) * TS + grp * TP + 1, K_, V_, xe, xo, po, pe, load);
      weights_turn(yes, yes, even, third * TS + grp * TP, K_ + KT, V_ + VTT, xo, xe, pe, po, nothing);
      end();
    }
    // the tiles that are left, while other waves' loads go to the other places
    const Tile odd = tile_of(tile0 - way + grp * TP + 1);
    const char* V_ = values + (~step & 1) * VS;
    weights_turn(no, yes, odd, (third == 0 ? 2 : third - 1) * TS + grp * TP + 1, V_, V_, xe, xo, po, pe, nothing);
    turn(no, no, yes, cap_poly, V_, V_ + VTT, xo, xe, 0.0f, pe, po, nothing);
  }
  while (step < again) idle();
#pragma clang loop unroll(disable)
  while (step < steps_n) {   // the tiles ahead of the window, few and seldom apart: step by step
    f32x16 xe, xo;
    Weights pe, po;
    const Tile even = mine_of(0), odd = mine_of(1);
    begin();
    const char* K_ = keys + (step & 1) * KS;
    turn(yes, no, no, cap_poly, K_, K_, xe, xo, 0.0f, po, pe, load_first);
    weights_turn(yes, no, even, third * TS + grp * TP, K_ + KT, K_, xo, xe, pe, po, nothing);
    end();
    const char* V_ = values + (~step & 1) * VS;
    weights_turn(no, yes, odd, (third == 0 ? 2 : third - 1) * TS + grp * TP + 1, V_, V_, xe, xo, po, pe, nothing);
    turn(no, no, yes, cap_poly, V_, V_ + VTT, xo, xe, 0.0f, pe, po, nothing);
  }
  if constexpr (NG > 1) {  // the second group's states, wave by wave, through the tiles' place
    __syncthreads();         // all waves are past their last tile
    float4v* sums = reinterpret_cast<float4v*>(tiles) + wid * (VT * 4 * 64 + 32) + lane;   // 16 bytes an access
    float* state = reinterpret_cast<float*>(sums - lane + VT * 4 * 64) + lane;
    if (grp == 1) {
      state[0] = m;
      state[64] = l;
#pragma unroll
      for (int t = 0; t < VT; ++t)
#pragma unroll
        for (int a = 0; a < 4; ++a)
          sums[(t * 4 + a) * 64] = float4v{oacc[t][4 * a], oacc[t][4 * a + 1], oacc[t][4 * a + 2], oacc[t][4 * a + 3]};
    }
    __syncthreads();
    if (grp == 1) return;
    const float m1 = state[0], top = fmaxf(m, m1);
    const float f0 = m == -INFINITY ? 0.0f : __builtin_amdgcn_exp2f(m - top);
    const float f1 = m1 == -INFINITY ? 0.0f : __builtin_amdgcn_exp2f(m1 - top);
    l = l * f0 + state[64] * f1;
#pragma unroll
    for (int t = 0; t < VT; ++t)
#pragma unroll
      for (int a = 0; a < 4; ++a) {
        const float4v other = sums[(t * 4 + a) * 64];
#pragma unroll
        for (int c = 0; c < 4; ++c) oacc[t][4 * a + c] = oacc[t][4 * a + c] * f0 + other[c] * f1;
      }
    m = top;
  }
  l += __shfl_xor(l, 32);
  if (sink2 != nullptr) l += __builtin_amdgcn_exp2f(sink2[h] - m);  // a learned score; a sink far above every key: 1 / inf = 0
  else if (sink) l += __builtin_amdgcn_exp2f(-m);  // the sink's score is 0 in either base; m is finite (a token sees itself)
  if (!tok_ok || !head_ok) return;
  float scale_out = 1.0f / l;
  if (gate != nullptr) scale_out *= sigmoidf_(ldf(gate + n * gate_stride + h));
  if (cross_out != nullptr || out32 != nullptr) {
    float* crow = cross_out != nullptr ? cross_out + ((n * H + h) * G + vg) * (long)Dvr : out32 + (n * H + h) * (long)Dvr;
#pragma unroll
    for (int t = 0; t < VT; ++t)
#pragma unroll
      for (int a = 0; a < 4; ++a) {
        if (t * 32 + 8 * a + 4 * hf >= Dvr) continue;
        *reinterpret_cast<float4v*>(crow + t * 32 + 8 * a + 4 * hf) =
            float4v{oacc[t][4 * a] * scale_out, oacc[t][4 * a + 1] * scale_out, oacc[t][4 * a + 2] * scale_out,
                    oacc[t][4 * a + 3] * scale_out};
      }
    return;
  }
  bf16s* orow = out + (n * H + h) * (long)Dvr;
#pragma unroll
  for (int t = 0; t < VT; ++t)
#pragma unroll
    for (int a = 0; a < 4; ++a) {
      if (t * 32 + 8 * a + 4 * hf >= Dvr) continue;  // padding channels (sizes are multiples of 8: four at a time)
      short4v pk;
#pragma unroll
      for (int c = 0; c < 4; ++c) pk[c] = (short)f2bf(oacc[t][4 * a + c] * scale_out);
      *reinterpret_cast<short4v*>(orow + t * 32 + 8 * a + 4 * hf) = pk;
    }
}

static void launch_scalar_attention(at::Tensor& out, const at::Tensor& q, const at::Tensor& kpool, const at::Tensor& vpool,
                                    const at::Tensor& block_tables, const at::Tensor& tok_seq, const at::Tensor& positions,
                                    const float* slp, const c10::optional<at::Tensor>& gate, long gstride, double scale,
                                    int64_t window, int64_t keep_first, double softcap, bool sink, int page_shift,
                                    long vrow, long vhead, const ScalarExtras& x) {
  const long N = q.size(0);
  const int H = (int)q.size(1), D = (int)q.size(2);
  const int G = (int)kpool.size(2), Dv = (int)vpool.size(3);
  if (launch_group_attention(out, q, kpool, vpool, block_tables, tok_seq, positions, slp, gate, gstride, scale, window,
                             keep_first, softcap, sink, page_shift, vrow, vhead, x))
    return;
  if (launch_row_attention(out, q, kpool, vpool, block_tables, tok_seq, positions, slp, gate, gstride, scale, window,
                           keep_first, softcap, sink, page_shift, vrow, vhead, x))
    return;
  const int VC = x.cross_out != nullptr ? G : 1;
  const int Dp = (D + 7) & ~7;
  const int R = H / G;
  int rc = RC_MAX;
  while (rc > 1 && (rc > R || N * G * VC * ((R + rc - 1) / rc) < 256)) rc >>= 1;  // enough blocks to cover the CUs
  auto lds_bytes = [&](int nw) { return (size_t)(rc * Dp + nw * (rc * 64 + 64) + nw * rc * (2 + Dv)) * sizeof(float); };
  // wide value rows (a latent of several hundred channels): fewer waves, then fewer heads per block
  int nwaves = ATT_WAVES;
  while (lds_bytes(nwaves) > 64 * 1024 && nwaves > 4) nwaves >>= 1;
  while (lds_bytes(nwaves) > 64 * 1024 && rc > 1) rc >>= 1;
  const int chunks = (R + rc - 1) / rc;
  const size_t smem = lds_bytes(nwaves);
  TORCH_CHECK(smem <= 64 * 1024, "head sizes too large for the scalar attention kernel");
  const int kvec = D % 8 == 0 ? 1 : 0;   // 16-byte (bfloat16) / 32-byte (float32) aligned key slices
  const int vvec_even = Dv % 2 == 0 ? 1 : 0;
  // value rows of a multiple of 8 channels whose loads are aligned take the 8-channels-per-lane value phase
  const bool v8 = Dv >= 8 && Dv % 8 == 0 && reinterpret_cast<uintptr_t>(vpool.data_ptr()) % 32 == 0 &&
                  vrow % 8 == 0 && vhead % 8 == 0;
  TORCH_CHECK(v8 || Dv <= 256, "value rows above 256 channels must be a multiple of 8 channels and aligned");
  const int vvec_ok = (vrow % 2 == 0 && vhead % 2 == 0) ? 1 : 0;
#define SCALAR_CASE(RC_)                                                                                            \
  if (v8) SCALAR_LAUNCH(RC_, true);                                                                                 \
  else SCALAR_LAUNCH(RC_, false)
#define SCALAR_LAUNCH(RC_, V8_)                                                                                     \
  hipLaunchKernelGGL((paged_attention_kernel<T, RC_, V8_>), dim3((unsigned)(N * G * chunks * VC)), dim3(64 * nwaves), smem,   \
                     stream(), (x.cross_out != nullptr || x.out32 != nullptr) ? (T*)nullptr : ptr<T>(out), ptr<T>(q), (long)q.stride(0), ptr<T>(kpool), ptr<T>(vpool),             \
                     block_tables.data_ptr<int>(), (int)block_tables.stride(0), tok_seq.data_ptr<int>(),            \
                     positions.data_ptr<int>(), slp, gate.has_value() ? ptr<T>(*gate) : (const T*)nullptr, gstride, \
                     H, G, D, Dv, page_shift, (float)scale, (int)window, (int)keep_first, kvec,                      \
                     vvec_even & vvec_ok, (float)softcap, sink ? 1 : 0, vrow, vhead, x.sink_logits, x.dist_bias, x.dist_rows,      \
                     (const T*)x.ksum, (const T*)x.vsum, x.sum_shift, x.sum_block, x.cross_out, x.chunk, x.key_fac,        \
                     x.vrep, x.out32)
  SERVING_DISPATCH_ACT(q, T, {
    if (rc == 4) { SCALAR_CASE(4); }
    else if (rc == 2) { SCALAR_CASE(2); }
    else { SCALAR_CASE(1); }
  });
#undef SCALAR_CASE
#undef SCALAR_LAUNCH
  HIP_CHECK_LAST();
}

// The matrix-core kernel for prompt portions in bfloat16 whose head sizes fit a tiling; false when it does not apply.
// In `x`, sink_logits and dist_bias are already in the base-2 domain (times log2 e), dist_bias one row per head.
static bool launch_mfma_attention(at::Tensor& out, const at::Tensor& q, const at::Tensor& kpool, const at::Tensor& vpool,
                                  const at::Tensor& block_tables, const at::Tensor& cu, const at::Tensor& start,
                                  const float* slp, const c10::optional<at::Tensor>& gate, long gstride, double scale,
                                  int64_t window, int64_t keep_first, double softcap, bool sink, int page_shift,
                                  int64_t num_tiles, int64_t num_tiles128, int64_t num_tiles64, const ScalarExtras& x, double even, int64_t longest, int fewest = 1) {
  const int H = (int)q.size(1), D = (int)q.size(2);
  const int G = (int)kpool.size(2), Dv = (int)vpool.size(3);
  // prompt portions in bfloat16 go to the matrix cores when the head sizes fit a tiling;
  // num_tiles = sum over sequences of ceil(new tokens / 32), 0 asks for the scalar kernel
  auto at16 = [](const void* p) { return reinterpret_cast<uintptr_t>(p) % 16 == 0; };
  const bool aligned = q.stride(0) % 8 == 0 && at16(q.data_ptr()) && at16(x.ksum) && at16(x.vsum);
  // head sizes that are multiples of 8 ride in the next larger tiling, zero-padded
  const bool mfma_shape = D % 8 == 0 && Dv % 8 == 0 && D <= 128 && Dv <= 128;
  if (!(num_tiles > 0 && is_bf16(q) && aligned && mfma_shape && vpool.is_contiguous())) return false;
  if (!at16(kpool.data_ptr()) || !at16(vpool.data_ptr())) {
    // Loads go straight into LDS from addresses of 16 bytes. Pools that lie otherwise lend the pages of the call's sequences to copies, which
    // the tables then number (4096 tokens of 16 heads on 4 of 128: 154 us, 135 without the copies, 5000 in the general kernel); not with data that is
    // numbered by page as well, nor beyond 1 GiB.
    const long pages = block_tables.numel(), per_page = (kpool.numel() + vpool.numel()) / std::max<long>(kpool.size(0), 1) * 2;
    if (x.ksum != nullptr || x.key_fac != nullptr || pages * per_page > (1L << 30)) return false;
    const at::Tensor ids = block_tables.reshape({-1}).clamp(0, kpool.size(0) - 1);   // places past a sequence's end hold anything
    return launch_mfma_attention(out, q, kpool.index_select(0, ids), vpool.index_select(0, ids),
                                 at::arange(pages, block_tables.options()).view(block_tables.sizes()), cu, start, slp, gate, gstride, scale,
                                 window, keep_first, softcap, sink, page_shift, num_tiles, num_tiles128, num_tiles64, x, even, longest, fewest);
  }
  {
    const int rep = H / G, nw = 4;
    // one query head per kv head: the waves of a block take four consecutive token tiles instead of four heads; two: two
    const int tile_waves = rep == 1 && num_tiles128 > 0 ? 2 : rep == 2 && num_tiles64 > 0 ? 1 : 0, heads = nw >> tile_waves;
    const int VC = x.cross_out != nullptr ? G : 1;
    const int tiles = (int)(tile_waves == 2 ? num_tiles128 : tile_waves == 1 ? num_tiles64 : num_tiles);
    const int rows = G * ((rep + heads - 1) / heads) * VC;
    const int sub = rows <= 8 && 8 % rows == 0 ? 8 / rows : 1;   // XCDs a row's tiles are spread over: whole rounds of them
    const dim3 grid((unsigned)((tiles + sub - 1) / sub * sub * rows));
    const int ds = D <= 32 ? 2 : D <= 48 ? 3 : D <= 64 ? 4 : D <= 96 ? 6 : 8, vt = (Dv + 31) / 32;
    // Two groups of waves take alternate key tiles where one block a CU is all there is: a second group then fills the
    // idle half of the CU, and a lone block's chain of tiles is half as long (2000 tokens, 16 heads on 4 of 128: 55 us with one group, 46 with two). Up to
    // 512 blocks it is a question of how even they are: a CU takes two after the other, and where long and short ones alternate, as in one long
    // prompt, that is better than both at once, of which the long one's last steps run alone; blocks of about one length, by a window or
    // many cached tokens, hide each other's waits when they run together. `even` is the mean length of their sequences' tiles of 32 tokens over
    // the longest; one group and two: 4096 tokens 129,
    // 114 (0.5), with a window of 1024 63, 71 (0.9); 3000 with the window (376 blocks, 0.84) 53, 64; 2200 with it (276, 0.8) 41, 35; 8 x 512
    // after 1000 73, 82 (0.83); 16 x 200 after 1500 (448, 0.95) 82, 92; 2 x 1200 with the window (304) 43, 36. Short blocks wait for their
    // first loads a good part of their time, and sooner run together: 4 x 1000 (512, 0.5) 39, 44, 3 x 1000 (384) 37, 38.
    const int ng = grid.x <= 256 || (grid.x <= 512 && even * grid.x <= (longest < 1536 ? 230 : 300)) ? 2 : 1;
    // the order of tiles matters where some wait for others, or share a CU with them
    const int sorted = cu.numel() > 2 && cu.numel() <= 65 && grid.x > 256;
    const bool more = x.ksum != nullptr || x.dist_bias != nullptr;
    // a sink, a cap that needs no running maximum and whose powers are ordinary numbers
    const double near = std::abs(scale) / softcap;
    const bool capped = sink && softcap > 0.0 && softcap * 1.4427 <= 96.0 && slp == nullptr && near > 1e-4 && near < 1e3;
    const size_t msmem = (size_t)ng * MFMA_TILES_PER_STEP *
                         (((ds + 1) / 2 + vt) * 4096 + (x.key_fac != nullptr ? 3 * 32 * sizeof(float) : 0));
// The common form exists for the sizes that serving meets most, 64 and 128 channels, and for the others with all there is.
#define MFMA_CASE(DS_, VT_)                                                                       \
  do {                                                                                            \
    constexpr bool ALWAYS = !((DS_ == 4 || DS_ == 8) && (VT_ == 2 || VT_ == 4));                  \
    if (ng == 2) MFMA_FORM(DS_, VT_, 2, ALWAYS);                                                  \
    else MFMA_FORM(DS_, VT_, 1, ALWAYS);                                                          \
  } while (0)
#define MFMA_FORM(DS_, VT_, NG_, ALWAYS_)                                                         \
  do {                                                                                            \
    if (more || ALWAYS_) MFMA_NG(DS_, VT_, NG_, 1);                                               \
    else if (capped) MFMA_NG(DS_, VT_, NG_, ALWAYS_ ? 1 : 2);                                     \
    else MFMA_NG(DS_, VT_, NG_, ALWAYS_ ? 1 : 0);                                                 \
  } while (0)
#define MFMA_NG(DS_, VT_, NG_, FORM_)                                                                                     \
  do {                                                                                                             \
    auto kfn = paged_attention_mfma_kernel<DS_, VT_, NG_, FORM_>;                                                         \
    if (msmem > 65536) /* more dynamic LDS than a kernel gets without asking */                                    \
      (void)hipFuncSetAttribute((const void*)kfn, hipFuncAttributeMaxDynamicSharedMemorySize, (int)msmem);         \
    hipLaunchKernelGGL(kfn, grid, dim3(64 * nw * NG_), msmem, stream(),                                            \
                       (x.cross_out != nullptr || x.out32 != nullptr) ? (bf16s*)nullptr : ptr<bf16s>(out),         \
                       ptr<bf16s>(q),                                                                              \
                       (long)q.stride(0), ptr<bf16s>(kpool), ptr<bf16s>(vpool), block_tables.data_ptr<int>(),      \
                       (int)block_tables.stride(0), cu.data_ptr<int>(), start.data_ptr<int>(), slp,                \
                       gate.has_value() ? ptr<bf16s>(*gate) : (const bf16s*)nullptr, gstride, H, G, D, Dv,         \
                       page_shift, (float)scale, (int)window, (int)keep_first, (float)softcap, sink ? 1 : 0,       \
                       tile_waves, x.sink_logits, x.dist_bias, x.dist_rows, (const bf16s*)x.ksum,                      \
                       (const bf16s*)x.vsum, x.sum_shift, x.sum_block, x.cross_out, x.chunk, x.key_fac, x.vrep,    \
                       x.out32, tiles, fewest, (int)cu.numel() - 1, sorted);                                                                         \
  } while (0)
#define MFMA_ROW(DS_)                     \
  do {                                    \
    if (vt == 1) MFMA_CASE(DS_, 1);       \
    else if (vt == 2) MFMA_CASE(DS_, 2);  \
    else if (vt == 3) MFMA_CASE(DS_, 3);  \
    else MFMA_CASE(DS_, 4);               \
  } while (0)
    if (ds == 2) MFMA_ROW(2);
    else if (ds == 3) MFMA_ROW(3);
    else if (ds == 4) MFMA_ROW(4);
    else if (ds == 6) MFMA_ROW(6);
    else MFMA_ROW(8);
#undef MFMA_ROW
#undef MFMA_CASE
#undef MFMA_FORM
#undef MFMA_NG
    HIP_CHECK_LAST();
    return true;
  }
}

at::Tensor paged_attention(at::Tensor q, at::Tensor kpool, at::Tensor vpool, at::Tensor block_tables, at::Tensor cu,
                           at::Tensor start, at::Tensor tok_seq, at::Tensor positions, double scale, int64_t window,
                           int64_t keep_first, c10::optional<at::Tensor> slopes, c10::optional<at::Tensor> gate,
                           int64_t num_tiles, double softcap, bool sink, int64_t num_tiles128, int64_t num_tiles64, int64_t singles,
                           bool singles_see_half, double even, int64_t longest, double even_apart, int64_t longest_apart) {
  check_act(q, "q");
  TORCH_CHECK(softcap >= 0.0, "softcap must not be negative (0 = none)");
  TORCH_CHECK(q.dim() == 3 && q.stride(2) == 1 && q.stride(1) == q.size(2), "q must be [N, H, D] with dense rows");
  // the value pool may be a view into wider rows (values that are leading channels of the keys): dense
  // channels, pages of `page` rows, any row and head stride
  TORCH_CHECK(kpool.dim() == 4 && vpool.dim() == 4 && kpool.is_contiguous() && vpool.stride(3) == 1 &&
              vpool.stride(0) == vpool.size(1) * vpool.stride(1), "pools must be [pages, page, G, D] with dense rows");
  TORCH_CHECK(kpool.scalar_type() == q.scalar_type() && vpool.scalar_type() == q.scalar_type(),
              "query and pools share one dtype");
  const long N = q.size(0);
  const int H = (int)q.size(1), D = (int)q.size(2);
  const int page = (int)kpool.size(1), G = (int)kpool.size(2), Dv = (int)vpool.size(3);
  TORCH_CHECK(kpool.size(3) == D && vpool.size(2) == G && vpool.size(1) == page && vpool.size(0) == kpool.size(0));
  TORCH_CHECK(H % G == 0 && Dv <= 512 && page > 0 && (page & (page - 1)) == 0);
  const long vrow = vpool.stride(1), vhead = G > 1 ? vpool.stride(2) : Dv;
  check_i32(block_tables, "block_tables"); check_i32(tok_seq, "tok_seq"); check_i32(positions, "positions");
  TORCH_CHECK(block_tables.dim() == 2 && tok_seq.numel() == N && positions.numel() == N);
  TORCH_CHECK(window >= 0 && keep_first >= 0);
  int page_shift = 0;
  while ((1 << page_shift) < page) ++page_shift;
  at::Tensor sl;
  const float* slp = nullptr;
  if (slopes.has_value()) {
    sl = f32c(*slopes);
    TORCH_CHECK(sl.numel() == H);
    slp = sl.data_ptr<float>();
  }
  long gstride = 0;
  if (gate.has_value()) {
    TORCH_CHECK(gate->scalar_type() == q.scalar_type() && gate->dim() == 2 && gate->size(0) == N &&
                gate->size(1) == H && gate->stride(1) == 1, "gate must be [N, H] of q's dtype");
    gstride = gate->stride(0);
  }
  at::Tensor out = at::empty({N, H, Dv}, q.options());
  if (N == 0) return out;
  check_i32(cu, "cu"); check_i32(start, "start");
  // A decode token beside prompt portions is a tile of its own in their kernel, 4 waves over all its keys, and costs little as
  // long as its blocks fit beside the others; a launch of its own stands in line (10 to 15 us). It goes apart where its blocks
  // would be the first beyond one, or two, for each CU and it sees half as many keys as a portion or more: 14 beside portions
  // of 1000 and 963, window 1024: 80 us together, 70 apart (32 heads on 8: 123, 96), without a window 2100 keys 150, 133, 16000 keys 1427, 1110.
  // `even` and `longest` then are those of the portions alone (`even_apart`, `longest_apart`).
  // Otherwise: 15 of 400 beside 4000, 8 heads on 4 of 64: 76 together, 86 apart; 15 beside 512 after 2000, window 512: 29, 40.
  int fewest = 1;
  if (singles > 0 && num_tiles > singles && vpool.is_contiguous()) {
    const int rep = H / G;
    const long tiles = rep == 1 && num_tiles128 > 0 ? num_tiles128 : rep == 2 && num_tiles64 > 0 ? num_tiles64 : num_tiles;
    const long rows = (long)G * (rep <= 4 ? 1 : (rep + 3) / 4), portions = (tiles - singles) * rows, both = tiles * rows;
    if (portions <= 512 && (both + 255) / 256 > (portions + 255) / 256 && singles_see_half &&
        launch_group_attention(out, q, kpool, vpool, block_tables, tok_seq, positions, slp, gate, gstride, scale, window, keep_first,
                               softcap, sink, page_shift, vrow, vhead, ScalarExtras(), SingleTokens{cu.data_ptr<int>(), cu.numel() - 1, singles})) {
      fewest = 2;
      num_tiles -= singles;
      num_tiles128 -= singles;
      num_tiles64 -= singles;
      even = even_apart;
      longest = longest_apart;
    }
  }
  if (launch_mfma_attention(out, q, kpool, vpool, block_tables, cu, start, slp, gate, gstride, scale, window, keep_first,
                            softcap, sink, page_shift, num_tiles, num_tiles128, num_tiles64, ScalarExtras(), even, longest, fewest))
    return out;
  launch_scalar_attention(out, q, kpool, vpool, block_tables, tok_seq, positions, slp, gate, gstride, scale, window,
                          keep_first, softcap, sink, page_shift, vrow, vhead, ScalarExtras());
  return out;
}

// Attention with its optional extras, for prompt portions and decode tokens alike: a learned sink per
// head, a per-distance bias table, block summaries ahead of the window, (cross) every query head's weights
// applied to every kv head's values, returned as float32 [N, H, G, Dv] for a talking-heads mix, visibility inside blocks
// of `chunk` positions, a factor per cached key, value pools with fewer heads than the key pool, float32 output.
at::Tensor paged_attention_ext(at::Tensor q, at::Tensor kpool, at::Tensor vpool, at::Tensor block_tables, at::Tensor cu,
                               at::Tensor start, at::Tensor tok_seq, at::Tensor positions, double scale, int64_t window,
                               int64_t keep_first, c10::optional<at::Tensor> slopes, c10::optional<at::Tensor> gate,
                               double softcap, bool sink, c10::optional<at::Tensor> sink_logits,
                               c10::optional<at::Tensor> dist_bias, c10::optional<at::Tensor> ksum,
                               c10::optional<at::Tensor> vsum, int64_t sum_block, bool cross, int64_t num_tiles,
                               int64_t num_tiles128, int64_t num_tiles64, int64_t chunk,
                               c10::optional<at::Tensor> key_fac, bool out_f32, double even, int64_t longest) {
  check_act(q, "q");
  TORCH_CHECK(softcap >= 0.0, "softcap must not be negative (0 = none)");
  TORCH_CHECK(q.dim() == 3 && q.stride(2) == 1 && q.stride(1) == q.size(2), "q must be [N, H, D] with dense rows");
  TORCH_CHECK(kpool.dim() == 4 && vpool.dim() == 4 && kpool.is_contiguous() && vpool.is_contiguous(),
              "pools must be contiguous [pages, page, G, D]");
  TORCH_CHECK(kpool.scalar_type() == q.scalar_type() && vpool.scalar_type() == q.scalar_type(),
              "query and pools share one dtype");
  const long N = q.size(0);
  const int H = (int)q.size(1), D = (int)q.size(2);
  const int page = (int)kpool.size(1), G = (int)kpool.size(2), Dv = (int)vpool.size(3);
  const int Gv = (int)vpool.size(2);
  TORCH_CHECK(kpool.size(3) == D && Gv > 0 && G % Gv == 0 && vpool.size(1) == page && vpool.size(0) == kpool.size(0),
              "the value pool must have the key pool's pages and a divisor of its heads");
  TORCH_CHECK(H % G == 0 && Dv <= 512 && page > 0 && (page & (page - 1)) == 0);
  check_i32(block_tables, "block_tables"); check_i32(tok_seq, "tok_seq"); check_i32(positions, "positions");
  TORCH_CHECK(block_tables.dim() == 2 && tok_seq.numel() == N && positions.numel() == N);
  TORCH_CHECK(window >= 0 && keep_first >= 0 && chunk >= 0);
  TORCH_CHECK(chunk == 0 || (window == 0 && keep_first == 0 && !ksum.has_value()),
              "fixed blocks of positions take the place of a window");
  TORCH_CHECK((Gv == G && !key_fac.has_value() && !out_f32) || (!cross && !ksum.has_value()),
              "cross values and block summaries go with plain key/value heads");
  int page_shift = 0;
  while ((1 << page_shift) < page) ++page_shift;
  at::Tensor sl, sk, db;
  const float* slp = nullptr;
  if (slopes.has_value()) {
    sl = f32c(*slopes);
    TORCH_CHECK(sl.numel() == H);
    slp = sl.data_ptr<float>();
  }
  long gstride = 0;
  if (gate.has_value()) {
    TORCH_CHECK(gate->scalar_type() == q.scalar_type() && gate->dim() == 2 && gate->size(0) == N &&
                gate->size(1) == H && gate->stride(1) == 1, "gate must be [N, H] of q's dtype");
    gstride = gate->stride(0);
  }
  ScalarExtras x;
  x.chunk = (int)chunk;
  x.vrep = G / Gv;
  if (key_fac.has_value()) {
    TORCH_CHECK(key_fac->is_cuda() && is_f32(*key_fac) && key_fac->is_contiguous() && key_fac->dim() == 3 &&
                key_fac->size(0) == kpool.size(0) && key_fac->size(1) == page && key_fac->size(2) == G,
                "key factors must be contiguous float32 [pages, page, G]");
    x.key_fac = key_fac->data_ptr<float>();
  }
  if (sink_logits.has_value()) {
    sk = f32c(*sink_logits);
    TORCH_CHECK(sk.is_cuda() && sk.numel() == H, "sink_logits must be [H]");
    x.sink_logits = sk.data_ptr<float>();
  }
  if (dist_bias.has_value()) {
    db = f32c(*dist_bias);
    TORCH_CHECK(db.is_cuda() && db.dim() == 2 && db.size(1) == H && db.size(0) >= 1, "dist_bias must be [rows, H]");
    x.dist_bias = db.data_ptr<float>();
    x.dist_rows = (int)db.size(0);
  }
  if (ksum.has_value()) {
    TORCH_CHECK(vsum.has_value() && window > 0 && sum_block >= 1, "block summaries need both pools, a window and a block length");
    const int rows = (int)ksum->size(1);
    TORCH_CHECK(ksum->dim() == 4 && vsum->dim() == 4 && ksum->is_contiguous() && vsum->is_contiguous() &&
                ksum->scalar_type() == q.scalar_type() && vsum->scalar_type() == q.scalar_type() &&
                ksum->size(0) == kpool.size(0) && vsum->size(0) == kpool.size(0) && vsum->size(1) == rows &&
                ksum->size(2) == G && ksum->size(3) == D && vsum->size(2) == G && vsum->size(3) == Dv &&
                rows > 0 && (rows & (rows - 1)) == 0 && (long)rows * sum_block >= page,
                "summary pools must be [pages, rows, G, D] / [.., Dv] of the pools' type, rows a power of two with "
                "rows * block >= page size");
    while ((1 << x.sum_shift) < rows) ++x.sum_shift;
    x.sum_block = (int)sum_block;
    x.ksum = ksum->data_ptr();
    x.vsum = vsum->data_ptr();
  }
  at::Tensor out = cross ? at::empty({N, H, G, Dv}, q.options().dtype(at::kFloat))
                         : at::empty({N, H, Dv}, out_f32 ? q.options().dtype(at::kFloat) : q.options());
  if (N == 0) return out;
  if (cross) x.cross_out = out.data_ptr<float>();
  else if (out_f32) x.out32 = out.data_ptr<float>();
  if (num_tiles > 0 && is_bf16(q)) {  // prompt portions in bfloat16: the matrix-core kernel, extras in the base-2 domain
    check_i32(cu, "cu"); check_i32(start, "start");
    constexpr double LOG2E = 1.4426950408889634;
    ScalarExtras x2 = x;
    at::Tensor sk2, db2;
    if (sink_logits.has_value()) {
      sk2 = sk * LOG2E;
      x2.sink_logits = sk2.data_ptr<float>();
    }
    if (dist_bias.has_value()) {
      db2 = (db * LOG2E).t().contiguous();   // [H, rows]
      x2.dist_bias = db2.data_ptr<float>();
    }
    if (launch_mfma_attention(out, q, kpool, vpool, block_tables, cu, start, slp, gate, gstride, scale, window,
                              keep_first, softcap, sink, page_shift, num_tiles, num_tiles128, num_tiles64, x2, even, longest))
      return out;
  }
  launch_scalar_attention(out, q, kpool, vpool, block_tables, tok_seq, positions, slp, gate, gstride, scale, window,
                          keep_first, softcap, sink, page_shift, (long)vpool.stride(1), (long)vpool.stride(2), x);
  return out;
}

// ------------------------------------------------------------------ block summaries
// One wave per (sequence, block completed in this step, kv head): the float32 mean of the block's `block` cached
// key rows and value rows goes to row b of the summary pools (page bt[b >> sum_shift], row b & mask).
template <typename T>
__global__ __launch_bounds__(64) void paged_pool_write_kernel(
    T* __restrict__ ksum, T* __restrict__ vsum, const T* __restrict__ kpool, const T* __restrict__ vpool,
    const int* __restrict__ block_tables, int bt_stride, const int* __restrict__ cu, const int* __restrict__ start,
    int G, int D, int Dv, int page_shift, int sum_shift, int block) {
  const int b = blockIdx.x, g = blockIdx.z;
  const int s0 = start[b], n = cu[b + 1] - cu[b];
  const int blk = s0 / block + (int)blockIdx.y;
  if (blk >= (s0 + n) / block) return;
  const int* bt = block_tables + (long)b * bt_stride;
  const int page_mask = (1 << page_shift) - 1, sum_mask = (1 << sum_shift) - 1;
  const long srow = ((long)bt[blk >> sum_shift] << sum_shift) + (blk & sum_mask);
  const float inv = 1.0f / (float)block;
  for (int d = threadIdx.x; d < D + Dv; d += 64) {
    const bool key = d < D;
    float acc = 0.0f;
    for (int i = 0; i < block; ++i) {
      const int j = blk * block + i;
      const long row = ((long)bt[j >> page_shift] << page_shift) + (j & page_mask);
      acc += key ? ldf(kpool + (row * G + g) * D + d) : ldf(vpool + (row * G + g) * Dv + (d - D));
    }
    if (key) stf(ksum + (srow * G + g) * D + d, acc * inv);
    else stf(vsum + (srow * G + g) * Dv + (d - D), acc * inv);
  }
}

void paged_pool_write(at::Tensor kpool, at::Tensor vpool, at::Tensor ksum, at::Tensor vsum, at::Tensor block_tables,
                      at::Tensor cu, at::Tensor start, int64_t block, int64_t most_blocks) {
  check_act(kpool, "kpool");
  TORCH_CHECK(kpool.dim() == 4 && vpool.dim() == 4 && ksum.dim() == 4 && vsum.dim() == 4 && kpool.is_contiguous() &&
              vpool.is_contiguous() && ksum.is_contiguous() && vsum.is_contiguous(), "pools must be contiguous");
  TORCH_CHECK(vpool.scalar_type() == kpool.scalar_type() && ksum.scalar_type() == kpool.scalar_type() &&
              vsum.scalar_type() == kpool.scalar_type(), "pools share one dtype");
  const int page = (int)kpool.size(1), G = (int)kpool.size(2), D = (int)kpool.size(3), Dv = (int)vpool.size(3);
  const int rows = (int)ksum.size(1);
  TORCH_CHECK(ksum.size(0) == kpool.size(0) && vsum.size(0) == kpool.size(0) && vsum.size(1) == rows &&
              ksum.size(2) == G && ksum.size(3) == D && vsum.size(2) == G && vsum.size(3) == Dv && vpool.size(2) == G &&
              vpool.size(1) == page, "summary pools do not fit the pools");
  TORCH_CHECK(block >= 1 && rows > 0 && (rows & (rows - 1)) == 0 && (page & (page - 1)) == 0 &&
              (long)rows * block >= page, "rows per page: a power of two with rows * block >= page size");
  check_i32(block_tables, "block_tables"); check_i32(cu, "cu"); check_i32(start, "start");
  const int B = (int)start.numel();
  if (B == 0 || most_blocks <= 0) return;
  int page_shift = 0, sum_shift = 0;
  while ((1 << page_shift) < page) ++page_shift;
  while ((1 << sum_shift) < rows) ++sum_shift;
  SERVING_DISPATCH_ACT(kpool, T, {
    hipLaunchKernelGGL(paged_pool_write_kernel<T>, dim3((unsigned)B, (unsigned)most_blocks, (unsigned)G), dim3(64), 0,
                       stream(), ptr<T>(ksum), ptr<T>(vsum), ptr<T>(kpool), ptr<T>(vpool), block_tables.data_ptr<int>(),
                       (int)block_tables.stride(0), cu.data_ptr<int>(), start.data_ptr<int>(), G, D, Dv, page_shift,
                       sum_shift, (int)block);
  });
  HIP_CHECK_LAST();
}

}  // namespace serving
}  // namespace cai
