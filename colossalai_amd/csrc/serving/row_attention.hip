// Split-key paged attention with a key block's rows in registers (decode tokens, float32 serving).
//
// One block per (token, kv head, group of up to RC query heads of that kv head); its waves take every nw-th key block.
// A row is covered by L lanes (a power of two) of 32 bytes each, so a wave's load instruction reads 64 / L whole rows,
// and a key block is NS such steps. All page lookups and then all row loads of a block are issued before the first
// product. Lane group g holds key g of every step, for the scores and for the weighted sum alike:
//   * the scores of a step meet across the L lanes of a row (DPP);
//   * every lane group runs an online softmax of its own over its keys — nothing crosses lane groups in the loop;
//   * the weighted sum uses the values in the same lanes. Where the values are the keys (or their leading channels)
//     they are the registers the scores were formed from: each cached row is read once.
// The lane groups' states meet in a butterfly, the waves' states in LDS, at the end. Few tokens with long contexts
// have their keys cut into parts, one block each, whose states row_merge_kernel puts together.
//
// What bounds it: the chain of dependent loads (position, page table, rows) and the block's end, about 10 us
// together, and beyond that the vector instructions of the products. bfloat16 calls of common sizes go to
// group_attention.hip; here are float32, shared key/value rows, key factors, float32 output and the other sizes. 16 x 1024
// keys of 16/4 heads of 128 with a cap and a sink took 17.8 us (29.3 before the base-2 scores and the halving butterfly), 1.9
// TB/s; 4 x 16384 took 51.5 us (242 with one block per token, kv head and head), 40 of it the parts at 3.4 TB/s and 7 the merge.
#include "paged_attention.h"

#include <algorithm>

namespace cai {
namespace serving {

typedef int int4v_ __attribute__((ext_vector_type(4)));

constexpr int ROW_WAVES = 8;
constexpr int MAX_PARTS = WAVE;  // of a token's keys: row_merge_kernel gives each part a lane

template <typename T> struct RowLane;   // CH channels = 32 bytes per lane, as two 16-byte pieces
template <> struct RowLane<bf16s> {
  static constexpr int CH = 16;
  DEV_INLINE static void unpack(const int4v_& p, float* o) {
#pragma unroll
    for (int e = 0; e < 4; ++e) {
      o[2 * e] = __builtin_bit_cast(float, p[e] << 16);
      o[2 * e + 1] = __builtin_bit_cast(float, p[e] & (int)0xffff0000);
    }
  }
};
template <> struct RowLane<float> {
  static constexpr int CH = 8;
  DEV_INLINE static void unpack(const int4v_& p, float* o) {
#pragma unroll
    for (int e = 0; e < 4; ++e) {
      const int bits = p[e];  // a bit cast of the vector element itself takes element 0
      o[e] = __builtin_bit_cast(float, bits);
    }
  }
};

// The domain of the scores. bfloat16: base 2, so that a weight is one v_exp_f32 and the cap an exponential and a
// reciprocal; float32 serving keeps the natural one with the library's functions.
template <typename T> struct Dom;
template <> struct Dom<bf16s> {
  static constexpr double NAT = 1.4426950408889634;    // what one nat is here
  static constexpr float UNIT = (float)NAT;
  DEV_INLINE static float exp_(float x) { return __builtin_amdgcn_exp2f(x); }
  // cap tanh(x / cap) for x and cap in units of this domain, a lane's N scores. tanh(y) = y P(y^2) for |y| <= 1/2, P the polynomial
  // through the Chebyshev nodes (1.3e-8 off); beyond, 1 - 2 / (exp(2 |y|) + 1) with y's sign, where an infinite
  // exponential is a quotient of 0 and a NaN stays one. That form alone is off by roundings of the cap, not of the score (cap
  // 30: 1.4e-6 at scores about 0.6 and 3, where these two are 0.9e-7 and 2.8e-7 off and the library's tanh 1.0e-7 and 3.8e-7), so a
  // score takes the form that is its own; mostly a whole wave's are small. 16 x 1024 keys with a cap take 17.8 us either way.
  template <int N>
  DEV_INLINE static void cap_(float (&x)[N], float cap, float inv_cap) {
    float far = 0.0f;
#pragma unroll
    for (int i = 0; i < N; ++i) far = fmaxf(far, fabsf(x[i]));
    const bool near = __all(far * inv_cap <= 0.5f);
#pragma unroll
    for (int i = 0; i < N; ++i) {
      const float y = x[i] * inv_cap, z = y * y;
      const float small = x[i] * fmaf(z, fmaf(z, fmaf(z, fmaf(z, 0.017131345f, -0.052984238f), 0.13324751f), -0.33333069f), 1.0f);
      if (near) {
        x[i] = small;
      } else {
        const float large = cap - 2.0f * cap * __builtin_amdgcn_rcpf(__builtin_amdgcn_exp2f(fabsf(y) * (2.0f * UNIT)) + 1.0f);
        x[i] = fabsf(y) <= 0.5f ? small : copysignf(large, y);
      }
    }
  }
};
template <> struct Dom<float> {
  static constexpr double NAT = 1.0;
  static constexpr float UNIT = 1.0f;
  DEV_INLINE static float exp_(float x) { return expf(x); }
  template <int N>
  DEV_INLINE static void cap_(float (&x)[N], float cap, float inv_cap) {
#pragma unroll
    for (int i = 0; i < N; ++i) x[i] = cap * tanhf(x[i] * inv_cap);
  }
};

typedef unsigned uint2v_ __attribute__((ext_vector_type(2)));

// Sums of two values over the two halves of the wave (rows of 16 lanes for swap16): lanes of the lower half (even
// rows) get a's sum, the others b's. A swap exchanges the upper half of a with the lower half of b.
DEV_INLINE float swap32_add(float a, float b) {
  const uint2v_ r = __builtin_amdgcn_permlane32_swap(__builtin_bit_cast(unsigned, a), __builtin_bit_cast(unsigned, b), false, false);
  const unsigned x = r[0], y = r[1];
  return __builtin_bit_cast(float, x) + __builtin_bit_cast(float, y);
}
DEV_INLINE float swap16_add(float a, float b) {
  const uint2v_ r = __builtin_amdgcn_permlane16_swap(__builtin_bit_cast(unsigned, a), __builtin_bit_cast(unsigned, b), false, false);
  const unsigned x = r[0], y = r[1];
  return __builtin_bit_cast(float, x) + __builtin_bit_cast(float, y);
}

template <typename T, int RC, int NS, bool SEP>
__global__ __launch_bounds__(64 * ROW_WAVES) void row_attention_kernel(
    T* __restrict__ out, float* __restrict__ out32, const T* __restrict__ q, long q_stride, const T* __restrict__ kpool,
    const T* __restrict__ vpool, const int* __restrict__ block_tables, int bt_stride, const int* __restrict__ tok_seq,
    const int* __restrict__ positions, const float* __restrict__ slopes, const T* __restrict__ gate, long gate_stride,
    const float* __restrict__ sink_logits, const float* __restrict__ key_fac, int H, int G, int D, int Dv, int page_shift,
    float scale, int window, int keep_first, int chunk, float softcap, int sink, int vrep, long vrow, long vhead,
    int lane_shift, int qvec, int splits, float* __restrict__ ws) {
  // scale: in units of the domain, rounded once (the product of two float32 factors leans a whole row's scores)
  constexpr int CH = RowLane<T>::CH, HC = CH / 2;
  extern __shared__ __align__(16) float lds[];
  const int wid = threadIdx.x >> 6, lane = threadIdx.x & 63, nw = blockDim.x >> 6;
  const int R = H / G, chunks = (R + RC - 1) / RC;
  // Heads of a group that are other blocks' come last: those blocks read the same rows, and a multiple of 8 blocks
  // apart they share an XCD's L2.
  const long parts = gridDim.x / chunks, item = blockIdx.x % parts;
  const int split = (int)(item % splits);           // which part of the keys
  const long n = item / splits / G;
  const int g = (int)(item / splits % G);
  const int h0 = g * R + (int)(blockIdx.x / parts) * RC;
  const int nh = min(RC, g * R + R - h0);
  const int L = 1 << lane_shift;
  const int ch = (lane & (L - 1)) * CH;             // this lane's first channel
  const int group = lane >> lane_shift, KPS = 64 >> lane_shift, KB = NS * KPS;
  const int pos = positions[n];
  const int* bt = block_tables + (long)tok_seq[n] * bt_stride;
  const int page_mask = (1 << page_shift) - 1;
  float* coef = lds;                                // [RC][ROW_WAVES]
  float* part = lds + RC * ROW_WAVES;               // [nw][RC][2 + Dv]

  float qf[RC][CH], slope[RC];
#pragma unroll
  for (int r = 0; r < RC; ++r) {
    slope[r] = (slopes != nullptr && r < nh) ? slopes[h0 + r] * Dom<T>::UNIT : 0.0f;
    const T* qp = q + n * q_stride + (long)(h0 + r) * D + ch;
    if (qvec) {
      const int4v_ none = {0, 0, 0, 0};
      RowLane<T>::unpack(r < nh && ch < D ? *reinterpret_cast<const int4v_*>(qp) : none, qf[r]);
      RowLane<T>::unpack(r < nh && ch + HC < D ? *reinterpret_cast<const int4v_*>(qp + HC) : none, qf[r] + HC);
    } else {
#pragma unroll
      for (int c = 0; c < CH; ++c) qf[r][c] = r < nh && ch + c < D ? ldf(qp + c) : 0.0f;
    }
#pragma unroll
    for (int c = 0; c < CH; ++c) qf[r][c] *= scale;
  }
  const int lo = first_visible(pos, window, chunk);
  const int n_keep = window > 0 ? min(keep_first, lo) : 0;
  const int total = n_keep + (pos - lo + 1);
  // this block's keys: whole key blocks of all its waves
  const int per = splits > 1 ? ((total + splits - 1) / splits + KB - 1) / KB * KB : total;
  const int first = split * per, last = min(total, first + per);
  const float cap = softcap * Dom<T>::UNIT, inv_cap = softcap > 0.0f ? 1.0f / cap : 0.0f;
  const T* vbase = SEP ? vpool + (long)(g / vrep) * vhead : nullptr;

  float m[RC], l[RC], acc[RC][CH];
#pragma unroll
  for (int r = 0; r < RC; ++r) {
    m[r] = -INFINITY;
    l[r] = 0.0f;
#pragma unroll
    for (int c = 0; c < CH; ++c) acc[r][c] = 0.0f;
  }
  const int4v_ zero = {0, 0, 0, 0};
  auto key_of = [&](int idx) { return idx < last ? (idx < n_keep ? idx : lo + (idx - n_keep)) : pos; };
  // pool rows of a block's keys; a key past the end reads the query's own row and is masked. Looked up one block ahead.
  int row[NS];
  auto lookup = [&](int base) {
#pragma unroll
    for (int s = 0; s < NS; ++s) {
      const int j = key_of(base + s * KPS + group);
      row[s] = (bt[j >> page_shift] << page_shift) + (j & page_mask);
    }
  };
  if (first + wid * KB < last) lookup(first + wid * KB);
  for (int base = first + wid * KB; base < last; base += nw * KB) {
    float fac[NS];
    int4v_ kr[NS][2], vr[SEP ? NS : 1][2];
#pragma unroll
    for (int s = 0; s < NS; ++s) {
      const bool some = base + s * KPS < last;      // the wave's step holds a key
      const T* kp = kpool + ((long)row[s] * G + g) * D + ch;
      kr[s][0] = some && ch < D ? *reinterpret_cast<const int4v_*>(kp) : zero;
      kr[s][1] = some && ch + HC < D ? *reinterpret_cast<const int4v_*>(kp + HC) : zero;
      fac[s] = key_fac != nullptr && some ? key_fac[(long)row[s] * G + g] : 1.0f;
      if constexpr (SEP) {
        const T* vp = vbase + (long)row[s] * vrow + ch;
        vr[s][0] = some && ch < Dv ? *reinterpret_cast<const int4v_*>(vp) : zero;
        vr[s][1] = some && ch + HC < Dv ? *reinterpret_cast<const int4v_*>(vp + HC) : zero;
      }
    }
    if (base + nw * KB < last) lookup(base + nw * KB);
    float sc[RC][NS];
#pragma unroll
    for (int s = 0; s < NS; ++s) {
      float kf[CH];
      RowLane<T>::unpack(kr[s][0], kf);
      RowLane<T>::unpack(kr[s][1], kf + HC);
#pragma unroll
      for (int r = 0; r < RC; ++r) {
        float d = 0.0f;
#pragma unroll
        for (int c = 0; c < CH; ++c) d += qf[r][c] * kf[c];
        sc[r][s] = d;
      }
    }
#define ROW_REDUCE(STAGE, EXPR)                        \
  if (lane_shift > STAGE) {                            \
    _Pragma("unroll") for (int r = 0; r < RC; ++r)     \
        _Pragma("unroll") for (int s = 0; s < NS; ++s) { const float v = sc[r][s]; sc[r][s] = EXPR; } \
  }
    ROW_REDUCE(0, dpp_add<0xB1>(v))           // lane xor 1
    ROW_REDUCE(1, dpp_add<0x4E>(v))           // lane xor 2
    ROW_REDUCE(2, dpp_add<0x141>(v))          // the other half of 8 lanes
    ROW_REDUCE(3, dpp_add<0x140>(v))          // the other half of 16 lanes
    ROW_REDUCE(4, v + __shfl_xor(v, 16))
    ROW_REDUCE(5, v + __shfl_xor(v, 32))
#undef ROW_REDUCE
#pragma unroll
    for (int r = 0; r < RC; ++r) {
      float top = m[r];
#pragma unroll
      for (int s = 0; s < NS; ++s) sc[r][s] *= fac[s];
      if (softcap > 0.0f) Dom<T>::cap_(sc[r], cap, inv_cap);
#pragma unroll
      for (int s = 0; s < NS; ++s) {
        float v = sc[r][s];
        v -= slope[r] * (float)(pos - key_of(base + s * KPS + group));
        sc[r][s] = base + s * KPS + group < last ? v : -INFINITY;
        top = fmaxf(top, sc[r][s]);
      }
      const float ref = top == -INFINITY ? 0.0f : top;   // no key in this lane group yet
      const float corr = Dom<T>::exp_(m[r] - ref);
      m[r] = top;
      float sum = 0.0f;
#pragma unroll
      for (int s = 0; s < NS; ++s) {
        sc[r][s] = Dom<T>::exp_(sc[r][s] - ref);
        sum += sc[r][s];
      }
      l[r] = l[r] * corr + sum;
#pragma unroll
      for (int c = 0; c < CH; ++c) acc[r][c] *= corr;
    }
#pragma unroll
    for (int s = 0; s < NS; ++s) {
      // keep the packed registers, not 2 CH floats per step, alive since the scores: unpack anew
      if constexpr (!SEP) asm volatile("" : "+v"(kr[s][0]), "+v"(kr[s][1]));
      float vf[CH];
      RowLane<T>::unpack(SEP ? vr[SEP ? s : 0][0] : kr[s][0], vf);
      RowLane<T>::unpack(SEP ? vr[SEP ? s : 0][1] : kr[s][1], vf + HC);
#pragma unroll
      for (int r = 0; r < RC; ++r)
#pragma unroll
        for (int c = 0; c < CH; ++c) acc[r][c] += sc[r][s] * vf[c];
    }
  }
  // The lane groups' states meet. Up to 8 lanes a row, the groups are spread over the three upper bits of the lane
  // number: each of these levels halves the channels a lane goes on with, so that 14 sums do instead of 48.
  const int PS = 2 + Dv;
#pragma unroll
  for (int r = 0; r < RC; ++r) {
    float top = m[r];
    for (int off = L; off < 64; off <<= 1) top = fmaxf(top, __shfl_xor(top, off));
    const float f = m[r] == -INFINITY ? 0.0f : Dom<T>::exp_(m[r] - top);
    float ll = l[r] * f;
    for (int off = L; off < 64; off <<= 1) ll += __shfl_xor(ll, off);
#pragma unroll
    for (int c = 0; c < CH; ++c) acc[r][c] *= f;
    float* mine = part + (wid * RC + r) * PS;
    if (lane == 0) { mine[0] = top; mine[1] = ll; }
    if (L <= 8) {
      float a8[CH / 2], a4[CH / 4], a2[CH / 8];
#pragma unroll
      for (int c = 0; c < CH / 2; ++c) a8[c] = swap32_add(acc[r][c], acc[r][c + CH / 2]);
#pragma unroll
      for (int c = 0; c < CH / 4; ++c) a4[c] = swap16_add(a8[c], a8[c + CH / 4]);
      const bool up = (lane & 8) != 0;
#pragma unroll
      for (int c = 0; c < CH / 8; ++c) {
        const float keep = up ? a4[c + CH / 8] : a4[c], give = up ? a4[c] : a4[c + CH / 8];
        a2[c] = keep + __shfl_xor(give, 8);
      }
      for (int off = L; off < 8; off <<= 1) {
#pragma unroll
        for (int c = 0; c < CH / 8; ++c) a2[c] += __shfl_xor(a2[c], off);
      }
      if ((lane & 7) < L) {
        const int at = ch + (lane >> 5) * (CH / 2) + (lane >> 4 & 1) * (CH / 4) + (lane >> 3 & 1) * (CH / 8);
#pragma unroll
        for (int c = 0; c < CH / 8; ++c)
          if (at + c < Dv) mine[2 + at + c] = a2[c];
      }
    } else {
      for (int off = L; off < 64; off <<= 1) {
#pragma unroll
        for (int c = 0; c < CH; ++c) acc[r][c] += __shfl_xor(acc[r][c], off);
      }
      if (group == 0) {
#pragma unroll
        for (int c = 0; c < CH; ++c)
          if (ch + c < Dv) mine[2 + ch + c] = acc[r][c];
      }
    }
  }
  __syncthreads();
  if (wid < nh) {  // wave r: what each wave's partial state counts in head r
    const int r = wid;
    const float mw = lane < nw ? part[(lane * RC + r) * PS] : -INFINITY;
    const float lw = lane < nw ? part[(lane * RC + r) * PS + 1] : 0.0f;
    float top = wave_reduce_max(mw);
    if (splits > 1) {  // this block's state for row_merge_kernel; a part without keys has a maximum of -inf
      const float f = mw == -INFINITY ? 0.0f : Dom<T>::exp_(mw - top);
      const float ll = wave_reduce_sum(lw * f);
      if (lane < nw) coef[r * ROW_WAVES + lane] = f;
      if (lane == 0) {
        float* state = ws + ((n * H + h0 + r) * splits + split) * (long)(2 + Dv);
        state[0] = top;
        state[1] = ll;
      }
    } else {
      if (sink_logits != nullptr) top = fmaxf(top, sink_logits[h0 + r] * Dom<T>::UNIT);
      const float f = mw == -INFINITY ? 0.0f : Dom<T>::exp_(mw - top);
      float ll = wave_reduce_sum(lw * f);
      if (sink_logits != nullptr) ll += Dom<T>::exp_(sink_logits[h0 + r] * Dom<T>::UNIT - top);
      else if (sink) ll += Dom<T>::exp_(-top);   // the sink's score is 0
      float c = f / ll;
      if (gate != nullptr) c *= sigmoidf_(ldf(gate + n * gate_stride + h0 + r));
      if (lane < nw) coef[r * ROW_WAVES + lane] = c;
    }
  }
  __syncthreads();
  for (int i = threadIdx.x; i < nh * Dv; i += blockDim.x) {
    const int r = i / Dv, dv = i % Dv;
    float o = 0.0f;
#pragma unroll 4
    for (int w = 0; w < nw; ++w) o += coef[r * ROW_WAVES + w] * part[(w * RC + r) * PS + 2 + dv];
    const long at = (n * H + h0 + r) * (long)Dv + dv;
    if (splits > 1) ws[((n * H + h0 + r) * splits + split) * (long)(2 + Dv) + 2 + dv] = o;
    else if (out32 != nullptr) out32[at] = o;
    else stf(out + at, o);
  }
}

// The states of a (token, head)'s parts [splits][2 + Dv] -> its output: one wave per (token, head), the parts' weights
// lane by lane, then channels.
template <typename T>
__global__ __launch_bounds__(256) void row_merge_kernel(
    T* __restrict__ out, float* __restrict__ out32, const float* __restrict__ ws, const T* __restrict__ gate, long gate_stride,
    const float* __restrict__ sink_logits, long rows, int H, int Dv, int sink, int splits) {
  const long row = (long)blockIdx.x * 4 + (threadIdx.x >> 6);
  const int lane = threadIdx.x & 63;
  if (row >= rows) return;
  const float* state = ws + row * splits * (long)(2 + Dv);
  const int h = (int)(row % H);
  const float m = lane < splits ? state[lane * (long)(2 + Dv)] : -INFINITY;   // splits <= MAX_PARTS
  const float l = lane < splits ? state[lane * (long)(2 + Dv) + 1] : 0.0f;
  float top = wave_reduce_max(m);
  if (sink_logits != nullptr) top = fmaxf(top, sink_logits[h] * Dom<T>::UNIT);
  const float f = m == -INFINITY ? 0.0f : Dom<T>::exp_(m - top);
  float ll = wave_reduce_sum(l * f);
  if (sink_logits != nullptr) ll += Dom<T>::exp_(sink_logits[h] * Dom<T>::UNIT - top);
  else if (sink) ll += Dom<T>::exp_(-top);   // the sink's score is 0
  float c = f / ll;
  if (gate != nullptr) c *= sigmoidf_(ldf(gate + row / H * gate_stride + h));
  // eight parts' loads at a time: one by one, 16 parts took 7.3 us
  for (int dv = lane; dv < Dv; dv += 64) {
    float o = 0.0f;
    for (int p0 = 0; p0 < splits; p0 += 8) {
      float v[8];
#pragma unroll
      for (int e = 0; e < 8; ++e) v[e] = state[min(p0 + e, splits - 1) * (long)(2 + Dv) + 2 + dv];
#pragma unroll
      for (int e = 0; e < 8; ++e)
        if (p0 + e < splits)
          o += __builtin_bit_cast(float, __builtin_amdgcn_readlane(__builtin_bit_cast(int, c), p0 + e)) * v[e];
    }
    if (out32 != nullptr) out32[row * (long)Dv + dv] = o;
    else stf(out + row * (long)Dv + dv, o);
  }
}

static void launch_row_merge(at::Tensor& out, const at::Tensor& q, const at::Tensor& ws, const c10::optional<at::Tensor>& gate,
                             long gate_stride, const ScalarExtras& x, int Dv, bool sink, int splits) {
  const long rows = q.size(0) * q.size(1);
  TORCH_CHECK(splits <= MAX_PARTS, "more parts of the keys than the merge takes");
  SERVING_DISPATCH_ACT(q, T, {
    hipLaunchKernelGGL((row_merge_kernel<T>), dim3((unsigned)((rows + 3) / 4)), dim3(256), 0, stream(),
                       x.out32 != nullptr ? (T*)nullptr : ptr<T>(out), x.out32, ws.data_ptr<float>(),
                       gate.has_value() ? ptr<T>(*gate) : (const T*)nullptr, gate_stride, x.sink_logits, rows, (int)q.size(1), Dv,
                       sink ? 1 : 0, splits);
  });
  HIP_CHECK_LAST();
}

bool launch_row_attention(at::Tensor& out, const at::Tensor& q, const at::Tensor& kpool, const at::Tensor& vpool,
                          const at::Tensor& block_tables, const at::Tensor& tok_seq, const at::Tensor& positions,
                          const float* slopes, const c10::optional<at::Tensor>& gate, long gate_stride, double scale,
                          int64_t window, int64_t keep_first, double softcap, bool sink, int page_shift, long vrow,
                          long vhead, const ScalarExtras& x) {
  const long N = q.size(0);
  const int H = (int)q.size(1), D = (int)q.size(2), G = (int)kpool.size(2), Dv = (int)vpool.size(3);
  if (x.dist_bias != nullptr || x.ksum != nullptr || x.cross_out != nullptr) return false;
  const int elem = is_bf16(q) ? 2 : 4, piece = 16 / elem, CH = 2 * piece;
  auto al16 = [](const void* p) { return reinterpret_cast<uintptr_t>(p) % 16 == 0; };
  if (D % piece != 0 || !al16(kpool.data_ptr()) || D > 64 * CH || Dv > 64 * CH) return false;
  const bool shared = vpool.data_ptr() == kpool.data_ptr() && vrow == (long)G * D && (G == 1 || vhead == D) && Dv <= D &&
                      x.vrep == 1;
  if (!shared && (Dv % piece != 0 || vrow % piece != 0 || vhead % piece != 0 || !al16(vpool.data_ptr()))) return false;
  int lane_shift = 0;
  while ((CH << lane_shift) < (D > Dv ? D : Dv)) ++lane_shift;
  const int R = H / G;
  // Most keys a token of this call can see: what its page table, window or block of positions holds.
  long keys = block_tables.size(1) << page_shift;
  if (window > 0) keys = std::min<long>(keys, window + keep_first);
  if (x.chunk > 0) keys = std::min<long>(keys, x.chunk);
  // Query heads per block and parts of the keys. Heads that share a block share its reads; heads in blocks of
  // their own meet in L2 and cost less per key, which wins while the chip is not full and the context is short (16
  // sequences of 1024 keys, 16/4 heads of 128: 18.9 us with one head a block, 19.7 with two and two parts; 4 x 16384: 53.9
  // against 44.0; 16 x 6000, 32/8 heads: 221 against 113; four heads do not fit into the registers: 166).
  // Then the keys are cut into parts while there are fewer blocks than CUs and a part still gives every wave a key
  // block: 4 x 16384 210 -> 44 us, 8 x 2048 26.6 -> 19.1, 1 x 4096 36 -> 18. More blocks than CUs are slower again (4 x 16384
  // with 512 blocks 76 us): a block costs about 10 us by itself. (All repeated on the same keys.) One or two blocks stop at the parts that the merge takes.
  int rc = R > 1 && (N * G * ((R + 1) / 2) >= 256 || keys >= 8192) ? 2 : 1;
  int splits = 1;
  const long blocks = N * G * ((R + rc - 1) / rc);
  const long pass = (long)ROW_WAVES * (rc == 1 || shared ? 8 : 4) * (64 >> lane_shift);   // keys of one key block of every wave
  while (blocks * splits * 2 <= 256 && keys > splits * pass && splits < MAX_PARTS) splits *= 2;
  auto lds_bytes = [&](int nw) { return (size_t)(rc * ROW_WAVES + nw * rc * (2 + Dv)) * sizeof(float); };
  int nwaves = ROW_WAVES;
  while (lds_bytes(nwaves) > 64 * 1024 && nwaves > 4) nwaves >>= 1;
  while (lds_bytes(nwaves) > 64 * 1024 && rc > 1) rc >>= 1;
  if (lds_bytes(nwaves) > 64 * 1024) return false;
  const int chunks = (R + rc - 1) / rc;
  at::Tensor ws;
  if (splits > 1) ws = at::empty({N * H * splits * (2 + Dv)}, q.options().dtype(at::kFloat));
  const int qvec = al16(q.data_ptr()) && q.stride(0) % piece == 0 ? 1 : 0;
#define ROW_LAUNCH(RC_, NS_, SEP_)                                                                                     \
  hipLaunchKernelGGL((row_attention_kernel<T, RC_, NS_, SEP_>), dim3((unsigned)(N * G * chunks * splits)), dim3(64 * nwaves), \
                     lds_bytes(nwaves), stream(), x.out32 != nullptr ? (T*)nullptr : ptr<T>(out), x.out32, ptr<T>(q),   \
                     (long)q.stride(0), ptr<T>(kpool), ptr<T>(vpool), block_tables.data_ptr<int>(),                     \
                     (int)block_tables.stride(0), tok_seq.data_ptr<int>(), positions.data_ptr<int>(), slopes,           \
                     gate.has_value() ? ptr<T>(*gate) : (const T*)nullptr, gate_stride, x.sink_logits, x.key_fac, H, G, \
                     D, Dv, page_shift, (float)(scale * Dom<T>::NAT), (int)window, (int)keep_first, x.chunk, (float)softcap, \
                     sink ? 1 : 0, x.vrep, vrow, vhead, lane_shift, qvec, splits,                                       \
                     splits > 1 ? ws.data_ptr<float>() : (float*)nullptr)
  SERVING_DISPATCH_ACT(q, T, {
    if (shared) {
      if (rc == 1) ROW_LAUNCH(1, 8, false);
      else ROW_LAUNCH(2, 8, false);
    } else {
      if (rc == 1) ROW_LAUNCH(1, 8, true);
      else ROW_LAUNCH(2, 4, true);
    }
  });
#undef ROW_LAUNCH
  HIP_CHECK_LAST();
  if (splits > 1) launch_row_merge(out, q, ws, gate, gate_stride, x, Dv, sink, splits);
  return true;
}

}  // namespace serving
}  // namespace cai
