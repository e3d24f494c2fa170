// Flash attention forward + backward for gfx950 (CDNA4), bf16, causal, GQA.
//
// MI355X-native design (not a CUDA port):
//  - mfma_f32_32x32x16_bf16 tiles; 64-wide waves; a wave owns 32 query rows (forward,
//    dQ) or 32 key/value rows (dK/dV); blocks of 4 waves, 2 for small forward grids.
//  - ALL operand tiles live in LDS in ONE layout, pieces of 16 rows of 32 channels (piece_at below), which global loads
//    write directly. Row-slice fragment reads (8 consecutive d at a fixed row) are
//    single 16 B loads; COLUMN fragment reads use gfx950's ds_read_b64_tr_b16.
//    HW-verified semantics (mfma_selftest.hip): each lane reads 64 bits at its own
//    address; within a 16-lane group, out[l][j] = pool[(l&15) + 16 j] where pool is
//    the group's reads in lane order. With lane addressing row=(m>>2), channels (m&3)*4
//    this delivers tile[row0+j][col m] per lane — a free 4x16 transpose.
//  - No intermediate passes through LDS: every product whose operand is a result (P · V,
//    P^T · dO, dS^T · Q, dS · K) is arranged so that the contracted index lies in a lane's
//    registers, and takes them in the order of the C layout (frag_born).
//  - The next tile's loads are spread over the current tile's products; two LDS
//    buffers, one barrier a tile.
//  - What differs from wave to wave but not inside one (masks on the diagonal, the last tile) is a scalar branch
//    with a body of its own; masks merged into the common body were half of its vector instructions.
//  - backward: delta preprocess, then ONE launch whose blocks take key/value tiles (dK/dV)
//    or query tiles (dQ); both form the scores again.
//
// What bounds it (B1 S8192 H32/8 D128 causal): with loads through registers and a maximum per tile, a tile took a wave 4034
// cycles, of which 557 went into issuing the loads, 638 into storing them, 150 into the barrier; the products and the
// softmax, 890 cycles each, overlapped little between the two waves of a SIMD, since it issues one instruction of all its waves
// at a time: 11 cycles for a product, 4 to 5 for a vector instruction, 8 for an exponential. The forward therefore places
// a half tile's exponentials between the products of its neighbours. A full chip is held by power then (1.9 GHz under this load);
// the backward has no registers for the same. Fragments read further ahead for P · V and other wave
// priorities (a fixed order of a SIMD's two waves) changed nothing.
//
// TFLOP/s, forward 2 products / backward 5 products of the visible pairs, loads through registers -> into LDS directly:
//   B4 S4096 H32 D128 causal          forward 768 -> 930, backward 599 -> 693
//   B1 S8192 H32/8 D128 causal        forward 888 -> 1040, backward 659 -> 761
//   B2 S4096 H16/8 D128               forward 928 -> 1072, backward 699 -> 807
//   B8 S1024 H12 D64 causal           forward 348 -> 424, backward 328 -> 395
//   B16 S512 H12 D64                  forward 524 -> 582, backward 430 -> 501
//   packed, 14 sequences of 256..4096, 32/8 heads   forward 608 -> 810, backward 535 -> 632
// and the forward with products and weights in turns, us (another card):
//   B4 S4096 H32/8 D128 causal 570 -> 550, B1 S8192 H32/8 514 -> 500, H4 159 -> 128 (half the chip); B8 S1024 H12 D64 32.0 -> 31.2,
//   packed, 16384 tokens of up to 4096, 32/8 of 128 384 -> 367, 12 of 64 102 -> 95, 8192 of up to 2048, 32/8 113 -> 103;
//   B1 S4096 H8/2 D64 unmasked 56.9 -> 53.3
// and with a quarter of its instructions taken out, waits and scalar ones (a step of 64 keys 380 -> 273; they were 25 % of what a SIMD issues), us:
//   B1 S8192 H4/1 D128 causal 126 -> 116, H12 D64 167 -> 162; B1 S2048 H12 D64 27.1 -> 24.8; B1 S4096 H8/2 D64 54 -> 50; B4 S4096 H32 D128 582 -> 572,
//   H32/8 at a full chip the same: power. Slower there: products of 16 x 16 x 32 (542 for 532, H4/1 148 for 127: more instructions), 64 rows a wave (610).
//
// Shapes: q [B,S,Hq,D], k/v [B,S,Hkv,D] ("bshd" — no transposes in the
// model), D in {64,128}. lse/delta are [B,Hq,S] fp32.
// Reference behavioral equivalent: flash-attn 2 package as consumed by
// colossalai/shardformer/layer/attn.py (ColoAttention).

#include <torch/extension.h>
#include <ATen/hip/HIPContext.h>

#include <algorithm>
#include <climits>
#include <type_traits>

#include "lds_tiles.h"

namespace cai {

typedef bf16x8_v bf16x8_t;

namespace fa {

constexpr int KVB = 64;     // kv rows per tile
constexpr int QW = 32;      // q rows per wave (fwd / dq); kv rows per wave (dkdv)
constexpr int NWB = 4;     // waves of a backward block
constexpr int NTB = 256;

DEV_INLINE bf16x8_t ld_g16(const unsigned short* p) {
  return *reinterpret_cast<const bf16x8_t*>(p);
}

// C-layout row for mfma_f32_32x32x16 register j (guide §3, HW-verified).
DEV_INLINE constexpr int crow(int j, int half) { return (j & 3) + 8 * (j >> 2) + 4 * half; }

// Whether a head's blocks of a causal packed batch that they do not look up (packed_tile) go by tile, late ones of all sequences first, and not sequence by sequence.
// Short sequences leave many tiles empty and end unevenly; keys and values of long ones, and of heads that share none, are
// met in L2 by the tiles that run together. By sequence / by tile, us, forward and backward: 186 sequences of up to 256 tokens, 16/4
// heads of 64: 48 / 39, 151 / 141; 54 of 900, 8/2 of 128: 58 / 49, 210 / 200; 46 of 1024, 32/8: 193 / 179, 534 / 531 (41: 188 / 185,
// 541 / 554); but 14 of 4096: 406 / 437, 1108 / 1147; 81 of 600, 12 heads of 64: 39 / 45, 110 / 116; 20 of 300, 8 heads: 9.3 / 10.4.
__host__ __device__ __forceinline__ bool by_tile(int tiles, long blocks, int group) { return tiles <= 8 && blocks > 512 && group > 1; }

// XCDs that share a row of tiles, so that all of them get as much: 1, 2, 4 or 8
__host__ __device__ __forceinline__ int row_parts(int n_y) { return n_y % 8 == 0 ? 1 : n_y % 4 == 0 ? 2 : n_y % 2 == 0 ? 4 : 8; }
// Blocks that deal() takes for n_y rows of n_x tiles: whole rounds of the XCDs
__host__ __device__ __forceinline__ long dealt_blocks(long n_x, int n_y) {
  const int parts = row_parts(n_y);
  return (n_x + parts - 1) / parts * parts * n_y;
}
// Tile x and row y of block f, false if it has none; x goes from a row's longest tile to its shortest. An XCD (f % 8) has whole rows, or every
// second, fourth or eighth tile of them, and takes W rows at a time, tile by tile, so that it ends with short tiles of many rows. With `pairs` the
// blocks are all there are: where two share a CU (32 on an XCD) they are a long one and a short one.
DEV_INLINE bool deal(int f, int n_x, int n_y, int W, bool pairs, int& x, int& y) {
  const int parts = row_parts(n_y), rows = n_y * parts / 8, tiles = (n_x + parts - 1) / parts, all = rows * tiles;
  int i = f >> 3;
  if (i >= all) return false;
  if (pairs && all <= 64) {   // all of its rows, whatever its L2 holds: in fours a long tile of the last rows met another one (B2 S4500 H5 D128 92 us for 80)
    W = rows;
    if (i >= 32) i = all - 1 - (i - 32);
  }
  const int first = i / (W * tiles) * W, wide = min(W, rows - first);
  i -= first * tiles;
  const int row = (f & 7) * rows + first + i % wide;
  x = i / wide * parts + row % parts;
  y = row / parts;
  return x < n_x;
}

// Tile i of a packed batch of up to MOST_PACKED sequences of at most `most` tiles of `rows` rows, those of more tiles first; false past the last one. Every
// lane has four sequences; how many tiles those of at least c tiles have is a sum over the lanes, and the c of tile i found by halving.
constexpr int MOST_PACKED = 256;
DEV_INLINE bool packed_tile(const int* __restrict__ CU, int B, int rows, int most, int i, int& b, int& tile, int& tiles) {
  const int lane = threadIdx.x & 63;
  int own[MOST_PACKED / 64];
#pragma unroll
  for (int k = 0; k < MOST_PACKED / 64; ++k) {
    const int at = 64 * k + lane;
    own[k] = 64 * k < B && at < B ? min((CU[at + 1] - CU[at] + rows - 1) / rows, most) : 0;
  }
  auto at_least = [&](int c) {
    int v = own[0] >= c ? own[0] : 0;
#pragma unroll
    for (int k = 1; k < MOST_PACKED / 64; ++k)
      if (64 * k < B) v += own[k] >= c ? own[k] : 0;
    // summed inside rows of 16 lanes, then over the rows
    v += __builtin_amdgcn_update_dpp(0, v, 0x111, 0xf, 0xf, false);
    v += __builtin_amdgcn_update_dpp(0, v, 0x112, 0xf, 0xf, false);
    v += __builtin_amdgcn_update_dpp(0, v, 0x114, 0xf, 0xf, false);
    v += __builtin_amdgcn_update_dpp(0, v, 0x118, 0xf, 0xf, false);
    v += __builtin_amdgcn_update_dpp(0, v, 0x142, 0xa, 0xf, false);
    v += __builtin_amdgcn_update_dpp(0, v, 0x143, 0xc, 0xf, false);
    return __builtin_amdgcn_readlane(v, 63);
  };
  int ahead = 0, hi = most + 1;   // at_least(tiles) > i >= at_least(hi) = ahead
  tiles = 1;
  if (at_least(1) <= i) return false;
  while (hi - tiles > 1) {
    const int mid = (tiles + hi) >> 1, n = at_least(mid);
    if (n > i) {
      tiles = mid;
    } else {
      hi = mid;
      ahead = n;
    }
  }
  int nth = (i - ahead) / tiles;   // of the sequences of as many tiles
  tile = i - ahead - nth * tiles;
#pragma unroll
  for (int k = 0; k < MOST_PACKED / 64; ++k) {
    const unsigned long long same = __ballot(own[k] == tiles);
    const int here = __builtin_popcountll(same);
    if (nth >= 0 && nth < here) {
      const int order = __builtin_amdgcn_mbcnt_hi((unsigned)(same >> 32), __builtin_amdgcn_mbcnt_lo((unsigned)same, 0));
      b = 64 * k + __builtin_ctzll(__ballot(own[k] == tiles && order == nth));
    }
    nth -= here;
  }
  return true;
}

// Sequence and head of row y of a dense batch: sequence by sequence, or with lengths and more than a tile (the forward: two) `by_head`, key head by key head over all
// sequences, so that no XCD has only long ones. Tiles of one row take about as long whatever their length, and neighbours in memory are read together (forward, us, by
// sequence and by head: B32 S128 H12 D64 9.3, 9.8; B16 S256 H12 10.1, 10.9, but B24 S256 H16/4 D128 24.6, 22.6). With lengths that differ little both take the same. us, forward and backward, lengths between a quarter and all: B16 S512 H12 D64 20.6 and 55.4 -> 18.8 and 52.9; B8 S2048 H12 D64 103 and 292 ->
// 90 and 231; B4 S4096 H8 D64 147 and 425 -> 100 and 261; causal, D128: B8 S2048 H32/8 244 and 760 -> 212 and 595, B2 S4096 H16/4 136 and 451 -> 118 and 366.
DEV_INLINE void row_of_batch(int y, int B, int H, int group, bool by_head, int& b, int& h) {
  if (by_head) {
    const int k = y / group;
    b = k % B;
    h = k / B * group + y % group;
  } else {
    b = y / H;
    h = y % H;
  }
}

// Which (q tile, sequence, head) a block of the forward works on, false if on none. Blocks of one (sequence, head) share an
// XCD's L2. Packed batches run head by head, each head over all sequences: the other way round
// the longest sequence is one XCD's work (10 sequences of 256..4096 tokens: 1488 against 463 us). Under a causal
// mask the late tiles see the most keys: they start first. Up to 512 blocks run at once, two on a CU: every second head of a dense batch goes the other way, so that the
// two are a long one and a short one. `dealt`: tiles of a row that deal() takes, of the packed batch or of a causal sequence.
template <bool VARLEN>
DEV_INLINE bool q_block(const int* __restrict__ CU, int rows, int B, int Hq, int group, int causal, int W, int dealt, int most, bool by_head, int& tile, int& b, int& h) {
  int y;
  if (dealt) {
    if (!deal((int)(blockIdx.y * gridDim.x + blockIdx.x), dealt, (VARLEN ? 1 : B) * Hq, W, true, tile, y)) return false;
    h = y;
    if (!VARLEN) row_of_batch(y, B, Hq, group, by_head, b, h);
    int tiles = dealt;
    if (VARLEN && !packed_tile(CU, B, rows, most, tile, b, tile, tiles)) return false;
    if (causal) tile = tiles - 1 - tile;
    return true;
  }
  xcd_swizzle_xy(tile, y);
  b = y % B;
  h = y / B;
  if (!VARLEN) row_of_batch(y, B, Hq, group, by_head, b, h);
  if (VARLEN && causal && by_tile((int)gridDim.x, (long)gridDim.x * gridDim.y, group)) {
    const int i = b * (int)gridDim.x + tile;
    tile = (int)gridDim.x - 1 - i / B;
    b = i % B;
  } else if (causal && (VARLEN || !(y & 1) || (int)(gridDim.x * gridDim.y) > 512)) {
    tile = (int)gridDim.x - 1 - tile;
  }
  return true;
}

// Logical index of block f of nblocks so that every XCD (block f runs on XCD f % 8) gets a contiguous range.
DEV_INLINE int xcd_chunk(int f, int nblocks) {
  const int q = nblocks >> 3, r = nblocks & 7, xcd = f & 7;
  return (xcd < r ? xcd * (q + 1) : r * (q + 1) + (xcd - r) * q) + (f >> 3);
}

// A tile's way from memory into LDS, without registers in between: a wave brings PER pieces, each with one load
// instruction, which is issued wherever the caller wants it between the products of the tile before. (All of a tile's loads
// issued together held the waves up for 557 of the 4034 cycles a tile took, at 64 bytes a cycle of address and cache
// work, and its LDS stores, which met in the banks, for another 638: B1 S8192 H32/8 D128 causal.)
// Rows past the matrix' end come as zeros: the buffer descriptor of a tile ends with its last row, and is made
// anew for each tile, so that a matrix may be of any size; rows less than 2^23 elements apart (offsets stay under 2^31).
template <int D, int ROWS, int WAVES>
struct TileLoad {
  static constexpr int RG = ROWS / 16, PIECES = RG * (D / 32), PER = PIECES / WAVES;
  static_assert(PIECES % WAVES == 0, "TileLoad: uneven pieces");
  const unsigned short* base;
  long stride;
  int rows;            // of the matrix
  unsigned off;        // bytes from a piece's first element to this lane's

  DEV_INLINE TileLoad(const unsigned short* base, long stride, int rows) : base(base), stride(stride), rows(rows) {
    const int r = (threadIdx.x & 63) >> 2, unit = (threadIdx.x & 3) ^ (r >> 2 & 3);
    off = (unsigned)(r * stride) * 2u + unit * 16;
  }
  // what the loads of the tile from row0 on share
  DEV_INLINE __amdgpu_buffer_rsrc_t tile(int row0) const {
    const int left = min(rows - row0, ROWS);
    const unsigned bytes = left > 0 ? (unsigned)((left - 1) * stride + D) * 2u : 0u;
    return __builtin_amdgcn_make_buffer_rsrc(const_cast<unsigned short*>(base + (left > 0 ? row0 * stride : 0)), 0, (int)bytes, 0x00027000);
  }
  // piece i (of PER) of wave w
  DEV_INLINE void piece(__amdgpu_buffer_rsrc_t t, char* __restrict__ lds, int w, int i) const {
    const int c = w + WAVES * i, rg = c % RG, cg = c / RG;
    __builtin_amdgcn_raw_ptr_buffer_load_lds(t, (lds_ptr)(lds + c * 1024), 16, (int)off, (int)(unsigned)((rg * 16 * stride + cg * 32) * 2), 0, 0);
  }
  DEV_INLINE void all(int row0, char* __restrict__ lds, int w) const {
    const auto t = tile(row0);
#pragma unroll
    for (int i = 0; i < PER; ++i) piece(t, lds, w, i);
  }
};

// A matrix' tiles one after the other, through a descriptor that is advanced instead of formed anew (six scalar instructions for some 20).
template <int D, int ROWS, int WAVES>
struct TileStream : TileLoad<D, ROWS, WAVES> {
  typedef TileLoad<D, ROWS, WAVES> Base;
  const unsigned short* at;    // of the next tile
  int left, whole, last;       // rows from there on; bytes of a tile, of the last one
  __amdgpu_buffer_rsrc_t now;
  DEV_INLINE TileStream(const unsigned short* base, long stride, int rows) : Base(base, stride, rows), at(base), left(rows) {
    whole = (int)((unsigned)((ROWS - 1) * stride + D) * 2u);
    last = (int)((unsigned)(((max(rows, 1) - 1) % ROWS) * stride + D) * 2u);
  }
  DEV_INLINE void skip(int tiles) {
    at += tiles * ROWS * Base::stride;
    left -= tiles * ROWS;
  }
  DEV_INLINE void next(bool all) {
    now = __builtin_amdgcn_make_buffer_rsrc(const_cast<unsigned short*>(at), 0, all ? whole : last, 0x00027000);
    at += ROWS * Base::stride;
  }
  DEV_INLINE void next() {
    now = __builtin_amdgcn_make_buffer_rsrc(const_cast<unsigned short*>(at), 0, left > ROWS ? whole : left > 0 ? last : 0, 0x00027000);
    skip(1);
  }
  DEV_INLINE void piece(char* __restrict__ lds, int w, int i) const { Base::piece(now, lds, w, i); }
};

}  // namespace fa

// ============================================================ forward kernel
//
// grid: (ceil(S / (32 NW)), B*Hq). LDS: two key and two value tiles.
//
// Mask generality (reference: colossalai/shardformer/layer/attn.py:139
// prepare_attn_kwargs CAUSAL / PADDED / PADDED_CAUSAL + varlen):
//  - VARLEN=false, CU=nullptr: dense [B,S,H,D].
//  - VARLEN=false, CU=seqlens[B]: right-padded batches; rows/cols beyond
//    seqlens[b] are masked; O=0 and LSE=-inf are written for pad rows so
//    the backward masks them via the existing lse==-inf guard.
//  - VARLEN=true, CU=cu_seqlens[n+1]: packed ragged batch [total,H,D]
//    passed with S=total and grid.y = n_seq*Hq; sequence b spans tokens
//    [CU[b], CU[b+1]); LSE/delta are [Hq, total].
//  - CUK (padded path only): SEPARATE kv-side valid counts — ring-attention
//    pieces where the q chunk and the arriving kv chunk cover different
//    parts of each padded sequence. null -> kv counts = CU.
// DEAL: whether `dealt` is looked at; with it in every kernel unmasked and small calls began 0.1 to 0.5 us later (B16 S200 H16 D64 11.0 -> 10.5 us, B32 S128
// H12 8.7 -> 8.5, B4 S1024 H8 D128 25.2 -> 24.2).
template <int D, int NW, bool VARLEN, bool DEAL>
__global__ __launch_bounds__(NW * 64, 2) void fa_fwd_kernel(
    const unsigned short* __restrict__ Q,
    const unsigned short* __restrict__ K,
    const unsigned short* __restrict__ V,
    unsigned short* __restrict__ O,
    float* __restrict__ LSE,
    const int* __restrict__ CU,
    const int* __restrict__ CUK,
    long qbs, long qts, long kbs, long kts,
    int B, int S, int Sk, int Hq, int Hkv, float scale, int causal, int W, int dealt, int most) {
  using namespace fa;
  extern __shared__ char smem[];
  constexpr int NT = NW * 64;
  constexpr int KB_BYTES = tile_bytes<KVB, D>();
  const int lane = threadIdx.x & 63;
  const int w = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);   // the same for a wave: what it decides is a scalar branch
  const int half = lane >> 5;
  const int ln = lane & 31;

  int tile, b, h;
  if (!q_block<VARLEN>(CU, NW * QW, B, Hq, Hq / Hkv, causal, W, DEAL ? dealt : 0, most, CU != nullptr && S > 2 * NWB * QW, tile, b, h)) return;
  const int hk = h / (Hq / Hkv);
  const int q0 = tile * (NW * QW);
  const int qw = q0 + w * QW;  // this wave's first q row

  long seq0 = 0;
  int Seff = S;
  if (VARLEN) {
    seq0 = CU[b];
    Seff = CU[b + 1] - (int)seq0;
    if (q0 >= Seff) return;
  } else if (CU != nullptr) {
    Seff = CU[b];
  }
  // kv extent: its own tensor length Sk (ring blocks where kv covers a
  // DIFFERENT — possibly longer — span than q), clipped by per-batch valid
  // counts: CUK when given, else CU only in the symmetric padded case
  int SeffK = VARLEN ? Seff
            : (CUK != nullptr ? CUK[b] : (CU != nullptr ? min(CU[b], Sk) : Sk));

  const unsigned short* q_base = VARLEN ? Q + seq0 * qts + (long)h * D : Q + (long)b * qbs + (long)h * D;
  const unsigned short* k_base = VARLEN ? K + seq0 * kts + (long)hk * D : K + (long)b * kbs + (long)hk * D;
  const unsigned short* v_base = VARLEN ? V + seq0 * kts + (long)hk * D : V + (long)b * kbs + (long)hk * D;
  const long o_stride = (long)Hq * D;  // O/LSE are always packed

  constexpr int DSL = D / 16;  // MFMA K-slices over the head dim

  // ---- Q fragments (B-operand of S^T = K·Q^T): lane holds q-col (ln),
  //      d-rows half*8+[0..7] per 16-d slice — one 16 B load per slice.
  // A negative scale moves into Q as an exact sign flip, so that the largest
  // product of a row is its largest score.
  const int q_my = max(min(qw + ln, Seff - 1), 0);
  bf16x8_t qf[DSL];
  {
    const unsigned short* qp = q_base + (long)q_my * qts + half * 8;
#pragma unroll
    for (int sl = 0; sl < DSL; ++sl) qf[sl] = ld_g16(qp + sl * 16);
    if (scale < 0.0f) {
#pragma unroll
      for (int sl = 0; sl < DSL; ++sl) qf[sl] = -qf[sl];
    }
  }

  // |scale| * log2(e); a scale of 0 must not meet a masked score of -inf in a product, one of NaN stays (fmaxf drops it)
  const float scale_abs = fabsf(scale) * 1.44269504f, scale2 = scale_abs < 1e-30f ? 1e-30f : scale_abs;
  f32x16 oacc[D / 32];                              // O^T: column = q row (ln), rows = channels
#pragma unroll
  for (int nb = 0; nb < D / 32; ++nb)
#pragma unroll
    for (int j = 0; j < 16; ++j) oacc[nb][j] = 0.0f;
  float m_run = -INFINITY, l_run = 0.0f;
  float mref = -3.0e38f;   // what the weights are taken against: m_run, and below every finite score until a row has one

  const int kv_tiles_all = (SeffK + KVB - 1) / KVB;
  const int kv_tiles = causal ? min(kv_tiles_all, (min(q0 + NW * QW, Seff) + KVB - 1) / KVB) : kv_tiles_all;

  // tiles this wave computes: those above its diagonal produce nothing (barriers stay uniform)
  const int my_tiles = qw >= Seff ? 0 : (causal ? min(kv_tiles, (qw + QW - 1) / KVB + 1) : kv_tiles);

  const int q_abs = qw + ln;
  char* Kbuf = smem;                 // [2] key tiles, then [2] value tiles
  char* Vbuf = smem + 2 * KB_BYTES;

  // The mask of 32 keys, of the few that need one: at the diagonal and at the end of the keys. Rows past the sequence's last one repeat it, or
  // see what keys there are; what becomes of them is overwritten at the end.
  const int last_key = causal ? min(q_abs, SeffK - 1) : SeffK - 1;   // the last key this row sees
  auto mask = [&](int k0, f32x16& s) __attribute__((always_inline)) {
    if (k0 + 32 > SeffK || (causal && k0 + 31 > qw)) {
      const int upto = last_key - k0 - 4 * half;
#pragma unroll
      for (int j = 0; j < 16; ++j) s[j] = crow(j, 0) > upto ? -INFINITY : s[j];
      asm volatile("" ::: "memory");   // a body of its own: merged into the common one, every tile would pay for it
    }
  };

  // ---- online softmax of 32 scores of q-row (qw+ln), half of them in this lane, in the base-2 domain (v_exp_f32 is exp2); the scale enters
  // with the fma that subtracts the reference m_run. m_run is a maximum the row has had, not always its newest: the
  // weights are taken against it as it stands, and only where their sum shows that some of them passed 2^12 (a row's first
  // finite score gives inf; NaN counts too) is the maximum formed, m_run raised and the weights taken
  // again. The sum is needed anyway, so most tiles need no maximum, no exchange between the half-waves and no
  // rescaling; float32 and bfloat16 hold a weight of 2^12 as precisely as one of 1, and its products with values of up to 2^100 are finite in any number.
  // P in the order it was born in is the B operand of O^T += V^T · P^T: slot half*8+e of a 16-k step holds
  // key 8*(e>>2) + 4*half + (e&3) of it, and the V column fragments are read in the same key
  // order. P never passes through LDS.
  struct Weights {
    bf16x8_t p[2];
  };
  // Two weights in two stages: the exponentials, then their sum and rounding.
  auto stage = [&](int k, const f32x16& s, int i, float (&w)[2], float& sum, Weights& p) __attribute__((always_inline)) {
    if (k == 0) {
#pragma unroll
      for (int e = 0; e < 2; ++e) w[e] = __builtin_amdgcn_exp2f(fmaf(s[i + e], scale2, -mref));
    } else {
#pragma unroll
      for (int e = 0; e < 2; ++e) {
        sum += w[e];
        p.p[i >> 3][(i & 7) + e] = (__bf16)w[e];
      }
    }
  };
  auto raise = [&](const f32x16& s, float rowsum, Weights& p) __attribute__((always_inline)) {
    if (__builtin_expect(!__all(rowsum <= 4096.0f), 0)) {
      float rowmax = s[0];
#pragma unroll
      for (int j = 1; j < 16; ++j) rowmax = fmaxf(rowmax, s[j]);
      rowmax = fmaxf(rowmax, __shfl_xor(rowmax, 32));
      rowmax = rowmax == -INFINITY ? -INFINITY : rowmax * scale2;  // no 0 * inf
      const float m_new = fmaxf(m_run, rowmax);
      const float corr = m_run == -INFINITY ? 0.0f : __builtin_amdgcn_exp2f(m_run - m_new);  // nothing summed yet: 0
#pragma unroll
      for (int nb = 0; nb < D / 32; ++nb)
#pragma unroll
        for (int j = 0; j < 16; ++j) oacc[nb][j] *= corr;
      l_run *= corr;
      m_run = m_new;
      mref = m_run == -INFINITY ? -3.0e38f : m_run;
      rowsum = 0.0f;
#pragma unroll
      for (int i = 0; i < 16; i += 2) {
        float w[2];
        stage(0, s, i, w, rowsum, p);
        stage(1, s, i, w, rowsum, p);
      }
    }
    l_run += rowsum;  // this lane's half of the row's keys; the halves meet at the end
  };

  const RowAt row_at(ln, half);
  const ColAt col_at(lane);
  TileStream<D, KVB, NW> kload(k_base, kts, SeffK), vload(v_base, kts, SeffK);
  constexpr int PER = TileLoad<D, KVB, NW>::PER;

  // The turn of 32 keys: the scores of the 32 after them into `sn` (keys from row kr of the tile at `K_`), their own weights from `s` into `p`, and what
  // the 32 ahead of them add, weights `pp` times the values from row vr at `V_`; none of these waits for another, and a
  // wave's instructions alternate between them. A product takes the matrix unit 32 cycles and the SIMD's issue 11; whatever else the SIMD's
  // waves issue (4 to 5 cycles, an exponential 8) fits beside it only if it stands between the products.
  // Fragments are read a group ahead of the products that take them, with one wait a group (a wait for each was 16 of a turn's 190 instructions) or, in unmasked and
  // small calls of four waves, as the compiler places them: few steps of two blocks a CU lose by the first group's wait more than they gain, longer ones nothing. us, one
  // and several: B24 S117 H16 D64 9.0, 8.5; B20 S100 H16 D128 12.5, 11.9; B8 S1024 H12 D64 35.9, 35.6; B4 S4096 H16/4 D128 493, 492; but causal (dealt) B4 S1024 H32/8
  // D128 46.5, 48.4, two waves B1 S1024 H16/4 D128 19.1, 19.6.
  constexpr bool ONE_WAIT = DEAL || NW == 2;
  constexpr int NB = D / 32, GROUPS = D / 32;   // a group: two fragments of keys, two of values
  auto turn = [&](auto with_scores, auto with_weights, auto with_values, const char* __restrict__ K_, int kr, const char* __restrict__ V_, int vr,
                  f32x16& sn, const f32x16& s, Weights& p, const Weights& pp, auto load) __attribute__((always_inline)) {
    bf16x8_t kf[DSL], vf[2 * NB];
    float w[8][2], sum = 0.0f;
    auto read = [&](int g) __attribute__((always_inline)) {
      if (g >= GROUPS) return;
#pragma unroll
      for (int i = 2 * g; i < 2 * g + 2; ++i) {
        if (with_scores) kf[i] = frag_row<KVB>(K_, row_at, kr, i);
        if (with_values) vf[i] = frag_born<KVB>(V_, col_at, vr + i / NB * 16, i % NB * 32);
      }
    };
    constexpr int READS = (decltype(with_scores)::value ? 2 : 0) + (decltype(with_values)::value ? 4 : 0);   // LDS instructions of a group
    constexpr int PRODUCTS = (decltype(with_scores)::value ? DSL : 0) + (decltype(with_values)::value ? 2 * NB : 0);
    auto weigh = [&](int n) __attribute__((always_inline)) {
      if (with_weights) {
#pragma unroll
        for (int k = n * 16 / PRODUCTS; k < (n + 1) * 16 / PRODUCTS; ++k) stage(k & 1, s, (k >> 1) * 2, w[k >> 1], sum, p);
      }
      __builtin_amdgcn_sched_barrier(0);
    };
    if (with_scores) {
#pragma unroll
      for (int j = 0; j < 16; ++j) sn[j] = 0.0f;
    }
    read(0);
    __builtin_amdgcn_sched_barrier(0);
    int n = 0;
#pragma unroll
    for (int g = 0; g < GROUPS; ++g) {
      read(g + 1);
      __builtin_amdgcn_sched_barrier(0);
      if (ONE_WAIT) reads_left<READS>(g + 1 < GROUPS);
#pragma unroll
      for (int i = 2 * g; i < 2 * g + 2; ++i) {
        if (with_scores) {
          sn = __builtin_amdgcn_mfma_f32_32x32x16_bf16(kf[i], qf[i], sn, 0, 0, 0);
          weigh(n++);
        }
        if (with_values) {
          oacc[i % NB] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(vf[i], pp.p[i / NB], oacc[i % NB], 0, 0, 0);
          weigh(n++);
        }
        load(i);
        __builtin_amdgcn_sched_barrier(0);
      }
    }
    if (with_weights) {
      // formed here: the compiler moves them to where they are used, behind the products
      asm volatile("" : "+v"(p.p[0]), "+v"(p.p[1]));
      raise(s, sum, p);
    }
  };
  constexpr std::true_type yes{};
  constexpr std::false_type no{};

  // Keys are a tile ahead of values: in step t a wave forms the scores of the tile's two halves, the weights of the half ahead of them and of the
  // first one, and adds what the halves of the tile before are worth; the next keys and this tile's values are on their way, all
  // issued in the first half of the step, so that they have arrived at its end (past the last key: zeros, without a read).
  if (kv_tiles > 0) {
    kload.all(0, Kbuf, w);
    vload.all(0, Vbuf, w);
  }
  loads_left<PER>();
  __syncthreads();
  int t = 0;
  kload.skip(1);
  auto begin = [&]() __attribute__((always_inline)) {
    kload.next();
    vload.next();
  };
  auto end = [&]() __attribute__((always_inline)) {
    loads_done();
    __syncthreads();
    ++t;
  };
  constexpr int PARTS = 2 * GROUPS;   // of the loads of a step, in its first turn
  auto load_keys = [&](char* __restrict__ K_, int i) __attribute__((always_inline)) {
#pragma unroll
    for (int n = i * PER / PARTS; n < (i + 1) * PER / PARTS; ++n) kload.piece(K_, w, n);
  };
  auto load = [&](char* __restrict__ K_, char* __restrict__ V_, int i) __attribute__((always_inline)) {
    load_keys(K_, i);
#pragma unroll
    for (int n = i * PER / PARTS; n < (i + 1) * PER / PARTS; ++n) vload.piece(V_, w, n);
  };
  auto nothing = [](int) {};
  if (my_tiles > 0) {
    f32x16 se, so;            // scores of an even and an odd half
    Weights pe, po;
    {
      begin();
      turn(yes, no, no, Kbuf, 0, Kbuf, 0, se, so, po, pe, [&](int i) __attribute__((always_inline)) { load_keys(Kbuf + KB_BYTES, i); });   // the first values are on their way
      mask(0, se);
      turn(yes, yes, no, Kbuf, 32, Kbuf, 0, so, se, pe, po, nothing);
      end();
    }
    // step t in buffer t % 2
    auto step = [&](auto masked, int odd) __attribute__((always_inline)) {
      char* K_ = Kbuf + odd * KB_BYTES;
      char* V_ = Vbuf + odd * KB_BYTES;
      char* Kn = Kbuf + (1 - odd) * KB_BYTES;
      char* Vn = Vbuf + (1 - odd) * KB_BYTES;   // of the step before
      begin();
      if (masked) mask(t * KVB - 32, so);
      turn(yes, yes, yes, K_, 0, Vn, 0, se, so, po, pe, [&](int i) __attribute__((always_inline)) { load(Kn, V_, i); });
      if (masked) mask(t * KVB, se);
      turn(yes, yes, yes, K_, 32, Vn, 32, so, se, pe, po, nothing);
      end();
    };
    // most steps meet no mask: they do not look for one either
    const int plain = min(my_tiles, min(SeffK >= 32 ? (SeffK + 32) / KVB : 0, causal ? (qw + KVB - 31) / KVB : my_tiles));
    while (t < plain) step(no, t & 1);
    while (t < my_tiles) step(yes, t & 1);
    const char* V_ = Vbuf + (~t & 1) * KB_BYTES;
    const int k0 = t * KVB - 32;
    if (k0 < SeffK && !(causal && k0 > qw + QW - 1)) {   // the last half shows something to the wave
      mask(k0, so);
      turn(no, yes, yes, V_, 0, V_, 0, se, so, po, pe, nothing);
      turn(no, no, yes, V_, 0, V_, 32, se, so, po, po, nothing);
    } else {
      turn(no, no, yes, V_, 0, V_, 0, se, so, po, pe, nothing);
    }
  }
  while (t < kv_tiles) {
    begin();
    char* K_ = Kbuf + (~t & 1) * KB_BYTES;
#pragma unroll
    for (int i = 0; i < PARTS; ++i) {
      if (t > 0) load(K_, Vbuf + (t & 1) * KB_BYTES, i);
      else load_keys(K_, i);
    }
    end();
  }

  // ---- epilogue: O /= l, store O and LSE. Rows beyond Seff (right-padded
  // batches) become O = 0, LSE = -inf, which the backward uses
  // to mask them; the buffer extent S is still fully written.
  const int row_lim = VARLEN ? Seff : S;
  l_run += __shfl_xor(l_run, 32);
  if (q_abs >= row_lim) return;
  const bool pad = q_abs >= Seff;
  if (pad) l_run = 0.0f;
  unsigned short* o_base = VARLEN ? O + (seq0 * Hq + h) * D : O + ((long)b * S * Hq + h) * D;
  float* lse_base = VARLEN ? LSE + (long)h * S + seq0 : LSE + ((long)b * Hq + h) * S;
  const float inv_l = (l_run > 0.0f) ? 1.0f / l_run : 0.0f;
#pragma unroll
  for (int nb = 0; nb < D / 32; ++nb)
#pragma unroll
    for (int jj = 0; jj < 4; ++jj) {
      short4v pk;
#pragma unroll
      for (int e = 0; e < 4; ++e) pk[e] = pad ? 0 : (short)f2bf(oacc[nb][jj * 4 + e] * inv_l);
      *reinterpret_cast<short4v*>(o_base + (long)q_abs * o_stride + nb * 32 + 8 * jj + 4 * half) = pk;
    }
  if (half == 0) {
    // back to nats: m_run is log2-domain
    lse_base[q_abs] = (l_run > 0.0f) ? m_run * 0.6931472f + __logf(l_run) : -INFINITY;
  }
}

// ==================================================== what a query row adds in the backward: -lse log2(e) and -rowsum(dO ⊙ O)
// One beside the other, so that one load of a wave brings those of 32 rows; a row that counts nothing (padding, or no
// visible key) has an addend of -inf.
__global__ __launch_bounds__(256) void fa_delta_kernel(
    const unsigned short* __restrict__ dO,
    const unsigned short* __restrict__ Oin,
    const float* __restrict__ LSE,
    float2v* __restrict__ stats,  // [B, H, S]
    long rows,  // B*S*H
    int S, int H, int D) {
  const int lane = threadIdx.x & 63;
  const int w = threadIdx.x >> 6;
  const int sub = lane >> 4;       // 4 rows per wave
  const int e16 = lane & 15;       // 16 lanes per row
  const int epl = D / 16;          // elems per lane (8 for D=128)
  const long waves_total = (long)gridDim.x * 4;  // 4 waves per block
  for (long r4 = blockIdx.x * 4L + w; r4 * 4 < rows; r4 += waves_total) {
    const long row = r4 * 4 + sub;
    if (row >= rows) continue;
    float acc = 0.0f;
    const unsigned short* dop = dO + row * D + e16 * epl;
    const unsigned short* op = Oin + row * D + e16 * epl;
    if (epl >= 8) {
      for (int k = 0; k < epl; k += 8) {
        short8 a = *reinterpret_cast<const short8*>(dop + k);
        short8 b = *reinterpret_cast<const short8*>(op + k);
#pragma unroll
        for (int j = 0; j < 8; ++j) acc += bf2f((unsigned short)a[j]) * bf2f((unsigned short)b[j]);
      }
    } else {  // D=64: 4 elems per lane — load width must match the slice
      short4v a = *reinterpret_cast<const short4v*>(dop);
      short4v b = *reinterpret_cast<const short4v*>(op);
#pragma unroll
      for (int j = 0; j < 4; ++j) acc += bf2f((unsigned short)a[j]) * bf2f((unsigned short)b[j]);
    }
#pragma unroll
    for (int off = 8; off > 0; off >>= 1) acc += __shfl_xor(acc, off);
    if (e16 == 0) {
      const long bidx = row / ((long)S * H);
      const long rem = row % ((long)S * H);
      const long s = rem / H;
      const long hh = rem % H;
      const long at = (bidx * H + hh) * S + s;
      const float lse = LSE[at];
      stats[at] = float2v{lse == -INFINITY ? -INFINITY : -lse * 1.44269504f, -acc};
    }
  }
}

// Query tiles, of all of a block's heads, whose rows' statistics a block of the backward can form itself, instead of a kernel ahead of it.
constexpr int OWN_TILES = 8;
template <int D, bool VARLEN>
constexpr bool CAN_OWN = D == 64 && !VARLEN;

// ============================================================ backward kernel
//
// One launch for dK/dV and dQ: the first n_kv blocks (a multiple of 8) take key/value tiles, the
// others query tiles, so that both kinds share the CUs and no second stream is needed. Both form the
// scores again; nothing is summed with atomics.
//
// In both parts the probabilities and their gradients are born with the row they are contracted
// over in the registers of a lane (the C layout's rows), so a packed run of eight registers is an
// operand of the next product as it stands and neither passes through LDS (frag_born reads the other
// operand's columns in the same order).
//
// What bounds it: the SIMDs' issue, 66 % of all cycles at 32 over 8 heads of 128, 8192 tokens, 30 % of that scalar instructions (78 for each 32 x 32
// scores), and waits for LDS reads right behind them; with the chip full then power (1.7 GHz). So descriptors are advanced, statistics come by one load
// into LDS, what a wave does not see is a loop of its own, and fragments are read a product pair ahead with one wait for each pair. us, before -> now:
//   B1 S8192 H32/8 D128 causal 1745 -> 1625, H4/1 362 -> 294, H12 D64 430 -> 394     B4 S4096 H32 D128 1900 -> 1738     B1 S2048 H12 D64 68 -> 53
//   B2 S4096 H16/8 D128 804 -> 752     B1 S4096 H8/2 D64 144 -> 127     B16 S512 H12 D64 63.5 -> 61     B2 S256 H4 D128 19 -> 16
//   packed, 16384 tokens of up to 4096, 32/8 of 128 1215 -> 1105, 12 of 64 278 -> 250; of up to 512, 16/4 of 64 145 -> 135
// Column fragments read ahead of the exponentials: nothing at 128 channels, 64 spill two registers by it in the first part (81 -> 78 us without, B8 S1024 H12).

// A block of 4 waves owns 128 key/value rows, 32 a wave, and streams the query tiles of its group's heads
// (32 rows, double-buffered). dK and dV stay in registers. What a query row adds (its -lse log2e and
// -delta) enters as the accumulator the product starts from and as the exponent's addend; a row of the sequence that sees
// no key has an addend of -inf. Rows past the sequence's end add nothing because those of Q and dO are zeros: their descriptors
// have to end with its last row. Their statistics are zeros by another such one, and so weights of 1, or (formed here) addends of -inf.
// GS blocks share a key/value tile's heads, as evenly as they go, where a model of the launch (launch_bwd) says that it pays; they leave
// float32 partial sums in PART [GS][2][B * Sk * Hkv * D] for fa_bwd_sum_kernel.
template <int D, bool VARLEN>
DEV_INLINE void bwd_dkdv(
    char* smem, int f, int nblocks,
    const unsigned short* __restrict__ Q, const unsigned short* __restrict__ K,
    const unsigned short* __restrict__ V, const unsigned short* __restrict__ dO, const float2v* __restrict__ STATS,
    const unsigned short* __restrict__ O, const float* __restrict__ LSE, unsigned short* __restrict__ dK, unsigned short* __restrict__ dV, float* __restrict__ PART, int GS,
    const int* __restrict__ CU, const int* __restrict__ CUK,
    long qbs, long qts, long kbs, long kts, long dkbs, long dkts,
    int tiles, int B, int S, int Sk, int Hq, int Hkv, float scale, int causal, int W, int dealt) {
  using namespace fa;
  constexpr int QB = 32;
  constexpr int TB = tile_bytes<QB, D>();
  constexpr int DSL = D / 16, NB = D / 32;
  char* Vlds = smem;                                     // [128 rows]
  char* Qbuf = smem + tile_bytes<NWB * QW, D>();         // [2] query tiles, [2] dO tiles
  char* dObuf = Qbuf + 2 * TB;
  char* stats_lds = dObuf + 2 * TB;                      // [2, or OWN_TILES][32 of -lse log2e, 32 of -delta]
  const bool own = CAN_OWN<D, VARLEN> && STATS == nullptr;   // no kernel ahead has formed them: all of the block's, in the order of its steps

  const int lane = threadIdx.x & 63;
  const int w = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);   // the same for a wave: what it decides is a scalar branch
  const int half = lane >> 5;
  const int ln = lane & 31;

  // key/value tile fastest, then the part of the group's heads, then (sequence, kv head): their
  // Q/dO streams meet in one XCD's L2. Under a causal mask the first tiles see the most queries.
  int tile, part, b, hk;
  const bool by_head = CU != nullptr && S > NWB * QW;
  if (dealt) {
    int y, all;
    if (!deal(f, dealt, (VARLEN ? 1 : B) * Hkv * GS, W, false, tile, y)) return;
    part = y % GS;
    hk = y / GS;
    if (!VARLEN) row_of_batch(y / GS, B, Hkv, 1, by_head, b, hk);
    if (VARLEN && !packed_tile(CU, B, NWB * QW, tiles, tile, b, tile, all)) return;
  } else {
    f = xcd_chunk(f, nblocks);
    tile = f % tiles;
    part = (f / tiles) % GS;
    const int y = f / (tiles * GS);
    if (y >= B * Hkv) return;
    b = y % B;
    hk = y / B;
    if (!VARLEN) row_of_batch(y, B, Hkv, 1, by_head, b, hk);
  }
  const int kv0 = tile * (NWB * QW);
  const int group = Hq / Hkv, h_first = part * group / GS;
  const int G = (part + 1) * group / GS - h_first;       // heads of this block: its share of the group, GS need not divide it
  const int kvw = kv0 + w * QW;  // this wave's first kv row

  long seq0 = 0;
  int Seff = S;
  if (VARLEN) {
    seq0 = CU[b];
    Seff = CU[b + 1] - (int)seq0;
    if (kv0 >= Seff) return;
  } else if (CU != nullptr) {
    Seff = CU[b];
  }
  // this part's OWN rows are kv (extent Sk); q streams over Seff
  const int SeffK = VARLEN ? Seff
            : (CUK != nullptr ? CUK[b] : (CU != nullptr ? min(CU[b], Sk) : Sk));

  const unsigned short* k_base = VARLEN ? K + seq0 * kts + (long)hk * D : K + (long)b * kbs + (long)hk * D;
  const unsigned short* v_base = VARLEN ? V + seq0 * kts + (long)hk * D : V + (long)b * kbs + (long)hk * D;
  const long do_stride = (long)Hq * D;

  // ---- K fragments (B operand of S = Q · K^T): lane column = kv (ln), d = sl*16+half*8+[0..7]
  const int kv_my = max(min(kvw + ln, SeffK - 1), 0);
  bf16x8_t kf[DSL];
  {
    const unsigned short* kp = k_base + (long)kv_my * kts + half * 8;
#pragma unroll
    for (int sl = 0; sl < DSL; ++sl) kf[sl] = ld_g16(kp + sl * 16);
  }
  // ---- V rows of the block (B operand of dP = dO · V^T): they do not fit into registers beside
  // the two accumulators, each wave reads its own 32 rows from LDS
  TileLoad<D, NWB * QW, NWB>(v_base, kts, SeffK).all(kv0, Vlds, w);

  f32x16 dk_acc[NB], dv_acc[NB];
#pragma unroll
  for (int nb = 0; nb < NB; ++nb)
#pragma unroll
    for (int j = 0; j < 16; ++j) {
      dk_acc[nb][j] = 0.0f;
      dv_acc[nb][j] = 0.0f;
    }

  const int qt_first = causal ? kv0 / QB : 0;
  const int nq = max((Seff + QB - 1) / QB - qt_first, 0);   // query tiles of a head
  const int steps = kv0 < SeffK ? nq * G : 0;
  const float scale2 = scale * 1.44269504f;

  const RowAt row_at(ln, half);
  const ColAt col_at(lane);
  const int first = qt_first * QB, last = first + nq * QB;   // query rows of a head, in tiles
  int f_head = -1;               // head of the block's that is fetched from
  TileStream<D, QB, NWB> qs(Q, qts, Seff), dos(dO, do_stride, Seff);
  const float2v* stats = STATS;
  int stats_whole = QB * 8, stats_last = ((max(Seff, 1) - 1) % QB + 1) * 8;
  __amdgpu_buffer_rsrc_t stats_now;
  const unsigned stats_off = ln * 8 + half * 4;
  // what the loads of the tile behind the one at `qt0` need, and of its rows' statistics; behind the last head's last one they bring zeros
  auto fetch = [&](int qt0) __attribute__((always_inline)) {
    bool all = qt0 + 2 * QB < last;
    if (__builtin_expect(qt0 + QB >= last, 0)) {
      all = nq > 1;
      if (++f_head < G) {
        const int h = hk * group + h_first + f_head;
        qs.at = (VARLEN ? Q + seq0 * qts + (long)h * D : Q + (long)b * qbs + (long)h * D) + (long)first * qts;
        dos.at = (VARLEN ? dO + (seq0 * Hq + h) * D : dO + ((long)b * S * Hq + h) * D) + (long)first * do_stride;   // dO packed
        stats = STATS + (VARLEN ? (long)h * S + seq0 : ((long)b * Hq + h) * S) + first;
      } else {
        qs.whole = qs.last = dos.whole = dos.last = stats_whole = stats_last = 0;
      }
    }
    qs.next(all);
    dos.next(all);
    stats_now = __builtin_amdgcn_make_buffer_rsrc(const_cast<float2v*>(stats), 0, all ? stats_whole : stats_last, 0x00027000);
    stats += QB;
  };
  const int stats_wave = own ? -1 : 0;
  auto bring_stats = [&](int buf) __attribute__((always_inline)) {
    if (w == stats_wave) __builtin_amdgcn_raw_ptr_buffer_load_lds(stats_now, (lds_ptr)(stats_lds + buf * 256), 4, (int)stats_off, 0, 0, 0);
  };
  typedef TileLoad<D, QB, NWB> Load;
  if (steps > 0) {
    fetch(last);
#pragma unroll
    for (int i = 0; i < Load::PER; ++i) {
      qs.piece(Qbuf, w, i);
      dos.piece(dObuf, w, i);
    }
    bring_stats(0);
    if (own) {
      constexpr int TPR = D / 8, AT_ONCE = NTB / TPR;   // threads of a row, rows
      const int c = threadIdx.x % TPR, sub = threadIdx.x / TPR;
      for (int at = 0; at < min(steps, OWN_TILES) * QB; at += AT_ONCE) {
        const int step = at / QB, head = step / nq, in = at % QB + sub, row = first + (step - head * nq) * QB + in;
        float dot = 0.0f, lse = -INFINITY;
        if (row < Seff) {
          const int h = hk * group + h_first + head;
          const long from = ((long)b * S + row) * do_stride + (long)h * D + c * 8;
          const bf16x8_t x = ld_g16(dO + from), y = ld_g16(O + from);
#pragma unroll
          for (int e = 0; e < 8; ++e) dot = fmaf((float)x[e], (float)y[e], dot);
          lse = LSE[((long)b * Hq + h) * S + row];
        }
#pragma unroll
        for (int o = 1; o < TPR; o <<= 1) dot += __shfl_xor(dot, o);
        if (c == 0) {
          float* to = reinterpret_cast<float*>(stats_lds + step * 256) + in;
          to[0] = lse == -INFINITY ? -INFINITY : -lse * 1.44269504f;
          to[QB] = -dot;
        }
      }
    }
  }
  loads_done();
  __syncthreads();

  int stats_at = 0;
  // A query tile, while the next one arrives in the other buffers.
  auto step = [&](int qt0, const char* __restrict__ Qlds, const char* __restrict__ dOlds, char* __restrict__ Qn,
                  char* __restrict__ dOn) __attribute__((always_inline)) {
    const float* stats = reinterpret_cast<const float*>(stats_lds + stats_at) + 4 * half;
    // ---- S[q][kv] = Q · K^T and dP[q][kv] - delta[q] = dO · V^T - delta: column = kv (ln), row = q
    f32x16 s, dp;
#pragma unroll
    for (int a = 0; a < 4; ++a) {
      const float4v d4 = *reinterpret_cast<const float4v*>(stats + QB + 8 * a);
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        dp[4 * a + e] = d4[e];
        s[4 * a + e] = 0.0f;
      }
    }
    __builtin_amdgcn_s_setprio(1);
    bf16x8_t qr[DSL], dor[DSL], vr[DSL], doc[2 * NB], qc[2 * NB];   // fragments, read ahead of their products with one wait for each pair of these
    auto rows = [&](int i) __attribute__((always_inline)) {
      if (i >= DSL) return;
      qr[i] = frag_row<QB>(Qlds, row_at, 0, i);
      dor[i] = frag_row<QB>(dOlds, row_at, 0, i);
      vr[i] = frag_row<NWB * QW>(Vlds + w * 2048, row_at, 0, i);
    };
    auto columns = [&](int i) __attribute__((always_inline)) {
      if (i >= 2 * NB) return;
      doc[i] = frag_born<QB>(dOlds, col_at, i / NB * 16, i % NB * 32);
      qc[i] = frag_born<QB>(Qlds, col_at, i / NB * 16, i % NB * 32);
    };
    rows(0);
#pragma unroll
    for (int sl = 0; sl < DSL; ++sl) {
      rows(sl + 1);
      __builtin_amdgcn_sched_barrier(0);
      reads_left<3>(sl + 1 < DSL);
      s = __builtin_amdgcn_mfma_f32_32x32x16_bf16(qr[sl], kf[sl], s, 0, 0, 0);
      dp = __builtin_amdgcn_mfma_f32_32x32x16_bf16(dor[sl], vr[sl], dp, 0, 0, 0);
#pragma unroll
      for (int i = sl * Load::PER / DSL; i < (sl + 1) * Load::PER / DSL; ++i) qs.piece(Qn, w, i);
    }
    __builtin_amdgcn_s_setprio(0);
    if (D == 128) columns(0);   // ahead of the exponentials; 64 channels have no registers for them there
    // ---- P = exp(scale s - lse); dS = P (dP - delta), its scale waits for the epilogue
    bf16x8_t pa[2], dsa[2];
    const int before = kvw + ln - qt0 - 4 * half;   // rows of the tile ahead of this key
    auto grads = [&](auto diagonal) __attribute__((always_inline)) {
#pragma unroll
      for (int a = 0; a < 4; ++a) {   // read here, the statistics take 4 registers and not 16 over the products
        const float4v l4 = *reinterpret_cast<const float4v*>(stats + 8 * a);
#pragma unroll
        for (int e = 0; e < 4; ++e) {
          const int j = 4 * a + e;
          float pv = __builtin_amdgcn_exp2f(fmaf(s[j], scale2, l4[e]));
          if (diagonal) pv = before > crow(j, 0) ? 0.0f : pv;
          pa[j >> 3][j & 7] = (__bf16)pv;
          dsa[j >> 3][j & 7] = (__bf16)(pv * dp[j]);
        }
      }
    };
    // two bodies: merged into one, every tile would pay for the mask of the few on the diagonal
    if (causal && qt0 < kvw + QW - 1) {
      grads(std::true_type());
      asm volatile("" ::: "memory");
    } else {
      grads(std::false_type());
    }
    // ---- dV += P^T · dO, dK += dS^T · Q (A: lane row = kv; B: columns of the tiles)
    if (D != 128) columns(0);
    __builtin_amdgcn_s_setprio(1);
#pragma unroll
    for (int at = 0; at < 2 * NB; ++at) {
      columns(at + 1);
      __builtin_amdgcn_sched_barrier(0);
      reads_left<4>(at + 1 < 2 * NB);
      dv_acc[at % NB] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(pa[at / NB], doc[at], dv_acc[at % NB], 0, 0, 0);
      dk_acc[at % NB] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(dsa[at / NB], qc[at], dk_acc[at % NB], 0, 0, 0);
#pragma unroll
      for (int i = at * Load::PER / (2 * NB); i < (at + 1) * Load::PER / (2 * NB); ++i) dos.piece(dOn, w, i);
    }
    __builtin_amdgcn_s_setprio(0);
  };
  // A head's first tiles show some waves nothing: they only bring the next one's rows, in a loop of its own, ahead of which the sums stay in their registers.
  int buf = 0;
  char *Qn, *dOn;
  auto begin = [&](int qt0) __attribute__((always_inline)) {
    fetch(qt0);
    Qn = Qbuf + (buf ^ 1) * TB;
    dOn = dObuf + (buf ^ 1) * TB;
    bring_stats(buf ^ 1);
  };
  auto finish = [&]() __attribute__((always_inline)) {
    buf ^= 1;
    stats_at = own ? stats_at + 256 : buf * 256;
    loads_done();
    __syncthreads();
  };
  const int from = kvw >= SeffK ? last : causal ? min(kvw, last) : 0;
  for (int head = 0; head < (steps > 0 ? G : 0); ++head) {
    int qt0 = first;
    for (; qt0 < from; qt0 += QB) {
      begin(qt0);
#pragma unroll
      for (int i = 0; i < Load::PER; ++i) {
        qs.piece(Qn, w, i);
        dos.piece(dOn, w, i);
      }
      finish();
    }
    for (; qt0 < last; qt0 += QB) {
      begin(qt0);
      step(qt0, Qbuf + buf * TB, dObuf + buf * TB, Qn, dOn);
      finish();
    }
  }

  // ---- epilogue: dK, dV of the rows of this tile. Padded rows get zeros.
  const int kv_lim = VARLEN ? Seff : Sk;
  const long n_part = (VARLEN ? (long)Sk : (long)B * Sk) * Hkv * D;
#pragma unroll
  for (int j = 0; j < 16; ++j) {
    const int kv_abs = kvw + crow(j, half);
    if (kv_abs >= kv_lim) continue;
    const bool live = kv_abs < SeffK;
    if (GS > 1) {
      const long row = VARLEN ? seq0 + kv_abs : (long)b * Sk + kv_abs;
      float* pk = PART + (long)part * 2 * n_part + (row * Hkv + hk) * D + ln;
#pragma unroll
      for (int nb = 0; nb < NB; ++nb) {
        pk[nb * 32] = live ? dk_acc[nb][j] * scale : 0.0f;
        pk[n_part + nb * 32] = live ? dv_acc[nb][j] : 0.0f;
      }
    } else {
      const long at = (VARLEN ? seq0 * dkts : (long)b * dkbs) + (long)hk * D + (long)kv_abs * dkts + ln;
#pragma unroll
      for (int nb = 0; nb < NB; ++nb) {
        dK[at + nb * 32] = live ? f2bf(dk_acc[nb][j] * scale) : 0;
        dV[at + nb * 32] = live ? f2bf(dv_acc[nb][j]) : 0;
      }
    }
  }
}

// A block of 4 waves owns 128 query rows, 32 a wave, and streams key/value tiles of 64 rows. K serves as
// rows (scores) and as columns (dQ), V as rows.
template <int D, bool VARLEN>
DEV_INLINE void bwd_dq(
    char* smem, int f, int nblocks,
    const unsigned short* __restrict__ Q, const unsigned short* __restrict__ K,
    const unsigned short* __restrict__ V, const unsigned short* __restrict__ dO,
    const float2v* __restrict__ STATS, const unsigned short* __restrict__ O, const float* __restrict__ LSE, unsigned short* __restrict__ dQ,
    const int* __restrict__ CU, const int* __restrict__ CUK,
    long qbs, long qts, long kbs, long kts, long dqbs, long dqts,
    int tiles, int B, int S, int Sk, int Hq, int Hkv, float scale, int causal, int W, int dealt) {
  using namespace fa;
  constexpr int TB = tile_bytes<KVB, D>();
  constexpr int DSL = D / 16, NB = D / 32;
  char* Kbuf = smem;           // [2] key tiles, [2] value tiles
  char* Vbuf = smem + 2 * TB;

  const int lane = threadIdx.x & 63;
  const int w = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);   // the same for a wave: what it decides is a scalar branch
  const int half = lane >> 5;
  const int ln = lane & 31;

  int y, tile, b, h;
  const bool by_head = CU != nullptr && S > NWB * QW;
  if (dealt) {
    int all = dealt;
    if (!deal(f, dealt, (VARLEN ? 1 : B) * Hq, W, false, tile, y)) return;
    h = y;
    if (!VARLEN) row_of_batch(y, B, Hq, Hq / Hkv, by_head, b, h);
    if (VARLEN && !packed_tile(CU, B, NWB * QW, tiles, tile, b, tile, all)) return;
    if (causal) tile = all - 1 - tile;  // late tiles see the most keys
  } else {
    f = xcd_chunk(f, nblocks);
    y = f / tiles;
    tile = f % tiles;
    if (y >= B * Hq) return;
    b = y % B;
    h = y / B;
    if (!VARLEN) row_of_batch(y, B, Hq, Hq / Hkv, by_head, b, h);
    if (VARLEN && causal && by_tile(tiles, nblocks, Hq / Hkv)) {
      const int i = b * tiles + tile;
      tile = tiles - 1 - i / B;
      b = i % B;
    } else if (causal) {
      tile = tiles - 1 - tile;
    }
  }
  const int hk = h / (Hq / Hkv);
  const int q0 = tile * (NWB * QW);
  const int qw = q0 + w * QW;

  long seq0 = 0;
  int Seff = S;
  if (VARLEN) {
    seq0 = CU[b];
    Seff = CU[b + 1] - (int)seq0;
    if (q0 >= Seff) return;
  } else if (CU != nullptr) {
    Seff = CU[b];
  }
  const int SeffK = VARLEN ? Seff
            : (CUK != nullptr ? CUK[b] : (CU != nullptr ? min(CU[b], Sk) : Sk));

  const unsigned short* q_base = VARLEN ? Q + seq0 * qts + (long)h * D : Q + (long)b * qbs + (long)h * D;
  const unsigned short* do_base =
      VARLEN ? dO + (seq0 * Hq + h) * D : dO + ((long)b * S * Hq + h) * D;  // dO packed
  const long do_stride = (long)Hq * D;
  const unsigned short* k_base = VARLEN ? K + seq0 * kts + (long)hk * D : K + (long)b * kbs + (long)hk * D;
  const unsigned short* v_base = VARLEN ? V + seq0 * kts + (long)hk * D : V + (long)b * kbs + (long)hk * D;

  // ---- Q, dO fragments (B operands): lane column = q (ln), d = sl*16+half*8+[0..7]
  const int q_my = max(min(qw + ln, Seff - 1), 0);
  bf16x8_t qf[DSL], dof[DSL];
  {
    const unsigned short* qp = q_base + (long)q_my * qts + half * 8;
    const unsigned short* dop = do_base + (long)q_my * do_stride + half * 8;
#pragma unroll
    for (int sl = 0; sl < DSL; ++sl) {
      qf[sl] = ld_g16(qp + sl * 16);
      dof[sl] = ld_g16(dop + sl * 16);
    }
  }
  const long stat = (VARLEN ? (long)h * S + seq0 : ((long)b * Hq + h) * S) + q_my;
  float2v own;
  if (!CAN_OWN<D, VARLEN> || STATS != nullptr) {
    own = STATS[stat];
  } else {   // a lane has half of its row's channels
    const unsigned short* op = O + (do_base - dO) + (long)q_my * do_stride + half * 8;
    float dot = 0.0f;
#pragma unroll
    for (int sl = 0; sl < DSL; ++sl) {
      const bf16x8_t y = ld_g16(op + sl * 16);
#pragma unroll
      for (int e = 0; e < 8; ++e) dot = fmaf((float)dof[sl][e], (float)y[e], dot);
    }
    const float lse = LSE[stat];
    own = float2v{lse == -INFINITY ? -INFINITY : -lse * 1.44269504f, -(dot + __shfl_xor(dot, 32))};
  }
  const float addend = qw + ln < Seff ? own[0] : -INFINITY, ndelta = own[1];
  const float scale2 = scale * 1.44269504f;

  f32x16 dq_acc[NB];
#pragma unroll
  for (int nb = 0; nb < NB; ++nb)
#pragma unroll
    for (int j = 0; j < 16; ++j) dq_acc[nb][j] = 0.0f;

  const int kv_tiles_all = (SeffK + KVB - 1) / KVB;
  const int kv_tiles = q0 >= Seff ? 0 : (causal ? min(kv_tiles_all, (min(q0 + NWB * QW, Seff) + KVB - 1) / KVB) : kv_tiles_all);

  const int last_key = causal ? min(qw + ln, SeffK - 1) : SeffK - 1;   // the last key this row sees
  const RowAt row_at(ln, half);
  const ColAt col_at(lane);
  typedef TileLoad<D, KVB, NWB> Load;
  TileStream<D, KVB, NWB> kload(k_base, kts, SeffK), vload(v_base, kts, SeffK);
  if (kv_tiles > 0) {
    kload.all(0, Kbuf, w);
    vload.all(0, Vbuf, w);
    kload.skip(1);
    vload.skip(1);
  }
  // keys from which on a wave's rows do not see all of 32, tiles of which they see something
  const int edge = min(SeffK - 31, causal ? qw - 30 : INT_MAX);
  const int my_tiles = qw >= Seff ? 0 : causal ? min(kv_tiles, (qw + QW - 1) / KVB + 1) : kv_tiles;
  loads_done();
  __syncthreads();

  // A key/value tile, while the next one arrives in the other buffers (past the last key: zeros, without a read).
  auto step = [&](int k0, const char* __restrict__ Klds, const char* __restrict__ Vlds, char* __restrict__ Kn,
                  char* __restrict__ Vn) __attribute__((always_inline)) {
    kload.next();
    vload.next();
#pragma unroll
    for (int kb = 0; kb < KVB / 32; ++kb) {
      // ---- S^T[kv][q] = K · Q^T and dP^T - delta = V · dO^T - delta: column = q (ln), row = kv
      f32x16 s, dp;
#pragma unroll
      for (int j = 0; j < 16; ++j) { s[j] = 0.0f; dp[j] = ndelta; }
      __builtin_amdgcn_s_setprio(1);
      bf16x8_t kr[DSL], vr[DSL], kc[2 * NB];
      auto rows = [&](int i) __attribute__((always_inline)) {
        if (i >= DSL) return;
        kr[i] = frag_row<KVB>(Klds, row_at, kb * 32, i);
        vr[i] = frag_row<KVB>(Vlds, row_at, kb * 32, i);
      };
      auto columns = [&](int g) __attribute__((always_inline)) {   // two fragments
        if (g >= NB) return;
#pragma unroll
        for (int i = 2 * g; i < 2 * g + 2; ++i) kc[i] = frag_born<KVB>(Klds, col_at, kb * 32 + i / NB * 16, i % NB * 32);
      };
      rows(0);
#pragma unroll
      for (int sl = 0; sl < DSL; ++sl) {
        rows(sl + 1);
        __builtin_amdgcn_sched_barrier(0);
        reads_left<2>(sl + 1 < DSL);
        s = __builtin_amdgcn_mfma_f32_32x32x16_bf16(kr[sl], qf[sl], s, 0, 0, 0);
        dp = __builtin_amdgcn_mfma_f32_32x32x16_bf16(vr[sl], dof[sl], dp, 0, 0, 0);
        const int at = kb * DSL + sl;
#pragma unroll
        for (int i = at * Load::PER / (2 * DSL); i < (at + 1) * Load::PER / (2 * DSL); ++i) {
          kload.piece(Kn, w, i);
          vload.piece(Vn, w, i);
        }
      }
      __builtin_amdgcn_s_setprio(0);
      columns(0);
      // ---- dS = exp(scale s - lse) (dP - delta), its scale waits for the epilogue
      bf16x8_t dsa[2];
      const int kb0 = k0 + kb * 32, upto = last_key - kb0 - 4 * half;
      auto grads = [&](auto edge) __attribute__((always_inline)) {
#pragma unroll
        for (int j = 0; j < 16; ++j) {
          float pv = __builtin_amdgcn_exp2f(fmaf(s[j], scale2, addend));
          if (edge) pv = crow(j, 0) > upto ? 0.0f : pv;
          dsa[j >> 3][j & 7] = (__bf16)(pv * dp[j]);
        }
      };
      if (kb0 >= edge) {
        grads(std::true_type());
        asm volatile("" ::: "memory");
      } else {
        grads(std::false_type());
      }
      // ---- dQ += dS · K (A: lane row = q; B: columns of K)
      __builtin_amdgcn_s_setprio(1);
#pragma unroll
      for (int g = 0; g < NB; ++g) {
        columns(g + 1);
        __builtin_amdgcn_sched_barrier(0);
        reads_left<4>(g + 1 < NB);
#pragma unroll
        for (int i = 2 * g; i < 2 * g + 2; ++i)
          dq_acc[i % NB] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(dsa[i / NB], kc[i], dq_acc[i % NB], 0, 0, 0);
      }
      __builtin_amdgcn_s_setprio(0);
    }
  };
  for (int t = 0; t < kv_tiles; ++t) {
    const int k0 = t * KVB, buf = t & 1;
    char* Kn = Kbuf + (buf ^ 1) * TB;
    char* Vn = Vbuf + (buf ^ 1) * TB;
    if (t < my_tiles) {
      step(k0, Kbuf + buf * TB, Vbuf + buf * TB, Kn, Vn);
    } else {
      kload.next();
      vload.next();
#pragma unroll
      for (int i = 0; i < Load::PER; ++i) {
        kload.piece(Kn, w, i);
        vload.piece(Vn, w, i);
      }
    }
    loads_done();
    __syncthreads();
  }

  // ---- epilogue: write dQ (pad rows accumulate nothing -> zeros)
  const int q_lim = VARLEN ? Seff : S;
  unsigned short* dq_base = VARLEN ? dQ + seq0 * dqts + (long)h * D : dQ + (long)b * dqbs + (long)h * D;
#pragma unroll
  for (int j = 0; j < 16; ++j) {
    const int q_abs = qw + crow(j, half);
    if (q_abs >= q_lim) continue;
#pragma unroll
    for (int nb = 0; nb < NB; ++nb) dq_base[(long)q_abs * dqts + nb * 32 + ln] = f2bf(dq_acc[nb][j] * scale);
  }
}

template <int D>
constexpr size_t bwd_lds() {
  using namespace fa;
  const size_t kv = tile_bytes<NWB * QW, D>() + 4 * tile_bytes<32, D>() + 4 * 32 * sizeof(float);
  const size_t q = 4 * tile_bytes<KVB, D>();
  return kv > q ? kv : q;
}

// Three waves a SIMD with 64 channels, 168 registers; left to itself the packed form took 174 and had two.
template <int D, bool VARLEN>
__global__ __launch_bounds__(fa::NTB, D == 64 ? 3 : 2) void fa_bwd_kernel(
    const unsigned short* __restrict__ Q, const unsigned short* __restrict__ K,
    const unsigned short* __restrict__ V, const unsigned short* __restrict__ dO,
    const float2v* __restrict__ STATS, const unsigned short* __restrict__ O, const float* __restrict__ LSE,
    unsigned short* __restrict__ dQ, unsigned short* __restrict__ dK, unsigned short* __restrict__ dV,
    float* __restrict__ PART, int GS, const int* __restrict__ CU, const int* __restrict__ CUK,
    long qbs, long qts, long kbs, long kts, long dqbs, long dqts, long dkbs, long dkts,
    int n_kv, int n_q, int kv_tiles, int q_tiles, int B, int S, int Sk, int Hq, int Hkv, float scale, int causal, int W, int dealt) {
  extern __shared__ char smem[];
  const int f = (int)(blockIdx.y * gridDim.x + blockIdx.x);   // more than one grid row only beyond 2^23 blocks
  if (f >= n_kv + n_q) return;
  if (f < n_kv)
    bwd_dkdv<D, VARLEN>(smem, f, n_kv, Q, K, V, dO, STATS, O, LSE, dK, dV, PART, GS, CU, CUK, qbs, qts, kbs, kts, dkbs, dkts,
                        kv_tiles, B, S, Sk, Hq, Hkv, scale, causal, W, dealt);
  else
    bwd_dq<D, VARLEN>(smem, f - n_kv, n_q, Q, K, V, dO, STATS, O, LSE, dQ, CU, CUK, qbs, qts, kbs, kts,
                      dqbs, dqts, q_tiles, B, S, Sk, Hq, Hkv, scale, causal, W, dealt);
}

// dK and dV from the float32 sums of the GS blocks that shared a tile's heads: four channels a thread.
__global__ __launch_bounds__(256) void fa_bwd_sum_kernel(unsigned short* __restrict__ dK, unsigned short* __restrict__ dV,
                                                         const float* __restrict__ PART, int GS, long n_part, int Sk,
                                                         int HD, long dkbs, long dkts) {
  const long i = ((long)blockIdx.x * 256 + threadIdx.x) * 4;
  if (i >= n_part) return;
  const long row = i / HD;
  const long at = row / Sk * dkbs + row % Sk * dkts + i % HD;
#pragma unroll
  for (int which = 0; which < 2; ++which) {
    float4v sum = {0.0f, 0.0f, 0.0f, 0.0f};
    for (int p = 0; p < GS; ++p) sum += *reinterpret_cast<const float4v*>(PART + (2L * p + which) * n_part + i);
    short4v o;
#pragma unroll
    for (int e = 0; e < 4; ++e) o[e] = (short)f2bf(sum[e]);
    *reinterpret_cast<short4v*>((which ? dV : dK) + at) = o;
  }
}

// =============================================================== host side

namespace {

// A tile's loads take 16 bytes at addresses of that alignment, with offsets of 32 bits inside the tile. Rows that lie
// otherwise, or 2^23 elements apart and more, are copied together first; k and v together, which share their strides.
bool loadable(const at::Tensor& t) {
  const int rows = (int)t.dim() - 3;
  return reinterpret_cast<uintptr_t>(t.data_ptr()) % 16 == 0 &&
         (t.size(rows) <= 1 || (t.stride(rows) % 8 == 0 && t.stride(rows) < (1L << 23))) &&
         (rows == 0 || t.size(0) <= 1 || t.stride(0) % 8 == 0);
}
void make_loadable(at::Tensor& t) {
  if (!loadable(t)) t = t.clone(at::MemoryFormat::Contiguous);
}
void make_loadable(at::Tensor& k, at::Tensor& v) {
  if (loadable(k) && loadable(v)) return;
  k = k.clone(at::MemoryFormat::Contiguous);
  v = v.clone(at::MemoryFormat::Contiguous);
}

void set_lds_limit(const void* kernel, size_t bytes) {
  if (bytes > 65536) {
    (void)hipFuncSetAttribute(kernel, hipFuncAttributeMaxDynamicSharedMemorySize, (int)bytes);
  }
}

// Waves (of 32 query rows) of a forward block. Four: two blocks share a CU, and their barriers do not
// hold each other up (8 waves in one block: 735 against 809 TFLOP/s at B4 S4096 H32 D128 causal). Two as long as blocks of two have a CU each, up to
// 128 of four: a wave has fewer neighbours to wait for, 8 to 20 % at 128 and 256 tokens, nothing at 2048. Beyond, two blocks of two share a CU
// and its loads are twice those of one block of four: 4/2 waves at 144 to 252 blocks 0.93 (128 tokens), 0.84 (512), 0.76 (2048); with a mask 0.9, 0.83, 0.98.
int fwd_waves(long blocks) { return blocks <= 128 ? 2 : 4; }

// Rows (heads of sequences) whose tiles an XCD takes side by side (deal): as many as end evenly and whose keys and values, of kv_bytes a kv head,
// still meet in its L2 (4 MB; twice that, as not all are in the same place). us, forward and backward, one row, four, eight, sixteen: B8 S1024 H12 D64 31
// and 81, 31 and 73, 30 and 73, 25 and 67; B4 S4096 H32 D128 568 and 1778, 548 and 1714, 555 and 1723, 571 and 1773; B4 S2048 H16/4 D128 91 and 288, 78
// and 276, 74 and 269, 74 and 272; B1 S8192 H12 D64 (two of three rows an XCD) 175 and 386, 123 and 338; B1 S8192 H32/8 D128 554 and 1645, 527 and 1579.
int rows_together(int group, long kv_bytes) { return (int)std::max(4L, group * std::min(16L, (8L << 20) / std::max(1L, kv_bytes))); }

// Whether rows that row_parts XCDs share are dealt tile by tile. Those of few tiles are not: the parts differ by a tile, or its place stays empty. us, in order and dealt,
// forward of 64 channels unless said: three tiles, 140 rows (2 XCDs a row) 11.4, 14.6, 99 rows (8) 10.8, 14.3; five of 128 channels, 66 rows (4) 20.9, 24.5; six, 63 rows (8)
// 14.8, 17.6; eight, 40 rows (1) 29, 22, 36 (2) 20.7, 15.8, 76 (2) 28.6, 28.3; 16 of 128, 30 (4) 55, 48; 32, 20 (2) 90, 61; 64, 9 (8) 152, 105. Backward: three of 128,
// 366 (4) 84, 113.
bool worth_dealing(long tiles, int n_y) { return tiles >= 4 * fa::row_parts(n_y); }

// The causal dense forward's rows, of more than 256 blocks: three tiles too where all blocks run at once. us, in order and dealt: B8 S384 H16/4 D128 17.5, 15.2, but
// B64 S384 H16/4 80, 87; B64 S36 H12 D64 6.5, 7.5; B24 S256 H12 14.2, 14.8.
bool deals(int S, int n_y, long blocks) {
  const long tiles = (S + 127) / 128;
  return blocks > 256 && (worth_dealing(tiles, n_y) || (tiles == 3 && n_y % 8 == 0 && blocks <= 512));
}

// Tiles of a packed batch that its blocks look up (packed_tile), an upper bound; 0: sequence by sequence or tile by tile. Sequences of one tile need no
// order, and small grids run at once in any. us, forward and backward, before and by lookup: 16384 tokens of up to 4096 in 12 sequences, 32/8 heads of
// 128 363 and 1110, 346 and 1072; 12 of 64 96 and 257, 80 and 235; 64 sequences of up to 900, 8/2 of 128 54 and 187, 37 and 138; 46 of 1024, 32/8 of 128 169
// and 493, 161 and 443; 56 of 500, 16/2 of 64 22 and 88, 22 and 62; 47 of 256, 16/4 of 64 12.3 and 37.1, 12.4 and 35.3; 39 of 128, 32/8 of 64 11.4, 12.8.
long packed_tiles(long T, int n_seq, long tiles, int rows, int H) {
  const long all = std::min(T / rows + n_seq, tiles * n_seq);
  return n_seq <= fa::MOST_PACKED && tiles > 1 && all * H > 512 ? all : 0;
}

// The forward's. Where tile by tile is the other order (by_tile) a look-up, longer than the one it takes the place of, pays with 128 channels, three tiles or more and 1024
// blocks. us, by tile and looked up: 16384 tokens of up to 160, 16/4 heads of 64 34, 39, 64/8 133, 156, 16/8 of 128 60, 66; of up to 400, 32/4 of 128 142, 129, 32/8
// 141, 134, 16/4 of 64 35.5, 37.3; 12000 of up to 700, 8/2 of 128 30.3, 32.4; 16384 of up to 1000, 32/4 of 128 183, 159, 32/8 199, 169, 16/4 of 64 45.3, 48.5, 64/8 192, 189.
long packed_tiles_fwd(long T, int n_seq, long tiles, int rows, int H, int group, int D, bool causal) {
  const long all = packed_tiles(T, n_seq, tiles, rows, H);
  return causal && fa::by_tile((int)tiles, tiles * n_seq * H, group) && (D == 64 || tiles <= 2 || all * H <= 1024) ? 0 : all;
}

// a grid dimension of 2^32 threads or more is cut short without an error
dim3 wide_grid(long blocks) {
  const long width = std::max(1L, std::min(blocks, 1L << 23));
  return dim3((unsigned)width, (unsigned)((blocks + width - 1) / width));
}

// q/k/v are [B,S,H,D] views that may be strided in dims 0/1 (e.g. views into
// a packed QKV GEMM output); dims 2/3 must be dense.
void check_fa_view(const at::Tensor& t, const char* name) {
  TORCH_CHECK(t.dim() == 4, "flash_attn: ", name, " must be [B,S,H,D]");
  TORCH_CHECK(t.scalar_type() == at::kBFloat16, "flash_attn: bf16 only");
  TORCH_CHECK(t.stride(3) == 1 && t.stride(2) == t.size(3), "flash_attn: ", name,
              " must be dense in [H,D] (strided B/S allowed)");
}

void check_fa_inputs(const at::Tensor& q, const at::Tensor& k, const at::Tensor& v) {
  check_fa_view(q, "q");
  check_fa_view(k, "k");
  check_fa_view(v, "v");
  const int D = (int)q.size(3);
  TORCH_CHECK(D == 64 || D == 128, "flash_attn: head dim must be 64 or 128");
  TORCH_CHECK(k.size(3) == D && v.size(3) == D);
  TORCH_CHECK(k.sizes() == v.sizes() && k.strides() == v.strides(), "flash_attn: k/v must match");
  TORCH_CHECK((int)q.size(2) % (int)k.size(2) == 0, "flash_attn: Hq must be a multiple of Hkv (GQA)");
}

}  // namespace

std::vector<at::Tensor> flash_attn_fwd(at::Tensor q, at::Tensor k, at::Tensor v, bool causal, double scale,
                                       c10::optional<at::Tensor> seqlens_opt,
                                       c10::optional<at::Tensor> seqlens_k_opt) {
  at::Tensor seqlens = seqlens_opt.has_value() ? *seqlens_opt : at::Tensor();
  at::Tensor seqlens_k = seqlens_k_opt.has_value() ? *seqlens_k_opt : at::Tensor();
  using namespace fa;
  check_fa_inputs(q, k, v);
  make_loadable(q);
  make_loadable(k, v);
  const int B = (int)q.size(0), S = (int)q.size(1), Hq = (int)q.size(2), D = (int)q.size(3);
  const int Hkv = (int)k.size(2);
  const int Sk = (int)k.size(1);  // kv may be a shorter ring piece
  const int* cu = nullptr;
  const int* cuk = nullptr;
  if (seqlens.defined() && seqlens.numel() > 0) {
    TORCH_CHECK(seqlens.scalar_type() == at::kInt && seqlens.numel() == B && seqlens.is_cuda(),
                "flash_attn: seqlens must be int32 [B] on device");
    cu = seqlens.data_ptr<int>();
  }
  if (seqlens_k.defined() && seqlens_k.numel() > 0) {
    TORCH_CHECK(cu != nullptr, "flash_attn: seqlens_k requires seqlens");
    TORCH_CHECK(seqlens_k.scalar_type() == at::kInt && seqlens_k.numel() == B && seqlens_k.is_cuda());
    cuk = seqlens_k.data_ptr<int>();
  }
  auto o = at::empty({B, S, Hq, D}, q.options());
  auto lse = at::empty({B, Hq, S}, q.options().dtype(at::kFloat));
  auto stream = at::hip::getCurrentHIPStream();
  const long qbs = q.stride(0), qts = q.stride(1), kbs = k.stride(0), kts = k.stride(1);

#define LAUNCH_FWD(DD, NW, DEAL)                                                                            \
  do {                                                                                            \
    const int tiles = (S + NW * QW - 1) / (NW * QW);                                                \
    const size_t lds = 4 * tile_bytes<KVB, DD>();                                                  \
    set_lds_limit((const void*)fa_fwd_kernel<DD, NW, false, DEAL>, lds);                                \
    hipLaunchKernelGGL((fa_fwd_kernel<DD, NW, false, DEAL>), DEAL ? wide_grid(dealt_blocks(tiles, B * Hq)) : dim3((unsigned)tiles, B * Hq), \
                       dim3(NW * 64), lds, stream.stream(),                                       \
                       (const unsigned short*)q.data_ptr(), (const unsigned short*)k.data_ptr(),  \
                       (const unsigned short*)v.data_ptr(), (unsigned short*)o.data_ptr(),        \
                       lse.data_ptr<float>(), cu, cuk, qbs, qts, kbs, kts,                        \
                       B, S, Sk, Hq, Hkv, (float)scale, causal ? 1 : 0, rows_together(Hq / Hkv, 4L * Sk * DD), DEAL ? tiles : 0, 0);  \
  } while (0)
#define LAUNCH_FWD_D(NW, DEAL)            \
  do {                                     \
    if (D == 128) LAUNCH_FWD(128, NW, DEAL); \
    else LAUNCH_FWD(64, NW, DEAL);           \
  } while (0)

  const long blocks = (S + 4 * QW - 1L) / (4 * QW) * B * Hq;   // of four waves
  if (fwd_waves(blocks) == 2) LAUNCH_FWD_D(2, false);
  else if (causal && deals(S, B * Hq, blocks)) LAUNCH_FWD_D(4, true);
  else LAUNCH_FWD_D(4, false);
#undef LAUNCH_FWD
#undef LAUNCH_FWD_D
  HIP_CHECK_LAST();
  return {o, lse};
}

// Packed ragged batch: q/k/v [total, H, D]; cu_seqlens int32 [n_seq+1].
// lse is [Hq, total]. (reference varlen surface: flash-attn 2's
// _flash_attn_varlen_forward as consumed by colossalai .../attn.py:139)
std::vector<at::Tensor> flash_attn_varlen_fwd(at::Tensor q, at::Tensor k, at::Tensor v,
                                              at::Tensor cu_seqlens, long max_seqlen,
                                              bool causal, double scale) {
  using namespace fa;
  TORCH_CHECK(q.dim() == 3 && k.dim() == 3 && v.dim() == 3, "varlen: q/k/v must be [total,H,D]");
  TORCH_CHECK(cu_seqlens.scalar_type() == at::kInt && cu_seqlens.is_cuda() && cu_seqlens.dim() == 1);
  const int T = (int)q.size(0), Hq = (int)q.size(1), D = (int)q.size(2);
  const int Hkv = (int)k.size(1);
  const int n_seq = (int)cu_seqlens.numel() - 1;
  TORCH_CHECK(D == 64 || D == 128, "flash_attn: head dim must be 64 or 128");
  TORCH_CHECK(q.stride(2) == 1 && q.stride(1) == D, "varlen: q must be dense in [H,D]");
  TORCH_CHECK(k.strides() == v.strides() && k.sizes() == v.sizes());
  make_loadable(q);
  make_loadable(k, v);
  auto o = at::empty({T, Hq, D}, q.options());
  auto lse = at::empty({Hq, T}, q.options().dtype(at::kFloat));
  auto stream = at::hip::getCurrentHIPStream();
  const long qts = q.stride(0), kts = k.stride(0);

#define LAUNCH_VFWD(DD, NW)                                                                           \
  do {                                                                                            \
    const size_t lds = 4 * tile_bytes<KVB, DD>();                                                  \
    const long tiles = (max_seqlen + NW * QW - 1) / (NW * QW), packed = packed_tiles_fwd(T, n_seq, tiles, NW * QW, Hq, Hq / Hkv, D, causal);  \
    set_lds_limit((const void*)fa_fwd_kernel<DD, NW, true, true>, lds);                                 \
    hipLaunchKernelGGL((fa_fwd_kernel<DD, NW, true, true>),                                             \
                       packed ? wide_grid(dealt_blocks(packed, Hq)) : dim3((unsigned)tiles, n_seq * Hq), dim3(NW * 64), lds, stream.stream(), \
                       (const unsigned short*)q.data_ptr(), (const unsigned short*)k.data_ptr(),  \
                       (const unsigned short*)v.data_ptr(), (unsigned short*)o.data_ptr(),        \
                       lse.data_ptr<float>(), cu_seqlens.data_ptr<int>(), nullptr,                \
                       0L, qts, 0L, kts,                                                          \
                       n_seq, T, T, Hq, Hkv, (float)scale, causal ? 1 : 0, rows_together(Hq / Hkv, max_seqlen * DD * 4L), (int)packed, (int)tiles);  \
  } while (0)

  // blocks' worth of waves that have tokens, a sequence's last wave half of them (8 heads on 2 of 128, 23 samples of 8 to 128 tokens: 6.8 us, blocks of four 7.3)
  const long whole = (max_seqlen + 4 * QW - 1) / (4 * QW) * n_seq, some = T / (4 * QW) + n_seq / 8;
  const int nw = fwd_waves(std::min(whole, some) * Hq);
  if (D == 128) { if (nw == 4) LAUNCH_VFWD(128, 4); else LAUNCH_VFWD(128, 2); }
  else { if (nw == 4) LAUNCH_VFWD(64, 4); else LAUNCH_VFWD(64, 2); }
#undef LAUNCH_VFWD
  HIP_CHECK_LAST();
  return {o, lse};
}

namespace {

// The backward launch of dense (VARLEN = false) and packed batches. `seqs` sequences of at most S_max queries and
// Sk_max keys; S, Sk are the extents the kernels index with (tokens of the whole batch when packed).
template <int D, bool VARLEN>
void launch_bwd(const at::Tensor& q, const at::Tensor& k, const at::Tensor& v, const at::Tensor& dout, const at::Tensor& out,
                const at::Tensor& lse, at::Tensor& dq, at::Tensor& dk, at::Tensor& dv, const int* cu, const int* cuk,
                long qbs, long qts, long kbs, long kts, long dqbs, long dqts, long dkbs, long dkts, int seqs, int S_max,
                int Sk_max, int S, int Sk, int Hq, int Hkv, float scale, bool causal, hipStream_t stream) {
  using namespace fa;
  const int rows = NWB * QW;
  const int kv_tiles = (Sk_max + rows - 1) / rows, q_tiles = (S_max + rows - 1) / rows;
  const int G = Hq / Hkv;
  // Blocks that share a tile's group of heads (GS; the heads need not divide evenly).
  // Under a causal mask the first tile takes twice the average, and what is left of it when all else is done runs almost alone. The time by GS, in steps
  // of 32 query rows by 128 keys: all blocks' over the 512 that run at once (768 with 64 channels), the dQ part's 3/4 of a step included and 6 steps around
  // each block, at 1.75 us (1.65); what the longest takes beyond that at 1.12; the partial sums, written and read at 4.8 TB/s, and their launch. Packed
  // batches are taken to be half as long as their longest on average, or T / sequences. us, GS 1, 2, 4, * chosen: B1 S8192 H32/8 D128 1748, 1731 *, -;
  // B1 S4096 635, 462 *, 472; B2 S4096 894 *, 914, 952; B4 S2048 H16/4 332, 259 *, 272; D64 B1 S8192 H16/4 821, 564, 501 *; B2 S4096 H32/8 582, 508 *, 522;
  // packed 43 of up to 1024, H8/2 D128 175, 122 *, 146; 64 of 900 158, 116 *, 141; 85 of 512, H16/4 D64 96 *, 114, 139; 12 of 2048, H32/8 374, 364 *, 415.
  // Without a mask the work is even and it only matters that every CU has a block; a second one each pays where a block keeps 128 steps (16 over 2 of
  // 64, B1 S8192: 1413 -> 1134; 8 over 4 of 64, B16 S512: 58 -> 67). A block keeps at least 16 steps, of its heads' full length, or the
  // sums cost more than they save. The float32 sums take 8 bytes for each channel of these blocks' 128 rows: 134 MB at most.
  const long kv_blocks = (VARLEN ? (Sk + rows - 1) / rows : (long)kv_tiles * seqs) * Hkv;
  const bool sums_ok = dk.stride(-3) % 4 == 0 && (VARLEN || dk.stride(0) % 4 == 0) &&
                       reinterpret_cast<uintptr_t>(dk.data_ptr()) % 8 == 0 && reinterpret_cast<uintptr_t>(dv.data_ptr()) % 8 == 0;
  const double tokens = VARLEN ? S : (double)seqs * S, length = VARLEN ? std::max(tokens / std::max(seqs, 1), 0.5 * S_max) : S_max;
  const double tiles = VARLEN ? tokens / rows + 0.5 * seqs : (double)q_tiles * seqs;
  auto causal_us = [&](int d) {
    const double all = (1.75 * Hq * tokens / rows * (length / 64 + 2) + 6 * tiles * (Hq + (double)Hkv * d)) / (D == 64 ? 768 : 512);
    const double longest = (double)((S_max + 31) / 32) * ((G + d - 1) / d) + 6;
    return (D == 64 ? 1.65 : 1.75) * all + 1.12 * std::max(0.0, longest - all) + (d > 1 ? 3 + 16.0 * d * tokens * Hkv * D / 4.8e6 : 0.0);
  };
  int gs = 1;
  double us = causal ? causal_us(1) : 0.0;
  for (int most = G; most > 1 && sums_ok;) {
    most = (most + 1) / 2;                     // heads of a block, and blocks that take
    const int d = (G + most - 1) / most;
    const long steps = (long)((S_max + 31) / 32) * (G / d);
    if (steps < 16 || kv_blocks * d > (causal ? 1024 : steps >= 128 ? 512 : 510)) break;
    if (causal) {
      const double by_d = causal_us(d);
      if (by_d >= us) continue;
      us = by_d;
    }
    gs = d;
  }
  const long n_part = (VARLEN ? (long)Sk : (long)seqs * Sk) * Hkv * D;
  at::Tensor part;
  if (gs > 1) part = at::empty({gs * 2 * n_part}, q.options().dtype(at::kFloat));
  const int each = VARLEN ? 1 : seqs;
  auto even = [&](int n_y) { return fa::row_parts(n_y) == 1 ? q_tiles > 1 : worth_dealing(q_tiles, n_y); };
  const long dealt = VARLEN ? packed_tiles(S, seqs, q_tiles, rows, Hq) : causal && S_max == Sk_max && even(each * Hkv * gs) && even(each * Hq) ? q_tiles : 0;
  const long n_kv = dealt ? (dealt_blocks(dealt, each * Hkv * gs) + 7) / 8 * 8 : ((long)kv_tiles * seqs * Hkv * gs + 7) / 8 * 8;
  const long n_q = dealt ? dealt_blocks(dealt, each * Hq) : (long)q_tiles * seqs * Hq, blocks = n_kv + n_q;
  TORCH_CHECK(blocks < (1L << 31) - (1L << 23), "flash_attn_bwd: too many tiles");
  // Where all blocks run at once and have few query tiles they form the rows' statistics themselves: one launch and one tensor less for the host, which
  // bounds such calls (B8 S197 H12 D64, forward and backward through autograd: 75.9 -> 69.3 us); on the device B8 S197 H12 15.5 -> 14.7, B8 S250 H8 14.6 -> 14.5,
  // B4 S128 H12 10.7 -> 9.6, but B2 S512 H8 (16 tiles) 19 -> 22. With 128 channels B2 S256 H4 16.2 -> 19.9, B3 S100 H6/3 16.2 -> 19.4.
  const bool own = CAN_OWN<D, VARLEN> && blocks <= 512 && (long)((S_max + 31) / 32) * ((G + gs - 1) / gs) <= OWN_TILES &&
                   reinterpret_cast<uintptr_t>(out.data_ptr()) % 16 == 0;
  at::Tensor stats;
  if (!own) {   // (pad rows of O are zero -> delta 0)
    stats = at::empty({lse.numel(), 2}, lse.options());
    const long all = out.numel() / D;
    hipLaunchKernelGGL(fa_delta_kernel, dim3(capped_grid((all + 15) / 16, 4096)), dim3(256), 0, stream,
                       (const unsigned short*)dout.data_ptr(), (const unsigned short*)out.data_ptr(),
                       lse.data_ptr<float>(), (float2v*)stats.data_ptr(), all, S, Hq, D);
    HIP_CHECK_LAST();
  }
  auto kernel = fa_bwd_kernel<D, VARLEN>;
  const size_t lds = bwd_lds<D>() + (own ? OWN_TILES * 256 : 0);
  set_lds_limit((const void*)kernel, lds);
  hipLaunchKernelGGL(kernel, wide_grid(blocks), dim3(NTB), lds, stream,
                     (const unsigned short*)q.data_ptr(), (const unsigned short*)k.data_ptr(),
                     (const unsigned short*)v.data_ptr(), (const unsigned short*)dout.data_ptr(),
                     own ? nullptr : (const float2v*)stats.data_ptr(), (const unsigned short*)out.data_ptr(), lse.data_ptr<float>(), (unsigned short*)dq.data_ptr(), (unsigned short*)dk.data_ptr(),
                     (unsigned short*)dv.data_ptr(), gs > 1 ? part.data_ptr<float>() : nullptr, gs, cu, cuk, qbs, qts, kbs,
                     kts, dqbs, dqts, dkbs, dkts, (int)n_kv, (int)n_q, kv_tiles, q_tiles, seqs, S, Sk, Hq, Hkv, scale, causal ? 1 : 0,
                     rows_together(G, 4L * Sk_max * D), (int)dealt);
  HIP_CHECK_LAST();
  if (gs > 1) {
    hipLaunchKernelGGL(fa_bwd_sum_kernel, dim3((unsigned)((n_part / 4 + 255) / 256)), dim3(256), 0, stream,
                       (unsigned short*)dk.data_ptr(), (unsigned short*)dv.data_ptr(), part.data_ptr<float>(), gs, n_part, Sk,
                       Hkv * D, dkbs, dkts);
    HIP_CHECK_LAST();
  }
}

}  // namespace

// dq/dk/dv may be caller-provided strided views (e.g. into a packed dQKV
// buffer) to avoid post-hoc gathers; pass empty tensors to allocate.
std::vector<at::Tensor> flash_attn_bwd(at::Tensor dout, at::Tensor q, at::Tensor k, at::Tensor v,
                                       at::Tensor out, at::Tensor lse, bool causal, double scale,
                                       at::Tensor dq, at::Tensor dk, at::Tensor dv,
                                       c10::optional<at::Tensor> seqlens_opt,
                                       c10::optional<at::Tensor> seqlens_k_opt) {
  at::Tensor seqlens = seqlens_opt.has_value() ? *seqlens_opt : at::Tensor();
  at::Tensor seqlens_k = seqlens_k_opt.has_value() ? *seqlens_k_opt : at::Tensor();
  using namespace fa;
  check_fa_inputs(q, k, v);
  TORCH_CHECK(dout.is_contiguous() && out.is_contiguous() && lse.is_contiguous(),
              "flash_attn_bwd: dout/out/lse must be contiguous");
  make_loadable(q);
  make_loadable(k, v);
  make_loadable(dout);
  const int B = (int)q.size(0), S = (int)q.size(1), Hq = (int)q.size(2), D = (int)q.size(3);
  const int Hkv = (int)k.size(2);
  const int* cu = nullptr;
  const int* cuk = nullptr;
  if (seqlens.defined() && seqlens.numel() > 0) {
    TORCH_CHECK(seqlens.scalar_type() == at::kInt && seqlens.numel() == B && seqlens.is_cuda(),
                "flash_attn: seqlens must be int32 [B] on device");
    cu = seqlens.data_ptr<int>();
  }
  if (seqlens_k.defined() && seqlens_k.numel() > 0) {
    TORCH_CHECK(cu != nullptr, "flash_attn: seqlens_k requires seqlens");
    TORCH_CHECK(seqlens_k.scalar_type() == at::kInt && seqlens_k.numel() == B && seqlens_k.is_cuda());
    cuk = seqlens_k.data_ptr<int>();
  }
  const int Sk = (int)k.size(1);  // kv may be a shorter ring piece
  if (dq.numel() == 0) dq = at::empty({B, S, Hq, D}, q.options());
  if (dk.numel() == 0) dk = at::empty({B, Sk, Hkv, D}, k.options());
  if (dv.numel() == 0) dv = at::empty({B, Sk, Hkv, D}, v.options());
  check_fa_view(dq, "dq");
  check_fa_view(dk, "dk");
  TORCH_CHECK(dk.strides() == dv.strides(), "flash_attn_bwd: dk/dv strides must match");
  auto stream = at::hip::getCurrentHIPStream();

#define LAUNCH_BWD(DD)                                                                                               \
  launch_bwd<DD, false>(q, k, v, dout, out, lse, dq, dk, dv, cu, cuk, q.stride(0), q.stride(1), k.stride(0), k.stride(1), \
                        dq.stride(0), dq.stride(1), dk.stride(0), dk.stride(1), B, S, Sk, S, Sk, Hq, Hkv, (float)scale,      \
                        causal, stream.stream())
  if (D == 128) LAUNCH_BWD(128);
  else LAUNCH_BWD(64);
#undef LAUNCH_BWD
  return {dq, dk, dv};
}

std::vector<at::Tensor> flash_attn_varlen_bwd(at::Tensor dout, at::Tensor q, at::Tensor k, at::Tensor v,
                                              at::Tensor out, at::Tensor lse, at::Tensor cu_seqlens,
                                              long max_seqlen, bool causal, double scale) {
  using namespace fa;
  TORCH_CHECK(q.dim() == 3 && k.dim() == 3 && v.dim() == 3, "varlen: q/k/v must be [total,H,D]");
  TORCH_CHECK(dout.is_contiguous() && out.is_contiguous() && lse.is_contiguous());
  make_loadable(q);
  make_loadable(k, v);
  make_loadable(dout);
  const int T = (int)q.size(0), Hq = (int)q.size(1), D = (int)q.size(2);
  const int Hkv = (int)k.size(1);
  const int n_seq = (int)cu_seqlens.numel() - 1;
  auto dq = at::empty({T, Hq, D}, q.options());
  auto dk = at::empty({T, Hkv, D}, k.options());
  auto dv = at::empty({T, Hkv, D}, v.options());
  auto stream = at::hip::getCurrentHIPStream();

#define LAUNCH_VBWD(DD)                                                                                              \
  launch_bwd<DD, true>(q, k, v, dout, out, lse, dq, dk, dv, cu_seqlens.data_ptr<int>(), nullptr, 0L, q.stride(0), 0L,     \
                       k.stride(0), 0L, dq.stride(0), 0L, dk.stride(0), n_seq, (int)max_seqlen, (int)max_seqlen, T, T, Hq,  \
                       Hkv, (float)scale, causal, stream.stream())
  if (D == 128) LAUNCH_VBWD(128);
  else LAUNCH_VBWD(64);
#undef LAUNCH_VBWD
  return {dq, dk, dv};
}

}  // namespace cai
