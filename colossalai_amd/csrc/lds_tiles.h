// Operand tiles of the attention kernels in LDS, filled by loads that go there without registers in between.
#pragma once

#include "common.h"

namespace cai {

// An operand tile in LDS: pieces of 16 rows of 32 channels, 1024 bytes each, all row groups of a channel group one after the
// other. In a piece the four 16-byte units of a row lie together, unit u at place u ^ (row / 4 % 4). A piece is what
// one load instruction of a wave brings straight into LDS (16 bytes a lane in lane order, a quad of lanes 64 neighbouring bytes of a
// row), and every access spreads over the 64 banks: a row fragment (ds_read_b128) takes one unit of 16 consecutive
// rows, which lie in 16 different places of 16 bytes; a transposing read takes rows 0-7 or 8-15 of a piece as a whole.
template <int ROWS>
__host__ __device__ constexpr int piece_at(int row, int col) { return ((col >> 5) * (ROWS / 16) + (row >> 4)) * 1024; }

template <int ROWS, int COLS>
__host__ __device__ constexpr int tile_bytes() { return ROWS * COLS * 2; }

// Where a lane's 8 channels 16 * sl + 8 * half of row `ln` (and every 32nd row from it) lie: `even` for even sl, `odd` for
// odd ones, beyond which a fragment's piece is a constant.
struct RowAt {
  int even, odd;
  DEV_INLINE RowAt(int ln, int half) {
    const int place = half ^ (ln >> 2 & 3), at = (ln >> 4) * 1024 + (ln & 15) * 64;
    even = at + place * 16;
    odd = at + (place ^ 2) * 16;
  }
};
template <int ROWS>
DEV_INLINE bf16x8_v frag_row(const char* tile, const RowAt& at, int row0, int sl) {
  return *reinterpret_cast<const bf16x8_v*>(tile + (sl & 1 ? at.odd : at.even) + piece_at<ROWS>(row0, sl * 16));
}

// Column fragment by transposing reads, in the order in which the C layout hands out its rows: lane l
// receives tile[k_base + 8*(e>>2) + 4*(l>>5) + (e&3)][col + (l&31)], e = 0..7, so
// that a packed run of eight C registers is the matching other operand.
struct ColAt {
  int lo, hi;
  DEV_INLINE explicit ColAt(int lane) {
    const int m = lane & 15, half = lane >> 5;
    const int unit = (lane >> 4 & 1) * 2 + (m >> 1 & 1), row = half * 4 + (m >> 2);
    lo = row * 64 + (unit ^ half) * 16 + (m & 1) * 8;
    hi = (row + 8) * 64 + (unit ^ half ^ 2) * 16 + (m & 1) * 8;
  }
};
template <int ROWS>
DEV_INLINE bf16x8_v frag_born(const char* tile, const ColAt& at, int k_base, int col) {
  const bf16x4_v lo = ld_tr16(tile, at.lo + piece_at<ROWS>(k_base, col));
  const bf16x4_v hi = ld_tr16(tile, at.hi + piece_at<ROWS>(k_base, col));
  return __builtin_shufflevector(lo, hi, 0, 1, 2, 3, 4, 5, 6, 7);
}

typedef __attribute__((address_space(3))) void* lds_ptr;
typedef const __attribute__((address_space(1))) void* global_ptr;

// every load of this wave has arrived (in LDS); a barrier behind it makes that true for the block
DEV_INLINE void loads_done() { __builtin_amdgcn_s_waitcnt(0x0f70); }   // vmcnt(0)

// at most N vector memory operations of this wave are on their way; what follows reads what the others brought
template <int N>
DEV_INLINE void loads_left() {
  asm volatile("" ::: "memory");
  __builtin_amdgcn_s_waitcnt((N & 15) | ((N >> 4) << 14) | 0x0f70);
  asm volatile("" ::: "memory");
  __builtin_amdgcn_sched_barrier(0);
}

// At most N of this wave's LDS reads (where `ahead`, else none) are on their way.
template <int N>
DEV_INLINE void reads_left(bool ahead) {
  if (ahead) __builtin_amdgcn_s_waitcnt(0xc07f | N << 8);
  else __builtin_amdgcn_s_waitcnt(0xc07f);
  __builtin_amdgcn_sched_barrier(0);
}

}  // namespace cai
