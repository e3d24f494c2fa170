// Index vectors of a ragged step from the few numbers that each sequence brings. Made as Python lists they took the host 0.9 ms for
// a prompt of 4096 tokens, and some thirty small launches for the dense layout another 0.25, while the GPU waited: the engine's whole
// prompt (six layers, 2048 wide) 4030 us, 3530 with these two kernels and copies that the host does not wait for.
// A thread an entry; each finds its sequence by halving, in vectors that stay in L2.
#include <c10/hip/HIPGuard.h>

#include <algorithm>

#include "serving_common.h"

namespace cai {
namespace serving {

// the last b of [0, B) whose first[b] is not beyond i (first[0] <= i, ascending)
DEV_INLINE int owner(const int* __restrict__ first, int B, long i) {
  int lo = 0, hi = B;
  while (hi - lo > 1) {
    const int mid = (lo + hi) >> 1;
    if (first[mid] <= i) lo = mid;
    else hi = mid;
  }
  return lo;
}

// buf: cu [B + 1], start [B], slots [B], tables [B, width] | tok_seq [N], positions [N], and where width > 0 rows [N]
__global__ __launch_bounds__(256) void ragged_index_kernel(int* __restrict__ buf, int B, int N, int width, int page_size) {
  const int i = blockIdx.x * 256 + threadIdx.x;
  if (i >= N) return;
  const int* cu = buf;
  const int* tables = buf + 3 * B + 1;
  int* tok = buf + 3 * B + 1 + (long)B * width;
  const int b = owner(cu, B, i), pos = buf[B + 1 + b] + i - cu[b];
  tok[i] = b;
  tok[(long)N + i] = pos;
  if (width > 0) tok[2L * N + i] = tables[(long)b * width + pos / page_size] * page_size + pos % page_size;
}

// The dense layout of whole contexts: each sequence's pages from its page `skip` on, one sequence after the other. of [4, B]: a sequence's first
// page there, its pages, its length, skip. rows [total]: pool row of each place (past the end: of the last one); tables [B, width].
__global__ __launch_bounds__(256) void dense_context_kernel(long* __restrict__ rows, int* __restrict__ tables,
                                                            const int* __restrict__ block_tables, long bt_stride,
                                                            const int* __restrict__ of, int B, long total, int width, int page_size) {
  const long i = (long)blockIdx.x * 256 + threadIdx.x;
  const int *first = of, *pages = of + B, *lens = of + 2 * B, *skip = of + 3 * B;
  if (i < total) {
    const int page = (int)(i / page_size), b = owner(first, B, page);
    const int pos = min((int)(i - (long)(first[b] - skip[b]) * page_size), lens[b] - 1);
    rows[i] = (long)block_tables[b * bt_stride + pos / page_size] * page_size + pos % page_size;
  } else if (i < total + (long)B * width) {
    const long k = i - total;
    const int b = (int)(k / width), c = (int)(k % width) - skip[b];
    tables[k] = c >= 0 && c < pages[b] ? first[b] + c : 0;
  }
}

void ragged_index(at::Tensor buf, int64_t B, int64_t N, int64_t width, int64_t page_size) {
  check_i32(buf, "buf");
  TORCH_CHECK(B > 0 && N > 0 && width >= 0 && N < (1L << 30) && B <= N && (width == 0 || (page_size > 0 && page_size < (1L << 31))) &&
              buf.numel() == 3 * B + 1 + 2 * N + (width > 0 ? B * width + N : 0), "ragged_index: sizes do not fit");
  const c10::hip::HIPGuard guard(buf.device().index());
  ragged_index_kernel<<<dim3((unsigned)((N + 255) / 256)), dim3(256), 0, stream()>>>(buf.data_ptr<int>(), (int)B, (int)N, (int)width,
                                                                                     (int)page_size);
  HIP_CHECK_LAST();
}

void dense_context(at::Tensor rows, at::Tensor tables, at::Tensor block_tables, at::Tensor of, int64_t page_size) {
  check_i32(tables, "tables"); check_i32(of, "of");
  TORCH_CHECK(block_tables.is_cuda() && block_tables.scalar_type() == at::kInt && block_tables.dim() == 2 && block_tables.stride(1) == 1 &&
              rows.is_cuda() && rows.scalar_type() == at::kLong && rows.is_contiguous() && tables.dim() == 2 && of.dim() == 2 &&
              of.size(0) == 4 && of.size(1) == tables.size(0) && block_tables.size(0) == tables.size(0) && page_size > 0 &&
              page_size < (1L << 31) && block_tables.size(1) >= tables.size(1), "dense_context: vectors do not fit");
  const long total = rows.numel(), all = total + tables.numel();
  TORCH_CHECK(total > 0 && all < (1L << 38), "dense_context: sizes do not fit");
  const c10::hip::HIPGuard guard(rows.device().index());
  dense_context_kernel<<<dim3((unsigned)((all + 255) / 256)), dim3(256), 0, stream()>>>(
      (long*)rows.data_ptr<int64_t>(), tables.data_ptr<int>(), block_tables.data_ptr<int>(), (long)block_tables.stride(0), of.data_ptr<int>(),
      (int)tables.size(0), total, (int)tables.size(1), (int)page_size);
  HIP_CHECK_LAST();
}

}  // namespace serving
}  // namespace cai
