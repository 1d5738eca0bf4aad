// Per-target source counts of a prefill chunk (aether_2b/modeling.py:316-319 HCA, :521-534 CSA): which
// blocks and which slice of the window each target sees, a closed form of its position.
//
// Bound by the launch (four int32 per target).  Filled on the device because the same arrays made on
// the host cost a chunk four pageable copies, each a synchronisation of the stream: with them the
// 8 x 256 target CSA chunk took 250 us for 152 us of kernels, a 3001-target HCA chunk 142 us for 80.
#include "aekv_common.h"

namespace aekv {
namespace {

constexpr int kThreads = 256;

__global__ __launch_bounds__(kThreads) void prefill_counts_kernel(int32_t rows, int32_t T, int64_t start, int64_t n_blocks,
                                                                  int64_t compression, int64_t sliding_window,
                                                                  int64_t window_base, int64_t k,
                                                                  int32_t* __restrict__ visible,
                                                                  int32_t* __restrict__ selected,
                                                                  int32_t* __restrict__ win_start,
                                                                  int32_t* __restrict__ win_len) {
  const int32_t r = static_cast<int32_t>(blockIdx.x) * kThreads + static_cast<int32_t>(threadIdx.x);
  if (r >= rows) return;
  const int64_t p = start + static_cast<uint32_t>(r) % static_cast<uint32_t>(T);
  const int64_t whole = p / compression;
  const int64_t vis = whole < n_blocks ? whole : n_blocks;
  const int64_t from = p - sliding_window + 1;
  const int64_t first = from > 0 ? from : 0;
  visible[r] = static_cast<int32_t>(vis);
  if (selected) selected[r] = static_cast<int32_t>(vis < k ? vis : k);
  win_start[r] = static_cast<int32_t>(first - window_base);
  win_len[r] = static_cast<int32_t>(p - first + 1);
}

}  // namespace
}  // namespace aekv

using namespace aekv;

extern "C" int aekv_prefill_counts(int64_t B, int64_t T, int64_t start, int64_t n_blocks, int64_t compression,
                                   int64_t sliding_window, int64_t window_base, int64_t k, int32_t* visible,
                                   int32_t* selected, int32_t* win_start, int32_t* win_len, void* stream) {
  const char* who = "aekv_prefill_counts";
  if (B < 0 || T < 0 || start < 0 || n_blocks < 0 || k < 0) return fail(AEKV_ERR_VALUE, "%s: negative size", who);
  if (compression < 1 || sliding_window < 1)
    return fail(AEKV_ERR_VALUE, "compression and sliding_window must be positive");
  if (B == 0 || T == 0) return AEKV_OK;
  if (T > (0x7fffffff - kThreads) / B) return fail(AEKV_ERR_UNSUPPORTED, "%s: B*T exceeds 2^31", who);
  if (!visible || !win_start || !win_len) return fail(AEKV_ERR_VALUE, "%s: null pointer", who);
  const int32_t rows = static_cast<int32_t>(B * T);
  hipLaunchKernelGGL(prefill_counts_kernel, dim3(static_cast<uint32_t>(ceil_div(rows, kThreads))), dim3(kThreads), 0,
                     as_stream(stream), rows, static_cast<int32_t>(T), start, n_blocks, compression, sliding_window,
                     window_base, k, visible, selected, win_start, win_len);
  return check_launch(who);
}
