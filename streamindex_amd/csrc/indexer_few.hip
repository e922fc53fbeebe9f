// Instantiates the selection pass of the few-row top-k (indexer_topk_few.h).
#include "indexer_topk_few.h"

namespace si {

// Registers follow the segment's length, the sort width top_k: at least
// 2 top_k keys, so that the window of the floor search is wide.
template <int E, bool KEYS>
static int launch_few_e(const FewSelectArgs& f, int64_t rows, unsigned segs, hipStream_t st) {
  const dim3 grid(static_cast<unsigned>(rows), segs);
  if (f.top_k <= 512) {
    hipLaunchKernelGGL((few_select_kernel<E, 1, KEYS>), grid, dim3(kFewThreads), 0, st, f);
  } else if (f.top_k <= 1024) {
    hipLaunchKernelGGL((few_select_kernel<E, 2, KEYS>), grid, dim3(kFewThreads), 0, st, f);
  } else if (f.top_k <= 2048) {
    hipLaunchKernelGGL((few_select_kernel<E, 4, KEYS>), grid, dim3(kFewThreads), 0, st, f);
  } else {
    return set_error(SI_ERR_UNSUPPORTED, "top_k > 2048 in the few-row selection");
  }
  return check_launch("few_select_kernel");
}

int launch_few_select(const FewSelectArgs& f, int64_t rows, bool keys, hipStream_t st) {
  if (keys) {
    if (f.n > kFewMergeMax) return set_error(SI_ERR_UNSUPPORTED, "too many segments in the few-row selection");
    if (f.n <= 4 * kFewThreads) return launch_few_e<4, true>(f, rows, 1, st);
    if (f.n <= 16 * kFewThreads) return launch_few_e<16, true>(f, rows, 1, st);
    return launch_few_e<32, true>(f, rows, 1, st);
  }
  const unsigned segs = static_cast<unsigned>((f.n + kFewSeg - 1) / kFewSeg);
  if (f.n <= 4 * kFewThreads) return launch_few_e<4, false>(f, rows, segs, st);
  return launch_few_e<16, false>(f, rows, segs, st);
}

}  // namespace si
