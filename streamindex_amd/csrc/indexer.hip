// Lightning-indexer C-ABI entries: argument validation and shape dispatch.
// Kernels: indexer_kernels.h (instantiated per head dim in indexer_inst_d*.hip).
#include <string>

#include "indexer_topk_few.h"

namespace si {

int g_topk_kernel_mode = 0;

// When the few-row top-k runs (few_worth): at most kFewMaxGroups four-row groups
// (one per CU), no causal ratio (its rows are short while they are few), and a
// scratch within kFewMaxScratch.  us a call (17 to 20 of them are the host's),
// one-wave-per-row kernel against this one, H = 64, D = 128, k = 512:
//   rows x keys   1 x 1,024   30 -> 22     4 x 16,384 (four batches)  203 -> 23
//   1 x 65,536   754 -> 27    1 x 262,144  2,910 -> 35
//   256 x 8,192  146 -> 45    512 x 32,768  460 -> 263
//   1,024 x 2,048   62 -> 55    1,024 x 32,000   511 -> 469   256 batches x 4,096  80 -> 54
// and past the line 1,536 x 2,048  79 -> 85, 2,048 x 32,000  818 -> 916: there
// the one-wave-per-row kernel fills the chip and saves the scores' round trip.
constexpr int64_t kFewMaxGroups = 256;
// (a bound on what a call allocates; 256 rows x 262,144 keys are just past it)
constexpr int64_t kFewMaxScratch = int64_t(256) << 20;

// Kernel and selection capacity for a top-k shape.  A compaction keeps
// between top_k and C - 192 keys; the capacity leaves room for several
// 64-key offers.  The four-M-block kernel (HB 2 and 4, D = 128, long rows)
// runs one workgroup per CU and stalls the CU while a row compacts, so it
// takes the largest capacity its LDS holds: compactions become rarer.
// Capacity 1536 rather than 1024 above top_k = 192 in the two-workgroup
// kernel: fewer compactions, still two workgroups per CU (measured 1.4 %
// faster at S = 64K, k = 512).  Shapes past what one wave holds (more than
// 128 heads, or 64 at D = 256) or past the four-row LDS budget (top_k above
// 2048, or 1536 at D = 256) run the head-split kernel.
static int plan_topk(const IndexerArgs& a, int D, TopkPlan* p) {
  if (D != 32 && D != 64 && D != 128 && D != 256)
    return set_error(SI_ERR_UNSUPPORTED, "unsupported indexer head dim D_I=" + std::to_string(D) +
                                             " (supported: 32, 64, 128, 256)");
  const int HB = (a.H + 31) / 32;
  if (HB > 8) return set_error(SI_ERR_UNSUPPORTED, "H_I > 256 is not supported");
  if (a.top_k > 4096) return set_error(SI_ERR_UNSUPPORTED, "top_k > 4096 is not supported");
  const int hb_one_wave = D == 256 ? 2 : 4;
  const int k_four_rows = D == 256 ? 1536 : 2048;
  if (HB <= hb_one_wave && a.top_k <= k_four_rows) {
    p->hb = HB;
    p->hs = 1;
    if (D == 128 && (HB == 2 || HB == 4) && a.top_k <= 1152 && topk_wide_preferred(a)) {
      p->kernel = TOPK_WIDE;
      p->cap = a.top_k <= 192 ? 1024 : (HB == 4 ? 2048 : 1536);
      return SI_OK;
    }
    p->kernel = TOPK_NARROW;
    p->cap = a.top_k <= 32 ? 256 : a.top_k <= 192 ? 512 : a.top_k <= 1152 ? 1536 : a.top_k <= 1536 ? 2048 : 4096;
    return SI_OK;
  }
  p->kernel = TOPK_SPLIT;
  if (D == 256) {
    p->hs = HB <= 4 ? 2 : 4;
    p->hb = HB <= 2 ? 1 : 2;
  } else {
    p->hs = 2;
    p->hb = HB <= 2 ? 1 : (HB <= 4 ? 2 : 4);
  }
  p->cap = a.top_k <= 1152 ? 1536 : 4608;
  return SI_OK;
}

template <int HB, int D>
static int launch_planned(const IndexerArgs& a, const TopkPlan& p, hipStream_t st) {
  if (p.kernel == TOPK_WIDE) {
    if constexpr (topk_wide_fits<HB, D, 1024>()) {
      if (p.cap == 1024) return launch_topk_wide<HB, D, 1024>(a, st);
      if (p.cap == 1536) return launch_topk_wide<HB, D, 1536>(a, st);
      if (p.cap == 2048) return launch_topk_wide<HB, D, 2048>(a, st);
    }
    return set_error(SI_ERR_UNSUPPORTED, "no four-M-block kernel for this plan");
  }
  switch (p.cap) {
    case 256: return launch_topk<HB, D, 256>(a, st);
    case 512: return launch_topk<HB, D, 512>(a, st);
    case 1536: return launch_topk<HB, D, 1536>(a, st);
    case 2048: return launch_topk<HB, D, 2048>(a, st);
    case 4096: return launch_topk<HB, D, 4096>(a, st);
    default: return set_error(SI_ERR_UNSUPPORTED, "no top-k kernel for this capacity");
  }
}

template <int D>
static int launch_split_planned(const IndexerArgs& a, const TopkPlan& p, hipStream_t st) {
#define SI_SPLIT(HS_, HBH_, C_) \
  if (p.hs == HS_ && p.hb == HBH_ && p.cap == C_) return launch_topk_split<HS_, HBH_, D, C_>(a, st);
  if constexpr (D == 256) {
    SI_SPLIT(2, 1, 4608)
    SI_SPLIT(2, 2, 1536)
    SI_SPLIT(2, 2, 4608)
    SI_SPLIT(4, 2, 1536)
    SI_SPLIT(4, 2, 4608)
  } else {
    SI_SPLIT(2, 1, 4608)
    SI_SPLIT(2, 2, 4608)
    SI_SPLIT(2, 4, 1536)
    SI_SPLIT(2, 4, 4608)
  }
#undef SI_SPLIT
  return set_error(SI_ERR_UNSUPPORTED, "no head-split kernel for this plan");
}

static int dispatch_topk(const IndexerArgs& a, int D, hipStream_t st) {
  TopkPlan p{};
  const int rc = plan_topk(a, D, &p);
  if (rc) return rc;
  if (p.kernel == TOPK_SPLIT) {
    switch (D) {
      case 32: return launch_split_planned<32>(a, p, st);
      case 64: return launch_split_planned<64>(a, p, st);
      case 128: return launch_split_planned<128>(a, p, st);
      default: return launch_split_planned<256>(a, p, st);
    }
  }
#define SI_CASE(HB_, D_) \
  if (p.hb == HB_ && D == D_) return launch_planned<HB_, D_>(a, p, st);
  SI_CASE(1, 32)
  SI_CASE(1, 64)
  SI_CASE(1, 128)
  SI_CASE(1, 256)
  SI_CASE(2, 32)
  SI_CASE(2, 64)
  SI_CASE(2, 128)
  SI_CASE(2, 256)
  SI_CASE(3, 32)
  SI_CASE(3, 64)
  SI_CASE(3, 128)
  SI_CASE(4, 32)
  SI_CASE(4, 64)
  SI_CASE(4, 128)
#undef SI_CASE
  return set_error(SI_ERR_UNSUPPORTED, "no top-k kernel for this plan");
}

// ---------------------------------------------------------------------------
// Few query rows, many keys: scores to a scratch, then a workgroup per row
// selects (indexer_topk_few.h).
// ---------------------------------------------------------------------------
struct FewPlan {
  bool use;
  int64_t sstride;  // floats per scratch score row
  int64_t segs;     // selection segments per row
  int64_t bytes;    // scratch: scores, then the segments' keys
};

// Whether the two passes are the faster ones (see kFewMaxGroups).  The lines, us of
// the one-wave-per-row kernel against the two passes on both sides:
//   * below 8 rows a batch each row reads the keys for itself, so its count of rows
//     is limited, not its groups: 256 x 1 row x 30,000 keys 426, 426 (D = 256: 691,
//     919; 128 x 1: 658, 497), 64 x 7 x 30,000 436, 510, 256 x 4 x 12,000 248, 501;
//   * a row costs more of the chip at D = 256 and from three head blocks on, which
//     the one-wave kernel fills with fewer rows: 1,024 x 30,000, D = 256 816, 911
//     (512 rows 691, 484); 128 x 8 x 12,000, H = 128 346, 401 (4,096 keys 137, 141);
//   * short rows of few picks, which the one-wave kernel hardly compacts: k = 16,
//     one row x 1,024 keys, H = 8 17, 20 (2,048 keys 24, 21); 1,024 rows x 3,000, H = 64
//     55, 64 (x 4,096, H = 8 55, 45); k = 128, one x 1,024, H = 32 18, 20 (2,048 27, 21).
static bool few_worth(const IndexerArgs& a, int D) {
  const int64_t rows = static_cast<int64_t>(a.B) * a.S;
  const int64_t groups = static_cast<int64_t>(a.B) * ((a.S + 3) / 4);
  const bool many = groups > kFewMaxGroups / 2;
  const int HB = (a.H + 31) / 32;
  if (groups > kFewMaxGroups) return false;
  if (a.S < 8 && rows > (D == 256 ? kFewMaxGroups / 2 : kFewMaxGroups)) return false;
  if (many && (D == 256 || (a.S >= 8 && HB >= 3 && a.T >= 8192))) return false;
  if (a.top_k >= 256 || HB >= 3) return a.T >= 1024;
  return a.T >= (many && a.top_k <= 64 ? 4096 : 2048);
}

static FewPlan few_plan(const IndexerArgs& a, int D) {
  FewPlan f{};
  TopkPlan p{};
  if (g_topk_kernel_mode != 0 || a.ratio > 0 || !few_worth(a, D)) return f;
  if (plan_topk(a, D, &p) != SI_OK || p.kernel == TOPK_SPLIT) return f;
  const int64_t rows = static_cast<int64_t>(a.B) * a.S;
  f.sstride = (static_cast<int64_t>(a.T) + 63) / 64 * 64;
  f.segs = (static_cast<int64_t>(a.T) + kFewSeg - 1) / kFewSeg;
  if (f.segs > 1 && f.segs * a.top_k > kFewMergeMax) return f;
  f.bytes = rows * f.sstride * 4 + (f.segs > 1 ? rows * f.segs * a.top_k * 8 : 0);
  if (f.bytes > kFewMaxScratch) return f;
  f.use = true;
  return f;
}

template <int HB, int D>
static int launch_few_score(const IndexerArgs& a, hipStream_t st) {
  return a.S < 8 ? launch_score_direct<HB, D>(a, st) : launch_score<HB, D>(a, st);
}

static int run_few(const IndexerArgs& a0, const FewPlan& f, int D, void* scratch, hipStream_t st) {
  IndexerArgs a = a0;
  a.scores = static_cast<float*>(scratch);
  a.ssb = a.S * f.sstride;
  a.sss = f.sstride;
  a.sst = 1;
  a.accumulate = 0;
  const int64_t rows = static_cast<int64_t>(a.B) * a.S;
  const int HB = (a.H + 31) / 32;
  int rc = -1;
#define SI_CASE(hb, d) \
  if (HB == hb && D == d) rc = launch_few_score<hb, d>(a, st);
  SI_CASE(1, 32)
  SI_CASE(1, 64)
  SI_CASE(1, 128)
  SI_CASE(1, 256)
  SI_CASE(2, 32)
  SI_CASE(2, 64)
  SI_CASE(2, 128)
  SI_CASE(2, 256)
  SI_CASE(3, 32)
  SI_CASE(3, 64)
  SI_CASE(3, 128)
  SI_CASE(4, 32)
  SI_CASE(4, 64)
  SI_CASE(4, 128)
#undef SI_CASE
  if (rc < 0) return set_error(SI_ERR_UNSUPPORTED, "no score kernel for this shape");
  if (rc) return rc;
  FewSelectArgs s{};
  s.scores = a.scores;
  s.sstride = f.sstride;
  s.n = a.T;
  s.S = a.S;
  s.top_k = a.top_k;
  s.mask = a.mask;
  s.msb = a.msb;
  s.mss = a.mss;
  s.mst = a.mst;
  s.out_idx = a.out_idx;
  s.out_scores = a.out_scores;
  if (f.segs > 1) s.seg_keys = reinterpret_cast<uint64_t*>(a.scores + rows * f.sstride);
  rc = launch_few_select(s, rows, false, st);
  if (rc || f.segs == 1) return rc;
  s.keys = s.seg_keys;
  s.n = static_cast<int>(f.segs * a.top_k);
  s.mask = nullptr;
  s.seg_keys = nullptr;
  return launch_few_select(s, rows, true, st);
}

// Materialised scores.  A launch covers up to four 32-head blocks (two at
// D = 256); wider rows run one launch per head group, each after the first
// adding its part to the scores already written (the same stream orders them).
static int dispatch_score(const IndexerArgs& a0, int D, hipStream_t st) {
  if (D != 32 && D != 64 && D != 128 && D != 256)
    return set_error(SI_ERR_UNSUPPORTED, "unsupported indexer head dim D_I=" + std::to_string(D) +
                                             " (supported: 32, 64, 128, 256)");
  if (a0.H > 256) return set_error(SI_ERR_UNSUPPORTED, "H_I > 256 is not supported");
  const int group = D == 256 ? 64 : 128;
  for (int h0 = 0; h0 < a0.H; h0 += group) {
    IndexerArgs a = a0;
    a.q = a0.q + static_cast<int64_t>(h0) * a0.qsh;
    a.w = a0.w_bf16 ? static_cast<const void*>(reinterpret_cast<const uint16_t*>(a0.w) + h0 * a0.wsh)
                    : static_cast<const void*>(reinterpret_cast<const float*>(a0.w) + h0 * a0.wsh);
    a.H = a0.H - h0 < group ? a0.H - h0 : group;
    a.accumulate = h0 > 0;
    const int HB = (a.H + 31) / 32;
    int rc = -1;
#define SI_CASE(hb, d) \
  if (HB == hb && D == d) rc = launch_score<hb, d>(a, st);
    SI_CASE(1, 32)
    SI_CASE(1, 64)
    SI_CASE(1, 128)
    SI_CASE(1, 256)
    SI_CASE(2, 32)
    SI_CASE(2, 64)
    SI_CASE(2, 128)
    SI_CASE(2, 256)
    SI_CASE(3, 32)
    SI_CASE(3, 64)
    SI_CASE(3, 128)
    SI_CASE(4, 32)
    SI_CASE(4, 64)
    SI_CASE(4, 128)
#undef SI_CASE
    if (rc < 0) return set_error(SI_ERR_UNSUPPORTED, "no score kernel for this shape");
    if (rc) return rc;
  }
  return SI_OK;
}

static int fill_common(IndexerArgs& a, const void* q, const int64_t* qs, const void* k, const int64_t* ks,
                       const void* w, int w_dtype, const int64_t* ws, int64_t B, int64_t S, int64_t T,
                       int64_t H, int64_t D) {
  if (!qs || !ks || !ws) return set_error(SI_ERR_INVALID, "null stride argument");
  if (B < 0 || S < 0 || T < 0 || H <= 0 || D <= 0) return set_error(SI_ERR_INVALID, "negative or zero dimension");
  // Empty tensors may carry a null data pointer; only non-empty ones are dereferenced.
  const bool rows = B > 0 && S > 0;
  if ((rows && (!q || !w)) || (B > 0 && T > 0 && !k)) return set_error(SI_ERR_INVALID, "null pointer argument");
  if (B > 0x7fffffff || S > 0x7fffffff || T > 0x7fffffff) return set_error(SI_ERR_UNSUPPORTED, "dimension exceeds int32");
  if (qs[3] != 1 || ks[2] != 1) return set_error(SI_ERR_INVALID, "q and k_idx need a contiguous last dimension");
  if ((qs[2] % 8) || (qs[1] % 8) || (qs[0] % 8) || (ks[1] % 8) || (ks[0] % 8))
    return set_error(SI_ERR_INVALID, "q/k_idx strides must be multiples of 8 elements (16-byte rows)");
  if (ks[1] < 0 || ks[1] >= (int64_t(1) << 23))  // tile loads address 128 rows with 32-bit byte offsets
    return set_error(SI_ERR_UNSUPPORTED, "k_idx row stride must be below 2^23 elements");
  if ((reinterpret_cast<uintptr_t>(q) | reinterpret_cast<uintptr_t>(k)) & 15)  // null is aligned
    return set_error(SI_ERR_INVALID, "q/k_idx must be 16-byte aligned");
  if (w_dtype != 0 && w_dtype != 1) return set_error(SI_ERR_INVALID, "weights dtype must be fp32 (0) or bf16 (1)");
  a.q = static_cast<const uint16_t*>(q);
  a.qsb = qs[0]; a.qss = qs[1]; a.qsh = qs[2];
  a.k = static_cast<const uint16_t*>(k);
  a.ksb = ks[0]; a.kst = ks[1];
  a.w = w; a.wsb = ws[0]; a.wss = ws[1]; a.wsh = ws[2];
  a.w_bf16 = w_dtype;
  a.B = static_cast<int>(B); a.S = static_cast<int>(S); a.T = static_cast<int>(T); a.H = static_cast<int>(H);
  return SI_OK;
}

}  // namespace si

using namespace si;

extern "C" int si_indexer_set_topk_kernel(int mode) {
  if (mode < 0 || mode > 2) return set_error(SI_ERR_INVALID, "top-k kernel mode must be 0 (auto), 1 or 2"), -1;
  const int prev = g_topk_kernel_mode;
  g_topk_kernel_mode = mode;
  return prev;
}

extern "C" int si_indexer_topk_plan(int64_t S, int64_t T, int64_t H, int64_t D, int64_t top_k,
                                    int64_t causal_ratio, int32_t* kernel, int32_t* capacity) {
  if (S < 0 || T < 0 || H <= 0 || D <= 0 || top_k <= 0 || causal_ratio < 0) return set_error(SI_ERR_INVALID, "bad dimension");
  if (S > 0x7fffffff || T > 0x7fffffff || H > 0x7fffffff || top_k > 0x7fffffff || causal_ratio > 0x7fffffff)
    return set_error(SI_ERR_UNSUPPORTED, "dimension exceeds int32");
  IndexerArgs a{};
  a.B = 1;
  a.S = static_cast<int>(S);
  a.T = static_cast<int>(T);
  a.H = static_cast<int>(H);
  a.top_k = static_cast<int>(top_k);
  a.ratio = static_cast<int>(causal_ratio);
  TopkPlan p{};
  const int rc = plan_topk(a, static_cast<int>(D), &p);
  if (rc) return rc;
  if (kernel) *kernel = p.kernel;
  if (capacity) *capacity = p.cap;
  return SI_OK;
}

extern "C" int64_t si_indexer_topk_scratch_bytes(int64_t B, int64_t S, int64_t T, int64_t H, int64_t D,
                                                 int64_t top_k, int64_t causal_ratio) {
  const int64_t lim = 0x7fffffff;
  if (B <= 0 || S <= 0 || T <= 0 || H <= 0 || top_k <= 0 || B > lim || S > lim || T > lim || H > lim || top_k > lim)
    return 0;
  IndexerArgs a{};
  a.B = static_cast<int>(B);
  a.S = static_cast<int>(S);
  a.T = static_cast<int>(T);
  a.H = static_cast<int>(H);
  a.top_k = static_cast<int>(top_k);
  a.ratio = causal_ratio > 0 ? 1 : 0;
  const FewPlan f = few_plan(a, static_cast<int>(D));
  return f.use ? f.bytes : 0;
}

extern "C" int si_indexer_topk(const void* q, const int64_t* q_strides, const void* k_idx,
                               const int64_t* k_strides, const void* weights, int w_dtype,
                               const int64_t* w_strides, const uint8_t* mask, const int64_t* mask_strides,
                               int64_t B, int64_t S, int64_t T, int64_t H, int64_t D, int64_t top_k,
                               int64_t causal_ratio, int64_t* out_idx, float* out_scores, void* stream) {
  return si_indexer_topk_scratch(q, q_strides, k_idx, k_strides, weights, w_dtype, w_strides, mask, mask_strides, B, S,
                                 T, H, D, top_k, causal_ratio, out_idx, out_scores, nullptr, 0, stream);
}

extern "C" int si_indexer_topk_scratch(const void* q, const int64_t* q_strides, const void* k_idx,
                                       const int64_t* k_strides, const void* weights, int w_dtype,
                                       const int64_t* w_strides, const uint8_t* mask, const int64_t* mask_strides,
                                       int64_t B, int64_t S, int64_t T, int64_t H, int64_t D, int64_t top_k,
                                       int64_t causal_ratio, int64_t* out_idx, float* out_scores, void* scratch,
                                       int64_t scratch_bytes, void* stream) {
  IndexerArgs a{};
  int rc = fill_common(a, q, q_strides, k_idx, k_strides, weights, w_dtype, w_strides, B, S, T, H, D);
  if (rc) return rc;
  if (top_k <= 0) return set_error(SI_ERR_INVALID, "top_k must be positive");
  if (causal_ratio < 0) return set_error(SI_ERR_INVALID, "causal_ratio must be positive");
  if (mask && causal_ratio > 0) return set_error(SI_ERR_INVALID, "specify either causal_mask or causal_ratio, not both");
  if (mask && !mask_strides) return set_error(SI_ERR_INVALID, "mask strides missing");
  if ((!out_idx || !out_scores) && B > 0 && S > 0) return set_error(SI_ERR_INVALID, "null output pointer");
  if (causal_ratio > 0x7fffffff) return set_error(SI_ERR_INVALID, "causal_ratio too large");
  a.top_k = static_cast<int>(top_k);
  a.ratio = static_cast<int>(causal_ratio);
  a.mask = mask;
  if (mask) { a.msb = mask_strides[0]; a.mss = mask_strides[1]; a.mst = mask_strides[2]; }
  a.out_idx = out_idx;
  a.out_scores = out_scores;
  if (a.B == 0 || a.S == 0) return SI_OK;
  if (scratch) {
    if (reinterpret_cast<uintptr_t>(scratch) & 15) return set_error(SI_ERR_INVALID, "scratch must be 16-byte aligned");
    const FewPlan f = few_plan(a, static_cast<int>(D));
    if (f.use && scratch_bytes >= f.bytes)
      return run_few(a, f, static_cast<int>(D), scratch, static_cast<hipStream_t>(stream));
  }
  return dispatch_topk(a, static_cast<int>(D), static_cast<hipStream_t>(stream));
}

extern "C" int si_csa_indexer_topk(const void* q, const int64_t* q_strides, const void* k_idx,
                                   const int64_t* k_strides, const void* weights, int w_dtype,
                                   const int64_t* w_strides, int64_t B, int64_t S, int64_t T, int64_t H,
                                   int64_t D, int64_t top_k, int64_t causal_ratio, int64_t n_win,
                                   int64_t idx_offset, int32_t* out_idx, const int64_t* out_strides,
                                   float* out_scores, void* stream) {
  IndexerArgs a{};
  int rc = fill_common(a, q, q_strides, k_idx, k_strides, weights, w_dtype, w_strides, B, S, T, H, D);
  if (rc) return rc;
  if (top_k <= 0) return set_error(SI_ERR_INVALID, "top_k must be positive");
  if (causal_ratio < 0 || causal_ratio > 0x7fffffff) return set_error(SI_ERR_INVALID, "bad causal_ratio");
  if (n_win < 0 || n_win > 0x7fffffff) return set_error(SI_ERR_INVALID, "n_win must be non-negative");
  if (idx_offset < 0 || idx_offset + T > 0x7fffffff)
    return set_error(SI_ERR_UNSUPPORTED, "idx_offset + T must fit in int32");
  if (!out_strides) return set_error(SI_ERR_INVALID, "null output strides");
  if (!out_idx && B > 0 && S > 0) return set_error(SI_ERR_INVALID, "null output pointer");
  if (out_strides[2] != 1) return set_error(SI_ERR_INVALID, "index rows must be contiguous");
  a.top_k = static_cast<int>(top_k);
  a.ratio = static_cast<int>(causal_ratio);
  a.out_idx = nullptr;
  a.out_scores = out_scores;
  a.out_idx32 = out_idx;
  a.o32sb = out_strides[0];
  a.o32ss = out_strides[1];
  a.n_win = static_cast<int>(n_win);
  a.idx_offset = static_cast<int>(idx_offset);
  if (a.B == 0 || a.S == 0) return SI_OK;
  return dispatch_topk(a, static_cast<int>(D), static_cast<hipStream_t>(stream));
}

extern "C" int si_indexer_score(const void* q, const int64_t* q_strides, const void* k_idx,
                                const int64_t* k_strides, const void* weights, int w_dtype,
                                const int64_t* w_strides, int64_t B, int64_t S, int64_t T, int64_t H,
                                int64_t D, float* scores, const int64_t* score_strides, void* stream) {
  IndexerArgs a{};
  int rc = fill_common(a, q, q_strides, k_idx, k_strides, weights, w_dtype, w_strides, B, S, T, H, D);
  if (rc) return rc;
  if (!score_strides || (!scores && B > 0 && S > 0 && T > 0)) return set_error(SI_ERR_INVALID, "null score output");
  a.scores = scores;
  a.ssb = score_strides[0]; a.sss = score_strides[1]; a.sst = score_strides[2];
  if (a.B == 0 || a.S == 0 || a.T == 0) return SI_OK;
  return dispatch_score(a, static_cast<int>(D), static_cast<hipStream_t>(stream));
}
