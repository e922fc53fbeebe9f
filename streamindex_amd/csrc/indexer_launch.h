// Launchers of the lightning-indexer kernels and the per-shape instantiation
// macro used by indexer_inst_d*.hip: launch_topk (indexer_topk_kernel,
// indexer_kernels.h), launch_topk_wide (four 32-head blocks per wave,
// indexer_topk_wide.h; the C-ABI dispatch picks it for long rows) and
// launch_score.  Both top-k kernels return the same results.
#pragma once

#include "indexer_kernels.h"
#include "indexer_topk_few.h"
#include "indexer_topk_wide.h"

namespace si {

// ---------------------------------------------------------------------------
// Launchers.
// ---------------------------------------------------------------------------
template <int HB, int D, int C>
int launch_topk(const IndexerArgs& a, hipStream_t st) {
  if constexpr (!topk_fits_lds<HB, D, C>()) {
    return set_error(SI_ERR_UNSUPPORTED, "top_k too large for this head dim (the selection buffers exceed LDS)");
  } else {
  if (a.top_k > WaveSelect<C>::MAX_TOPK) return set_error(SI_ERR_UNSUPPORTED, "top_k exceeds the selection capacity");
  constexpr int NW = TopkShape<C>::NW;
  const int nqb = (a.S + NW - 1) / NW;
  const int64_t nblk = static_cast<int64_t>(nqb) * a.B;
  if (nblk > 0x7fffffffLL) return set_error(SI_ERR_UNSUPPORTED, "grid too large");
  if (a.mask) {
    hipLaunchKernelGGL((indexer_topk_kernel<HB, D, C, true>), dim3(static_cast<unsigned>(nblk)), dim3(NW * 64),
                       0, st, a);
  } else {
    hipLaunchKernelGGL((indexer_topk_kernel<HB, D, C, false>), dim3(static_cast<unsigned>(nblk)), dim3(NW * 64),
                       0, st, a);
  }
  return check_launch("indexer_topk_kernel");
  }
}

template <int HB, int D>
int launch_score(const IndexerArgs& a, hipStream_t st) {
  // 8 rows per workgroup (two waves per SIMD) up to two head blocks at
  // D <= 128; wider rows need a SIMD's registers for one wave.
  constexpr int NW = (HB <= 2 && D <= 128) ? 8 : 4;
  constexpr int TILE_N = 128;
  const int nqb = (a.S + NW - 1) / NW;
  const int64_t nblk = static_cast<int64_t>(nqb) * a.B;
  if (nblk > 0x7fffffffLL) return set_error(SI_ERR_UNSUPPORTED, "grid too large");
  // One workgroup runs on a CU at a time.  With fewer row groups than CUs the
  // keys are split as well: over the splits, the rounds of the grid times a
  // workgroup's tiles plus its prologue (the row's Q, about two tile times).
  const int tiles = (a.T + TILE_N - 1) / TILE_N;
  IndexerArgs c = a;
  c.score_tiles = tiles;
  int64_t best = (nblk + 255) / 256 * (tiles + 2);
  for (int y = 2; y <= 64 && y <= tiles && nblk < 512; ++y) {
    const int per = (tiles + y - 1) / y;
    const int64_t cost = (nblk * ((tiles + per - 1) / per) + 255) / 256 * (per + 2);
    if (cost < best) {
      best = cost;
      c.score_tiles = per;
    }
  }
  const int ny = (tiles + c.score_tiles - 1) / c.score_tiles;
  hipLaunchKernelGGL((indexer_score_kernel<HB, D, NW, TILE_N>),
                     dim3(static_cast<unsigned>(nblk), static_cast<unsigned>(ny)), dim3(NW * 64), 0, st, c);
  return check_launch("indexer_score_kernel");
}

template <int HB, int D>
int launch_score_direct(const IndexerArgs& a, hipStream_t st) {
  // Tiles per workgroup: two workgroups per CU first, then longer runs, which
  // load the row's Q (half a K tile at 64 heads) less often.
  const int64_t rows = static_cast<int64_t>(a.B) * a.S;
  const int all = (a.T + DirectShape<D>::TILE_N - 1) / DirectShape<D>::TILE_N;
  int64_t per = rows * all / 512;
  per = per < 1 ? 1 : (per > 16 ? 16 : per);
  const int64_t nwg = (all + per - 1) / per;
  hipLaunchKernelGGL((indexer_score_direct_kernel<HB, D>), dim3(static_cast<unsigned>(nwg), static_cast<unsigned>(rows)),
                     dim3(DirectShape<D>::NW * 64), 0, st, a, static_cast<int>(per));
  return check_launch("indexer_score_direct_kernel");
}

#define SI_INSTANTIATE_INDEXER(HB, D)                                   \
  template int launch_score<HB, D>(const IndexerArgs&, hipStream_t);    \
  template int launch_score_direct<HB, D>(const IndexerArgs&, hipStream_t); \
  template int launch_topk<HB, D, 256>(const IndexerArgs&, hipStream_t);  \
  template int launch_topk<HB, D, 512>(const IndexerArgs&, hipStream_t);  \
  template int launch_topk<HB, D, 1024>(const IndexerArgs&, hipStream_t); \
  template int launch_topk<HB, D, 1536>(const IndexerArgs&, hipStream_t); \
  template int launch_topk<HB, D, 2048>(const IndexerArgs&, hipStream_t); \
  template int launch_topk<HB, D, 4096>(const IndexerArgs&, hipStream_t);    \
  template int launch_topk_wide<HB, D, 1024>(const IndexerArgs&, hipStream_t); \
  template int launch_topk_wide<HB, D, 1536>(const IndexerArgs&, hipStream_t); \
  template int launch_topk_wide<HB, D, 2048>(const IndexerArgs&, hipStream_t);

}  // namespace si
