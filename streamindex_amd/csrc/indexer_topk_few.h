// Exact top-k for calls with few query rows and many keys (decode steps,
// chunks of a longer prompt), in two passes over a caller-provided scratch.
//
// indexer_topk_kernel gives a query row one wave, which walks all T keys: with
// fewer row groups than the chip has workgroup slots, most CUs idle while the
// call takes T / 64 tile times.  Here the keys are split over the chip instead:
//   1. scores: [rows, T] fp32 into the scratch, by indexer_score_kernel over
//      T chunks (8 query rows share a K tile), or, below 8 query rows per
//      batch, by indexer_score_direct_kernel, whose waves share one query row
//      and split the keys.
//   2. few_select_kernel: one workgroup per row holds the row's ordered
//      scores in registers, finds a floor that keeps between top_k and SORTN
//      keys, and orders those keys.  Rows longer
//      than kFewSeg keys run one workgroup per segment and a second launch of
//      the same kernel over the segments' sorted keys.
// Scores are formed by the same fp32 operations in the same order as in
// indexer_topk_kernel and ranked by the same 64-bit keys, so the results are
// identical bit for bit.
// Bound: latency (few rows), then the MFMA rate of the score pass.  At B = 4,
// S = 1, T = 16,384, H = 64, k = 512: scores 7 us, selection 8.4 us, against
// 203 us in indexer_topk_kernel; 256 rows x 8,257 keys: 42 + 10 against 163 us.
// Dispatch and its figures: few_plan (indexer.hip).
#pragma once

#include "indexer_kernels.h"

namespace si {

// Selection workgroup.  Its code runs once, straight through, so it is bound
// by instruction fetch and latency: 16 keys per thread and 16 waves take
// fewer cycles than 64 keys per thread and 4 waves, whose unrolled passes over
// the keys are four times the code.
constexpr int kFewThreads = 1024;
constexpr int kFewWaves = kFewThreads / kWave;
constexpr int kFewSeg = 16 * kFewThreads;       // keys of one selection workgroup
constexpr int kFewMergeMax = 32 * kFewThreads;  // keys of the merging workgroup

// Scores of one query row per grid row (y): the waves of a workgroup take the
// 32-key blocks of a K tile, so a row's keys spread over blockIdx.x
// workgroups of `tiles` tiles each.  K tiles, and the row's Q, come
// through LDS like the other kernels' (a fragment load straight from memory
// touches 32 lines per instruction: 11 against 7 us at
// B = 4, T = 16,384).
template <int D>
struct DirectShape {
  static constexpr int NW = D <= 128 ? 4 : 2;  // waves, and 32-key blocks per tile
  static constexpr int TILE_N = 32 * NW;
};

template <int HB, int D>
__global__ __launch_bounds__(DirectShape<D>::NW * 64) void indexer_score_direct_kernel(IndexerArgs a, int tiles) {
  constexpr int NW = DirectShape<D>::NW;
  constexpr int NT = NW * 64;
  constexpr int TILE_N = DirectShape<D>::TILE_N;
  constexpr int KS = D / 16;
  constexpr int QROWS = HB * 32;
  constexpr int TILE_BYTES = TILE_N * D * 2;
  __shared__ __attribute__((aligned(16))) char lds[QROWS * D * 2 + 2 * TILE_BYTES];
  __shared__ __attribute__((aligned(16))) float wl[QROWS];
  char* const kt = lds + QROWS * D * 2;
  const int lane = threadIdx.x & 63;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int row = blockIdx.y;
  const int b = row / a.S, s = row % a.S;
  const int it0 = static_cast<int>(blockIdx.x) * tiles;
  const int all = (a.T + TILE_N - 1) / TILE_N;
  const int it1 = it0 + tiles < all ? it0 + tiles : all;  // it0 < all: the grid covers the row's tiles

  const uint16_t* qrow = a.q + b * a.qsb + static_cast<int64_t>(s) * a.qss;
  const uint16_t* kb = a.k + b * a.ksb;
  KTileLoader<D, TILE_N, NT> ld;
  ld.init(a.kst);
  ld.issue(kb, a.kst, it0 * TILE_N, a.T, kt);
  constexpr int CPR = D / 8;
#pragma unroll
  for (int i = 0; i < (QROWS * CPR + NT - 1) / NT; ++i) {  // (zero past H)
    const int e = i * NT + static_cast<int>(threadIdx.x);
    if (QROWS * CPR % NT == 0 || e < QROWS * CPR) {
      const int h = e / CPR, c = e % CPR;
      const u32x4 v = h < a.H ? *reinterpret_cast<const u32x4*>(qrow + h * a.qsh + c * 8) : u32x4{0u, 0u, 0u, 0u};
      *reinterpret_cast<u32x4*>(lds + kt_off<D>(h, c)) = v;
    }
  }
  for (int h = threadIdx.x; h < QROWS; h += NT) {
    float wv = 0.f;
    if (h < a.H) {
      const int64_t off = b * a.wsb + static_cast<int64_t>(s) * a.wss + h * a.wsh;
      wv = a.w_bf16 ? bf16_bits_to_f32(reinterpret_cast<const uint16_t*>(a.w)[off])
                    : reinterpret_cast<const float*>(a.w)[off];
    }
    wl[h] = wv;
  }
  tile_barrier();
  QueryFrags<HB, D> qfr;
#pragma unroll
  for (int mb = 0; mb < HB; ++mb) {
    const int h = mb * 32 + (lane & 31);
#pragma unroll
    for (int ks = 0; ks < KS; ++ks)
      qfr.qf[mb][ks] = *reinterpret_cast<const bf16x8*>(lds + kt_off<D>(h, ks * 2 + (lane >> 5)));
#pragma unroll
    for (int c = 0; c < 4; ++c) {
      const f32x4 w4 = *reinterpret_cast<const f32x4*>(&wl[mb * 32 + 8 * c + 4 * (lane >> 5)]);
#pragma unroll
      for (int v = 0; v < 4; ++v) qfr.wf[mb][4 * c + v] = w4[v];
    }
  }
  float* orow = a.scores + b * a.ssb + static_cast<int64_t>(s) * a.sss;
  for (int it = it0; it < it1; ++it) {
    const char* tile = kt + ((it - it0) & 1) * TILE_BYTES;
    if (it + 1 < it1) ld.issue(kb, a.kst, (it + 1) * TILE_N, a.T, kt + ((it + 1 - it0) & 1) * TILE_BYTES);
    bf16x8 kf[KS];
    qfr.load_b(tile, wave, lane, kf);
    const float p = qfr.partial(kf);
    const SwapPair r = permlane32_swap(__float_as_uint(p), __float_as_uint(p));
    const float v = __uint_as_float(r.x) + __uint_as_float(r.y);
    const int t = it * TILE_N + wave * 32 + (lane & 31);
    if (lane < 32 && t < a.T) orow[t] = v;
    tile_barrier();
  }
}

struct FewSelectArgs {
  const float* scores;  // [rows, sstride] (score input)
  int64_t sstride;
  const uint64_t* keys;  // [rows, n] selection keys (key input)
  int n;                 // keys per row
  int S;
  int top_k;
  const uint8_t* mask;   // optional [B,S,n]
  int64_t msb, mss, mst;
  uint64_t* seg_keys;    // [rows, segments, top_k] when the row has several segments, else null
  int64_t* out_idx;      // [rows, top_k]
  float* out_scores;
};

// Reduction of the values lanes 0..15 hold (the other 16-lane rows hold the
// same), returned uniformly.
template <typename F>
__device__ __forceinline__ uint32_t row16_reduce(uint32_t x, F op) {
  x = op(x, static_cast<uint32_t>(__builtin_amdgcn_mov_dpp(static_cast<int>(x), 0xB1, 0xf, 0xf, false)));
  x = op(x, static_cast<uint32_t>(__builtin_amdgcn_mov_dpp(static_cast<int>(x), 0x4E, 0xf, 0xf, false)));
  x = op(x, static_cast<uint32_t>(__builtin_amdgcn_mov_dpp(static_cast<int>(x), 0x141, 0xf, 0xf, false)));
  x = op(x, static_cast<uint32_t>(__builtin_amdgcn_mov_dpp(static_cast<int>(x), 0x140, 0xf, 0xf, false)));
  return static_cast<uint32_t>(__builtin_amdgcn_readfirstlane(static_cast<int>(x)));
}

__device__ __forceinline__ float wave_sum_f32(float x) {
#pragma unroll
  for (int d = 1; d < kWave; d <<= 1) x += __shfl_xor(x, d, kWave);
  return x;
}

// Inclusive sum over the lanes up to this one.
__device__ __forceinline__ int wave_prefix_sum(int x, int lane) {
#pragma unroll
  for (int d = 1; d < kWave; d <<= 1) {
    const int y = __shfl_up(x, d, kWave);
    x += lane >= d ? y : 0;
  }
  return x;
}

// One workgroup per (row, segment).  E: keys of the segment per thread; ES:
// kept keys per thread (SORTN = 1024 ES keys, at least 2 top_k).  KEYS: the
// input is 64-bit selection keys (the merge of the segments), not scores.
//
// A row is one workgroup's serial chain, so the steps are chosen for their
// latency:
//   * the floor that keeps [top_k, SORTN] keys: the first probe is the quantile
//     of a normal distribution with the scores' mean and variance (a score
//     sums many heads), later ones search as WaveSelect::compact_to does (a
//     probe is 2,000 cycles; from a cold start it takes five);
//   * the order: kept keys go to the bins of a histogram that is linear in the
//     score, each key then ranks itself among the few of its bin.  Rows with
//     crowded bins (ties, outliers) take the bitonic sort instead (11,000
//     cycles at 1,024 keys).
template <int E, int ES, bool KEYS>
__global__ __launch_bounds__(kFewThreads) void few_select_kernel(FewSelectArgs a) {
  constexpr int W = kFewWaves;
  constexpr int WAVE_KEYS = ES * kWave;
  constexpr int SORTN = W * WAVE_KEYS;
  constexpr int BPT = 2 * ES;  // bins per thread: two bins per kept key
  constexpr int BINS = BPT * kFewThreads;
  constexpr int CROWD = 24;    // most keys of a bin that rank themselves
  static_assert(E % 4 == 0, "scores are loaded four at a time");
  __shared__ __attribute__((aligned(16))) uint64_t sbuf[SORTN], rbuf[SORTN];
  __shared__ __attribute__((aligned(16))) int hist[BINS + 1];
  __shared__ __attribute__((aligned(16))) int cnt[2][kFewWaves];
  __shared__ __attribute__((aligned(16))) uint32_t wmax[kFewWaves];
  __shared__ __attribute__((aligned(16))) float wsum[kFewWaves], wsq[kFewWaves];
  static_assert(kFewWaves == 16, "the waves' values are combined within a 16-lane row");

  const int tid = threadIdx.x;
  const int lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int64_t row = blockIdx.x;
  const int t0 = static_cast<int>(blockIdx.y) * kFewSeg;
  auto index = [&](int j) { return t0 + ((j >> 2) * kFewThreads + tid) * 4 + (j & 3); };

  // ---- the segment's ordered scores (0: no key) ----------------------------
  uint32_t hi[E];
  uint32_t lo[KEYS ? E : 1];
  if constexpr (KEYS) {
    const uint64_t* src = a.keys + row * a.n;
#pragma unroll
    for (int j = 0; j < E; ++j) {
      const int t = index(j);
      const uint64_t k = src[t < a.n ? t : a.n - 1];
      hi[j] = t < a.n ? key_hi(k) : 0u;
      lo[j] = static_cast<uint32_t>(k);
    }
  } else {
    // (score rows are padded to whole 64-key groups, so a group of four that
    // starts inside the row is inside the scratch)
    const float* src = a.scores + row * a.sstride;
    f32x4 x[E / 4];
#pragma unroll
    for (int j = 0; j < E; j += 4) {
      const int t = index(j);
      x[j / 4] = *reinterpret_cast<const f32x4*>(src + (t < a.n ? t : 0));
    }
    if (a.mask) {
      const uint8_t* mrow = a.mask + (row / a.S) * a.msb + (row % a.S) * a.mss;
#pragma unroll
      for (int j = 0; j < E; ++j) {
        const int t = index(j);
        const bool ok = mrow[static_cast<int64_t>(t < a.n ? t : a.n - 1) * a.mst] != 0 && t < a.n;
        hi[j] = ok ? f32_to_ord(x[j / 4][j & 3]) : 0u;
      }
    } else {
#pragma unroll
      for (int j = 0; j < E; ++j) hi[j] = index(j) < a.n ? f32_to_ord(x[j / 4][j & 3]) : 0u;
    }
  }
  auto key = [&](int j) -> uint64_t {
    const uint32_t l = KEYS ? lo[KEYS ? j : 0] : ~static_cast<uint32_t>(index(j));
    return (static_cast<uint64_t>(hi[j]) << 32) | l;
  };

  // Sum over the workgroup of a wave-uniform count, returned uniformly.  The
  // two buffers make one barrier per sum enough: a buffer is written again
  // only after the next sum's barrier, which every wave passes after its reads.
  int par = 0;
  auto block_sum = [&](int c) {
    par ^= 1;
    if (lane == 0) cnt[par][wave] = c;
    __syncthreads();
    return static_cast<int>(row16_reduce(static_cast<uint32_t>(cnt[par][lane & 15]),
                                         [](uint32_t x, uint32_t y) { return x + y; }));
  };
  // Sum of cnt[par] over the waves below this one.
  auto waves_below = [&]() {
    return static_cast<int>(row16_reduce((lane & 15) < wave ? static_cast<uint32_t>(cnt[par][lane & 15]) : 0u,
                                         [](uint32_t x, uint32_t y) { return x + y; }));
  };
  // (counted per lane, then summed over the wave: a ballot per key keeps a mask
  // register pair per key, more than there are)
  auto count = [&](auto keep) {
    uint32_t c = 0;
#pragma unroll
    for (int j = 0; j < E; ++j) c += keep(j) ? 1u : 0u;
    return block_sum(static_cast<int>(wave_sum_u32(c)));
  };

  // ---- keys held, their greatest score, mean and variance -------------------
  uint32_t mx = 0, held = 0;
  float fsum = 0.f, fsq = 0.f;
#pragma unroll
  for (int j = 0; j < E; ++j) {
    mx = hi[j] > mx ? hi[j] : mx;
    const bool in = hi[j] != 0u;
    const float f = in ? ord_to_f32(hi[j]) : 0.f;
    held += in ? 1u : 0u;
    fsum += f;
    fsq = __builtin_fmaf(f, f, fsq);
  }
  mx = wave_max_u32(mx);
  fsum = wave_sum_f32(fsum);
  fsq = wave_sum_f32(fsq);
  if (lane == 0) {
    wmax[wave] = mx;
    wsum[wave] = fsum;
    wsq[wave] = fsq;
  }
#pragma unroll
  for (int i = 0; i < BPT; ++i) hist[i * kFewThreads + tid] = 0;
  const int n = block_sum(static_cast<int>(wave_sum_u32(held)));  // (its barrier also publishes the above)
  auto max_op = [](uint32_t x, uint32_t y) { return x > y ? x : y; };
  auto sum_op = [](uint32_t x, uint32_t y) { return __float_as_uint(__uint_as_float(x) + __uint_as_float(y)); };
  mx = row16_reduce(wmax[lane & 15], max_op);

  // ---- the floor: kept keys are those whose score word is at least floor_hi
  // or, after a mass tie, the keys >= floor_key --------------------------------
  uint32_t floor_hi = 1u;  // every key
  uint64_t floor_key = 0;
  int kept = n;
  if (n > SORTN) {
    const int kk = a.top_k;
    const int target = kk + (SORTN - kk) / 2;
    uint64_t lo_ = 0, hi_ = static_cast<uint64_t>(mx) + 1;
    int c_lo = n, c_hi = 0;
    bool found = false;
    // Upper target/n quantile of the normal distribution (Abramowitz & Stegun
    // 26.2.22); only the first probe depends on it.
    uint32_t first = 0;
    {
      const float inv = __builtin_amdgcn_rcpf(static_cast<float>(n));
      const float mean = __uint_as_float(row16_reduce(__float_as_uint(wsum[lane & 15]), sum_op)) * inv;
      const float var = __uint_as_float(row16_reduce(__float_as_uint(wsq[lane & 15]), sum_op)) * inv - mean * mean;
      const float tail = static_cast<float>(target) * inv;
      const float q = tail < 0.5f ? tail : 1.f - tail;
      const float u = __builtin_sqrtf(-2.f * __logf(q));
      const float z = u - (2.30753f + 0.27061f * u) / (1.f + u * (0.99229f + 0.04481f * u));
      const float guess = mean + (tail < 0.5f ? z : -z) * __builtin_sqrtf(var);
      if (guess == guess) first = __builtin_amdgcn_readfirstlane(f32_to_ord(guess));
    }
    for (int it = 0; it < 48 && hi_ - lo_ > 1; ++it) {
      const uint64_t span = hi_ - lo_;
      uint64_t step;
      if (it == 0 && first > 0u) {
        step = first;
      } else if (it & 1) {
        step = span >> 1;
      } else {
        const float f = static_cast<float>(c_lo - target) * __builtin_amdgcn_rcpf(static_cast<float>(c_lo - c_hi));
        const float half_span = static_cast<float>(static_cast<uint32_t>(span >> 1));
        step = static_cast<uint64_t>(static_cast<uint32_t>(half_span * __builtin_fminf(f, 1.0f))) << 1;
      }
      step = step < 1 ? 1 : (step > span - 1 ? span - 1 : step);
      const uint32_t mid = static_cast<uint32_t>(lo_ + step);
      kept = count([&](int j) { return hi[j] >= mid; });
      if (kept >= kk && kept <= SORTN) {
        found = true;
        floor_hi = mid;
        break;
      }
      if (kept > SORTN) {
        lo_ = mid;
        c_lo = kept;
      } else {
        hi_ = mid;
        c_hi = kept;
      }
    }
    if (!found) {
      // many keys share one score: bisect the full key (all distinct, so a
      // count changes by one per key and the window is always hit)
      uint64_t plo = lo_ << 32;
      uint64_t phi = hi_ >= (1ull << 32) ? ~0ull : (hi_ << 32);
      for (int it = 0; it < 64 && phi - plo > 1; ++it) {
        floor_key = plo + ((phi - plo) >> 1);
        kept = count([&](int j) { return key(j) >= floor_key; });
        if (kept >= kk && kept <= SORTN) break;
        if (kept > SORTN) plo = floor_key; else phi = floor_key;
      }
    }
  }

  // ---- the kept keys, dense in LDS (in any order), zero-filled to SORTN ---------
  {
    // Each thread appends its own keys.  (The opaque copies keep the compiler
    // from holding a lane mask per key from the count to the append.)
    auto gather = [&](auto keep, auto keep2) {
      int c = 0;
#pragma unroll
      for (int j = 0; j < E; ++j) c += keep(j) ? 1 : 0;
      const int upto = wave_prefix_sum(c, lane);
      par ^= 1;
      if (lane == kWave - 1) cnt[par][wave] = upto;
      __syncthreads();
      int pos = upto - c + waves_below();
#pragma unroll
      for (int j = 0; j < E; ++j) {
        if (keep2(j)) sbuf[pos++] = key(j);
      }
    };
    if (floor_key == 0) {
      uint32_t f = floor_hi;
      asm volatile("" : "+v"(f));
      gather([&](int j) { return hi[j] >= floor_hi; }, [&](int j) { return hi[j] >= f; });
    } else {
      uint64_t f = floor_key;
      asm volatile("" : "+v"(f));
      gather([&](int j) { return key(j) >= floor_key; }, [&](int j) { return key(j) >= f; });
    }
    for (int i = kept + tid; i < SORTN; i += kFewThreads) sbuf[i] = 0ull;
    __syncthreads();
  }

  // ---- the order by bins: bin 0 holds the greatest score -----------------------
  uint64_t v[ES];
  uint32_t mn = 0;  // complement of the least kept score word
#pragma unroll
  for (int j = 0; j < ES; ++j) {
    v[j] = sbuf[j * kFewThreads + tid];
    const uint32_t m = v[j] != 0ull ? ~key_hi(v[j]) : 0u;
    mn = m > mn ? m : mn;
  }
  mn = wave_max_u32(mn);
  if (lane == 0) wmax[wave] = mn;
  __syncthreads();
  mn = row16_reduce(wmax[lane & 15], max_op);
  const float top = ord_to_f32(mx);
  const float scale = static_cast<float>(BINS - 1) / (top - ord_to_f32(~mn));
  bool binned = scale > 0.f && scale < __FLT_MAX__;  // (not for a range that is zero, infinite or NaN)
  if (binned) {
    int bin[ES], slot[ES];
#pragma unroll
    for (int j = 0; j < ES; ++j) {
      // (an empty slot's score is NaN: the minimum takes the bound)
      bin[j] = static_cast<int>(__builtin_fminf((top - ord_to_f32(key_hi(v[j]))) * scale, static_cast<float>(BINS - 1)));
      slot[j] = v[j] != 0ull ? atomicAdd(&hist[bin[j]], 1) : 0;
    }
    __syncthreads();
    // counts -> first rank of each bin
    int own[BPT], sum = 0;
    uint32_t most = 0;
#pragma unroll
    for (int i = 0; i < BPT; ++i) {
      own[i] = hist[tid * BPT + i];
      sum += own[i];
      most = static_cast<uint32_t>(own[i]) > most ? own[i] : most;
    }
    const int upto = wave_prefix_sum(sum, lane);
    most = wave_max_u32(most);
    par ^= 1;
    if (lane == kWave - 1) {
      cnt[par][wave] = upto;
      wmax[wave] = most;
    }
    __syncthreads();
    int first = upto - sum + waves_below();
    binned = row16_reduce(wmax[lane & 15], max_op) <= CROWD;
    if (binned) {
#pragma unroll
      for (int i = 0; i < BPT; ++i) {
        hist[tid * BPT + i] = first;
        first += own[i];
      }
      if (tid == kFewThreads - 1) hist[BINS] = first;
      __syncthreads();
      int lo_r[ES], hi_r[ES];
#pragma unroll
      for (int j = 0; j < ES; ++j) {
        lo_r[j] = hist[bin[j]];
        hi_r[j] = hist[bin[j] + 1];
        if (v[j] != 0ull) rbuf[lo_r[j] + slot[j]] = v[j];
      }
      __syncthreads();
#pragma unroll
      for (int j = 0; j < ES; ++j) {
        if (v[j] != 0ull) {
          int r = lo_r[j];
          for (int m = lo_r[j]; m < hi_r[j]; ++m) r += rbuf[m] > v[j] ? 1 : 0;
          sbuf[r] = v[j];
        }
      }
      __syncthreads();
    }
  }

  if (!binned) {
  // ---- bitonic sort, descending: rank e = WAVE_KEYS wave + ES lane + j ---------
  // Each wave sorts its WAVE_KEYS keys in registers; the levels above exchange whole
  // registers between waves through LDS.  A block that runs ascending is
  // handled as the descending sort of the complemented keys.
#pragma unroll
  for (int j = 0; j < ES; ++j) v[j] = sbuf[wave * WAVE_KEYS + j * kWave + lane];
  auto flip = [&](bool asc) {
    const uint64_t x = asc ? ~0ull : 0ull;
#pragma unroll
    for (int j = 0; j < ES; ++j) v[j] ^= x;
  };
  flip(wave & 1);
  wave_sort_desc<ES>(v, lane);
  flip(wave & 1);
  for (int size = 2; size <= W; size <<= 1) {  // in waves
    const bool asc = size < W && (wave & size) != 0;
    for (int stride = size >> 1; stride > 0; stride >>= 1) {
      __syncthreads();  // the previous exchange's reads (and the loads above) are done
#pragma unroll
      for (int j = 0; j < ES; ++j) sbuf[wave * WAVE_KEYS + j * kWave + lane] = v[j];
      __syncthreads();
      const bool keep_max = ((wave & stride) == 0) != asc;
      const int pw = wave ^ stride;
#pragma unroll
      for (int j = 0; j < ES; ++j) {
        const uint64_t o = sbuf[pw * WAVE_KEYS + j * kWave + lane];
        v[j] = (o > v[j]) == keep_max ? o : v[j];
      }
    }
    flip(asc);
    bitonic_level<ES, WAVE_KEYS, WAVE_KEYS, WAVE_KEYS / 2>(v, lane);
    flip(asc);
  }
  __syncthreads();
#pragma unroll
  for (int j = 0; j < ES; ++j) sbuf[wave * WAVE_KEYS + lane * ES + j] = v[j];
  __syncthreads();
  }

  // ---- output -------------------------------------------------------------------
  if (a.seg_keys) {
    uint64_t* out = a.seg_keys + (row * gridDim.y + blockIdx.y) * a.top_k;
    for (int e = tid; e < a.top_k; e += kFewThreads) out[e] = sbuf[e];
    return;
  }
  for (int e = tid; e < a.top_k; e += kFewThreads) {
    const uint64_t k = sbuf[e];
    a.out_idx[row * a.top_k + e] = k ? static_cast<int64_t>(key_idx(k)) : int64_t(-1);
    a.out_scores[row * a.top_k + e] = k ? ord_to_f32(key_hi(k)) : -__builtin_inff();
  }
}

}  // namespace si
