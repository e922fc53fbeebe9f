// Backward of the HCA composition (included by sparse_attn_bwd.hip).
//
// HCA's keys are not scattered: query s attends to the window s-n_win+1 .. s
// and to every compressed entry i < (s+1)/m.  The general backward writes one
// dkv row per (query, slot) and sorts and sums them by key; here 128 keys and a
// block of consecutive queries meet in one workgroup, which sums their dkv in
// MFMA accumulators, so nothing is written per pair:
//   1. hca_bwd_idx_kernel: index rows whose window part starts at a multiple of
//      32 keys, so that slot tile i of query s holds the aligned key tile
//      (s-n_win+1)/32 + i whatever s is.  A masked slot names a key that the
//      query attends to (as ~key): its row is gathered in the slot's place, so
//      that 0 times a value that is not finite comes only from the query's own keys.
//   2. sparse_attn_bwd_rows_kernel on those rows: dq, dsink terms, and P / dS of
//      every tile (8 KiB each) in its register layout.
//   3. hca_bwd_dkv_kernel: per (128 keys, RB query rows) the sum over the rows'
//      heads of dS q + P dO, fp32, to a partial buffer.  Sums that are not finite
//      are taken again with each stage apart, for the keys its row attends to only
//      (S = 16,384, D = 576: a step 4.2 ms, 5.1 with one infinity, 9.0 with NaN in every row).
//   4. hca_bwd_reduce_kernel: each key's partials in block order.
// Every sum has a fixed order, so repeated calls are bit-identical.
//
// Bound: step 2 (its gathers and coefficients) and step 3's chain per row (see
// its comment).  Measured at S = 16,384, 64 heads, D = 576, n_win = m = 128: rows
// 1.80, dkv 1.41, reduction 0.07 ms, against 1.76 + 1.45 + 1.26 + 0.11 ms (rows,
// dkv rows, reduction, sort) of the general backward over 3.2M pairs; forward
// and backward 5.51 -> 4.14 ms.
#pragma once

namespace si {

constexpr int kHcaShift = 7;  // 128 keys (four 32-key tiles) per group
constexpr int kHcaKeys = 1 << kHcaShift;

struct HcaBwdArgs {
  int n_win, m, T;
  int wtiles;      // 32-key window tiles of an index row
  int RB;          // query rows of a block
  int b0;          // first batch of this chunk
  int s0, s1;      // query rows of this chunk (s0 a multiple of RB)
  int GW, ncg;     // window / compressed key groups of a block
  float* part;     // [nb, blocks, GW + ncg, kHcaKeys, D]
  float* acc;      // [N, D] fp32 sums of the batch's earlier chunks
  uint16_t* dkv;   // [B, N, D]
  int64_t dsb, dsn;
  int first, last;  // first / last chunk of the batch
};

// First window group that row block blk meets (keys below 0 count).
__device__ __forceinline__ int hca_group_lo(const HcaBwdArgs& h, int blk) {
  return (blk * h.RB - h.n_win + 1) >> kHcaShift;
}

// Query rows of (block, group j): the block's rows inside the chunk that have a
// key of the group.
__device__ __forceinline__ void hca_item_rows(const HcaBwdArgs& h, int blk, int j, int& r0, int& r1) {
  r0 = blk * h.RB > h.s0 ? blk * h.RB : h.s0;
  r1 = (blk + 1) * h.RB < h.s1 ? (blk + 1) * h.RB : h.s1;
  if (j < h.GW) {
    const int kg = hca_group_lo(h, blk) + j;
    const int lo = kHcaKeys * kg, hi = lo + kHcaKeys - 1 + h.n_win;  // rows lo .. hi-1 see the group's keys
    if (kg < 0) r1 = r0;
    r0 = r0 > lo ? r0 : lo;
    r1 = r1 < hi ? r1 : hi;
  } else {
    const int64_t lo = static_cast<int64_t>(h.m) * (kHcaKeys * (j - h.GW) + 1) - 1;
    if (r0 < lo) r0 = lo < r1 ? static_cast<int>(lo) : r1;
  }
}

// Index rows [rows, 32 wtiles + T] of queries s0 .. and their used lengths [rows],
// shared by all batches: window column j of query s holds key 32 floor((s-n_win+1)/32) + j
// where that lies in the window, else ~key of the window's key next to it (a row
// that the same tile gathers anyway; with key s everywhere the rows kernel took 0.6 %
// longer), then legal compressed entry i as S + i.
__global__ __launch_bounds__(256) void hca_bwd_idx_kernel(int32_t* idx, int32_t* row_len, int s0, int S, int n_win, int T,
                                                          int m, int wtiles) {
  const int r = blockIdx.x;
  const int s = s0 + r;
  const int K = 32 * wtiles + T;
  const int first = s - n_win + 1;
  const int base = (first >> 5) * 32;
  const int legal = (s + 1) / m < T ? (s + 1) / m : T;
  const int low = first > 0 ? first : 0;
  for (int j = threadIdx.x; j < K; j += 256) {
    int v;
    if (j < 32 * wtiles) {
      const int t = base + j;
      v = t < low ? ~low : t > s ? ~s : t;
    } else {
      const int i = j - 32 * wtiles;
      v = i < legal ? S + i : ~S;  // (past the row's length, never read)
    }
    idx[static_cast<int64_t>(r) * K + j] = v;
  }
  if (threadIdx.x == 0) row_len[r] = 32 * wtiles + legal;
}

template <int D>
struct HcaDkvShape {
  static constexpr int CPR = D / 8;
  static constexpr int CPP = CPR + 2;          // chunks per LDS row: padded as in DkvShape
  static constexpr int QROW = CPP * 16;
  static constexpr int PART = 16 * QROW;       // 16 heads of Q or of dO
  static constexpr int BUF = 2 * PART;         // Q then dO
  static constexpr int NW = 8;                      // waves, two per SIMD
  static constexpr int COPIES = 2 * 16 * CPP / 64;  // 64-lane copies of a stage (CPP is even)
  static constexpr int CPW = (COPIES + NW - 1) / NW;  // copies per wave
  // 16-dimension blocks: MBW each for waves 0..3, the rest in equal shares for
  // waves 4..7, so that the two waves of a SIMD hold MBT / 4 together.
  static constexpr int MBT = D / 16;
  static constexpr int MBW = (MBT + 7) / 8;
  static constexpr int MBW2 = MBT > 4 * MBW ? (MBT - 4 * MBW) / 4 : 0;
  static_assert(MBT <= 4 * MBW || (MBT - 4 * MBW) % 4 == 0, "blocks of waves 4..7");
  // Coefficients: [tile][P, dS][4-key group][head][16 bytes], the key groups 320
  // bytes apart (256 would put a transposing read's four in one bank)
  static constexpr int CG = 320;
  static constexpr int CW4 = 4 * CG;
  static constexpr int COEF = 4 * 2 * CW4;
};

// 16 bytes per lane from memory to LDS (64 lanes: consecutive slots from dst).
__device__ __forceinline__ void hca_copy16(const uint16_t* src, char* dst) {
  __builtin_amdgcn_global_load_lds(src, (lds_void_t*)dst, 16, 0, 0);
}

// dkv^T [D x 128 keys] += [Q^T | dO^T] [D x 32] . [dS; P] [32 x 128 keys] per
// stage: one query row, 16 heads, whose dS against Q and P against dO make one
// 32-deep MFMA step.  The operands are read as in
// sparse_attn_bwd_dkv_rows_kernel.  Two waves per SIMD: one's copies, waits and
// fragment reads run beside the other's MFMAs.  128 keys per group: a row is
// copied and read 3 times at S = 16K (4.5 times with 64 keys and 32-head stages:
// 1.55 ms, this 1.41).  A stage takes 3,900 clocks for 1,152 of MFMA per SIMD:
// the copies, the fragment reads behind the barrier and the MFMAs follow one
// another.  Counters: matrix cores busy 39 % of the CUs' busy cycles, LDS 29 % (46 %
// of that bank conflicts), 1.73 GB from the fabric.  Two more stages in flight (a ring of four) measured 1.39, touching
// the lines two rows ahead or spreading the copies over the blocks nothing.
// (waves per SIMD: two workgroups fit a CU up to D = 256, one above)
template <int D, bool F16>
__global__ __launch_bounds__(512, D <= 256 ? 4 : 2) void hca_bwd_dkv_kernel(AttnBwdArgs a, HcaBwdArgs h) {
  using HS = HcaDkvShape<D>;
  constexpr int MBW = HS::MBW;
  __shared__ __attribute__((aligned(16))) char qd_lds[2 * HS::BUF];
  __shared__ __attribute__((aligned(16))) char coef_lds[HS::COEF];
  __shared__ int nonfinite_lds[HS::NW];

  const int lane = threadIdx.x & 63;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  __builtin_assume(wave >= 0 && wave < HS::NW);
  const int g = lane >> 4;
  const int i16 = lane & 15;
  const int per = h.GW + h.ncg;
  const int blk0 = h.s0 / h.RB;
  const int nblk = (h.s1 + h.RB - 1) / h.RB - blk0;
  const int item = xcd_block_order();  // neighbouring items share their rows' Q and dO
  const int j = item % per;
  const int blk = blk0 + (item / per) % nblk;
  const int b = h.b0 + item / (per * nblk);
  int r0, r1;
  hca_item_rows(h, blk, j, r0, r1);
  if (r0 >= r1) return;
  const bool window = j < h.GW;
  const int kt = 4 * (window ? hca_group_lo(h, blk) + j : j - h.GW);  // first 32-key tile of the group
  const int blk_lo = wave < 4 ? wave * MBW : 4 * MBW + (wave - 4) * HS::MBW2;  // this wave's dimension blocks

  // Copies of a stage: LDS chunk e (16 bytes) is chunk e % CPP of head
  // (e / CPP) % 16 of Q (e < 16 CPP) or dO; the pad chunks re-read chunk 0.
  int voff[HS::CPW];  // byte offset from the stage's first head
#pragma unroll
  for (int i = 0; i < HS::CPW; ++i) {
    const int n = i * HS::NW + wave;
    const int e = n * 64 + lane;
    const int c = e % HS::CPP;
    voff[i] = static_cast<int>(((e / HS::CPP) % 16) * (e < 16 * HS::CPP ? a.qsh : a.gsh) + (c < HS::CPR ? c : 0) * 8) * 2;
  }
  const int nq = (a.H + 15) / 16;  // 16-head parts of a row
  struct Stage {
    int s, part;
  };
  auto next = [&](Stage x) { return x.part + 1 < nq ? Stage{x.s, x.part + 1} : Stage{x.s + 1, 0}; };
  auto copy_stage = [&](const Stage& x, int buf) {
    const int h0 = x.part * 16;
    const char* qs = reinterpret_cast<const char*>(a.q + b * a.qsb + static_cast<int64_t>(x.s) * a.qss + h0 * a.qsh);
    const char* gs = reinterpret_cast<const char*>(a.dout + b * a.gsb + static_cast<int64_t>(x.s) * a.gss + h0 * a.gsh);
    char* dst = qd_lds + buf * HS::BUF;
    const bool whole = h0 + 16 <= a.H;
#pragma unroll
    for (int i = 0; i < HS::CPW; ++i) {
      const int n = i * HS::NW + wave;
      if (n < HS::COPIES) {
        const int e = n * 64 + lane;
        const bool isq = e < 16 * HS::CPP;
        int off = voff[i];
        if (!whole) {
          // heads past H re-read head H-1 (their P and dS are 0)
          const int hd = (e / HS::CPP) % 16;
          const int over = h0 + hd - (a.H - 1);
          if (over > 0) off -= over * static_cast<int>(isq ? a.qsh : a.gsh) * 2;
        }
        hca_copy16(reinterpret_cast<const uint16_t*>((isq ? qs : gs) + off), dst + n * 1024);
      }
    }
  };
  // Coefficients of a stage: tiles kt .. kt+3, 16 heads (one producer wave), 16
  // bytes a thread: wave 2 k + 0 / 1 takes P / dS of tile kt + k; zero where the
  // query row has no such tile.
  const int64_t nr = h.s1 - h.s0;
  u32x4 cf;
  auto load_coef = [&](const Stage& x) {
    const int64_t lrow = (b - h.b0) * nr + (x.s - h.s0);
    const uint16_t* row = a.coef + (lrow * a.HG + (x.part >> 2)) * a.ntiles * kCoefTile;
    int ti = kt + (wave >> 1);
    bool ok;
    if (window) {
      ti -= (x.s - h.n_win + 1) >> 5;
      ok = ti >= 0 && ti < h.wtiles;
    } else {
      ok = static_cast<int64_t>(h.m) * (ti * 32 + 1) <= x.s + 1 && ti * 32 < h.T;  // its first entry is legal
      ti += h.wtiles;
    }
    const int off = ((wave & 1) * 4 + (x.part & 3)) * 512 + lane * 8;
    cf = ok ? *reinterpret_cast<const u32x4*>(row + static_cast<int64_t>(ti) * kCoefTile + off) : u32x4{0u, 0u, 0u, 0u};
  };
  char* const cst = coef_lds + wave * HS::CW4 + (lane >> 4) * HS::CG + (lane & 15) * 16;  // where they go

  // k of the MFMA step: 0..15 the 16 heads of Q / dS, 16..31 those of dO / P.  Lane
  // group g holds k = 8 g .. 8 g + 7: heads 8 (g & 1) .. of the first or second.
  const int kh = 8 * (g & 1) + (i16 >> 2);
  const uint32_t qd0 = lds_addr(qd_lds) + (g >> 1) * HS::PART + kh * HS::QROW + 8 * (i16 & 3) + blk_lo * 32;
  const uint32_t cf0 = lds_addr(coef_lds) + (g < 2 ? HS::CW4 : 0) + (i16 & 3) * HS::CG + kh * 16;

  // Whether query s attends to this lane's key of key block nb.
  auto attends = [&](int s, int nb) {
    const int key = kt * 32 + nb * 16 + i16;
    return window ? key <= s && key > s - h.n_win : key < h.T && static_cast<int64_t>(h.m) * (key + 1) <= s + 1;
  };

  // The stages with NB dimension blocks (a compile-time count: LDS reads in
  // flight must not cross control flow, where their registers could be copied
  // before the data lands).
  auto stages = [&](auto NBC) {
    constexpr int NB = decltype(NBC)::value;
    f32x4 acc[NB > 0 ? NB : 1][8];
    // The sums over all stages.  APART: each stage's part is formed apart and added for
    // the keys that its row attends to only.
    auto sum_stages = [&](auto APARTC) {
      constexpr bool APART = decltype(APARTC)::value;
#pragma unroll
      for (int m = 0; m < NB; ++m)
#pragma unroll
        for (int nb = 0; nb < 8; ++nb) acc[m][nb] = f32x4{0.f, 0.f, 0.f, 0.f};
      Stage cur{r0, 0};
      copy_stage(cur, 0);
      load_coef(cur);
      int buf = 0;
      for (; cur.s < r1; buf ^= 1) {
        const int s = cur.s;
        __builtin_amdgcn_s_waitcnt(vm_lgkm0(0));  // this stage's copies and coefficients landed (issued a stage ago)
        *reinterpret_cast<u32x4*>(cst) = cf;
        attn_tile_barrier();
        // (the other buffer was last read in the previous stage, which every wave has left)
        cur = next(cur);
        if (cur.s < r1) {
          copy_stage(cur, buf ^ 1);
          load_coef(cur);
        }
        if constexpr (NB > 0 && !APART) {
          // Key blocks nb: 16 (nb & 1) of tile nb >> 1.
          v4i16 blo[8], bhi[8];
          attn_static_for<0, 8>([&](auto NC) {
            constexpr int nb = decltype(NC)::value;
            constexpr int off = (nb >> 1) * 2 * HS::CW4 + 8 * (nb & 1);
            blo[nb] = tr_read<off>(cf0);
            bhi[nb] = tr_read<off + 64>(cf0);
          });
          const uint32_t qa = qd0 + buf * HS::BUF;
          v4i16 alo[2], ahi[2];
          auto a_read = [&](auto JC) {
            constexpr int m = decltype(JC)::value;
            alo[m & 1] = tr_read<m * 32>(qa);
            ahi[m & 1] = tr_read<m * 32 + 4 * HS::QROW>(qa);
          };
          a_read(std::integral_constant<int, 0>{});
          lds_wait_n<2>();
          bf16x8 bfr[8];
#pragma unroll
          for (int nb = 0; nb < 8; ++nb) {
            reg_tie(blo[nb]);
            reg_tie(bhi[nb]);
            bfr[nb] = __builtin_bit_cast(bf16x8, __builtin_shufflevector(blo[nb], bhi[nb], 0, 1, 2, 3, 4, 5, 6, 7));
          }
          attn_static_for<0, NB>([&](auto JC) {
            constexpr int m = decltype(JC)::value;
            if constexpr (m + 1 < NB) {
              a_read(std::integral_constant<int, m + 1>{});
              lds_wait_n<2>();
            } else {
              lds_wait_n<0>();
            }
            reg_tie(alo[m & 1]);
            reg_tie(ahi[m & 1]);
            const bf16x8 af = __builtin_bit_cast(bf16x8, __builtin_shufflevector(alo[m & 1], ahi[m & 1], 0, 1, 2, 3, 4, 5, 6, 7));
#pragma unroll
            for (int nb = 0; nb < 8; ++nb) acc[m][nb] = mfma16x16x32<F16>(af, bfr[nb], acc[m][nb]);
          });
        }
        if constexpr (NB > 0 && APART) {
          // (two key blocks at a time, so that this takes no more registers than the above)
          const uint32_t qa = qd0 + buf * HS::BUF;
          attn_static_for<0, NB>([&](auto JC) {
            constexpr int m = decltype(JC)::value;
            attn_static_for<0, 4>([&](auto NC) {
              constexpr int n = decltype(NC)::value;
              v4i16 alo = tr_read<m * 32>(qa);
              v4i16 ahi = tr_read<m * 32 + 4 * HS::QROW>(qa);
              v4i16 xlo = tr_read<n * 2 * HS::CW4>(cf0);
              v4i16 xhi = tr_read<n * 2 * HS::CW4 + 64>(cf0);
              v4i16 ylo = tr_read<n * 2 * HS::CW4 + 8>(cf0);
              v4i16 yhi = tr_read<n * 2 * HS::CW4 + 8 + 64>(cf0);
              lds_wait_n<0>();
              reg_tie(alo);
              reg_tie(ahi);
              reg_tie(xlo);
              reg_tie(xhi);
              reg_tie(ylo);
              reg_tie(yhi);
              const bf16x8 af = __builtin_bit_cast(bf16x8, __builtin_shufflevector(alo, ahi, 0, 1, 2, 3, 4, 5, 6, 7));
              const bf16x8 xf = __builtin_bit_cast(bf16x8, __builtin_shufflevector(xlo, xhi, 0, 1, 2, 3, 4, 5, 6, 7));
              const bf16x8 yf = __builtin_bit_cast(bf16x8, __builtin_shufflevector(ylo, yhi, 0, 1, 2, 3, 4, 5, 6, 7));
              f32x4 x = mfma16x16x32<F16>(af, xf, f32x4{0.f, 0.f, 0.f, 0.f});
              f32x4 y = mfma16x16x32<F16>(af, yf, f32x4{0.f, 0.f, 0.f, 0.f});
              mfma_result_fence(x, y);
              const bool bx = attends(s, 2 * n), by = attends(s, 2 * n + 1);
#pragma unroll
              for (int c = 0; c < 4; ++c) {
                acc[m][2 * n][c] = bx ? acc[m][2 * n][c] + x[c] : acc[m][2 * n][c];
                acc[m][2 * n + 1][c] = by ? acc[m][2 * n + 1][c] + y[c] : acc[m][2 * n + 1][c];
              }
              reg_tie(acc[m][2 * n]);  // (added here, not after later parts)
              reg_tie(acc[m][2 * n + 1]);
            });
          });
        }
        attn_tile_barrier();  // every wave is done with this stage's coefficients and buffer
      }
    };
    sum_stages(std::false_type{});
    f32x4 z = f32x4{0.f, 0.f, 0.f, 0.f};  // NaN where a sum is not finite
#pragma unroll
    for (int m = 0; m < NB; ++m) {
#pragma unroll
      for (int nb = 0; nb < 8; nb += 2) mfma_result_fence(acc[m][nb], acc[m][nb + 1]);
      if (blk_lo + m < HS::MBT) {  // (at D = 32 waves 2 and 3 hold no block of the row)
#pragma unroll
        for (int nb = 0; nb < 8; ++nb)
#pragma unroll
          for (int c = 0; c < 4; ++c) z[c] = __builtin_fmaf(acc[m][nb][c], 0.f, z[c]);
      }
    }
    // (before the stores: an LDS read waits for the memory operations in flight.  The
    // barrier also ends every wave's use of the buffers.)
    const bool bad = __builtin_amdgcn_ballot_w64((z[0] + z[1]) + (z[2] + z[3]) != 0.f) != 0;
    if (lane == 0) nonfinite_lds[wave] = bad ? 1 : 0;
    attn_tile_barrier();
    int any = 0;
#pragma unroll
    for (int w = 0; w < HS::NW; ++w) any |= nonfinite_lds[w];
    if (__builtin_amdgcn_readfirstlane(any) != 0) {
      // The coefficients of the keys that a row does not attend to are 0, and 0
      // times an infinity or NaN of the row's Q or dO is NaN.
      sum_stages(std::true_type{});
    }
    // lane (key 16 nb + i16 of the group, g) holds dimensions 16 mbi + 4 g + 0..3
    float* out = h.part + static_cast<int64_t>(item) * kHcaKeys * D;
#pragma unroll
    for (int m = 0; m < NB; ++m) {
      if (blk_lo + m < HS::MBT) {
#pragma unroll
        for (int nb = 0; nb < 8; ++nb)
          *reinterpret_cast<f32x4*>(out + (nb * 16 + i16) * D + (blk_lo + m) * 16 + 4 * g) = acc[m][nb];
      }
    }
  };
  if (wave < 4) stages(std::integral_constant<int, MBW>{});
  else stages(std::integral_constant<int, HS::MBW2>{});
}

// dkv of one key from its partials (blocks in order), the sums of the earlier
// chunks first.  Keys without a partial in a middle chunk keep their sum.
template <int D, bool F16>
__global__ __launch_bounds__(256) void hca_bwd_reduce_kernel(HcaBwdArgs h, int S) {
  const int N = S + h.T;
  const int n = static_cast<int>(blockIdx.x) % N;
  const int b = h.b0 + static_cast<int>(blockIdx.x) / N;
  const int d = static_cast<int>(threadIdx.x) * 4;
  const int per = h.GW + h.ncg;
  const int blk0 = h.s0 / h.RB;
  const int nblk = (h.s1 + h.RB - 1) / h.RB - blk0;
  const bool window = n < S;
  const int grp = (window ? n : n - S) >> kHcaShift;
  const int64_t lo = window ? kHcaKeys * grp : static_cast<int64_t>(h.m) * (kHcaKeys * grp + 1) - 1;
  const int64_t hi = window ? lo + kHcaKeys - 1 + h.n_win : h.s1;
  int64_t from = lo > h.s0 ? lo : h.s0, to = hi < h.s1 ? hi : h.s1;  // rows with a key of the group
  if (window ? h.GW == 0 : grp >= h.ncg) to = from;
  if (from >= to && !h.first && !h.last) return;
  if (d >= D) return;
  f32x4 sum = f32x4{0.f, 0.f, 0.f, 0.f};
  float* acc = h.acc + static_cast<int64_t>(n) * D + d;  // (a batch in several chunks is alone in them)
  if (!h.first) sum = *reinterpret_cast<const f32x4*>(acc);
  if (from < to) {
    const int q0 = static_cast<int>(from) / h.RB, q1 = static_cast<int>(to - 1) / h.RB;  // inclusive
    auto part = [&](int q) {
      const int j = window ? grp - hca_group_lo(h, q) : h.GW + grp;
      const int64_t item = (static_cast<int64_t>(b - h.b0) * nblk + (q - blk0)) * per + j;
      return *reinterpret_cast<const f32x4*>(h.part + (item * kHcaKeys + ((window ? n : n - S) & (kHcaKeys - 1))) * D + d);
    };
    for (int q = q0; q <= q1; q += 8) {
      f32x4 v[8];
#pragma unroll
      for (int u = 0; u < 8; ++u) v[u] = part(q + u <= q1 ? q + u : q1);
#pragma unroll
      for (int u = 0; u < 8; ++u)
#pragma unroll
        for (int c = 0; c < 4; ++c) sum[c] += q + u <= q1 ? v[u][c] : 0.f;
    }
  }
  if (!h.last) {
    *reinterpret_cast<f32x4*>(acc) = sum;
  } else {
    uint2 w;
    w.x = pack2<F16>(sum[0], sum[1]);
    w.y = pack2<F16>(sum[2], sum[3]);
    *reinterpret_cast<uint2*>(h.dkv + b * h.dsb + static_cast<int64_t>(n) * h.dsn + d) = w;
  }
}

// ---- host side ----------------------------------------------------------------
struct HcaPlan {
  int64_t rows;  // query rows of a chunk (a multiple of RB, or S)
  int64_t nb;    // batches of a chunk (1 where a batch takes several chunks)
  int RB, wtiles, ntiles, GW, ncg;
  size_t dsink_rows, acc, idx, row_len, coef, part, total;
};

static void hca_plan_for(int64_t B, int64_t S, int64_t H, int64_t D, int64_t n_win, int64_t T, int RB, int64_t rows,
                         int64_t nb, HcaPlan* p) {
  const int64_t HG = (H + 63) / 64;
  p->rows = rows;
  p->nb = nb;
  p->RB = RB;
  p->wtiles = n_win > 0 ? static_cast<int>((n_win + 31 + 31) / 32) : 0;
  p->ntiles = p->wtiles + static_cast<int>((T + 31) / 32);
  p->GW = n_win > 0 ? static_cast<int>((RB + n_win - 2) / kHcaKeys + 2) : 0;
  p->ncg = static_cast<int>((T + kHcaKeys - 1) / kHcaKeys);
  size_t off = 0;
  auto take = [&](int64_t bytes) {
    const size_t at = off;
    off = (off + static_cast<size_t>(bytes) + 255) & ~static_cast<size_t>(255);
    return at;
  };
  const int64_t blocks = (rows + RB - 1) / RB;
  p->dsink_rows = take(B * S * 64 * HG * 4);
  p->acc = take(rows < S ? (S + T) * D * 4 : 0);
  p->idx = take(rows * (32 * p->wtiles + T) * 4);
  p->row_len = take(rows * 4);
  p->coef = take(nb * rows * HG * p->ntiles * kCoefTile * 2);
  p->part = take(nb * blocks * (p->GW + p->ncg) * kHcaKeys * D * 4);
  p->total = off;
}

// The plan of row blocks of RB rows with the fewest chunks that fits `bytes`; false
// when none does: all batches, else equal groups of whole batches, else equal parts
// of one batch's rows (which add up dkv in the workspace).  Equal, because a short
// last chunk costs what a whole one does on the CUs that it leaves idle.
static bool hca_plan_rb(int64_t B, int64_t S, int64_t H, int64_t D, int64_t n_win, int64_t T, int RB, size_t bytes,
                        HcaPlan* p) {
  hca_plan_for(B, S, H, D, n_win, T, RB, S, B, p);
  if (p->total <= bytes) return true;
  // The greatest x below `end` with fits(x) (0: none), then ceil(end / chunks of x).
  auto share = [&](int64_t end, auto fits) {
    int64_t lo = 0, hi = end;
    while (hi - lo > 1) {
      const int64_t mid = (lo + hi) / 2;
      if (fits(mid)) lo = mid; else hi = mid;
    }
    if (lo == 0) return int64_t{0};
    const int64_t chunks = (end + lo - 1) / lo;
    return (end + chunks - 1) / chunks;
  };
  auto batches = [&](int64_t nb) {
    hca_plan_for(B, S, H, D, n_win, T, RB, S, nb, p);
    return p->total <= bytes;
  };
  auto blocks = [&](int64_t n) {
    hca_plan_for(B, S, H, D, n_win, T, RB, n * RB, 1, p);
    return p->total <= bytes;
  };
  const int64_t nb = share(B, batches);
  if (nb > 0) return batches(nb);
  const int64_t n = share((S + RB - 1) / RB, blocks);
  return n > 0 && blocks(n);
}

// Row blocks of 64 (the fewest partials), smaller where a chunk of them has fewer
// items than the CUs hold workgroups twice over (two a CU up to D = 256), down to 128
// stages (of 16 heads of a row) a block: a workgroup of the dkv kernel runs a block's
// stages one after another.  us a layer step with a floor of 32 rows against this one:
// 4 x 256 tokens, H = 128, D = 576, n_win = m = 16 612 -> 479 (general backward 508);
// backward of 64K tokens in chunks of 1,024 (381 MB), D = 576 35.0 -> 27.1 ms (45.7);
// 1,024 items and not 512 at S = 8,192, H = 64, D = 64, n_win = m = 16 887 -> 783 us (835).
static bool hca_plan(int64_t B, int64_t S, int64_t H, int64_t D, int64_t n_win, int64_t T, size_t bytes, HcaPlan* p) {
  bool ok = false;
  for (int RB = 64; RB >= 8; RB /= 2) {
    HcaPlan q{};
    if (hca_plan_rb(B, S, H, D, n_win, T, RB, bytes, &q)) {
      ok = true;
      *p = q;
      if (q.nb * ((q.rows + RB - 1) / RB) * (q.GW + q.ncg) >= (D <= 256 ? 1024 : 512)) break;
    }
    if (RB <= 32 && RB * ((H + 15) / 16) <= 128) break;
  }
  return ok;
}

template <int D, bool F16>
static int launch_hca_bwd(AttnBwdArgs a, const HcaPlan& pl, char* ws, HcaBwdArgs h, float* dsink, hipStream_t st) {
  const int S = a.S;
  const int K = 32 * pl.wtiles + h.T;
  int32_t* idx = reinterpret_cast<int32_t*>(ws + pl.idx);
  int32_t* row_len = reinterpret_cast<int32_t*>(ws + pl.row_len);
  int rc;
  a.isb = 0;
  a.iss = K;
  a.isk = 1;
  a.rlsb = 0;
  a.rlss = 1;
  a.K = K;
  a.ntiles = pl.ntiles;
  a.masked_keys = 1;
  a.dsink_rows = reinterpret_cast<float*>(ws + pl.dsink_rows);
  a.coef = reinterpret_cast<uint16_t*>(ws + pl.coef);
  h.wtiles = pl.wtiles;
  h.RB = pl.RB;
  h.GW = pl.GW;
  h.ncg = pl.ncg;
  h.part = reinterpret_cast<float*>(ws + pl.part);
  h.acc = reinterpret_cast<float*>(ws + pl.acc);
  for (int64_t b0 = 0; b0 < a.B; b0 += pl.nb) {
    const int64_t nb = a.B - b0 < pl.nb ? a.B - b0 : pl.nb;
    for (int64_t s0 = 0; s0 < S; s0 += pl.rows) {
      h.b0 = static_cast<int>(b0);
      h.s0 = static_cast<int>(s0);
      h.s1 = static_cast<int>(S - s0 < pl.rows ? S : s0 + pl.rows);
      h.first = s0 == 0;
      h.last = h.s1 == S;
      if (b0 == 0 || pl.rows < S) {  // (whole batches share one chunk's index rows)
        hipLaunchKernelGGL(hca_bwd_idx_kernel, dim3(static_cast<unsigned>(h.s1 - h.s0)), dim3(256), 0, st, idx, row_len, h.s0,
                           S, h.n_win, h.T, h.m, pl.wtiles);
        if ((rc = check_launch("hca_bwd_idx_kernel"))) return rc;
      }
      a.idx = idx - s0 * K;  // (indexed by s)
      a.row_len = row_len - s0;
      a.row0 = b0 * S + s0;
      a.nrows = static_cast<int>(nb * (h.s1 - h.s0));
      const unsigned grid = static_cast<unsigned>(static_cast<int64_t>(a.nrows) * a.HG);
      hipLaunchKernelGGL((sparse_attn_bwd_rows_kernel<D, false, F16>), dim3(grid), dim3(kBwdThreads), 0, st, a);
      if ((rc = check_launch("sparse_attn_bwd_rows_kernel"))) return rc;
      const int64_t blocks = (h.s1 + h.RB - 1) / h.RB - h.s0 / h.RB;
      const unsigned items = static_cast<unsigned>(nb * blocks * (h.GW + h.ncg));
      if (items > 0) {
        hipLaunchKernelGGL((hca_bwd_dkv_kernel<D, F16>), dim3(items), dim3(HcaDkvShape<D>::NW * 64), 0, st, a, h);
        if ((rc = check_launch("hca_bwd_dkv_kernel"))) return rc;
      }
      hipLaunchKernelGGL((hca_bwd_reduce_kernel<D, F16>), dim3(static_cast<unsigned>(nb * (S + h.T))), dim3((D / 4 + 63) / 64 * 64), 0,
                         st, h, S);
      if ((rc = check_launch("hca_bwd_reduce_kernel"))) return rc;
    }
  }
  hipLaunchKernelGGL(sparse_attn_bwd_dsink_kernel, dim3(static_cast<unsigned>(a.H)), dim3(256), 0, st, a.dsink_rows,
                     static_cast<int64_t>(a.B) * S, 64 * a.HG, dsink);
  return check_launch("sparse_attn_bwd_dsink_kernel");
}

}  // namespace si
