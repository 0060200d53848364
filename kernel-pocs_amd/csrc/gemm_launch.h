// Tile configurations of the MFMA GEMM core and their launches, shared by the
// bf16 (gemm.hip) and fp16 (gemm_f16.hip) instantiations.
#pragma once

#include "gemm_core.h"
#include "gemm_w4.h"

namespace fgemm {

// Tile configurations.
enum Cfg {
  CFG_BIG = 0,       // 256 x 256: 2 x 2 waves (128 x 128 per wave), or 4 x 2 (see launch_cfg)
  CFG_SKINNY_N = 1,  // N <= 32-ish (rank-r outputs): 64 x 64 tiles (2 x 2 waves) for a K-contiguous
                     // A, else 256 x 32 (4 x 1 waves)
  CFG_SKINNY_M = 2,  // 32 x 256, 1 x 4 waves: M <= 32-ish (LoRA A gradients)
  CFG_SKINNY_N64 = 3,  // 32 < N <= 64: 64 x 64 tiles for a K-contiguous A, 256 x 64 for
                       // token-major operands, else 256 x 32
  CFG_NARROW_128 = 4,  // 64 < N <= 128, K-contiguous A: 64 x 128 tiles (2 x 2 waves)
  CFG_NARROW_256 = 5,  // 192 < N <= 256, K-contiguous A: 64 x 256 tiles (2 x 2 waves)
  CFG_NARROW_192 = 6,  // 128 < N <= 192, K-contiguous A: 96 x 192 tiles (3 x 2 waves, 32 x 96 per wave)
};

// One launcher per epilogue family, each in a translation unit of its own
// (the engines' instantiations compile in parallel).
int launch_store_bf16(int cfg, int al, int bl, const GemmArgs& a, hipStream_t s);
int launch_store_f32(int cfg, int al, int bl, const GemmArgs& a, hipStream_t s);
int launch_atomic_f32(int cfg, int al, int bl, const GemmArgs& a, hipStream_t s);
int launch_glu_fwd(int epi, int al, int bl, const GemmArgs& a, hipStream_t s);
int launch_glu_bwd(int epi, int al, int bl, const GemmArgs& a, hipStream_t s);
int launch_rope(const GemmArgs& a, hipStream_t s);
int launch_rows(int epi, const GemmArgs& a, hipStream_t s);  // few rows, K-contiguous operands

inline int64_t total_k(const GemmArgs& a) {
  int64_t k = 0;
  for (int i = 0; i < a.n_segs; ++i) k += a.segs[i].k;
  return k;
}

// Few rows against K-contiguous weights: the row engine (gemm_rows.hip).  Up
// to 64 rows of a gate/up product (80 us; 256 x 256 tiles 94, the row engine
// 172 at 128) and 32 of a plain one (43 us at 32 rows, K = 14336, N = 4096; 256 x
// 256 tiles split over K take 45 at any row count up to 128, the row engine 77
// at 64).  Columns a workgroup of a plain product, 0: 32 x 256 tiles.
// Every workgroup reads all of A from L2, which passes the weights' own time
// where there are many rows and columns; 64 columns a workgroup read it a
// quarter as often but leave fewer of them, and 32 x 256 tiles are faster once
// they fill the chip.  Measured on MI355X, us with 32 x 256 tiles / 16 / 64
// columns, K = 4096: [16, 28672] 81 / 67 / 54, [32, 28672] 84 / 81 / 62, [32,
// 32000] 86 / 92, [1, 40960] 86 / 63 / 73, [17, 40960] 89 / 94, [16, 50264] 97 /
// 113 / 99, [8, 65536] 128 / 116 / 108, [1, 128256] 208 / 179 / 190, [8, 128256]
// 212 / 219 / 194, [16, 128256] 219 / 263 / 199, [32, 128256] 229 / 350 / 244;
// K = 8192: [8, 128256] 364 / 402 / 401; K = 64: [16, 65536] 9 / 16 / 10; K =
// 512: [1, 65536] 18 / 23 / 16, K = 1024: [8, 65536] 30 / 39 / 29.
inline int rows_columns(const GemmArgs& a) {
  const int64_t mn = a.M * a.N, k = total_k(a);
  if (a.N <= 128 * 256) return mn <= 896 * 1024 ? 16 : 0;  // 32 x 256 tiles on half the CUs or fewer
  if (a.M > 16 || k <= 128) return 0;
  if (mn <= 512 * 1024 && k >= 2048) return 16;
  return k <= 4096 ? 64 : 0;
}

inline bool rows_engine(int epi, const GemmArgs& a) {
  if (a.split_k != 1 || a.N <= a.M) return false;
  if (epi == EPI_STORE_BF16) return a.M <= 32 && rows_columns(a) > 0;
  return glu_fwd_epi(epi) && a.M <= 64 && !a.ep.vpart && !a.f16;
}
int launch_f16(int epi, int cfg, int al, int bl, const GemmArgs& a, hipStream_t s);  // fp16 operands

#ifndef SKINNY_NSTAGE
#define SKINNY_NSTAGE 2
#endif
#ifndef SKINNY_BKT
#define SKINNY_BKT 64
#endif
#ifndef SKINNY_WPE
#define SKINNY_WPE 2
#endif
// cache policy of a buffer load whose data is read once: nontemporal (the NT
// bit, 2, of the gfx950 buffer instruction's cache-policy field)
constexpr int CP_STREAM = 2;

// Column tiles of unequal K work (column-ranged segments of different
// lengths, e.g. [dQ B_q | dK B_k | dV B_v] with K = 4096, 1024, 1024) are
// dispatched heaviest first, so that the long tiles do not start in the last
// round; equal work keeps the default order.
static void order_columns(GemmArgs& a, int64_t out_bn, int64_t tn) {
  a.n_col_order = 0;
  if (tn < 2 || tn > MAX_COL_ORDER) return;
  int64_t work[MAX_COL_ORDER];
  int idx[MAX_COL_ORDER];
  bool uniform = true;
  for (int j = 0; j < tn; ++j) {
    const int64_t lo = j * out_bn, hi = lo + out_bn;
    work[j] = 0;
    for (int s = 0; s < a.n_segs; ++s)
      if (a.segs[s].n_hi > lo && a.segs[s].n_lo < hi) work[j] += a.segs[s].k;
    uniform = uniform && work[j] == work[0];
    idx[j] = j;
  }
  if (uniform) return;
  for (int i = 1; i < tn; ++i)  // stable insertion sort, heaviest first
    for (int j = i; j > 0 && work[idx[j]] > work[idx[j - 1]]; --j) {
      const int t = idx[j];
      idx[j] = idx[j - 1];
      idx[j - 1] = t;
    }
  a.n_col_order = (int)tn;
  for (int j = 0; j < tn; ++j) a.col_order[j] = (uint8_t)idx[j];
}

static bool plain_store(const GemmArgs& a) { return a.ep.beta == 0.f && a.ep.act == ACT_NONE && a.ep.alpha_group == 0; }

// Launches the 4-wave engine with its epilogue through LDS, or returns false:
// it needs 16-byte vectors, and of the 16-bit stores takes the plain one.  A^T B
// added to an fp32 C stays on 8 waves, whose two waves a SIMD cover each other's
// reads of C, where the reduction is short or an activation follows.  Measured
// on MI355X, 8 against 4 waves: [8192, 4096] K = 64 71 / 76 us, with GELU 71 /
// 90, [512, 4096] K = 64 19 / 23, [1024, 1024] K = 1024 39 / 45, [4096, 4096] K
// = 4096 152 / 131.  So does a short A^T B in 16 bits of more than one round of
// tiles: [8192, 4096] K = 64 27 / 31, K = 256 35 / 42; [4096, 4096] K = 512 28 /
// 28, [2048, 4096] K = 16 14.2 / 13.5.
template <class T, int BMODE, int EPI, bool AT, bool BT>
static bool launch_w4_staged(const GemmArgs& a, dim3 grid, hipStream_t s) {
  if constexpr (w4_staged_epi(EPI)) {
    if (!a.ep.vec_ok) return false;
    if constexpr (EPI == EPI_STORE_F32) {
      if (!plain_store(a)) {
        if (AT && a.ep.beta != 0.f && (a.ep.act != ACT_NONE || total_k(a) <= 1024)) return false;
        gemm_w4_kernel<T, BMODE, EPI, true, AT, BT, false><<<grid, 256, 0, s>>>(a);
        return true;
      }
    }
    if (EPI == EPI_STORE_BF16 && (!plain_store(a) || (AT && total_k(a) <= 256 && grid.x > 256))) return false;
    gemm_w4_kernel<T, BMODE, EPI, true, AT, BT><<<grid, 256, 0, s>>>(a);
    return true;
  }
  return false;
}

template <class T, int BM, int BN, int WM, int WN, int AL, int BL, int BMODE, int EPI>
static int launch_cfg(GemmArgs a, hipStream_t s) {
  constexpr int OUT_BN = (BMODE == B_DUAL) ? BN / 2 : BN;
  const int64_t tm = (a.M + BM - 1) / BM;
  const int64_t tn = (a.N + OUT_BN - 1) / OUT_BN;
  if (tm * tn > 0x7fffffffLL) return forge_set_error(FORGE_ERR_INVALID, "gemm: too many tiles");
  order_columns(a, OUT_BN, tn);
  dim3 grid((unsigned)(tm * tn), 1, (unsigned)a.split_k);
  constexpr bool CAN_STAGE = staged_ok(BM, BN, WM, WN, EPI);
  const bool staged = CAN_STAGE && a.ep.vec_ok;
  if constexpr (BM == 256 && BN == 256 && AL == ROW && BL == COL) {
    // both operands K-contiguous: the 4-wave engine (128 x 128 per wave,
    // accumulators in AGPRs, a ring of five LDS half-slots fed by LDS-DMA)
    bool done = launch_w4_staged<T, BMODE, EPI, false, false>(a, grid, s);
    if constexpr (EPI == EPI_STORE_BF16) {
      // beta reads C before the single rounding: the fp32-staged epilogue of
      // the 8-wave engine moves it as 16-byte vectors (rank-r products added
      // to a base product: K is short and C's traffic is the cost)
      if (!done && a.ep.vec_ok && a.ep.beta != 0.f) {
        gemm_dma_kernel<T, BM, BN, 4, 2, EPI, 64, 2, true, 2><<<grid, 512, 0, s>>>(a);
        done = true;
      }
    }
    if (!done) gemm_w4_kernel<T, BMODE, EPI, false><<<grid, 256, 0, s>>>(a);
  } else if constexpr (BM == 64 && (BN == 64 || BN == 128 || BN == 256) && AL == ROW &&
                       (BL == COL || BL == ROW) && BMODE == B_SINGLE) {
    // narrow outputs (N <= 256: X A^T, dY B) with A K-contiguous: 64-row
    // tiles as wide as the output (so X streams once) with 4 waves; a 3-stage
    // ring (48 / 72 KB of LDS: three / two workgroups per CU) or, at 64 x 256,
    // two stages in 80 KB (two per CU).  M/64 tiles fill the chip without a
    // split-K pass.  B may be [N][K] or, read with the transposing LDS loads,
    // [K][N] as stored.
    // (measured cold on MI355X: 4 or 5 stages at 64 x 64 were no faster)
    constexpr int NS = BN == 256 ? 2 : 3;
    constexpr int WPE_N = BN == 64 ? 3 : 2;
    // (nontemporal loads of A, read by one column of tiles, measured 0.2% slower)
    gemm_dma_kernel<T, BM, BN, WM, WN, EPI, 64, NS, false, WPE_N, false, BL == ROW>
        <<<grid, WM * WN * 64, 0, s>>>(a);
  } else if constexpr (BM == 96 && BN == 192 && AL == ROW && BL == COL && BMODE == B_SINGLE) {
    // 129..192 output columns (the three stacked rank-64 LoRA-A products of
    // LoRA-QKV): 96-row tiles of 3 x 2 waves and a 3-stage ring (108 KB, one
    // workgroup per CU; 240 tiles at 22954 tokens, one round on 256 CUs),
    // with no padded columns.  Measured cold on MI355X against 64 x 192 tiles
    // with two stages (two workgroups per CU): [22954, 4096] x [4096, 192]
    // 116 -> 94 us, [4096, 4096] x [4096, 192] 78 -> 61 us, bitwise-equal
    // output; 4 stages no faster than 3; 64 x 64 or 64 x 128 tiles slower.
    gemm_dma_kernel<T, 96, 192, 3, 2, EPI, 64, 3, false, 2><<<grid, 384, 0, s>>>(a);
  } else if constexpr (AL == ROW && BL == ROW && BMODE == B_SINGLE && BM == 256 && BN == 256 &&
                       (EPI == EPI_STORE_BF16 || EPI == EPI_STORE_F32)) {
    // B as stored [K][N]: the 4-wave engine with transposing fragment reads of
    // B; a 16-bit C that is read (beta) or activated, and stores by elements:
    // the 8-wave LDS-DMA engine
    // (every fp32 C with vectors is the 4-wave engine's)
    constexpr bool DMA_STAGE = EPI == EPI_STORE_BF16;
    if (launch_w4_staged<T, BMODE, EPI, false, true>(a, grid, s)) {
    } else if (DMA_STAGE && a.ep.vec_ok)
      gemm_dma_kernel<T, BM, BN, 4, 2, EPI, 64, 2, DMA_STAGE, 2, false, true><<<grid, 512, 0, s>>>(a);
    else
      gemm_dma_kernel<T, BM, BN, 4, 2, EPI, 64, 2, false, 2, false, true><<<grid, 512, 0, s>>>(a);
  } else if constexpr (AL == COL && BL == ROW && BMODE == B_SINGLE && BM == 256 && BN == 256) {
    // both operands token-major (A^T B reduced over tokens): as above, with
    // transposing fragment reads of both
    constexpr int DWM = 4, DWN = 2;
    constexpr bool DMA_STAGE = staged_ok(BM, BN, DWM, DWN, EPI);
    if (launch_w4_staged<T, BMODE, EPI, true, true>(a, grid, s)) {
    } else if (DMA_STAGE && a.ep.vec_ok)
      gemm_dma_kernel<T, BM, BN, DWM, DWN, EPI, 64, 2, DMA_STAGE, 2, true, true><<<grid, DWM * DWN * 64, 0, s>>>(a);
    else
      gemm_dma_kernel<T, BM, BN, DWM, DWN, EPI, 64, 2, false, 2, true, true><<<grid, DWM * DWN * 64, 0, s>>>(a);
  } else if constexpr (AL == COL && BL == ROW && BMODE == B_SINGLE && ((BM == 256 && BN <= 64) || (BM == 32 && BN == 256))) {
    // skinny token reductions (LoRA weight gradients): as the skinny
    // K-contiguous case, with token-major operands
    // the wide operand (A of 256 x N tiles, B of 32 x 256) is read once, so
    // its loads are nontemporal and leave the caches to the narrow one
    // (LoRA-MLP step 0.35%, LoRA-QKV step 0.7% faster, same box)
    constexpr int CPA_T = BM == 256 ? CP_STREAM : 0, CPB_T = BM == 256 ? 0 : CP_STREAM;
    gemm_dma_kernel<T, BM, BN, WM, WN, EPI, 64, SKINNY_NSTAGE, false, SKINNY_WPE, true, true, CPA_T, CPB_T>
        <<<grid, WM * WN * 64, 0, s>>>(a);
  } else if constexpr (BM == 256 && BN <= 64 && AL == ROW && BL == COL && BMODE == B_SINGLE) {
    // skinny output, K-contiguous operands (X A^T, dY B with B^T given): the
    // big operand streams through the LDS-DMA ring; ~72-80 KB of LDS lets two
    // workgroups share a CU, so two K tiles per CU are in flight
    gemm_dma_kernel<T, BM, BN, WM, WN, EPI, SKINNY_BKT, SKINNY_NSTAGE, false, SKINNY_WPE><<<grid, WM * WN * 64, 0, s>>>(a);
  } else {
    if (staged)
      gemm_kernel<T, BM, BN, WM, WN, AL, BL, EPI, CAN_STAGE><<<grid, WM * WN * 64, 0, s>>>(a);
    else
      gemm_kernel<T, BM, BN, WM, WN, AL, BL, EPI, false><<<grid, WM * WN * 64, 0, s>>>(a);
  }
  FORGE_CHECK_LAUNCH();
  return FORGE_OK;
}

template <class T, int AL, int BL, int BMODE, int EPI>
static int launch_layout(int cfg, const GemmArgs& a, hipStream_t s) {
  switch (cfg) {
    case CFG_BIG: return launch_cfg<T, 256, 256, 2, 2, AL, BL, BMODE, EPI>(a, s);
    case CFG_SKINNY_N:
      if constexpr (BMODE == B_SINGLE) {
        if constexpr (AL == ROW) return launch_cfg<T, 64, 64, 2, 2, AL, BL, BMODE, EPI>(a, s);
        return launch_cfg<T, 256, 32, 4, 1, AL, BL, BMODE, EPI>(a, s);
      }
      break;
    case CFG_NARROW_128:
      if constexpr (BMODE == B_SINGLE && AL == ROW) return launch_cfg<T, 64, 128, 2, 2, AL, BL, BMODE, EPI>(a, s);
      break;
    case CFG_NARROW_256:
      if constexpr (BMODE == B_SINGLE && AL == ROW) return launch_cfg<T, 64, 256, 2, 2, AL, BL, BMODE, EPI>(a, s);
      break;
    case CFG_NARROW_192:  // B as [N][K] only (a 192-wide k-row is not a whole number of transposing reads)
      if constexpr (BMODE == B_SINGLE && AL == ROW && BL == COL) return launch_cfg<T, 96, 192, 3, 2, AL, BL, BMODE, EPI>(a, s);
      break;
    case CFG_SKINNY_M:
      if constexpr (BMODE == B_SINGLE) return launch_cfg<T, 32, 256, 1, 4, AL, BL, BMODE, EPI>(a, s);
      break;
    case CFG_SKINNY_N64:
      if constexpr (BMODE == B_SINGLE) {
        if constexpr (AL == ROW) return launch_cfg<T, 64, 64, 2, 2, AL, BL, BMODE, EPI>(a, s);
        if constexpr (AL == COL && BL == ROW) return launch_cfg<T, 256, 64, 4, 1, AL, BL, BMODE, EPI>(a, s);
        return launch_cfg<T, 256, 32, 4, 1, AL, BL, BMODE, EPI>(a, s);
      }
      break;
  }
  return forge_set_error(FORGE_ERR_UNSUPPORTED, "gemm: tile config %d", cfg);
}

template <class T, int EPI>
static int launch_epi(int cfg, int al, int bl, const GemmArgs& a, hipStream_t s) {
  if (al == ROW && bl == COL) return launch_layout<T, ROW, COL, B_SINGLE, EPI>(cfg, a, s);
  if (al == ROW && bl == ROW) return launch_layout<T, ROW, ROW, B_SINGLE, EPI>(cfg, a, s);
  if (al == COL && bl == ROW) return launch_layout<T, COL, ROW, B_SINGLE, EPI>(cfg, a, s);
  if (al == COL && bl == COL) return launch_layout<T, COL, COL, B_SINGLE, EPI>(cfg, a, s);
  return forge_set_error(FORGE_ERR_INVALID, "gemm: layout");
}

}  // namespace fgemm
