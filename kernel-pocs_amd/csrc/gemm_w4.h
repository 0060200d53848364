// Big-tile MFMA engine: 256 x 256 x BKT block tiles computed by 4 waves of
// 128 x 128, one wave per SIMD.
//
// Why 4 waves of 128 x 128: a wave's LDS fragment reads per MFMA fall with
// the size of its output tile.  A 128 x 128 wave tile reads 8 A + 8 B
// fragments per 64 MFMAs; the 64 x 128 wave tiles of 8 waves half as many
// again, which with the LDS-DMA writes held the LDS port, not the matrix
// cores, as the limit (MFMA busy 63% on MI355X).  The 256 fp32 accumulators
// per lane need the whole AGPR file, so each SIMD holds exactly one wave (512
// registers: 256 VGPRs + 256 AGPRs).
//
// Why v_mfma_f32_16x16x32: under MFMA load the chip is held by its power, and
// this shape does the same work for less.  Register-only loops on random bf16
// data, back to back: 2100 TFLOP/s against 1820 with 32x32x16 (2460 both on
// zeros).  The GEMMs, back to back, 32x32x16 -> 16x16x32: [8192, 4096] K =
// 14336 838 -> 806 us, [4096, 4096] K = 128256 3137 -> 2900, [4096, 128256] K =
// 4096 3423 -> 3330 (hipBLASLt on the same box: 650, 2740 and 3000).  With a
// few tiles in flight, where power does not matter, a K tile takes 1.08 us
// either way.
//
// With one wave per SIMD nothing else covers a stall, so the main loop keeps
// the matrix core fed across K-tile boundaries:
//   * fragments are double-buffered in registers: the 16 reads of the next
//     32-deep k-step are interleaved with the 64 MFMAs of this one;
//   * the workgroup barrier of each K tile sits before the tile's LAST
//     k-step (whose fragments are already in registers), so the barrier, the
//     first fragment reads of the next tile and the DMA issue for the freed
//     LDS slot all overlap that k-step's MFMAs instead of draining the pipe;
//   * global -> LDS moves by LDS-DMA (buffer_load ... lds) into a ring of
//     half-tiles.  A DMA whose tile does not exist is still issued, with every
//     offset out of range (the hardware returns zeros without a fetch);
//   * the addresses of the next DMA are two scalar additions; segment
//     switches, partial last tiles and the end of the list take a path out of
//     the loop's way.  (Walking (segment, tile) cursors there, with 64-bit
//     multiplies and two far branches between the last MFMA and the barrier,
//     cost 1 to 3% of the whole product.)
#pragma once

#include "gemm_core.h"
#include "gemm_w4_epi.h"

namespace fgemm {

constexpr int SG_VMEM_READ = 0x020;

// s_waitcnt vmcnt <= N and lgkmcnt == 0 (expcnt not waited on).
template <int N>
__device__ __forceinline__ void wait_vm_lgkm0() {
  static_assert(N >= 0 && N < 64, "vmcnt range");
  __builtin_amdgcn_s_waitcnt((N & 15) | ((N >> 4) << 14) | (7 << 4));
}

// Bare workgroup barrier (no release fence: __syncthreads() would make the
// compiler wait for every outstanding LDS-DMA, vmcnt(0)).  The empty asm
// statements keep LDS accesses from moving across it at compile time.
__device__ __forceinline__ void bare_barrier() {
  asm volatile("" ::: "memory");
  __builtin_amdgcn_s_barrier();
  asm volatile("" ::: "memory");
}

// LDS-DMA loader of one 256-row K-contiguous operand tile for the 4-wave
// engine.  As DmaLoader (XOR-swizzled 16-byte chunks, OOB offsets read
// zeros), but the segment-tail mask is a per-lane select instead of a
// branch, so that the DMA issue can be interleaved with MFMAs.
template <int BKT, bool DUAL>
struct W4Loader {
  static constexpr int BROWS = 256, NT = 256;
  static constexpr int RB = BKT * 2;          // LDS bytes per row
  static constexpr int CPR = RB / 16;         // 16-byte chunks per row
  static constexpr int RPI = 64 / CPR;        // rows per wave instruction
  static constexpr int IPW = BROWS / RPI / 4; // instructions per wave per tile
  static_assert(!DUAL || RPI <= 32, "dual: an instruction's rows inside one 32-row group");
  uint32_t voff[IPW];  // byte offset of this lane's chunk in the panel (OOB = zero-fill)
  const char* base[2];
  int64_t ld_bytes;
  int kch[2];          // first k of this lane's chunk, by instruction parity
  int64_t k_split;     // dual: gate rows k < k_split, up rows k >= k_split (0: none)

  // 32-row groups alternate gate / up.  A wave's rows are a whole number of
  // 64-row pairs, so the pointer an instruction reads depends on j alone:
  // a compile-time choice (computed from the wave index, the compiler kept
  // both descriptors in a scratch array and issued every DMA through a
  // waterfall loop with vmcnt(0): the dual GEMM ran 2.6x slower).
  static_assert((IPW * RPI) % 64 == 0, "wave slab = whole gate/up group pairs");
  static __device__ __forceinline__ constexpr int sel_of(int j) { return DUAL ? ((j * RPI) / 32) % 2 : 0; }

  template <class RowSrc>
  __device__ __forceinline__ void setup(const void* p0, const void* p1, int64_t ld, int64_t panel_off,
                                        RowSrc row_src, int64_t ksplit = 0) {
    ld_bytes = ld * 2;
    k_split = DUAL ? ksplit : 0;
    const int64_t pan = panel_off * ld_bytes;
    base[0] = p0 ? (const char*)p0 + pan : nullptr;
    // (up rows: k is counted from the segment start, their column is k - k_split;
    // every lane that reads them has k >= k_split, so no address before p1 is read)
    base[1] = DUAL ? (p1 ? (const char*)p1 + pan - k_split * 2 : nullptr) : base[0];
    const int lane = threadIdx.x % 64, wave = threadIdx.x / 64;
    // A lane's chunk depends on its instruction only through the parity of
    // the instruction's first row / RPI (BKT 64: swz = (row >> 1) & 7 with 8
    // rows per instruction; BKT 32: not at all), so two values cover it.
    static_assert(IPW % 2 == 0, "instruction parity = j parity");
#pragma unroll
    for (int j = 0; j < IPW; ++j) {
      const int q = (wave * IPW + j) * RPI + lane / CPR;   // tile row
      const int chunk = (lane % CPR) ^ swz<BKT>(q);        // source chunk of LDS slot lane % CPR
      const int sel = sel_of(j);
      const int64_t row = base[sel] ? row_src(q, sel) : -1;
      voff[j] = row < 0 ? OOB : (uint32_t)(row * ld_bytes + chunk * 16);
      if (j < 2) kch[j] = chunk * 8;
    }
  }

  // Addresses and tail masks of one K-tile DMA at k0 (kvalid valid k; <= 0:
  // every chunk reads zeros); load_one issues instruction j of it, next()
  // moves to the following tile of the segment (the masks stay).
  struct Prep {
    const char* p0;
    const char* p1;
    bool kin[2][2];  // [gate / up rows][instruction parity]
    __device__ __forceinline__ void next() {
      p0 += BKT * 2;
      if constexpr (DUAL) p1 += BKT * 2;
    }
  };
  __device__ __forceinline__ Prep prep(int64_t k0, int64_t kvalid) const {
    Prep p;
    p.p0 = base[0] + k0 * 2;
    p.p1 = base[1] + k0 * 2;
    const int64_t ks = k_split - k0;  // the split in tile coordinates
#pragma unroll
    for (int par = 0; par < 2; ++par) {
      p.kin[0][par] = kch[par] < kvalid && (k_split == 0 || kch[par] < ks);
      p.kin[1][par] = kch[par] < kvalid && kch[par] >= ks;
    }
    return p;
  }
  __device__ __forceinline__ void load_one(const Prep& p, int j, char* dst) const {
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x / 64);
    const uint32_t off = p.kin[sel_of(j)][j % 2] ? voff[j] : OOB;
    const __amdgpu_buffer_rsrc_t r = make_rsrc(sel_of(j) ? p.p1 : p.p0);
    __builtin_amdgcn_raw_ptr_buffer_load_lds(r,
                                             (__attribute__((address_space(3))) void*)(dst + (wave * IPW + j) * 1024),
                                             16, off, 0, 0, 0);
  }
};

// The same for a token-major operand (A stored [K][M], B stored [K][N]): the
// half-tile is 64 k-rows of 256 elements as they lie in memory, and the
// fragments are read with ds_read_b64_tr_b16 (the lane layout stands with
// tr_frag).  A 16x16x32 fragment's 16-lane group g takes k 8 g .. 8 g + 7 of 16
// rows: 32 bytes of each of four k-rows a read.  k-rows are 512 bytes, so the
// XOR of a k-row's 16-byte chunks puts those four in different 64-byte
// windows of the 256-byte bank cycle, and the two groups of a half-wave (k-rows
// 8 apart) in different halves of them.
// Against 8 waves of 32x32x16 (gemm_dma_kernel), MI355X: [8192, 4096] K = 14336 with
// B as [K][N] 850 -> 743 us (733 with both K-contiguous), A^T B [32768, 4096] K =
// 4096 1000 -> 945.
__device__ __forceinline__ int swz_w4t(int q) { return 4 * (q & 3) + 2 * ((q >> 3) & 1); }

template <int BKT>
struct W4LoaderT {
  static constexpr int RB = 512;               // LDS bytes per k-row
  static constexpr int CPR = RB / 16;          // 16-byte chunks per k-row
  static constexpr int RPI = 64 / CPR;         // k-rows per wave instruction
  static constexpr int IPW = BKT / RPI / 4;    // instructions per wave per tile
  uint32_t voff[IPW];  // byte offset of this lane's chunk from the tile's first k-row (OOB = zero-fill)
  const char* base;
  int64_t ld_bytes;
  int q0;              // this lane's k-row of instruction 0

  // row_ok(r): row panel_off + r exists (extents are multiples of 8, so a
  // chunk's 8 rows exist or not together)
  template <class RowOk>
  __device__ __forceinline__ void setup(const void* p, int64_t ld, int64_t panel_off, RowOk row_ok) {
    ld_bytes = ld * 2;
    base = p ? (const char*)p + panel_off * 2 : nullptr;
    const int lane = threadIdx.x % 64, wave = threadIdx.x / 64;
    q0 = wave * IPW * RPI + lane / CPR;
#pragma unroll
    for (int j = 0; j < IPW; ++j) {
      const int q = q0 + j * RPI;
      const int chunk = (lane % CPR) ^ swz_w4t(q);  // source chunk of LDS slot lane % CPR
      voff[j] = (base && row_ok(chunk * 8)) ? (uint32_t)(q * ld_bytes + chunk * 16) : OOB;
    }
  }

  struct Prep {
    const char* p0;
    int64_t step;  // bytes of a K tile
    int kvalid;    // k-rows of the tile that exist
    __device__ __forceinline__ void next() { p0 += step; }
  };
  __device__ __forceinline__ Prep prep(int64_t k0, int64_t kvalid) const {
    return {base + k0 * ld_bytes, BKT * ld_bytes, (int)(kvalid < BKT ? kvalid : BKT)};
  }
  __device__ __forceinline__ void load_one(const Prep& p, int j, char* dst) const {
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x / 64);
    const uint32_t off = q0 + j * RPI < p.kvalid ? voff[j] : OOB;
    const __amdgpu_buffer_rsrc_t r = make_rsrc(p.p0);
    __builtin_amdgcn_raw_ptr_buffer_load_lds(r,
                                             (__attribute__((address_space(3))) void*)(dst + (wave * IPW + j) * 1024),
                                             16, off, 0, 0, 0);
  }
};

// Byte offset, in a token-major half-tile, of what this lane supplies to the
// fragment of rows r0 .. r0 + 15 (r0 a multiple of 128) at k 0..3; rows 16 i
// further: ^ (i << 5); k-row q further: + q * 512 (q = 4, or a multiple of 32).
__device__ __forceinline__ int w4t_lane_offset(int r0, int lane) {
  const int l = lane % 16, q = 8 * (lane / 16) + l / 4, r = r0 + 4 * (l % 4);
  return q * 512 + (((r / 8) ^ swz_w4t(q)) * 16) + (r % 8) * 2;
}

// Ring of NHALF half-slots of 32 KB (256 rows x 64 k of one operand).  K
// tile x keeps A in half-slot (2x) % NHALF and B in (2x + 1) % NHALF.  With
// NHALF = 5 (160 KB) the barrier of iteration t frees tile t's two halves,
// which take B of tile t+2 and A of tile t+3: the copy engine always has the
// older half of the next tile in flight when new work arrives, so the L2 ->
// LDS stream never drains (with two whole-tile stages every period paid the
// copy time plus the L2 latency: 811 against ~610 us on the 8192 x 4096 x
// 14336 product, MI355X).
constexpr int W4_NHALF = 5;
constexpr int W4_HALF = 256 * 64 * 2;  // bytes per half-slot

template <class T, int BMODE, int EPI, bool STAGED, bool AT = false, bool BT = false, bool PLAIN = true>
__global__ __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(1, 1)))
void gemm_w4_kernel(GemmArgs args) {
  constexpr int BM = 256, BN = 256, WAVES_M = 2, WAVES_N = 2, BKT = 64;
  constexpr int TM = BM / WAVES_M, TN = BN / WAVES_N;  // 128 x 128 per wave
  constexpr int FM = TM / 16, FN = TN / 16;            // 16 x 16 blocks per wave
  constexpr int KS = BKT / 32;                         // k-steps per K tile
  constexpr int RB = BKT * 2;                          // LDS bytes per row
  constexpr int NH = W4_NHALF;
  static_assert(KS == 2, "one fragment slot per k-step of a tile");
  constexpr int RING = NH * W4_HALF;
  static_assert(RING >= W4_STAGE_BYTES && RING >= W4_DUAL_BYTES, "the staged epilogue reuses the ring");
  constexpr int SMEM = RING;
  __shared__ __attribute__((aligned(1024))) char smem[SMEM];

  const int64_t M = args.M;
  constexpr int OUT_BN = (BMODE == B_DUAL) ? BN / 2 : BN;
  const int64_t tiles_m = (M + BM - 1) / BM;
  const int64_t tiles_n = (args.N + OUT_BN - 1) / OUT_BN;
  int tmi, tni;
  tile_coords(tiles_m, tiles_n, tmi, tni, args);
  const int64_t m0 = (int64_t)tmi * BM;
  const int64_t n0 = (int64_t)tni * OUT_BN;
  const int lane = threadIdx.x % 64;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x / 64);
  const int wm = wave % WAVES_M;
  const int wn = wave / WAVES_M;

  int seg_tiles[MAX_SEGS];
  int total_tiles = 0;
  for (int s = 0; s < args.n_segs; ++s) {
    const Seg& sg = args.segs[s];
    const bool active = sg.n_hi > n0 && sg.n_lo < n0 + OUT_BN;
    seg_tiles[s] = active ? (int)((sg.k + BKT - 1) / BKT) : 0;
    total_tiles += seg_tiles[s];
  }
  const int per = (total_tiles + args.split_k - 1) / args.split_k;
  const int t_begin = blockIdx.z * per;
  const int t_end = min(total_tiles, t_begin + per);

  f32x4 acc[FM][FN];
#pragma unroll
  for (int i = 0; i < FM; ++i)
#pragma unroll
    for (int j = 0; j < FN; ++j) acc[i][j] = f32x4{0.f, 0.f, 0.f, 0.f};

  static_assert(!(BT && BMODE == B_DUAL), "dual B operands are K-contiguous");
  using LoaderA = std::conditional_t<AT, W4LoaderT<BKT>, W4Loader<BKT, false>>;
  using LoaderB = std::conditional_t<BT, W4LoaderT<BKT>, W4Loader<BKT, BMODE == B_DUAL>>;
  using PrepA = typename LoaderA::Prep;
  using PrepB = typename LoaderB::Prep;
  LoaderA la;
  LoaderB lb;
  PrepA pa_cur;  // A of tile t+2 (dst half-slot ha_dst)
  PrepB pb_cur;  // B of tile t+1 (dst half-slot hb_dst)
  auto setup_a = [&](int s) {
    const Seg& sg = args.segs[s];
    if constexpr (AT) la.setup(sg.a, sg.lda, m0, [&](int r) { return m0 + r < M; });
    else la.setup(sg.a, sg.a, sg.lda, m0, [&](int q, int) -> int64_t { return m0 + q < M ? q : -1; });
  };
  auto setup_b = [&](int s) {
    const Seg& sg = args.segs[s];
    if constexpr (BT) {
      lb.setup(sg.b, sg.ldb, n0 - sg.n_lo, [&](int r) {
        const int64_t n = n0 + r;
        return n < args.N && n >= sg.n_lo && n < sg.n_hi;
      });
    } else if constexpr (BMODE == B_DUAL) {
      lb.setup(sg.b, sg.b2, sg.ldb, n0, [&](int q, int) -> int64_t {
        const int t4 = (q % 128) / 32;
        const int rel = (q / 128) * 64 + (t4 / 2) * 32 + q % 32;
        return n0 + rel < args.N ? rel : -1;
      }, sg.k_split);
    } else {
      const int64_t off = n0 - sg.n_lo;
      lb.setup(sg.b, sg.b, sg.ldb, off, [&](int q, int) -> int64_t {
        const int64_t n = n0 + q;
        return (n < args.N && n >= sg.n_lo && n < sg.n_hi) ? q : -1;
      });
    }
  };
  // A and B walk the flat K-tile list [t_begin, t_end); `at` points a loader at
  // tile t of it (past the end: nothing is read) and returns how many tiles
  // after it next() alone reaches: whole ones of the same segment.
  const int n_t = t_end - t_begin;
  int seg_a = -1, seg_b = -1;  // segments that la and lb are set up for
  constexpr int FOREVER = 1 << 30;
  auto at = [&](int t, auto& loader, auto& setup, int& seg, auto& out) -> int {
    if (t >= n_t) {
      out = loader.prep(0, 0);
      return FOREVER;
    }
    int s = 0, rel = t_begin + t;
    while (rel >= seg_tiles[s]) rel -= seg_tiles[s++];
    if (s != seg) setup(s);
    seg = s;
    const int64_t k = args.segs[s].k, k0 = (int64_t)rel * BKT;
    out = loader.prep(k0, k - k0);
    // (a k_split segment's masks change from tile to tile)
    const int whole = (BMODE == B_DUAL && args.segs[s].k_split) ? 0 : (int)(k / BKT) - 1 - rel;
    return whole < 0 ? 0 : (whole < n_t - 1 - t ? whole : n_t - 1 - t);
  };
  auto at_a = [&](int t, PrepA& out) { return at(t, la, setup_a, seg_a, out); };
  auto at_b = [&](int t, PrepB& out) { return at(t, lb, setup_b, seg_b, out); };

  constexpr int IPH = LoaderA::IPW;  // DMA instructions per wave per half-tile
  static_assert(IPH == LoaderB::IPW, "equal halves");
  auto half_ptr = [&](int h) { return smem + h * W4_HALF; };

  // per-lane fragment offsets: row (wave tile + lane % 16), chunk 4 ks + lane / 16, swizzled
  const int g = swz<BKT>(lane % 16) ^ (lane / 16);  // chunk ^ swz = 4 ks ^ g
  const int a_row = (wm * TM + lane % 16) * RB;
  const int b_row = (wn * TN + lane % 16) * RB;
  const int a_tr = AT ? w4t_lane_offset(wm * TM, lane) : 0;
  const int b_tr = BT ? w4t_lane_offset(wn * TN, lane) : 0;
  bf16x8 af[KS][FM], bfr[KS][FN];
  auto read_tr = [&](const char* half, int off, int ks, int i) {
    const char* p = smem + (((int)(half - smem) + off) ^ (i << 5)) + ks * 32 * 512;
    return tr_frag(p, p + 4 * 512);
  };
  auto read_a = [&](const char* pa, int ks, int i) {
    if constexpr (AT) return read_tr(pa, a_tr, ks, i);
    else return *reinterpret_cast<const bf16x8*>(pa + a_row + i * 16 * RB + (((4 * ks) ^ g) << 4));
  };
  auto read_b = [&](const char* pb, int ks, int j) {
    if constexpr (BT) return read_tr(pb, b_tr, ks, j);
    else return *reinterpret_cast<const bf16x8*>(pb + b_row + j * 16 * RB + (((4 * ks) ^ g) << 4));
  };
  // fragment read `idx` of k-step ks of the tile in half-slots (pa, pb), in
  // the order the MFMAs consume them: A0, B0 .. B7, A1 .. A7
  auto frag_read = [&](const char* pa, const char* pb, int ks, int idx) {
    if (idx == 0) af[ks][0] = read_a(pa, ks, 0);
    else if (idx <= FN) bfr[ks][idx - 1] = read_b(pb, ks, idx - 1);
    else af[ks][idx - FN] = read_a(pa, ks, idx - FN);
  };
  // MFMAs 4p .. 4p + 3 of a k-step, (i, j) row-major.  The operands are
  // swapped (block (i, j) is computed as B_j A_i^T), so a lane accumulates
  // four consecutive output columns of one row (the layout gemm_w4_epi.h
  // stages with 8-byte writes).
  auto mfma_group = [&](int ks, int p) {
#pragma unroll
    for (int u = 0; u < 4; ++u) {
      const int m = 4 * p + u, i = m / FN, j = m % FN;
      acc[i][j] = mfma16<T>(bfr[ks][j], af[ks][i], acc[i][j]);
    }
  };
  constexpr int NGRP = FM * FN / 4;  // 16 groups of four MFMAs per k-step ...
  static_assert(NGRP == FM + FN && NGRP == 2 * IPH, "... 16 fragment reads and 8 DMA instructions");

  // Per period (barrier(t-1) .. barrier(t)) the second k-step of tile t-1
  // issues the DMA of B of tile t+1 (its deadline is barrier(t)) and the first
  // of tile t that of A of tile t+2 (deadline barrier(t+1)), one instruction
  // after every other group, so that no stretch carries a burst (16 in a
  // quarter of a tile held the in-order issue: loop time per K tile 3300
  // cycles against the MFMAs' 2048).
  if (n_t > 0) {
    // prologue: A0, B0, A1 and B1 into half-slots 0 .. 3 (the wait below counts
    // the IPH instructions of each); A2 follows in tile 0's k-steps
    at_a(0, pa_cur);
#pragma unroll
    for (int d = 0; d < IPH; ++d) la.load_one(pa_cur, d, half_ptr(0));
    at_b(0, pb_cur);
#pragma unroll
    for (int d = 0; d < IPH; ++d) lb.load_one(pb_cur, d, half_ptr(1));
    at_a(1, pa_cur);
#pragma unroll
    for (int d = 0; d < IPH; ++d) la.load_one(pa_cur, d, half_ptr(2));
    int run_b = at_b(1, pb_cur);
#pragma unroll
    for (int d = 0; d < IPH; ++d) lb.load_one(pb_cur, d, half_ptr(3));
    // iterations that need no more than next(), for both operands
    int run = at_a(2, pa_cur);
    run = run < run_b ? run : run_b;
    char* ha_dst = half_ptr(4);
    wait_vm_lgkm0<2 * IPH>();  // tile 0 (halves 0, 1) landed (this wave's part)
    bare_barrier();
#pragma unroll
    for (int p = 0; p < NGRP; ++p) frag_read(half_ptr(0), half_ptr(1), 0, p);
    // nothing but these reads outstanding at the loop entry, so the waits
    // inside the loop can count them precisely
    wait_vm_lgkm0<63>();
    int ha = 0;  // half-slot of tile t's A (B is the next one)
    for (int t = 0; t < n_t; ++t) {
      const int hb = ha + 1 == NH ? 0 : ha + 1;
      const char* pa_t = half_ptr(ha);
      const char* pb_t = half_ptr(hb);
      // Program order is pinned (sched_barrier): the fragment reads of the
      // other k-step and the DMA instructions are issued between groups of
      // four MFMAs, in their shadow.  (The reads two a group at first, so that
      // all have landed by the wait before the barrier, measured equal; the
      // DMA in the first half of each k-step, or the barrier 2 or 4 groups into
      // the second one, 1 to 3% slower.)
#pragma unroll
      for (int p = 0; p < NGRP; ++p) {
        mfma_group(0, p);
        if (p % 2) la.load_one(pa_cur, p / 2, ha_dst);
        frag_read(pa_t, pb_t, 1, p);
        __builtin_amdgcn_sched_barrier(0);
      }
      // Second k-step: its fragments are in registers.  Wait until this wave's
      // reads of tile t are done and its part of tile t+1 has landed (A of
      // tile t+2 may stay in flight), then one barrier: after it tile t+1 is
      // whole in LDS and tile t's half-slots (ha, hb) are free for B of tile
      // t+2 and A of tile t+3.
      wait_vm_lgkm0<IPH>();
      bare_barrier();
      if (__builtin_expect(--run >= 0, 1)) {
        pa_cur.next();
        pb_cur.next();
      } else {  // a segment's last, partial tile, the next segment, or the end
        run_b = at_b(t + 2, pb_cur);
        run = at_a(t + 3, pa_cur);
        run = run < run_b ? run : run_b;
      }
      char* hb_dst = half_ptr(ha);
      ha_dst = half_ptr(hb);
      const int ha1 = hb + 1 == NH ? 0 : hb + 1;  // tile t+1's halves
      const int hb1 = ha1 + 1 == NH ? 0 : ha1 + 1;
      const char* pa_n = half_ptr(ha1);  // (after the last tile: slots nobody reads; in bounds)
      const char* pb_n = half_ptr(hb1);
#pragma unroll
      for (int p = 0; p < NGRP; ++p) {
        mfma_group(1, p);
        if (p % 2) lb.load_one(pb_cur, p / 2, hb_dst);
        frag_read(pa_n, pb_n, 0, p);
        __builtin_amdgcn_sched_barrier(0);
      }
      ha = ha1;
    }
    wait_vmcnt<0>();  // no zero-fill DMA may land in the staged epilogue's LDS
  }
  // The epilogue's per-lane addresses are formed here: hoisted above the main
  // loop (which holds 128 VGPRs of fragments), they spill inside it.
  int elane = lane, ewave = wave;
  asm volatile("" : "+v"(elane), "+s"(ewave));
  const int ewm = ewave % WAVES_M, ewn = ewave / WAVES_M;
  if constexpr (STAGED) {
    static_assert(w4_staged_epi(EPI), "staged epilogue: 16-bit or fp32 outputs");
    static_assert(RING >= W4_F32_BYTES, "the fp32 epilogue's slabs reuse the ring");
    __bf16* lds = reinterpret_cast<__bf16*>(smem);
    if constexpr (EPI == EPI_STORE_F32)
      w4_epilogue_f32<PLAIN>(args, acc, m0, n0, elane, ewm, ewn, reinterpret_cast<float*>(smem));
    else if constexpr (BMODE == B_DUAL)
      w4_epilogue_staged_dual<EPI>(args, acc, m0, n0, elane, ewm, ewn, lds);
    else  // (STORE_BF16 is launched staged at beta = 0 only)
      w4_epilogue_staged<T, EPI>(args, acc, m0, n0, elane, ewm, ewn, lds);
  } else {
    w4_epilogue_direct<T, BMODE, EPI>(args, acc, m0, n0, elane, ewm, ewn);
  }
}

}  // namespace fgemm
