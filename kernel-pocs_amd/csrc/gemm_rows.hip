// GEMMs with at most 64 output rows and K-contiguous operands (A [M][K], B
// [N][K]): the products of a decode step, where every weight is read once for
// a few rows and the weights' bytes set the time.
//
// A workgroup owns 16 or 64 output columns (dual B: up to 32 gate and 32 up) and
// all rows; its waves split K in chunks of U 32-deep k-steps, dealt out in
// turn so that the workgroup streams each weight row front to back.  Weights
// go from memory straight to the registers that v_mfma_f32_16x16x32 reads (no
// wave reads a weight that another one needs, so LDS would only add a copy);
// the A fragments come from L2.  The waves' fp32 sums are added in wave order
// through LDS: deterministic.  With 256 x 256 (or 32 x 256) tiles a decode
// step ran on 112 and 16 workgroups.  Measured on MI355X, hidden 4096,
// intermediate 14336, weights not cached: gate/up with SwiGLU at 1 / 16 / 64
// rows 92 / 92 / 93 -> 48 / 50 / 80 us, down projection at 1 / 16 / 32 rows
// 250 / 253 / 256 -> 25 / 32 / 43 us (the weights alone at a read-only pass's
// 5.1 TB/s: 46 and 23 us).  Bound by HBM at few rows, by the A fragments' L2
// traffic (every workgroup reads all of A) at many.
#include "gemm_core.h"
#include "gemm_launch.h"

namespace fgemm {

// MB: blocks of 16 rows; CB: blocks of 16 columns; ND: 2 for the dual gate / up B, else 1.
// Lane l of a wave feeds weight row n0 + l % 16 and output row 16 b + l % 16
// (two k-steps share 64 k: 16 (l / 16) .. + 7, then + 8 .. + 15, in both
// operands), and accumulates columns 4 (l / 16) .. + 3 of row 16 b + l % 16.
template <class T, int MB, int CB, int NW, int EPI>
__global__ __launch_bounds__(NW * 64) void gemm_rows_kernel(GemmArgs args) {
  constexpr int ND = glu_fwd_epi(EPI) ? 2 : 1;
  constexpr int U = MB <= 2 ? 8 : 4;  // k-steps whose loads are in flight
  __shared__ __attribute__((aligned(16))) f32x4 red[NW][CB * ND][MB][64];
  const int lane = threadIdx.x % 64, wave = __builtin_amdgcn_readfirstlane(threadIdx.x / 64);
  const int64_t M = args.M, N = args.N, n0 = (int64_t)blockIdx.x * (16 * CB);
  const int r16 = lane % 16, kg = 16 * (lane / 16);
  f32x4 acc[CB * ND][MB];
#pragma unroll
  for (int d = 0; d < CB * ND; ++d)
#pragma unroll
    for (int b = 0; b < MB; ++b) acc[d][b] = f32x4{0.f, 0.f, 0.f, 0.f};

  int turn = 0;  // chunks dealt out so far, over all segments
  for (int s = 0; s < args.n_segs; ++s) {
    const Seg& sg = args.segs[s];
    if (sg.n_hi <= n0 || sg.n_lo >= n0 + 16 * CB) continue;
    // (a lane whose row does not exist reads zeros; the base, row n0 - n_lo, may
    // lie before the operand, where no lane reads)
    const int64_t brow = n0 - sg.n_lo;
    uint32_t boff[CB];
#pragma unroll
    for (int c = 0; c < CB; ++c) {
      const int64_t n = n0 + 16 * c + r16;
      boff[c] = n < N && n >= sg.n_lo && n < sg.n_hi ? (uint32_t)(((16 * c + r16) * sg.ldb + kg) * 2) : OOB;
    }
    uint32_t aoff[MB];
#pragma unroll
    for (int b = 0; b < MB; ++b)
      aoff[b] = 16 * b + r16 < M ? (uint32_t)(((16 * b + r16) * sg.lda + kg) * 2) : OOB;
    const __amdgpu_buffer_rsrc_t ra = make_rsrc(sg.a);
    const __amdgpu_buffer_rsrc_t rb0 = make_rsrc(sg.b + brow * sg.ldb);
    // up rows of a k_split segment start at column k - k_split
    const int64_t ks1 = ND == 2 ? sg.k_split : 0;
    const __amdgpu_buffer_rsrc_t rb1 = make_rsrc(ND == 2 ? sg.b2 + brow * sg.ldb - ks1 : sg.b);
    // (a null operand reads as zeros, as in the other engines' loaders)
    const bool has_a = sg.a, has_b0 = sg.b, has_b1 = ND == 1 || sg.b2;
    const int n_chunk = (int)((sg.k + 32 * U - 1) / (32 * U));
    const int first = ((wave - turn) % NW + NW) % NW;
    turn += n_chunk;
    auto load = [&](__amdgpu_buffer_rsrc_t r, uint32_t off, int k) {
      return __builtin_bit_cast(bf16x8, __builtin_amdgcn_raw_buffer_load_b128(r, (int)off, 2 * k, 0));
    };
    auto chunk = [&](int k0, bool whole) {
      bf16x8 bf[U][CB * ND], af[U][MB];
#pragma unroll
      for (int u = 0; u < U; ++u) {
        const int k = k0 + 64 * (u / 2) + 8 * (u % 2);
        const bool in = whole || k + kg < sg.k;
        // (a k_split segment: gate rows read k < k_split, up rows the rest)
        const bool in0 = whole || (in && has_b0 && (ks1 == 0 || k + kg < ks1));
        const bool in1 = whole || (in && has_b1 && k + kg >= ks1);
#pragma unroll
        for (int c = 0; c < CB; ++c) {
          bf[u][c * ND] = load(rb0, in0 ? boff[c] : OOB, k);
          if constexpr (ND == 2) bf[u][c * ND + 1] = load(rb1, in1 ? boff[c] : OOB, k);
        }
#pragma unroll
        for (int b = 0; b < MB; ++b) af[u][b] = load(ra, whole || (in && has_a) ? aoff[b] : OOB, k);
      }
      // every load of the chunk is issued before the first wait (left to the
      // scheduler, half of them were)
      __builtin_amdgcn_sched_barrier(0);
#pragma unroll
      for (int u = 0; u < U; ++u)
#pragma unroll
        for (int d = 0; d < CB * ND; ++d)
#pragma unroll
          for (int b = 0; b < MB; ++b) acc[d][b] = mfma16<T>(bf[u][d], af[u][b], acc[d][b]);
    };
    for (int c = first; c < n_chunk; c += NW) {
      const int k0 = c * 32 * U;
      if (ks1 == 0 && has_a && has_b0 && has_b1 && k0 + 32 * U <= sg.k) chunk(k0, true);
      else chunk(k0, false);
    }
  }
#pragma unroll
  for (int d = 0; d < CB * ND; ++d)
#pragma unroll
    for (int b = 0; b < MB; ++b) red[wave][d][b][lane] = acc[d][b];
  __syncthreads();
  const EpiArgs& ep = args.ep;
  for (int i = threadIdx.x; i < CB * MB * 64; i += NW * 64) {
    const int c = i / (MB * 64), b = i / 64 % MB, l = i % 64;
    const int64_t m = 16 * b + l % 16, n = n0 + 16 * c + 4 * (l / 16);
    f32x4 v[ND];
#pragma unroll
    for (int d = 0; d < ND; ++d) {
      v[d] = red[0][c * ND + d][b][l];
#pragma unroll
      for (int w = 1; w < NW; ++w) v[d] += red[w][c * ND + d][b][l];
    }
    if (m >= M) continue;
#pragma unroll
    for (int q = 0; q < 4; ++q) {
      if (n + q >= N) break;
      if constexpr (ND == 2) {
        const float e = v[0][q], g = v[1][q];
        if (ep.e) {
          ep.e[m * ep.ld_eg + n + q] = (__bf16)e;
          ep.g[m * ep.ld_eg + n + q] = (__bf16)g;
        }
        ((__bf16*)ep.c)[m * ep.ldc + n + q] = (__bf16)glu_fwd_h<EPI>(e, g);
      } else {
        float a = ep.alpha;
        if (ep.alpha_group > 0) {
          const int64_t grp = (n + q) / ep.alpha_group;
          a = ep.alphas[grp < 4 ? grp : 3];
        }
        T* cp = (T*)ep.c + m * ep.ldc + n + q;
        float o = a * v[0][q];
        if (ep.beta != 0.f) o += ep.beta * (float)*cp;
        if (ep.act) o = epi_act(ep.act, o);
        *cp = (T)o;
      }
    }
  }
}

template <class T, int MB, int CB, int NW, int EPI>
static int launch_one(const GemmArgs& a, hipStream_t s) {
  const int64_t blocks = (a.N + 16 * CB - 1) / (16 * CB);
  if (blocks > 0x7fffffffLL) return forge_set_error(FORGE_ERR_INVALID, "gemm: too many tiles");
  gemm_rows_kernel<T, MB, CB, NW, EPI><<<(unsigned)blocks, NW * 64, 0, s>>>(a);
  FORGE_CHECK_LAUNCH();
  return FORGE_OK;
}

// Single B: 16 columns a workgroup (32 leave CUs without one at N = 4096: 32
// -> 43 us at 16 rows), or 64 (rows_columns); 4, 8 and 16 waves measured equal
// there, and more shorten the K loop where there are few workgroups.
template <class T, int MB>
static int launch_single(const GemmArgs& a, hipStream_t s) {
  if constexpr (MB == 1)
    if (rows_columns(a) == 64) return launch_one<T, MB, 4, 4, EPI_STORE_BF16>(a, s);
  if (a.N < 16 * 64) return launch_one<T, MB, 1, 16, EPI_STORE_BF16>(a, s);
  return launch_one<T, MB, 1, 8, EPI_STORE_BF16>(a, s);
}

// Dual B: 32 + 32 columns a workgroup halve the A traffic from L2 (64 rows,
// 14336 columns: 107 -> 80 us; 16 rows 53 -> 50) where that leaves at least
// 128 workgroups.
template <int MB, int EPI>
static int launch_dual(const GemmArgs& a, hipStream_t s) {
  if (a.N < 32 * 128) return launch_one<bf16_t, MB, 1, 4, EPI>(a, s);
  return launch_one<bf16_t, MB, 2, 4, EPI>(a, s);
}

template <int EPI>
static int launch_glu(const GemmArgs& a, hipStream_t s) {
  if (a.M <= 16) return launch_dual<1, EPI>(a, s);
  if (a.M <= 32) return launch_dual<2, EPI>(a, s);
  return launch_dual<4, EPI>(a, s);
}

int launch_rows(int epi, const GemmArgs& a, hipStream_t s) {
  if (!rows_engine(epi, a)) return forge_set_error(FORGE_ERR_INVALID, "gemm: %lld rows", (long long)a.M);
  switch (epi) {
    case EPI_STORE_BF16:
      if (a.f16) return a.M <= 16 ? launch_single<fp16_t, 1>(a, s) : launch_single<fp16_t, 2>(a, s);
      return a.M <= 16 ? launch_single<bf16_t, 1>(a, s) : launch_single<bf16_t, 2>(a, s);
    case EPI_SWIGLU_FWD: return launch_glu<EPI_SWIGLU_FWD>(a, s);
    case EPI_GEGLU_TANH_FWD: return launch_glu<EPI_GEGLU_TANH_FWD>(a, s);
    case EPI_GEGLU_ERF_FWD: return launch_glu<EPI_GEGLU_ERF_FWD>(a, s);
  }
  return forge_set_error(FORGE_ERR_UNSUPPORTED, "gemm: epilogue %d on %lld rows", epi, (long long)a.M);
}

}  // namespace fgemm
