// Host launchers for the MFMA GEMM core: the generic forge_gemm entry point
// and the fused LoRA entry points (LoRA-MLP gate/up + SwiGLU / GeGLU, LoRA-MLP
// down-projection backward + SwiGLU / GeGLU backward, LoRA-QKV + RoPE).
#include "gemm_launch.h"

namespace fgemm {

// 33 .. 64 rows of K-contiguous operands take the big tiles instead of two rows
// of 32-row ones (a register engine) where the caller split them over K, and,
// of the products whose big-tile epilogue moves vectors, where the 32-row tiles
// no longer fit on 256 CUs at once and where a short product is added to a
// 16-bit C (whose traffic is the cost).  Measured on MI355X, 64 rows, 32-row
// against big tiles: [4096], K = 14336 240 / 45 us split 16 ways, 260 unsplit;
// unsplit, K = 4096: [4096] 61 / 76, with SiLU 62 / 140, fp32 atomics 68 / 182,
// [32000] 92 / 93, [40960] 152 / 98, [128256] 341 / 228; added to C, K = 64:
// [4096] 13 / 10, K = 256 [14336] 15 / 14, K = 1024 [1024] 23 / 28.
static bool few_rows_big(int64_t N, int epi, const GemmArgs& a) {
  if (a.split_k > 1) return epi == EPI_STORE_F32;
  const bool linear = a.ep.act == ACT_NONE && a.ep.alpha_group == 0;
  if (!a.ep.vec_ok || (epi != EPI_STORE_F32 && !(epi == EPI_STORE_BF16 && linear))) return false;
  const bool short_k = total_k(a) <= 256;
  if (2 * ((N + 255) / 256) > 256) return linear || !short_k;
  return epi == EPI_STORE_BF16 && a.ep.beta != 0.f && short_k;
}

// Picks a tile shape from the output shape (a K-contiguous A takes the
// 64-row narrow tiles up to N = 256).
static int pick_cfg(int64_t N, int al, int bl, int epi, const GemmArgs& a) {
  const int64_t M = a.M;
  if (al == ROW && (bl == COL || bl == ROW) && N <= 256 && M > N)
    return N <= 64 ? CFG_SKINNY_N64 : N <= 128 ? CFG_NARROW_128 : (N <= 192 && bl == COL) ? CFG_NARROW_192 : CFG_NARROW_256;
  if (N <= 32 && M > N) return CFG_SKINNY_N;
  if (N <= 64 && M > N) return CFG_SKINNY_N64;
  if (M > 32 && M <= 64 && N > 256 && al == ROW && bl == COL && few_rows_big(N, epi, a)) return CFG_BIG;
  if (M <= 64 && N > M) return CFG_SKINNY_M;
  return CFG_BIG;
}

// Largest operand pitch (elements of 2 bytes): 256 rows of it span < 2^31 bytes.
constexpr int64_t kMaxLd = (int64_t(1) << 31) / (256 * 2) - 1;

static int check_segs(const GemmArgs& a, int al, int bl) {
  if (a.n_segs < 1 || a.n_segs > MAX_SEGS)
    return forge_set_error(FORGE_ERR_INVALID, "gemm: 1..%d segments", MAX_SEGS);
  for (int i = 0; i < a.n_segs; ++i) {
    const Seg& s = a.segs[i];
    // K-contiguous operands (A ROW, B COL) are fetched in 8-element chunks
    // along K; transposed operands check every k row individually.
    const bool kchunks = (al == ROW) || (bl == COL);
    if (s.k < 0 || (kchunks && s.k % 8 != 0))
      return forge_set_error(FORGE_ERR_INVALID, "gemm: segment %d K=%lld must be a multiple of 8", i,
                             (long long)s.k);
    if (!aligned16(s.a) || (s.b && !aligned16(s.b)) || (s.b2 && !aligned16(s.b2)))
      return forge_set_error(FORGE_ERR_INVALID, "gemm: segment %d operand not 16-byte aligned", i);
    if (s.lda % 8 != 0 || s.ldb % 8 != 0)
      return forge_set_error(FORGE_ERR_INVALID, "gemm: segment %d leading dims must be multiples of 8", i);
    // A lane's operand offset inside a tile is a 32-bit byte offset from the
    // tile's first row (buffer loads): up to 256 rows of the pitch must stay
    // below 2^31 bytes.
    if (s.lda > kMaxLd || s.ldb > kMaxLd)
      return forge_set_error(FORGE_ERR_INVALID, "gemm: segment %d leading dimension above %lld elements", i,
                             (long long)kMaxLd);
  }
  return FORGE_OK;
}

int run(int64_t width, int al, int bl, int epi, const GemmArgs& args, hipStream_t s) {
  if (int e = check_segs(args, al, bl)) return e;
  // 16-byte vector epilogue when every buffer it touches allows it
  GemmArgs a = args;
  {
    const EpiArgs& ep = a.ep;
    bool ok = aligned16(ep.c) && ep.ldc % 8 == 0;
    if (ep.e || ep.g) ok = ok && aligned16(ep.e) && aligned16(ep.g) && ep.ld_eg % 8 == 0;
    if (ep.cos || ep.sin)
      ok = ok && aligned16(ep.cos) && aligned16(ep.sin) && ep.cs_ld % 8 == 0 && ep.head_dim % 16 == 0;
    a.ep.vec_ok = ok ? 1 : 0;
  }
  // transposed-operand tiles are fetched as 8-row blocks of 16-byte vectors
  if (al == COL && a.M % 8 != 0)
    return forge_set_error(FORGE_ERR_INVALID, "gemm: A^T layout needs M %% 8 == 0 (M=%lld)", (long long)a.M);
  if (bl == ROW && a.N % 8 != 0)
    return forge_set_error(FORGE_ERR_INVALID, "gemm: [K][N] B layout needs N %% 8 == 0 (N=%lld)", (long long)a.N);
  if (a.M == 0 || a.N == 0) return FORGE_OK;
  if (al == ROW && bl == COL && rows_engine(epi, a)) return launch_rows(epi, a, s);
  const int cfg = pick_cfg(width > 0 ? width : a.N, al, bl, epi, a);
  if (a.f16) return launch_f16(epi, cfg, al, bl, a, s);
  switch (epi) {
    case EPI_STORE_BF16: return launch_store_bf16(cfg, al, bl, a, s);
    case EPI_STORE_F32: return launch_store_f32(cfg, al, bl, a, s);
    case EPI_ATOMIC_F32: return launch_atomic_f32(cfg, al, bl, a, s);
    case EPI_ROPE:
      if (al == ROW && bl == COL) return launch_rope(a, s);
      break;
    default:
      if (glu_fwd_epi(epi)) return launch_glu_fwd(epi, al, bl, a, s);
      if (glu_bwd_epi(epi)) return launch_glu_bwd(epi, al, bl, a, s);
  }
  return forge_set_error(FORGE_ERR_UNSUPPORTED, "gemm: epilogue %d with layouts (%d, %d)", epi, al, bl);
}

}  // namespace fgemm

using namespace fgemm;

static int gemm_entry(int dtype, int64_t M, int64_t N, const forge_gemm_segment* segs, int n_segs,
                      int a_layout, int b_layout, void* c, int64_t ldc, int c_dtype,
                      float alpha, float beta, int epilogue, int split_k, void* stream) {
  if (M < 0 || N < 0) return forge_set_error(FORGE_ERR_INVALID, "gemm: negative shape");
  if (n_segs < 1 || n_segs > MAX_SEGS)
    return forge_set_error(FORGE_ERR_INVALID, "gemm: 1..%d segments", MAX_SEGS);
  if (split_k < 1) split_k = 1;
  GemmArgs a = {};
  a.M = M;
  a.N = N;
  a.f16 = dtype == FORGE_DTYPE_F16;
  a.n_segs = n_segs;
  bool ranged = false;
  int64_t width = 0;  // widest column range of a segment
  for (int i = 0; i < n_segs; ++i) {
    a.segs[i].a = (const __bf16*)segs[i].a;
    a.segs[i].lda = segs[i].lda;
    a.segs[i].b = (const __bf16*)segs[i].b;
    a.segs[i].b2 = nullptr;
    a.segs[i].ldb = segs[i].ldb;
    a.segs[i].k = segs[i].k;
    if (segs[i].n_lo == 0 && segs[i].n_hi == 0) {
      a.segs[i].n_lo = 0;
      a.segs[i].n_hi = N;
    } else {
      if (segs[i].n_lo < 0 || segs[i].n_hi <= segs[i].n_lo || segs[i].n_hi > N)
        return forge_set_error(FORGE_ERR_INVALID, "gemm: segment %d columns [%lld, %lld) outside [0, %lld)", i,
                               (long long)segs[i].n_lo, (long long)segs[i].n_hi, (long long)N);
      a.segs[i].n_lo = segs[i].n_lo;
      a.segs[i].n_hi = segs[i].n_hi;
      ranged = true;
    }
    if (a.segs[i].n_hi - a.segs[i].n_lo > width) width = a.segs[i].n_hi - a.segs[i].n_lo;
  }
  a.split_k = split_k;
  a.ep.c = c;
  a.ep.ldc = ldc;
  a.ep.alpha = alpha;
  a.ep.beta = beta;
  int epi;
  if (epilogue == FORGE_EPI_ATOMIC_F32) {
    if (c_dtype != FORGE_DTYPE_F32)
      return forge_set_error(FORGE_ERR_INVALID, "gemm: atomic epilogue needs an fp32 C");
    epi = EPI_ATOMIC_F32;
  } else if (epilogue == FORGE_EPI_STORE || epilogue == FORGE_EPI_SILU || epilogue == FORGE_EPI_RELU ||
             epilogue == FORGE_EPI_GELU) {
    a.ep.act = epilogue == FORGE_EPI_SILU ? ACT_SILU
             : epilogue == FORGE_EPI_RELU ? ACT_RELU
             : epilogue == FORGE_EPI_GELU ? ACT_GELU : ACT_NONE;
    if (a.ep.act != ACT_NONE && split_k != 1)
      return forge_set_error(FORGE_ERR_INVALID, "gemm: an activation epilogue needs split_k == 1");
    if (c_dtype == dtype) {
      if (split_k != 1)
        return forge_set_error(FORGE_ERR_INVALID, "gemm: split_k needs an fp32 C (partials) or the atomic epilogue");
      epi = EPI_STORE_BF16;
    } else if (c_dtype == FORGE_DTYPE_F32) {
      epi = EPI_STORE_F32;
      if (split_k > 1) {  // partial sums: split z owns C[z] = c + z * M * ldc
        if (beta != 0.f) return forge_set_error(FORGE_ERR_INVALID, "gemm: split-K partials need beta == 0");
        a.ep.split_stride = M * ldc;
      }
    } else {
      return forge_set_error(FORGE_ERR_UNSUPPORTED, "gemm: C dtype %d", c_dtype);
    }
  } else {
    return forge_set_error(FORGE_ERR_INVALID, "gemm: epilogue %d", epilogue);
  }
  // column-ranged segments: tiles sized for the widest range, so that
  // independent products side by side get tiles of their own
  return run(ranged ? width : 0, a_layout, b_layout, epi, a, (hipStream_t)stream);
}

extern "C" int forge_gemm(int64_t M, int64_t N, const forge_gemm_segment* segs, int n_segs,
                          int a_layout, int b_layout, void* c, int64_t ldc, int c_dtype,
                          float alpha, float beta, int epilogue, int split_k, void* stream) {
  return gemm_entry(FORGE_DTYPE_BF16, M, N, segs, n_segs, a_layout, b_layout, c, ldc, c_dtype, alpha, beta, epilogue,
                    split_k, stream);
}

extern "C" int forge_gemm_f16(int64_t M, int64_t N, const forge_gemm_segment* segs, int n_segs,
                              int a_layout, int b_layout, void* c, int64_t ldc, int c_dtype,
                              float alpha, float beta, int epilogue, int split_k, void* stream) {
  return gemm_entry(FORGE_DTYPE_F16, M, N, segs, n_segs, a_layout, b_layout, c, ldc, c_dtype, alpha, beta, epilogue,
                    split_k, stream);
}
