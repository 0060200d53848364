// Generic GEMM: C[M, N] = act(alpha * sum_k A(m, k) B(k, n) + beta * C + bias[n]).
//
// Any strides (so every layout: X W^T, dY W, dY^T X), fp32 / fp16 / bf16
// operands, fp32 accumulation with one fmaf per k in increasing k order
// (deterministic, and exact to fp32 rounding).  It is the path for what the
// MFMA core does not take: fp32 models, and 16-bit operands whose extents or
// row pitches are not multiples of 8, and for short ones.  16-bit products that
// the core does take (mfma_segment below) run there: same products, fp32 accumulation, one
// rounding, another summation order.
//
// Why: this kernel does one fmaf per multiply (no matrix instruction) and is
// bound by its LDS reads at 70 TFLOP/s; [2048, 2048] x [2048, 8192] in fp16
// takes 989 us here, 67 us on the MFMA core with W as stored [N][K] and
// 75-90 us with W as stored [K][N] (MI355X).
//
// Tiling: 64 x 64 output tiles, 16-deep K tiles staged in LDS as fp32,
// 256 threads with 4 x 4 outputs each.  Operand loads are coalesced along
// whichever of the two strides is unit (checked once per launch).
#include "common.h"
#include "gelu.h"

namespace {

struct GenArgs {
  int64_t M, N, K;
  const void* a;
  int64_t a_sm, a_sk;
  const void* b;
  int64_t b_sk, b_sn;
  void* c;
  int64_t ldc;
  const void* bias;
  float alpha, beta;
  int act;  // FORGE_GEMM_ACT_*: activation applied to the result
};

__device__ __forceinline__ float gen_act(int act, float v) {
  if (act == FORGE_GEMM_ACT_SILU) return v * __builtin_amdgcn_rcpf(1.0f + __expf(-v));
  if (act == FORGE_GEMM_ACT_RELU) return v > 0.f ? v : 0.f;
  if (act == FORGE_GEMM_ACT_GELU) {  // tanh form, as the MFMA core's GELU epilogue
    float a, d;
    fgelu::gelu_and_grad<true>(v, a, d);
    return a;
  }
  return v;
}

constexpr int GBM = 64, GBN = 64, GBK = 16;

template <class T, class TC>
__global__ __launch_bounds__(256) void generic_gemm_kernel(GenArgs g, int64_t tiles_n) {
  __shared__ float As[GBK][GBM + 4];
  __shared__ float Bs[GBK][GBN + 4];
  const int64_t tile = blockIdx.x;
  const int64_t m0 = (tile / tiles_n) * GBM, n0 = (tile % tiles_n) * GBN;
  const int tid = threadIdx.x, tx = tid % 16, ty = tid / 16;
  const T* A = static_cast<const T*>(g.a);
  const T* B = static_cast<const T*>(g.b);
  const bool a_kfast = g.a_sk == 1;  // row-major A: neighbouring threads walk k
  const bool b_nfast = g.b_sn == 1;  // row-major B ([K][N]): neighbouring threads walk n
  float acc[4][4];
#pragma unroll
  for (int i = 0; i < 4; ++i)
#pragma unroll
    for (int j = 0; j < 4; ++j) acc[i][j] = 0.f;

  for (int64_t k0 = 0; k0 < g.K; k0 += GBK) {
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      const int e = tid + 256 * i;  // 1024 elements per operand tile
      int r, ka;
      if (a_kfast) { r = e / GBK; ka = e % GBK; } else { ka = e / GBM; r = e % GBM; }
      const int64_t m = m0 + r, k = k0 + ka;
      As[ka][r] = (m < g.M && k < g.K) ? to_f32<T>(A[m * g.a_sm + k * g.a_sk]) : 0.f;
      int cn, kb;
      if (b_nfast) { kb = e / GBN; cn = e % GBN; } else { cn = e / GBK; kb = e % GBK; }
      const int64_t n = n0 + cn, k2 = k0 + kb;
      Bs[kb][cn] = (n < g.N && k2 < g.K) ? to_f32<T>(B[k2 * g.b_sk + n * g.b_sn]) : 0.f;
    }
    __syncthreads();
#pragma unroll
    for (int kk = 0; kk < GBK; ++kk) {
      float av[4], bv[4];
#pragma unroll
      for (int i = 0; i < 4; ++i) av[i] = As[kk][ty * 4 + i];
#pragma unroll
      for (int j = 0; j < 4; ++j) bv[j] = Bs[kk][tx * 4 + j];
#pragma unroll
      for (int i = 0; i < 4; ++i)
#pragma unroll
        for (int j = 0; j < 4; ++j) acc[i][j] = fmaf(av[i], bv[j], acc[i][j]);
    }
    __syncthreads();
  }

  TC* C = static_cast<TC*>(g.c);
  const T* bias = static_cast<const T*>(g.bias);
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    const int64_t m = m0 + ty * 4 + i;
    if (m >= g.M) continue;
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      const int64_t n = n0 + tx * 4 + j;
      if (n >= g.N) continue;
      float v = g.alpha * acc[i][j];
      if (g.beta != 0.f) v += g.beta * to_f32<TC>(C[m * g.ldc + n]);
      if (bias) v += to_f32<T>(bias[n]);
      if (g.act) v = gen_act(g.act, v);
      C[m * g.ldc + n] = from_f32<TC>(v);
    }
  }
}

template <class T>
int launch_generic(const GenArgs& g, int c_dtype, hipStream_t s) {
  const int64_t tm = (g.M + GBM - 1) / GBM, tn = (g.N + GBN - 1) / GBN;
  if (tm * tn > 0x7fffffffLL) return forge_set_error(FORGE_ERR_INVALID, "gemm_generic: too many tiles");
  const dim3 grid((unsigned)(tm * tn));
  if (c_dtype == FORGE_DTYPE_F32)
    generic_gemm_kernel<T, float><<<grid, 256, 0, s>>>(g, tn);
  else
    generic_gemm_kernel<T, T><<<grid, 256, 0, s>>>(g, tn);
  FORGE_CHECK_LAUNCH();
  return FORGE_OK;
}

// Short reductions into outputs that this kernel covers in one round of 64 x 64
// tiles take less here than one of the core's tiles takes to start: measured on
// MI355X, core / here: [8, 8] K = 8 10.3 / 4.5 us, [1024, 1024] K = 32 11.9 /
// 7.2, K = 64 11.9 / 10.0, K = 128 14 / 16; A as [K][M] and B as [N][K] (staged
// through registers there) K = 128 23.6 / 16.9; [256, 8] K = 32, A as [K][M]
// 8.9 / 6.5.  The core's narrow tiles and its row engine start sooner: [8, 64]
// K = 16 5.6 / 4.8, K = 32 5.4 / 6.1, [1024, 16] K = 64 6.5 / 9.0, [16, 64] K =
// 8, B as [N][K] 3.8 / 4.7.
bool short_product(const GenArgs& g, int al, int bl) {
  if (((g.M + GBM - 1) / GBM) * ((g.N + GBN - 1) / GBN) > 256) return false;
  if (al == 0 && bl == 1 && g.M <= 32 && g.N > g.M) return false;
  if (g.K <= 16) return true;
  const bool narrow = g.M != g.N && (g.M <= 64 || g.N <= 64 || (al == 0 && g.N <= 128));
  if (narrow) return g.K <= 32 && ((al == 1 && g.M > g.N) || (g.M > 64 && g.N > 64));
  return g.K <= (al == 1 && bl == 1 ? 128 : 64);
}

// The product as one segment of the MFMA core (fp16 or bf16 operands), or
// false.  The core fetches 16-byte chunks along each operand's unit-stride
// dimension, so that dimension's extent and the other's stride must be
// multiples of 8 (and a pitch at most 2^31 / 512 elements, so that a tile's
// byte offsets fit 31 bits); it has no bias.
bool mfma_segment(const GenArgs& g, forge_gemm_segment& seg, int& al, int& bl) {
  if (g.bias || g.K == 0 || !aligned16(g.a) || !aligned16(g.b)) return false;
  constexpr int64_t kMaxPitch = (int64_t(1) << 31) / 512 - 1;
  if (g.a_sk == 1) al = 0, seg.lda = g.a_sm;       // [M][K]
  else if (g.a_sm == 1) al = 1, seg.lda = g.a_sk;  // [K][M]
  else return false;
  if (g.b_sk == 1) bl = 1, seg.ldb = g.b_sn;       // [N][K]
  else if (g.b_sn == 1) bl = 0, seg.ldb = g.b_sk;  // [K][N]
  else return false;
  if (seg.lda % 8 || seg.ldb % 8 || seg.lda < 0 || seg.ldb < 0 || seg.lda > kMaxPitch || seg.ldb > kMaxPitch) return false;
  if ((al == 0 || bl == 1) && g.K % 8) return false;
  if ((al == 1 && g.M % 8) || (bl == 0 && g.N % 8)) return false;
  if (short_product(g, al, bl)) return false;
  seg.a = g.a;
  seg.b = g.b;
  seg.k = g.K;
  seg.n_lo = seg.n_hi = 0;
  return true;
}

}  // namespace

extern "C" int forge_gemm_generic(int64_t M, int64_t N, int64_t K, int dtype, const void* a, int64_t a_sm,
                                  int64_t a_sk, const void* b, int64_t b_sk, int64_t b_sn, void* c, int64_t ldc,
                                  int c_dtype, float alpha, float beta, const void* bias, int act,
                                  void* stream) {
  if (M < 0 || N < 0 || K < 0) return forge_set_error(FORGE_ERR_INVALID, "gemm_generic: negative shape");
  if (dtype != FORGE_DTYPE_F32 && dtype != FORGE_DTYPE_F16 && dtype != FORGE_DTYPE_BF16)
    return forge_set_error(FORGE_ERR_UNSUPPORTED, "gemm_generic: dtype %d", dtype);
  if (c_dtype != FORGE_DTYPE_F32 && c_dtype != dtype)
    return forge_set_error(FORGE_ERR_UNSUPPORTED, "gemm_generic: C dtype %d with operands %d", c_dtype, dtype);
  if (act != FORGE_GEMM_ACT_NONE && act != FORGE_GEMM_ACT_SILU && act != FORGE_GEMM_ACT_RELU &&
      act != FORGE_GEMM_ACT_GELU)
    return forge_set_error(FORGE_ERR_UNSUPPORTED, "gemm_generic: activation %d", act);
  if (M == 0 || N == 0) return FORGE_OK;
  if (!c || (K > 0 && (!a || !b))) return forge_set_error(FORGE_ERR_INVALID, "gemm_generic: null operand");
  GenArgs g{M, N, K, a, a_sm, a_sk, b, b_sk, b_sn, c, ldc, bias, alpha, beta, act};
  hipStream_t s = (hipStream_t)stream;
  forge_gemm_segment seg;
  int al, bl;
  if (dtype != FORGE_DTYPE_F32 && mfma_segment(g, seg, al, bl)) {
    const int epi = act == FORGE_GEMM_ACT_SILU ? FORGE_EPI_SILU
                  : act == FORGE_GEMM_ACT_RELU ? FORGE_EPI_RELU
                  : act == FORGE_GEMM_ACT_GELU ? FORGE_EPI_GELU : FORGE_EPI_STORE;
    return (dtype == FORGE_DTYPE_F16 ? forge_gemm_f16 : forge_gemm)(M, N, &seg, 1, al, bl, c, ldc, c_dtype, alpha, beta,
                                                                    epi, 1, stream);
  }
  switch (dtype) {
    case FORGE_DTYPE_F32: return launch_generic<float>(g, c_dtype, s);
    case FORGE_DTYPE_F16: return launch_generic<fp16_t>(g, c_dtype, s);
    default: return launch_generic<bf16_t>(g, c_dtype, s);
  }
}
