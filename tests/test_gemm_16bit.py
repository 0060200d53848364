"""forge_gemm_generic on fp16 / bf16 operands: the forms the MFMA core takes
(unit stride along one dimension of each operand, extents and pitches that
are multiples of 8, 16-byte aligned) and, beside each, the forms just outside
that rule, which stay on the general kernel.

Oracle: the product in float64.  Bound per element: one rounding to the
storage type (half an ulp, 2^-11 / 2^-8 of the result, plus half the smallest
subnormal) and fp32 accumulation in any order (K 2^-24 sum |a| |b|)."""
import pytest
import torch

from forge_hip import _lib as L

# unit roundoff: 2^-p of a p-bit significand (11 and 8 bits)
ULP = {torch.float16: 2.0 ** -11, torch.bfloat16: 2.0 ** -8}


def _operand(rows, cols, form, dtype, gen):
    """[rows, cols] values in a given storage form."""
    t = torch.randn(rows, cols, generator=gen).to(dtype).cuda()
    if form == "row":
        return t
    if form == "col":  # unit stride along rows
        return t.t().contiguous().t()
    if form == "pitch":  # padded pitch, a multiple of 8
        return torch.nn.functional.pad(t, (0, 16))[:, :cols]
    if form == "pitch_odd":
        return torch.nn.functional.pad(t, (0, 3))[:, :cols]
    if form == "offset":  # base 2 bytes past a 16-byte boundary
        buf = torch.empty(rows * cols + 8, dtype=dtype, device="cuda")[1:1 + rows * cols].view(rows, cols)
        return buf.copy_(t)
    if form == "strided":  # no unit stride
        buf = torch.empty(rows, cols, 2, dtype=dtype, device="cuda")[:, :, 0]
        return buf.copy_(t)
    if form == "expanded":  # every row the same memory
        return t[:1].expand(rows, cols)
    raise AssertionError(form)


def _check(a, b, dtype, alpha=1.0, beta=0.0, act=L.GEMM_ACT_NONE, bias=None, c_dtype=None):
    M, K = a.shape
    N = b.shape[1]
    c_dtype = c_dtype or dtype
    c = torch.randn(M, N, device="cuda").to(c_dtype)
    ad, bd = a.double(), b.double()
    ref = alpha * (ad @ bd) + beta * c.double()
    if bias is not None:
        ref = ref + bias.double()
    if act == L.GEMM_ACT_SILU:
        ref = torch.nn.functional.silu(ref)
    L.check(L.forge_gemm_generic(M, N, K, L.dtype_code(dtype), a.data_ptr(), a.stride(0), a.stride(1), b.data_ptr(),
                                 b.stride(0), b.stride(1), c.data_ptr(), N, L.dtype_code(c_dtype), alpha, beta,
                                 L.ptr(bias), act, L.stream_of(c)), "forge_gemm_generic")
    ulp = ULP.get(c_dtype, 2.0 ** -24)
    # (1.1: the activation's slope; 1e-6: its own fp32 evaluation)
    bound = ulp * ref.abs() * 1.01 + 1.1 * abs(alpha) * K * 2.0 ** -24 * (ad.abs() @ bd.abs()) + 2.0 ** -25 + 1e-6
    assert ((c.double() - ref).abs() <= bound).all(), (M, N, K, ((c.double() - ref).abs() - bound).max().item())


# tile edges of the configurations the shape rule picks (64 x 64 .. 256 x 256,
# 32 x 256, 256 x 32), their remainders, and K from one chunk to many tiles
SHAPES = [(8, 8, 8), (40, 24, 16), (256, 256, 64), (264, 520, 72), (64, 512, 1000), (1000, 16, 2048),
          (16, 1000, 520), (520, 264, 136), (1000, 136, 264), (264, 192, 64)]


@pytest.mark.gpu
@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16])
@pytest.mark.parametrize("shape", SHAPES)
@pytest.mark.parametrize("fa", ["row", "col"])
@pytest.mark.parametrize("fb", ["row", "col"])
def test_layouts(dtype, shape, fa, fb):
    gen = torch.Generator().manual_seed(1)
    M, N, K = shape
    a, b = _operand(M, K, fa, dtype, gen), _operand(K, N, fb, dtype, gen)
    _check(a, b, dtype, alpha=0.5)
    _check(a, b, dtype, alpha=2.0, beta=1.0)
    _check(a, b, dtype, c_dtype=torch.float32, beta=0.5)


@pytest.mark.gpu
@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16])
@pytest.mark.parametrize("fa,fb", [("pitch", "row"), ("pitch_odd", "col"), ("offset", "row"), ("row", "offset"),
                                   ("strided", "col"), ("expanded", "col"), ("row", "pitch"), ("col", "pitch_odd")])
@pytest.mark.parametrize("M,N,K", [(72, 264, 128), (71, 263, 129), (1, 300, 40), (300, 1, 40)])
def test_storage_forms(dtype, fa, fb, M, N, K):
    gen = torch.Generator().manual_seed(2)
    _check(_operand(M, K, fa, dtype, gen), _operand(K, N, fb, dtype, gen), dtype)


@pytest.mark.gpu
@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16])
def test_bias_and_activation(dtype):
    gen = torch.Generator().manual_seed(3)
    a, b = _operand(72, 128, "row", dtype, gen), _operand(128, 264, "col", dtype, gen)
    _check(a, b, dtype, alpha=0.05, act=L.GEMM_ACT_SILU)
    _check(a, b, dtype, bias=torch.randn(264, generator=gen).to(dtype).cuda())


@pytest.mark.gpu
def test_fp16_range():
    """Subnormal operands are not flushed, and a result past the fp16 range
    is infinite, as a rounding of the fp32 sum."""
    a = torch.full((64, 64), 2.0 ** -24, dtype=torch.float16, device="cuda")
    b = torch.full((64, 64), 0.125, dtype=torch.float16, device="cuda")
    c = torch.empty(64, 64, dtype=torch.float16, device="cuda")
    for lhs, rhs, want in ((a, b, 2.0 ** -21), (b * 8 * 2048, b * 8, float("inf"))):
        L.check(L.forge_gemm_generic(64, 64, 64, L.DTYPE_F16, lhs.data_ptr(), 64, 1, rhs.data_ptr(), 64, 1,
                                     c.data_ptr(), 64, L.DTYPE_F16, 1.0, 0.0, None, L.GEMM_ACT_NONE,
                                     L.stream_of(c)), "forge_gemm_generic")
        assert (c.float() == want).all()


@pytest.mark.gpu
@pytest.mark.parametrize("M,N", [(8, 8), (64, 64), (1024, 1024), (1032, 1024), (72, 264), (16, 264), (264, 16), (264, 128)])
@pytest.mark.parametrize("K", [8, 16, 24, 32, 40, 64, 72, 128, 136])
def test_short_reductions(M, N, K):
    """Either side of the lines between the general kernel and the core."""
    gen = torch.Generator().manual_seed(K)
    for fa, fb in (("row", "row"), ("row", "col"), ("col", "col")):
        a, b = _operand(M, K, fa, torch.float16, gen), _operand(K, N, fb, torch.float16, gen)
        _check(a, b, torch.float16, alpha=0.5, beta=1.0)
