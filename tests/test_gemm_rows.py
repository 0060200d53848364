"""The few-rows GEMM engine (csrc/gemm_rows.hip) at its edges: 1 to 64 rows
around each block of 16, columns and K that are not whole tiles, K shorter
than one chunk and long enough that every wave has several, column-ranged
segments, the gate/up product with LoRA segments that share one K range, and
the row counts just past it.

Oracle: the product in float64; bound: one rounding to C's type and fp32
accumulation in any order (K 2^-24 sum |a| |b|); the gated activation carries
the bound of its two factors."""
import pytest
import torch

from forge_hip import _lib as L
from kernels._lora_ops import COL, ROW, gemm

U = {torch.float16: 2.0 ** -11, torch.bfloat16: 2.0 ** -8}


def _mat(rows, cols, gen, dtype=torch.bfloat16, pad=0):
    t = torch.randn(rows, cols + pad, generator=gen).to(dtype).cuda()
    return t[:, :cols]


@pytest.mark.gpu
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("M", [1, 15, 16, 17, 32, 33, 64])
@pytest.mark.parametrize("N,K,pad", [(72, 8, 0), (1000, 264, 8), (1040, 4104, 0), (2056, 72, 16)])
def test_rows(dtype, M, N, K, pad):
    gen = torch.Generator().manual_seed(M * N)
    a, b = _mat(M, K, gen, dtype, pad), _mat(N, K, gen, dtype)
    c = torch.randn(M, N, generator=gen).to(dtype).cuda()
    ref = 0.5 * (a.double() @ b.double().t()) + 2.0 * c.double()
    seg = (L.GemmSegment * 1)(L.GemmSegment(a.data_ptr(), a.stride(0), b.data_ptr(), K, K, 0, 0))
    fn = L.forge_gemm_f16 if dtype == torch.float16 else L.forge_gemm
    L.check(fn(M, N, seg, 1, ROW, COL, c.data_ptr(), N, L.dtype_code(dtype), 0.5, 2.0, L.EPI_STORE, 1,
               L.stream_of(c)), "forge_gemm")
    bound = U[dtype] * ref.abs() * 1.01 + K * 2.0 ** -24 * (a.double().abs() @ b.double().abs().t()) + 1e-6
    assert ((c.double() - ref).abs() <= bound).all()


@pytest.mark.gpu
@pytest.mark.parametrize("M", [3, 20])
def test_column_ranges(M):
    """Segments that cover columns [0, 40), [40, 100) and all of them; ranges
    that start and end inside a block of 16 columns."""
    gen = torch.Generator().manual_seed(M)
    N, K = 100, 320
    a, x, y, z = _mat(M, K, gen), _mat(40, K, gen), _mat(60, K, gen), _mat(N, 16, gen)
    t = _mat(M, 16, gen)
    c = gemm(M, N, [(a, K, x, K, K, 0, 40), (a, K, y, K, K, 40, 100), (t, 16, z, 16, 16)], ROW, COL)
    w = torch.cat([x, y]).double()
    ref = a.double() @ w.t() + t.double() @ z.double().t()
    mag = a.double().abs() @ w.abs().t() + t.double().abs() @ z.double().abs().t()
    assert ((c.double() - ref).abs() <= 2.0 ** -8 * 1.01 * ref.abs() + K * 2.0 ** -24 * mag).all()


@pytest.mark.gpu
@pytest.mark.parametrize("M", [1, 16, 31, 48, 64, 65])
@pytest.mark.parametrize("H,I,r", [(256, 264, 0), (264, 4136, 8), (2048, 4104, 24), (64, 512, 64)])
@pytest.mark.parametrize("act", [L.ACT_SILU, L.ACT_GELU_TANH, L.ACT_GELU_ERF])
def test_gate_up(M, H, I, r, act):
    gen = torch.Generator().manual_seed(M + I)
    x, wg, wu = _mat(M, H, gen), _mat(I, H, gen) * H ** -0.5, _mat(I, H, gen) * H ** -0.5
    xa, bg, bu = _mat(M, 2 * max(r, 8), gen), _mat(I, max(r, 8), gen), _mat(I, max(r, 8), gen)
    e, g, h = (torch.empty(M, I, dtype=torch.bfloat16, device="cuda") for _ in range(3))
    args = (M, H, I, r, x.data_ptr(), H, wg.data_ptr(), wu.data_ptr(), H, xa.data_ptr() if r else None, 2 * r,
            bg.data_ptr() if r else None, bu.data_ptr() if r else None, r)
    L.check(L.forge_lora_mlp_gate_up(*args, e.data_ptr(), g.data_ptr(), h.data_ptr(), I, act, L.stream_of(x)), "gate_up")
    re, rg = x.double() @ wg.double().t(), x.double() @ wu.double().t()
    if r:
        re, rg = re + xa[:, :r].double() @ bg.double().t(), rg + xa[:, r:].double() @ bu.double().t()
    for got, ref in ((e, re), (g, rg)):
        assert ((got.double() - ref).abs() <= 2.0 ** -8 * 1.01 * ref.abs() + 1e-4).all()
    a = {L.ACT_SILU: torch.nn.functional.silu(re), L.ACT_GELU_TANH: torch.nn.functional.gelu(re, approximate="tanh"),
         L.ACT_GELU_ERF: torch.nn.functional.gelu(re)}[act]
    # GELU forms round e, g and the activation first: four roundings of at most 2^-8, slope of the activation <= 1.13
    assert ((h.double() - a * rg).abs() <= 4.6 * 2.0 ** -8 * (a.abs() + re.abs() * 0.3) * rg.abs() + 1e-3).all()
    h2 = torch.empty_like(h)  # inference: h alone
    L.check(L.forge_lora_mlp_gate_up(*args, None, None, h2.data_ptr(), I, act, L.stream_of(x)), "gate_up")
    assert torch.equal(h, h2)


@pytest.mark.gpu
@pytest.mark.parametrize("M", [1, 20, 40, 64, 65])
def test_null_operands_read_as_zeros(M):
    """A missing operand contributes nothing, whatever the row count (the row
    engine up to 64 rows, 256 x 256 tiles past them); K of one partial chunk
    and of several whole ones."""
    gen = torch.Generator().manual_seed(M)
    H, I, r = 2056, 520, 16
    x, wg, wu = _mat(M, H, gen), _mat(I, H, gen) * H ** -0.5, _mat(I, H, gen) * H ** -0.5
    xa, b = _mat(M, 2 * r, gen), _mat(I, r, gen)
    zero = torch.zeros_like(b)

    def gate_up(wgate, wup, bg, bu, rank=r):
        e, g, h = (torch.empty(M, I, dtype=torch.bfloat16, device="cuda") for _ in range(3))
        L.check(L.forge_lora_mlp_gate_up(M, H, I, rank, x.data_ptr(), H, L.ptr(wgate), L.ptr(wup), H,
                                         xa.data_ptr() if rank else None, 2 * r, L.ptr(bg), L.ptr(bu), r, e.data_ptr(),
                                         g.data_ptr(), h.data_ptr(), I, L.ACT_SILU, L.stream_of(x)), "gate_up")
        return e, g, h

    for got, want in ((gate_up(wg, wu, None, b), gate_up(wg, wu, zero, b)),
                      (gate_up(wg, wu, b, None), gate_up(wg, wu, b, zero)),
                      (gate_up(wg, None, None, None, 0), gate_up(wg, torch.zeros_like(wu), None, None, 0))):
        for a, c in zip(got, want):
            assert torch.equal(a, c)
    c = torch.full((M, I), 7.0, dtype=torch.bfloat16, device="cuda")
    for a, w in ((None, wg), (x, None)):
        seg = (L.GemmSegment * 1)(L.GemmSegment(L.ptr(a), H, L.ptr(w), H, H, 0, 0))
        L.check(L.forge_gemm(M, I, seg, 1, ROW, COL, c.data_ptr(), I, L.DTYPE_BF16, 1.0, 0.0, L.EPI_STORE, 1,
                             L.stream_of(c)), "forge_gemm")
        assert not c.any()
        c.fill_(7.0)


@pytest.mark.gpu
@pytest.mark.parametrize("M", [33, 64])
@pytest.mark.parametrize("N,K", [(264, 64), (1000, 512), (32768, 72), (32776, 72)])
@pytest.mark.parametrize("c_dtype,epi", [(torch.bfloat16, L.EPI_STORE), (torch.bfloat16, L.EPI_SILU),
                                         (torch.float32, L.EPI_STORE), (torch.float32, L.EPI_SILU),
                                         (torch.float32, L.EPI_ATOMIC_F32)])
def test_unsplit_33_to_64_rows(M, N, K, c_dtype, epi):
    """Either side of the lines of the rule that picks 32-row or 256-row
    tiles: column counts, K, epilogues, a C that is added to, and a pitch
    that rules out vectors."""
    gen = torch.Generator().manual_seed(N)
    a, b = _mat(M, K, gen), _mat(N, K, gen) * K ** -0.5
    prod, mag = a.double() @ b.double().t(), a.double().abs() @ b.double().abs().t()
    seg = (L.GemmSegment * 1)(L.GemmSegment(a.data_ptr(), K, b.data_ptr(), K, K, 0, 0))
    for beta, pad in ((0.0, 0), (1.0, 0), (0.0, 3)):
        c = torch.randn(M, N + pad, generator=gen).to(c_dtype).cuda()
        c0 = c.double()[:, :N]
        L.check(L.forge_gemm(M, N, seg, 1, ROW, COL, c.data_ptr(), N + pad, L.dtype_code(c_dtype), 1.0, beta, epi, 1,
                             L.stream_of(c)), "forge_gemm")
        ref = prod + (c0 if epi == L.EPI_ATOMIC_F32 else beta * c0)
        if epi == L.EPI_SILU:
            ref = torch.nn.functional.silu(ref)
        ulp = U.get(c_dtype, 2.0 ** -24)
        # (1.1: the activation's slope; 1e-6: its own fp32 evaluation)
        bound = ulp * ref.abs() * 1.01 + 1.1 * (K + 2) * 2.0 ** -24 * (mag + c0.abs()) + 1e-6
        assert ((c.double()[:, :N] - ref).abs() <= bound).all(), (beta, pad)


@pytest.mark.gpu
@pytest.mark.parametrize("M,N,K", [(28, 32768, 72), (29, 32768, 72), (16, 32768, 520), (15, 32776, 2048), (16, 32784, 2048),
                                   (1, 32776, 2040), (1, 32776, 128), (16, 40968, 4096), (16, 40968, 4104), (17, 32776, 520)])
def test_many_columns(M, N, K):
    """Either side of each line of the rule that picks 16 or 64 columns a
    workgroup or 32-row tiles; a second segment, a C that is added to."""
    gen = torch.Generator().manual_seed(K)
    for dtype in (torch.bfloat16, torch.float16):
        a, t = _mat(M, K - 8, gen, dtype), _mat(M, 8, gen, dtype)
        b = (torch.randn(N, K - 8, device="cuda") * K ** -0.5).to(dtype)
        z = torch.randn(N, 8, device="cuda").to(dtype)
        c = torch.randn(M, N, device="cuda").to(dtype)
        ref = a.double() @ b.double().t() + t.double() @ z.double().t() + c.double()
        mag = a.double().abs() @ b.double().abs().t() + t.double().abs() @ z.double().abs().t() + c.double().abs()
        segs = (L.GemmSegment * 2)(L.GemmSegment(a.data_ptr(), K - 8, b.data_ptr(), K - 8, K - 8, 0, 0),
                                   L.GemmSegment(t.data_ptr(), 8, z.data_ptr(), 8, 8, 0, 0))
        fn = L.forge_gemm_f16 if dtype == torch.float16 else L.forge_gemm
        L.check(fn(M, N, segs, 2, ROW, COL, c.data_ptr(), N, L.dtype_code(dtype), 1.0, 1.0, L.EPI_STORE, 1,
                   L.stream_of(c)), "forge_gemm")
        assert ((c.double() - ref).abs() <= U[dtype] * ref.abs() * 1.01 + (K + 2) * 2.0 ** -24 * mag + 1e-6).all()
