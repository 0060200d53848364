"""Outputs on 256 x 256 tiles that are split over K (kernels/_lora_ops.py
split_for, kernels/_generic_lora.py gmm / gmm_sum) and the fp32 epilogue their
partial slices are stored with.

Oracle: the product in float64; bounds: one rounding to C's type and fp32
accumulation in any order (K 2^-24 sum |a| |b|)."""
import pytest
import torch

from forge_hip import _lib as L
from kernels._generic_lora import gmm, gmm_sum
from kernels._lora_ops import COL, ROW, gemm, split_for

U = {torch.float16: 2.0 ** -11, torch.bfloat16: 2.0 ** -8, torch.float32: 2.0 ** -24}


def _close(c, ref, mag, K):
    bound = U[c.dtype] * ref.abs() * 1.01 + K * 2.0 ** -24 * mag + 1e-7
    assert ((c.double() - ref).abs() <= bound).all(), ((c.double() - ref).abs() - bound).max().item()


def test_split_rule():
    assert split_for(8192, 4096, 224) == 1 and split_for(2048, 8192, 32) == 1  # the chip is full
    assert split_for(1003, 4096, 224) == 4
    for m in (65, 256, 300, 1003, 4096):
        for n in (264, 4096, 128256):
            for kt in (1, 3, 64, 2004):
                s = split_for(m, n, kt)
                tiles = -(-m // 256) * -(-n // 256)
                assert s == 1 or (kt // s >= 4 and tiles * s <= 512)


@pytest.mark.gpu
@pytest.mark.parametrize("M,N,K", [(65, 264, 2048), (256, 512, 1024), (1003, 4096, 4096), (300, 776, 4104)])
def test_split_products(M, N, K):
    g = torch.Generator().manual_seed(0)
    for dtype in (torch.bfloat16, torch.float16):
        a = torch.randn(M, K, generator=g).to(dtype).cuda()
        b = torch.randn(N, K, generator=g).to(dtype).cuda()
        xa = torch.randn(M, 16, generator=g).to(dtype).cuda()
        bb = torch.randn(N, 16, generator=g).to(dtype).cuda()
        if dtype == torch.bfloat16:
            assert split_for(M, N, -(-K // 64) + 1) > 1
            c = gemm(M, N, [(a, K, b, K, K), (xa, 16, bb, 16, 16)], ROW, COL, alpha=0.5)
            _close(c, 0.5 * (a.double() @ b.double().t() + xa.double() @ bb.double().t()),
                   0.5 * (a.double().abs() @ b.double().abs().t() + xa.double().abs() @ bb.double().abs().t()), K + 16)
        else:
            _close(gmm(a, b.t(), alpha=0.5), 0.5 * (a.double() @ b.double().t()),
                   0.5 * (a.double().abs() @ b.double().abs().t()), K)
            _close(gmm_sum([(a, b.t()), (xa, bb.t())]), a.double() @ b.double().t() + xa.double() @ bb.double().t(),
                   a.double().abs() @ b.double().abs().t() + xa.double().abs() @ bb.double().abs().t(), K + 16)
            w, v = b.t().contiguous(), bb.t().contiguous()  # [K, N] as stored
            _close(gmm_sum([(a, w), (xa, v)]), a.double() @ w.double() + xa.double() @ v.double(),
                   a.double().abs() @ w.double().abs() + xa.double().abs() @ v.double().abs(), K + 16)


@pytest.mark.gpu
def test_gmm_sum_of_mixed_layouts_adds_products():
    g = torch.Generator().manual_seed(1)
    a, b = torch.randn(70, 40, generator=g).half().cuda(), torch.randn(40, 264, generator=g).half().cuda()
    x, y = torch.randn(70, 12, generator=g).half().cuda(), torch.randn(12, 264, generator=g).half().cuda()  # K % 8 != 0
    ref = a.double() @ b.double() + x.double() @ y.double()
    # the first product is rounded to fp16 before the second is added
    assert ((gmm_sum([(a, b), (x, y)]).double() - ref).abs()
            <= 2.0 ** -10 * ((a.double() @ b.double()).abs() + ref.abs()) + 1e-4).all()


@pytest.mark.gpu
@pytest.mark.parametrize("M,N,K", [(256, 256, 64), (300, 264, 136), (65, 512, 72), (257, 1000, 64)])
@pytest.mark.parametrize("beta", [0.0, 0.5])
@pytest.mark.parametrize("pitch", [0, 8, 1])
def test_fp32_store(M, N, K, beta, pitch):
    """Whole and ragged tiles, with and without C read, and a pitch that
    rules out 16-byte stores."""
    g = torch.Generator().manual_seed(2)
    a = torch.randn(M, K, generator=g).bfloat16().cuda()
    b = torch.randn(N, K, generator=g).bfloat16().cuda()
    buf = torch.randn(M, N + pitch, generator=g).cuda()
    before = buf.clone()
    seg = (L.GemmSegment * 1)(L.GemmSegment(a.data_ptr(), K, b.data_ptr(), K, K, 0, 0))
    L.check(L.forge_gemm(M, N, seg, 1, ROW, COL, buf.data_ptr(), N + pitch, L.DTYPE_F32, 2.0, beta, L.EPI_STORE, 1,
                         L.stream_of(buf)), "forge_gemm")
    _close(buf[:, :N], 2.0 * (a.double() @ b.double().t()) + beta * before[:, :N].double(),
           2.0 * (a.double().abs() @ b.double().abs().t()) + beta * before[:, :N].double().abs(), K)
    assert torch.equal(buf[:, N:], before[:, N:])


@pytest.mark.gpu
@pytest.mark.parametrize("scales", [(1.0, 2.0), (2.0, 2.0), (0.5, 2.0), (2.0, 3.0), (-1.0, 1.0)])
@pytest.mark.parametrize("M,N,K", [(1, 264, 512), (31, 72, 136), (72, 264, 520), (300, 776, 4104), (264, 8, 64)])
@pytest.mark.parametrize("rank", [8, 64, 72, 12])
def test_lora_terms_of_a_sum(scales, M, N, K, rank):
    """Two base products and two LoRA terms in both weight layouts, into a
    column slice.  Scales of 1 and 2 join the product where the rank lets
    them (one rounding, also where s * B alone would overflow fp16); the
    others are added to the rounded base (two roundings more)."""
    g = torch.Generator().manual_seed(4)
    draw = lambda *shape: torch.randn(*shape, generator=g).half().cuda()
    a, x = draw(M, K), [draw(M, rank) for _ in scales]
    x[1] *= 2.0 ** -10
    for nt in (True, False):
        w = draw(N, K).t() if nt else draw(K, N)
        b = [draw(N, rank).t() if nt else draw(rank, N) for _ in scales]
        b[1] = (b[1] * 4096).clamp(-40000, 40000)
        buf = torch.full((M, N + 16), 7.0, dtype=torch.float16, device="cuda")
        c = gmm_sum([(a, w), (a, w)], [(p, q, s) for p, q, s in zip(x, b, scales)], out=buf[:, 8:8 + N])
        base = 2 * (a.double() @ w.double())
        terms = [s * (p.double() @ q.double()) for p, q, s in zip(x, b, scales)]
        ref = base + sum(terms)
        mag = 2 * (a.double().abs() @ w.double().abs())
        mag += sum(abs(s) * (p.double().abs() @ q.double().abs()) for p, q, s in zip(x, b, scales))
        one = rank % 8 == 0 and all(s in (1.0, 2.0) for s in scales)
        seen = ref.abs() if one else base.abs() + (base + terms[0]).abs() + ref.abs() + base.abs() / 2
        bound = 2.0 ** -11 * 1.02 * seen + (2 * K + 4 * rank) * 2.0 ** -24 * mag + 1e-6
        assert ((c.double() - ref).abs() <= bound).all(), (nt, ((c.double() - ref).abs() - bound).max().item())
        assert (buf[:, :8] == 7).all() and (buf[:, 8 + N:] == 7).all()


@pytest.mark.gpu
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("M,N,K", [(264, 272, 8), (256, 512, 64), (264, 520, 200), (512, 264, 1096), (776, 1000, 328)])
@pytest.mark.parametrize("a_layout", [ROW, COL])
@pytest.mark.parametrize("split", [1, 3])
def test_token_major_big_tiles(dtype, M, N, K, a_layout, split):
    """256 x 256 tiles with B stored [K][N] and A either way: two segments of
    unequal K (with A^T not a multiple of 8), padded pitches and partial tiles."""
    g = torch.Generator().manual_seed(5)
    ks = (K, 72) if a_layout == ROW else (K - 3, 65)
    segs, ref, mag = [], 0, 0
    for k in ks:
        a, b = torch.randn(M, k, generator=g).to(dtype), torch.randn(k, N, generator=g).to(dtype)
        ref, mag = ref + a.double() @ b.double(), mag + a.double().abs() @ b.double().abs()
        b = torch.nn.functional.pad(b, (0, 8)).cuda()
        if a_layout == ROW:
            a, lda = torch.nn.functional.pad(a, (0, -k % 8)).cuda(), k + -k % 8
        else:
            a, lda = torch.nn.functional.pad(a.t(), (0, 16)).cuda(), M + 16
        segs.append((a, lda, b, N + 8, k))
    ref, mag = ref.cuda(), mag.cuda()
    arr = (L.GemmSegment * 2)(*(L.GemmSegment(a.data_ptr(), la, b.data_ptr(), lb, k, 0, 0) for a, la, b, lb, k in segs))
    fn = L.forge_gemm_f16 if dtype == torch.float16 else L.forge_gemm
    for out_dtype in (dtype, torch.float32):
        if out_dtype == dtype and split > 1:
            continue
        c = torch.full((split, M, N), float("nan"), dtype=out_dtype, device="cuda")
        L.check(fn(M, N, arr, 2, a_layout, ROW, c.data_ptr(), N, L.dtype_code(out_dtype), 0.5, 0.0, L.EPI_STORE, split,
                   L.stream_of(c)), "forge_gemm")
        _close(c[0] if split == 1 else c.sum(0), 0.5 * ref, mag, sum(ks))


@pytest.mark.gpu
@pytest.mark.parametrize("al,bl,N", [(ROW, COL, 518), (ROW, COL, 512), (ROW, ROW, 520), (COL, ROW, 520)])
@pytest.mark.parametrize("K", [64, 264, 1032])
def test_fp32_forms(al, bl, N, K):
    """An fp32 C that is added to, activated and both, whole tiles and ragged
    ones (N that is not a multiple of 4 included), short and long reductions."""
    M = 264
    gen = torch.Generator().manual_seed(K)
    a = torch.randn(M, K, generator=gen).to(torch.bfloat16)
    b = (torch.randn(K, N, generator=gen) * K ** -0.5).to(torch.bfloat16)
    prod, mag = a.double() @ b.double(), a.double().abs() @ b.double().abs()
    ad, bd = (a if al == ROW else a.t().contiguous()).cuda(), (b if bl == ROW else b.t().contiguous()).cuda()
    seg = (L.GemmSegment * 1)(L.GemmSegment(ad.data_ptr(), ad.stride(0), bd.data_ptr(), bd.stride(0), K, 0, 0))
    acts = ((L.EPI_STORE, lambda v: v), (L.EPI_SILU, torch.nn.functional.silu), (L.EPI_RELU, torch.relu),
            (L.EPI_GELU, lambda v: torch.nn.functional.gelu(v, approximate="tanh")))
    for epi, act in acts:
        for alpha, beta in ((0.5, 0.0), (1.0, 2.0)):
            c0 = torch.randn(M, 520, generator=gen)
            c = c0.cuda()
            L.check(L.forge_gemm(M, N, seg, 1, al, bl, c.data_ptr(), 520, L.DTYPE_F32, alpha, beta, epi, 1,
                                 L.stream_of(c)), "forge_gemm")
            ref = act(alpha * prod + beta * c0.double()[:, :N])
            # (1.13: the activations' largest slope; 2e-6: their own fp32 evaluation)
            bound = 1.13 * ((K + 2) * 2.0 ** -24 * (abs(alpha) * mag + abs(beta) * c0.abs()[:, :N])) + 2e-6 + \
                2.0 ** -22 * ref.abs()
            got = c.cpu()
            assert ((got.double()[:, :N] - ref).abs() <= bound).all(), (epi, beta)
            assert torch.equal(got[:, N:], c0[:, N:])  # past the last column


@pytest.mark.gpu
def test_fp32_partials_with_column_alphas():
    """Stacked LoRA-A products wider than the narrow tiles, split over K: each
    projection's scale is applied to its own columns."""
    M, K, r, n = 300, 1024, 96, 4
    gen = torch.Generator().manual_seed(3)
    x = torch.randn(M, K, generator=gen).to(torch.bfloat16).cuda()
    stack = torch.randn(n * r, K, generator=gen).to(torch.bfloat16).cuda()
    scales = [0.5, 1.0, 2.0, -3.0]
    out = torch.empty(M, n * r, dtype=torch.bfloat16, device="cuda")
    work = torch.empty(4, M, n * r, device="cuda")
    import ctypes
    ptrs = (ctypes.c_void_p * n)(*[stack[p * r:].data_ptr() for p in range(n)])
    L.check(L.forge_lora_a(M, K, r, n, x.data_ptr(), K, ptrs, K, (ctypes.c_float * n)(*scales), out.data_ptr(), n * r,
                           work.data_ptr(), 4, L.stream_of(x)), "forge_lora_a")
    s = torch.tensor(scales, device="cuda", dtype=torch.float64).repeat_interleave(r)
    _close(out, x.double() @ stack.double().t() * s, x.double().abs() @ stack.double().abs().t() * s.abs(), K)


@pytest.mark.gpu
@pytest.mark.parametrize("K", [256, 264])
def test_token_major_to_16_bits(K):
    """Either side of the reduction length that changes the engine of A^T B
    (289 tiles)."""
    M, N = 4104, 4112
    g = torch.Generator().manual_seed(K)
    for dtype in (torch.bfloat16, torch.float16):
        a, b = torch.randn(K, M, generator=g).to(dtype).cuda(), torch.randn(K, N, generator=g).to(dtype).cuda()
        c = torch.empty(M, N, dtype=dtype, device="cuda")
        seg = (L.GemmSegment * 1)(L.GemmSegment(a.data_ptr(), M, b.data_ptr(), N, K, 0, 0))
        fn = L.forge_gemm if dtype == torch.bfloat16 else L.forge_gemm_f16
        L.check(fn(M, N, seg, 1, COL, ROW, c.data_ptr(), N, L.dtype_code(dtype), 0.5, 0.0, L.EPI_STORE, 1,
                   L.stream_of(c)), "forge_gemm")
        _close(c, 0.5 * (a.double().t() @ b.double()), 0.5 * (a.double().abs().t() @ b.double().abs()), K)
