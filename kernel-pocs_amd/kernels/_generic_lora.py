"""LoRA-MLP and LoRA-QKV for fp32 / fp16 inputs on the generic GEMM.

The fused paths (kernels/lora_mlp/_impl.py, kernels/lora_qkv/_impl.py) run
on the bf16 MFMA core.  The reference's entry points also take fp32 (and
fp16) tensors - its tests call lora_mlp_v3 / lora_mlp_v6 / lora_qkv_v2_3 in
fp32 (kernels/lora_mlp/tests/test_lora_mlp.py:507-549, :1348-1456;
kernels/lora_qkv/tests/test_v2_2_v2_3_v3.py) - where its big GEMMs are plain
cuBLAS fp32 products.  This module is that path here: every product is
forge_gemm_generic (fp32 accumulation, one rounding to the storage type, any
strides, so transposed operands are read in place).  Aligned fp16 products run
on the MFMA core: those whose tiles leave CUs idle are split over K (`gmm`),
and the LoRA terms of a base product join it as K segments (`gmm_sum`).  The
activation is the SwiGLU / GeGLU kernel and RoPE the RoPE kernel, all in the
input's dtype.
The math is the reference's PyTorch formulation
(kernels/lora_mlp/reference/lora_mlp_pytorch.py:100-225,
kernels/lora_qkv/reference/lora_qkv_pytorch.py:34-214):
  proj(X) = X W^T + s (X A^T) B^T
  MLP backward: DW = dY Wd + s_d (dY B_d) A_d; (dgate, dup) from the
  activation's backward; LoRA gradients s (dZ B)^T X and s dZ^T (X A^T).
"""
from __future__ import annotations

from typing import Optional

import torch

from forge_hip import _lib as L
from kernels._lora_ops import COL, ROW, array_type, skinny_split, split_for, split_k_for, split_product

GENERIC_DTYPES = (torch.float32, torch.float16)


def check_dtypes(what: str, *ts) -> torch.dtype:
    """The one dtype of the given tensors (None entries skipped)."""
    dts = {t.dtype for t in ts if t is not None}
    if len(dts) != 1:
        raise TypeError(f"{what}: tensors must share one dtype, got {sorted(str(d) for d in dts)}")
    return dts.pop()


_MAX_PITCH = (1 << 31) // 512 - 1


def _mfma_layouts(a: torch.Tensor, b: torch.Tensor):
    """(a_layout, b_layout, K segment) of a @ b for the MFMA core, or None:
    fp16 operands that it reads in 16-byte chunks along their unit-stride
    dimension (the rule of forge_gemm_generic, csrc/gemm_generic.hip; its line
    for small products is the library's to draw).  (One query of each
    property: a small layer's step is the host's time, 2 us a look.)"""
    if a.dtype != torch.float16:
        return None
    M, K = a.shape
    N = b.shape[1]
    pa, pb = a.data_ptr(), b.data_ptr()
    if K == 0 or (pa | pb) & 15:
        return None
    (am, ak), (bk, bn) = a.stride(), b.stride()
    if ak == 1:
        al, lda = ROW, am
    elif am == 1:
        al, lda = COL, ak
    else:
        return None
    if bk == 1:
        bl, ldb = COL, bn
    elif bn == 1:
        bl, ldb = ROW, bk
    else:
        return None
    if (lda | ldb) & 7 or lda > _MAX_PITCH or ldb > _MAX_PITCH:
        return None
    if (al == ROW or bl == COL) and K % 8 or al == COL and M % 8 or bl == ROW and N % 8:
        return None
    return al, bl, (pa, lda, pb, ldb, K, 0, 0)


def _split(M: int, N: int, K: int, al: int, bl: int) -> int:
    """Split-K factor of one MFMA product: by the rules of the bf16 paths for
    skinny outputs (rank-r products and gradients) and for big tiles that do
    not fill the chip."""
    if al == COL:  # reduced over tokens: A^T B
        big = M > 64 and N > 64
        tiles = (-(-M // 256) if M > 64 else 1) * (-(-N // 256) if N > 64 else 1)
        return split_k_for(K, tiles, target_wgs=256 if big else 512)
    if N <= 64 and M > N:
        return skinny_split(M, N, K)
    if N > 256 and N % 8 == 0 and (M > 64 or M > 32 and bl == COL):
        return split_for(M, N, -(-K // 64))
    return 1


_MAX_SEGS = 6  # K segments of one product (csrc/gemm_core.h)


def _one_product(terms, out: Optional[torch.Tensor]) -> Optional[torch.Tensor]:
    """sum of a @ b over terms as one fp16 product of as many K segments, or
    None where the MFMA core does not take them all in the same layouts, or an
    `out` that is not fp16 with unit stride along its rows (left to gmm)."""
    if len(terms) > _MAX_SEGS:
        return None
    M, N = terms[0][0].shape[0], terms[0][1].shape[1]
    if out is not None and (out.dtype != torch.float16 or out.stride(1) != 1 and N != 1):
        return None
    segs, first = [], None
    for i, (a, b) in enumerate(terms):
        if i and a is terms[i - 1][0] and b is terms[i - 1][1]:  # the second of a term with scale 2
            segs.append(segs[-1])
            continue
        lay = _mfma_layouts(a, b)
        if lay is None or first is not None and lay[:2] != first:
            return None
        first = lay[:2]
        segs.append(lay[2])
    if M == 0 or N == 0:
        return None
    al, bl = first
    if out is None:
        out = torch.empty(M, N, dtype=torch.float16, device=terms[0][0].device)
    split = _split(M, N, sum(-(-sg[4] // 64) * 64 for sg in segs), al, bl)
    arr = array_type(L.GemmSegment, len(segs))(*segs)
    if split > 1:
        return split_product(M, N, arr, True, al, bl, split, out)
    L.check(L.forge_gemm_f16(M, N, arr, len(segs), al, bl, out.data_ptr(), out.stride(0), L.DTYPE_F16, 1.0, 0.0,
                             L.EPI_STORE, 1, L.stream_of(out)), "forge_gemm_f16")
    return out


def gmm_sum(pairs, lora=(), out: Optional[torch.Tensor] = None) -> torch.Tensor:
    """sum of a @ b over pairs + sum of s * a @ b over lora's (a, b, s): one
    product over all of them (one rounding) where the MFMA core takes them,
    else one product after another, added in the storage type.

    A LoRA term joins with s = 1 as a K segment and with s = 2 as that segment
    twice: the sum is exact in the fp32 accumulators, and no operand is scaled
    in fp16 (where it could overflow or lose bits).  The 64-deep K tile that a
    segment costs is 1 us, the read-modify-write product that it replaces 33 us
    at [2048, 8192] (MI355X).  Other scales keep that product and its alpha, and
    so do terms past six segments (LoRA-QKV's dX, three base products and three
    terms, joins at scale 1 only): a LoRA-MLP step of 2048 tokens, 2048 -> 8192,
    takes 679 us at scale 1, 692 at 2 and 827 at 0.5 or 3."""
    total = None
    if pairs[0][0].dtype == torch.float16:
        terms = list(pairs)
        for a, b, s in lora:
            if s != 1 and s != 2:
                break
            terms += [(a, b)] * int(s)
        else:
            total = _one_product(terms, out)
            if total is not None:
                return total
        if lora:
            total = _one_product(pairs, out)
    if total is None:
        total = out
        for i, (a, b) in enumerate(pairs):
            total = gmm(a, b, out=total, beta=1.0 if i else 0.0)
    for a, b, s in lora:
        gmm(a, b, out=total, alpha=s, beta=1.0)
    return total


def gmm(a: torch.Tensor, b: torch.Tensor, out: Optional[torch.Tensor] = None, alpha: float = 1.0,
        beta: float = 0.0) -> torch.Tensor:
    """alpha * a @ b (+ beta * out): a [M, K], b [K, N] of one dtype with any
    strides (transposed views are read in place), out [M, N] row-major."""
    M, K = a.shape
    N = b.shape[1]
    if out is None:
        out = torch.empty(M, N, dtype=a.dtype, device=a.device)
    if M == 0 or N == 0:
        return out
    if K == 0:
        if beta == 0.0:
            out.zero_()
        else:
            out.mul_(beta)
        return out
    assert out.stride(1) == 1 or N == 1
    # (no product is split into fewer than 4 K tiles a split; the host's time
    # for this look is what a small layer's step takes)
    if K > 7 * 64 and beta == 0.0 and a.dtype == torch.float16 and out.dtype == torch.float16:
        lay = _mfma_layouts(a, b)
        split = _split(M, N, K, lay[0], lay[1]) if lay is not None else 1
        if split > 1:
            return split_product(M, N, array_type(L.GemmSegment, 1)(lay[2]), True, lay[0], lay[1], split, out, alpha)
    L.check(L.forge_gemm_generic(M, N, K, L.dtype_code(a.dtype), a.data_ptr(), a.stride(0), a.stride(1),
                                 b.data_ptr(), b.stride(0), b.stride(1), out.data_ptr(), out.stride(0),
                                 L.dtype_code(out.dtype), float(alpha), float(beta), None, L.GEMM_ACT_NONE,
                                 L.stream_of(out)),
            "forge_gemm_generic")
    return out


def _proj(X, W, A, B, s, out=None):
    """X W^T + s (X A^T) B^T -> (out, xa = X A^T or None)."""
    if A is None or B is None:
        return gmm(X, W.t(), out=out), None
    xa = gmm(X, A.t())
    return gmm_sum([(X, W.t())], [(xa, B.t(), s)], out=out), xa


def _act_fwd(e, g, activation):
    M, n = e.shape
    h = torch.empty_like(e)
    if activation == "silu":
        L.check(L.forge_swiglu_fwd(L.dtype_code(e.dtype), e.data_ptr(), g.data_ptr(), n, h.data_ptr(), n, M, n,
                                   1.0, 1.0, L.stream_of(e)), "forge_swiglu_fwd")
    else:
        L.check(L.forge_geglu_fwd(L.dtype_code(e.dtype), e.data_ptr(), g.data_ptr(), n, h.data_ptr(), n, M, n,
                                  int(activation == "gelu_tanh"), L.stream_of(e)), "forge_geglu_fwd")
    return h


def _act_bwd(DW, e, g, activation):
    """(dup, dgate) of the gated activation at (e, g) for dout = DW."""
    M, n = e.shape
    dgate, dup = torch.empty_like(e), torch.empty_like(e)
    if activation == "silu":
        L.check(L.forge_swiglu_bwd(L.dtype_code(e.dtype), DW.data_ptr(), n, e.data_ptr(), g.data_ptr(), n,
                                   dgate.data_ptr(), dup.data_ptr(), n, M, n, 1.0, 1.0, L.stream_of(e)),
                "forge_swiglu_bwd")
    else:
        L.check(L.forge_geglu_bwd(L.dtype_code(e.dtype), DW.data_ptr(), n, e.data_ptr(), g.data_ptr(), n,
                                  dgate.data_ptr(), dup.data_ptr(), n, M, n, int(activation == "gelu_tanh"),
                                  L.stream_of(e)), "forge_geglu_bwd")
    return dup, dgate


def _c(t):
    return None if t is None else (t if t.stride(-1) == 1 else t.contiguous())


def mlp_forward(X2, W_gate, A_gate, B_gate, s_gate, W_up, A_up, B_up, s_up, W_down, A_down, B_down, s_down,
                save_eg=True, aux=None, activation="silu"):
    """(out [M, H], e, g) as the fused path returns them; aux receives the
    unscaled LoRA-A products (X Ag^T, X Au^T, h Ad^T) for the backward."""
    check_dtypes("LoRA-MLP", X2, W_gate, A_gate, B_gate, W_up, A_up, B_up, W_down, A_down, B_down)
    L.require_gpu(X2, W_gate, W_up, W_down)
    X2 = _c(X2)
    e, xag = _proj(X2, W_gate, A_gate, B_gate, s_gate)
    g, xau = _proj(X2, W_up, A_up, B_up, s_up)
    h = _act_fwd(e, g, activation)
    out, xd = _proj(h, W_down, A_down, B_down, s_down)
    if aux is not None and xag is not None and xd is not None:
        aux.update(generic=True, xag=xag, xau=xau, xd=xd)
    if not save_eg:
        e = g = None
    return out, e, g


def mlp_backward(dY2, X2, e, g, W_gate, A_gate, B_gate, s_gate, W_up, A_up, B_up, s_up, W_down, A_down, B_down,
                 s_down, aux=None, activation="silu"):
    """(dX, dAg, dBg, dAu, dBu, dAd, dBd): lora_mlp_pytorch.py:153-225 with
    the activation's backward from the SwiGLU / GeGLU kernel."""
    dY2, X2, e, g = _c(dY2), _c(X2), _c(e), _c(g)
    td = gmm(dY2, B_down)                                   # dY Bd [M, r]
    DW = gmm_sum([(dY2, W_down)], [(td, A_down, s_down)])   # [M, I]
    h = _act_fwd(e, g, activation)
    df, de = _act_bwd(DW, e, g, activation)                 # d up, d gate
    dAd = gmm(td.t(), h, alpha=s_down)                      # [r, I]
    xd = aux["xd"] if aux and aux.get("generic") else gmm(h, A_down.t())
    dBd = gmm(dY2.t(), xd, alpha=s_down)                    # [H, r]
    vu, vg = gmm(df, B_up), gmm(de, B_gate)                 # [M, r]
    dAu, dAg = gmm(vu.t(), X2, alpha=s_up), gmm(vg.t(), X2, alpha=s_gate)
    if aux and aux.get("generic"):
        xau, xag = aux["xau"], aux["xag"]
    else:
        xau, xag = gmm(X2, A_up.t()), gmm(X2, A_gate.t())
    dBu, dBg = gmm(df.t(), xau, alpha=s_up), gmm(de.t(), xag, alpha=s_gate)
    dX = gmm_sum([(df, W_up), (de, W_gate)], [(vu, A_up, s_up), (vg, A_gate, s_gate)])
    return dX, dAg, dBg, dAu, dBu, dAd, dBd


def qkv_forward(X2, W_q, W_k, W_v, A_q, B_q, s_q, A_k, B_k, s_k, A_v, B_v, s_v, rope=None, aux=None):
    """out [M, Hq + 2 Hkv] (Q | K | V columns) as the fused path returns it;
    rope = {cos, sin, positions, head_dim} (tables in X's dtype) rotates Q and K."""
    check_dtypes("LoRA-QKV", X2, W_q, W_k, W_v, A_q, B_q, A_k, B_k, A_v, B_v)
    L.require_gpu(X2, W_q, W_k, W_v)
    X2 = _c(X2)
    M = X2.shape[0]
    Hq, Hkv = W_q.shape[0], W_k.shape[0]
    out = torch.empty(M, Hq + 2 * Hkv, dtype=X2.dtype, device=X2.device)
    xas = []
    for (W, A, B, s), c0, c1 in zip(((W_q, A_q, B_q, s_q), (W_k, A_k, B_k, s_k), (W_v, A_v, B_v, s_v)),
                                    (0, Hq, Hq + Hkv), (Hq, Hq + Hkv, Hq + 2 * Hkv)):
        xas.append(_proj(X2, W, A, B, s, out=out[:, c0:c1])[1])
    if aux is not None and xas[0] is not None:
        aux.update(generic=True, xa=xas)
    if rope is not None:
        D = rope["head_dim"]
        cos, sin, pos = rope["cos"], rope["sin"], rope.get("positions")
        q, k = out[:, :Hq], out[:, Hq:Hq + Hkv]
        L.check(L.forge_rope(L.dtype_code(out.dtype),
                             q.data_ptr(), 0, D, out.stride(0), k.data_ptr(), 0, D, out.stride(0),
                             q.data_ptr(), 0, D, out.stride(0), k.data_ptr(), 0, D, out.stride(0),
                             cos.data_ptr(), 0, cos.stride(0), sin.data_ptr(), 0, sin.stride(0),
                             L.dtype_code(cos.dtype), cos.shape[0],
                             None if pos is None else pos.data_ptr(), 1, Hq // D, Hkv // D, M, D, 0,
                             L.stream_of(out)), "forge_rope")
    return out


def qkv_backward(dQ, dK, dV, X2, W_q, W_k, W_v, A_q, B_q, s_q, A_k, B_k, s_k, A_v, B_v, s_v, aux=None):
    """(dX, dA_q, dB_q, dA_k, dB_k, dA_v, dB_v): lora_qkv_pytorch.py:170-214."""
    X2 = _c(X2)
    dQ, dK, dV = _c(dQ), _c(dK), _c(dV)
    dYBs = [gmm(dQ, B_q), gmm(dK, B_k), gmm(dV, B_v)]       # [M, r]
    dX = gmm_sum([(dQ, W_q), (dK, W_k), (dV, W_v)],
                 [(dYB, A, s) for dYB, A, s in zip(dYBs, (A_q, A_k, A_v), (s_q, s_k, s_v))])
    grads = []
    xas = aux["xa"] if aux and aux.get("generic") else [None, None, None]
    for dY, dYB, A, s, xa in zip((dQ, dK, dV), dYBs, (A_q, A_k, A_v), (s_q, s_k, s_v), xas):
        xa = xa if xa is not None else gmm(X2, A.t())
        grads += [gmm(dYB.t(), X2, alpha=s), gmm(dY.t(), xa, alpha=s)]
    return (dX, *grads)
