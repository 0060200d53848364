"""The streaming cross-entropy engine where it can go wrong: rows that start
and end off a 16-byte boundary, rows shorter than one vector or one pass of
the workgroup, both workgroup sizes, the polynomial soft cap against its
exponential form, argmax ties after saturation, and rows of infinities and
NaN.

Oracle: float64 torch.  Bounds: one rounding of the gradient to the logits'
type (2^-8, 2^-11, 2^-24 of it) and an fp32 exponent error of a few 2^-24 of
|x log2 e| <= 100, so 1e-5 of p."""
import pytest
import torch
import torch.nn.functional as F

from kernels.cross_entropy.experiments.v2 import forge_cross_entropy

U = {torch.bfloat16: 2.0 ** -8, torch.float16: 2.0 ** -11, torch.float32: 2.0 ** -24}


def _rows(n, V, dtype, pitch, offset, std, gen):
    """[n, V] logits in a buffer of the given pitch, `offset` elements in."""
    buf = torch.zeros(n * pitch + offset + 8, dtype=dtype, device="cuda")
    x = buf[offset:offset + n * pitch].view(n, pitch)[:, :V]
    x.copy_((torch.randn(n, V, generator=gen) * std).to(dtype))
    return buf, x


def _reference(x, t, softcap, smoothing, weight):
    z = x.double().requires_grad_(True)
    v = softcap * torch.tanh(z / softcap) if softcap else z
    loss = F.cross_entropy(v, t, ignore_index=-100, label_smoothing=smoothing,
                           weight=weight.double() if weight is not None else None)
    return loss.detach(), torch.autograd.grad(loss, z)[0], v.detach()


@pytest.mark.gpu
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16, torch.float32])
@pytest.mark.parametrize("V,pitch,offset", [(1, 1, 0), (5, 5, 3), (13, 16, 1), (1003, 1003, 0), (4099, 4104, 5),
                                            (8192, 8192, 1), (16391, 16391, 2)])
@pytest.mark.parametrize("softcap,smoothing,weighted", [(None, 0.0, False), (30.0, 0.0, False), (None, 0.1, False),
                                                        (30.0, 0.1, True), (3.0, 0.0, False), (50.0, 0.1, False)])
def test_ragged_rows(dtype, V, pitch, offset, softcap, smoothing, weighted):
    gen = torch.Generator().manual_seed(V + offset)
    n = 7
    buf, x = _rows(n, V, dtype, pitch, offset, 4.0, gen)
    before = buf.clone()
    t = torch.randint(0, V, (n,), generator=gen).cuda()
    t[0], t[1] = 0, V - 1
    t[3] = -100
    w = torch.rand(V, generator=gen).cuda() + 0.5 if weighted else None
    loss, grad, v = _reference(x, t, softcap, smoothing, w)
    leaf = x.detach().requires_grad_(True)
    got = forge_cross_entropy(leaf, t, weight=w, softcap=softcap, label_smoothing=smoothing)
    assert abs(got.double() - loss) <= U[dtype] * abs(loss) + 2e-6 * (1 + v.abs().max())
    p = torch.softmax(v, -1) / 6 * (1.5 if weighted else 1.0)
    tiny = 2.0 ** -24 if dtype == torch.float16 else 1e-9
    # (2^-22 of p - onehot: the cap's slope 1 - tanh^2, with tanh good to 2^-23)
    near = p.scatter(1, t.clamp(min=0)[:, None], 1.5 / 6 if weighted else 1 / 6)
    bound = U[dtype] * grad.abs() * 1.01 + 2e-5 * p + 2.0 ** -22 * near + tiny
    assert ((x.double() - grad).abs() <= bound).all()
    outside = torch.ones_like(buf, dtype=torch.bool)
    outside[offset:offset + n * pitch].view(n, pitch)[:, :V] = False
    assert torch.equal(buf[outside], before[outside])  # neighbours of the rows untouched


@pytest.mark.gpu
@pytest.mark.parametrize("dtype,V", [(torch.bfloat16, 140001), (torch.float32, 70003), (torch.bfloat16, 262144)])
@pytest.mark.parametrize("evaluate", [False, True])
def test_long_rows(dtype, V, evaluate):
    gen = torch.Generator().manual_seed(V)
    _, x = _rows(3, V, dtype, V, 0, 3.0, gen)
    t = torch.randint(0, V, (3,), generator=gen).cuda()
    loss, grad, v = _reference(x, t, None, 0.0, None)
    if evaluate:
        t[1] = v[1].argmax()
        o = forge_cross_entropy(x.clone(), t, return_token_accuracy=True, return_predicted_tokens=True)
        first = (x == x.amax(-1, keepdim=True)).int().argmax(-1)
        assert torch.equal(o.predicted_tokens, first)
        assert abs(o.token_accuracy.item() - (first == t).float().mean().item()) < 1e-6
        return
    got = forge_cross_entropy(x.requires_grad_(True), t)
    assert abs(got.double() - loss) <= U[dtype] * abs(loss) + 1e-5
    x = x.detach()
    assert ((x.double() - grad).abs() <= U[dtype] * grad.abs() * 1.01 + 2e-5 * torch.softmax(v, -1) / 3 + 1e-12).all()


@pytest.mark.gpu
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16, torch.float32])
@pytest.mark.parametrize("level", [0.5, 3.9, 4.5, 40.0, -40.0])
def test_softcap_argmax(dtype, level):
    """The prediction is the first of the largest capped values in the
    logits' fp32 cap, saturated ones included."""
    gen = torch.Generator().manual_seed(5)
    V, sc = 3001, 30.0
    x = (torch.randn(4, V, generator=gen) + level * sc).to(dtype).cuda()
    x[0, 7] = x[0, 100] = x[0].max()
    t = torch.zeros(4, dtype=torch.int64, device="cuda")
    o = forge_cross_entropy(x, t, softcap=sc, return_predicted_tokens=True)
    capped = sc * torch.tanh(x.float() / sc)
    best = capped.gather(1, o.predicted_tokens[:, None])[:, 0]
    # torch's fp32 tanh may differ from the kernel's by an ulp
    assert (best >= capped.amax(-1) * (1 - 2.0 ** -22 * (1 if level > 0 else -1))).all()
    if abs(level) >= 40:  # every value caps to +-sc: the first column
        assert (o.predicted_tokens == 0).all()


@pytest.mark.gpu
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float32])
@pytest.mark.parametrize("softcap", [None, 30.0])
def test_infinities_and_nan(dtype, softcap):
    V = 2053
    gen = torch.Generator().manual_seed(6)
    x = torch.randn(4, V, generator=gen).to(dtype).cuda()
    x[1, 5:900] = -float("inf")  # masked columns
    x[2, 11] = float("nan")
    if softcap:
        x[3, 17] = float("inf")  # caps to softcap
    t = torch.tensor([1, 2, 3, 17], device="cuda")
    ref = x.double()
    v = softcap * torch.tanh(ref / softcap) if softcap else ref
    logp = torch.log_softmax(v, -1)
    o = forge_cross_entropy(x.clone().requires_grad_(True), t, softcap=softcap, reduction="none")
    want = -logp.gather(1, t[:, None])[:, 0]
    assert torch.isnan(o[2]) and torch.isnan(want[2])
    keep = torch.tensor([0, 1, 3], device="cuda")
    assert ((o[keep].double() - want[keep]).abs() <= U[dtype] * want[keep].abs() + 1e-5).all()


@pytest.mark.gpu
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16, torch.float32])
@pytest.mark.parametrize("softcap", [3.0, 40.0, 100.0, 1000.0])
def test_negative_softcap(dtype, softcap):
    """softcap * tanh(x / softcap) is even in softcap: the functional entry
    takes a negative value for its magnitude, argmax included."""
    gen = torch.Generator().manual_seed(8)
    x = (torch.randn(3, 4099, generator=gen) * 30).to(dtype).cuda()
    t = torch.tensor([1, 4098, 2000], device="cuda")
    out = []
    for sc in (softcap, -softcap):
        leaf = x.clone().requires_grad_(True)
        o = forge_cross_entropy(leaf, t, softcap=sc, return_predicted_tokens=True)
        o.loss.backward()
        assert torch.isfinite(o.loss)
        out.append((o.loss.detach(), leaf.grad, o.predicted_tokens))
    for a, b in zip(*out):
        assert torch.equal(a, b)


@pytest.mark.gpu
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("softcap", [3.0, 30.0, 50.0])
def test_softcap_slope(dtype, softcap):
    """Gradients of logits of up to 8 times the cap, where its slope 1 - tanh^2
    falls to 5e-7: relative to the slope itself (2e-6 from its own evaluation
    and 1e-5 of p), not to 1."""
    V = 2048
    level = torch.linspace(0.0, 8.0, V)
    x = torch.stack([level, -level, level.flip(0)]).mul(softcap).to(dtype).cuda()
    t = torch.tensor([V - 1, V - 1, 700], device="cuda")  # 8 sc, -8 sc and 5.3 sc
    z = x.double().requires_grad_(True)
    v = softcap * torch.tanh(z / softcap)
    F.cross_entropy(v, t, reduction="sum").backward()
    leaf = x.clone().requires_grad_(True)
    forge_cross_entropy(leaf, t, softcap=softcap, reduction="sum").backward()
    p = torch.softmax(v.detach(), -1)
    slope = 1.0 / torch.cosh(x.double() / softcap) ** 2
    # (exponent errors of 2^-22 of |v| log2 e <= 72 in p and its normalisation)
    error = slope * (4e-5 * p + 4e-6 * F.one_hot(t, V))
    tiny = 2.0 ** -24 if dtype == torch.float16 else 1e-30
    assert ((leaf.grad.double() - z.grad).abs() <= U[dtype] * z.grad.abs() * 1.01 + error + tiny).all()


@pytest.mark.gpu
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("softcap", [30.0, 3e4])
def test_softcap_of_mixed_sizes(dtype, softcap):
    """Small logits beside saturated ones: each gradient is as accurate as in a
    row of small logits alone (a cap with an absolute error of 2^-23 of the
    softcap moves p by 3.6e-3 at 3e4)."""
    gen = torch.Generator().manual_seed(9)
    V = 512
    x = torch.randn(3, V, generator=gen)
    x[:, 3::64] = -0.9 * min(2 * softcap, 6e4)  # saturated, and of no weight in the softmax
    x = x.to(dtype).cuda()
    t = torch.tensor([0, 5, 511], device="cuda")
    z = x.double().requires_grad_(True)
    v = softcap * torch.tanh(z / softcap)
    F.cross_entropy(v, t, reduction="sum").backward()
    leaf = x.clone().requires_grad_(True)
    forge_cross_entropy(leaf, t, softcap=softcap, reduction="sum").backward()
    p = torch.softmax(v.detach(), -1)
    error = 1e-5 * p + 4e-6 * F.one_hot(t, V) + (2.0 ** -24 if dtype == torch.float16 else 1e-30)
    assert ((leaf.grad.double() - z.grad).abs() <= U[dtype] * z.grad.abs() * 1.01 + error).all()


@pytest.mark.gpu
@pytest.mark.parametrize("softcap,smoothing", [(None, 0.0), (None, 0.1), (30.0, 0.0)])
def test_fp32_mean_is_the_sum_divided(softcap, smoothing):
    """fp32 gradients of the mean are those of the sum divided by the token
    count with one rounding, the target's too, where p - 1 cancels."""
    gen = torch.Generator().manual_seed(10)
    n, V = 7, 4099
    x = (torch.randn(n, V, generator=gen) * 2).cuda()
    t = torch.randint(0, V, (n,), generator=gen).cuda()
    x[torch.arange(4), t[:4]] += 20.0  # confident rows: p within 1e-5 of 1
    grads = []
    for reduction in ("mean", "sum"):
        leaf = x.clone().requires_grad_(True)
        forge_cross_entropy(leaf, t, softcap=softcap, label_smoothing=smoothing, reduction=reduction).backward()
        grads.append(leaf.grad.cpu())
    want = grads[1] / torch.full_like(grads[1], n)  # (a scalar divisor may become a product with its reciprocal)
    if softcap is None:
        assert torch.equal(grads[0], want)
    else:  # the cap's slope comes after the division in one and before it in the other: four roundings of 2^-24
        assert ((grads[0] - want).abs() <= 2.0 ** -22 * want.abs() + 1e-44).all()


@pytest.mark.gpu
@pytest.mark.parametrize("dtype,V,n", [(torch.bfloat16, 16384, 3), (torch.bfloat16, 16385, 3), (torch.float32, 8192, 3),
                                       (torch.float32, 8193, 3), (torch.bfloat16, 17, 3001), (torch.float32, 2, 600)])
@pytest.mark.parametrize("softcap", [None, 30.0])
def test_workgroup_sizes(dtype, V, n, softcap):
    """Either side of the row size that changes the workgroup, and more rows
    than threads for the workgroup that sums the losses."""
    gen = torch.Generator().manual_seed(V)
    x = (torch.randn(n, V, generator=gen) * 3).to(dtype).cuda()
    t = torch.randint(0, V, (n,), generator=gen).cuda()
    loss, grad, v = _reference(x, t, softcap, 0.0, None)
    leaf = x.clone().requires_grad_(True)
    o = forge_cross_entropy(leaf, t, softcap=softcap, return_predicted_tokens=True, return_token_accuracy=True)
    o.loss.backward()
    assert abs(o.loss.double() - loss) <= U[dtype] * abs(loss) + 1e-5
    error = 2e-5 * torch.softmax(v, -1) / n + 2.0 ** -22 * F.one_hot(t, V) / n
    assert ((leaf.grad.double() - grad).abs() <= U[dtype] * grad.abs() * 1.01 + error + 1e-12).all()
    first = (x == x.amax(-1, keepdim=True)).int().argmax(-1)
    assert torch.equal(o.predicted_tokens, first)
    assert abs(o.token_accuracy.item() - (first == t).float().mean().item()) < 1e-6
