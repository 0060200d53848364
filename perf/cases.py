"""The work that the framework's speed is measured on.

Each case is one call that a fine-tuning or serving program makes, with the sizes it meets: the
gated activations, RoPE, RMSNorm, cross-entropy, the fused linear + cross-entropy head, the fused
LoRA-MLP and LoRA-QKV layers, and the merged-weight MLP of a serving program. A training case is
forward and backward through the public autograd entry points.
"""
import math
import sys
from pathlib import Path

import torch
import torch.nn.functional as F

sys.path.insert(0, str(Path(__file__).resolve().parents[1] / "kernel-pocs_amd"))

from kernels.cross_entropy.experiments.v2 import (  # noqa: E402
    forge_cross_entropy,
    forge_fused_linear_cross_entropy,
)
from kernels.geglu import geglu  # noqa: E402
from kernels.lora_mlp.experiments.v5.lora_mlp_kernel_v5 import (  # noqa: E402
    lora_mlp_v5_inference,
    prepare_inference_weights,
)
from kernels.lora_mlp.experiments.v6.lora_mlp_kernel_v6 import LoRAMLPv6  # noqa: E402
from kernels.lora_mlp.geglu_mlp import LoRAMLPGeGLU  # noqa: E402
from kernels.lora_qkv.experiments.v4.lora_qkv_kernel_v4 import lora_qkv_rope  # noqa: E402
from kernels.rmsnorm.forge_rmsnorm_v4 import apply_rmsnorm_v4  # noqa: E402
from kernels.rope import apply_rope  # noqa: E402
from kernels.swiglu import swiglu  # noqa: E402

DTYPES = {"fp32": torch.float32, "bf16": torch.bfloat16, "fp16": torch.float16}
BYTES = {"fp32": 4, "bf16": 2, "fp16": 2}
IGNORE = -100


def listed():
    return [
        # the smallest call of a training step: RoPE on a short bf16 batch, where launches and host time count
        {"name": "rope_short", "op": "rope", "batch": 1, "seq": 128, "heads": 32, "kv_heads": 8, "head_dim": 128,
         "base": 500000.0, "dtype": "bf16"},
        # SwiGLU of a 7B-class MLP in fp32
        {"name": "swiglu_fp32", "op": "glu", "act": "silu", "rows": 2048, "cols": 11008, "dtype": "fp32"},
        # RoPE of a long GQA batch
        {"name": "rope_gqa", "op": "rope", "batch": 4, "seq": 4096, "heads": 32, "kv_heads": 8, "head_dim": 128,
         "base": 500000.0, "dtype": "bf16"},
        # a decoder layer's norm over a long batch, weight gradient included
        {"name": "rmsnorm", "op": "rmsnorm", "rows": 8192, "cols": 4096, "dtype": "bf16"},
        # the loss of a training step over a 128k vocabulary
        {"name": "ce_128k", "op": "ce", "rows": 8192, "vocab": 128256, "softcap": 0.0, "smoothing": 0.0,
         "evaluate": False, "dtype": "bf16"},
        # the same with capped logits over a 256k vocabulary (Gemma-2's head)
        {"name": "ce_softcap_256k", "op": "ce", "rows": 2048, "vocab": 256000, "softcap": 30.0, "smoothing": 0.0,
         "evaluate": False, "dtype": "bf16"},
        # head and loss in one call, lm_head frozen as in LoRA fine-tuning
        {"name": "linear_ce", "op": "flce", "rows": 4096, "hidden": 4096, "vocab": 128256, "train_head": False,
         "dtype": "bf16"},
        # the LoRA-MLP training step at the full batch
        {"name": "lora_mlp", "op": "mlp", "act": "silu", "rows": 8192, "hidden": 4096, "inter": 14336, "rank": 16,
         "dtype": "bf16"},
        # the same layer on one short, ragged batch
        {"name": "lora_mlp_short", "op": "mlp", "act": "silu", "rows": 1003, "hidden": 4096, "inter": 14336,
         "rank": 16, "dtype": "bf16"},
        # an fp16 model's LoRA-MLP
        {"name": "lora_mlp_fp16", "op": "mlp", "act": "silu", "rows": 2048, "hidden": 2048, "inter": 8192,
         "rank": 16, "dtype": "fp16"},
        # LoRA-QKV with RoPE on packed sequences of different lengths
        {"name": "lora_qkv_varlen", "op": "qkv", "rows": 16384, "seqs": 8, "hidden": 4096, "heads": 32,
         "kv_heads": 8, "head_dim": 128, "rank": 64, "dtype": "bf16"},
        # a serving program's MLP on merged weights: one decode step of a small batch
        {"name": "mlp_decode", "op": "infer", "rows": 16, "hidden": 4096, "inter": 14336, "dtype": "bf16"},
    ]


def _log(rng, lo, hi):
    """A whole number from lo to hi, spread over its logarithm: as often odd as it comes."""
    return min(hi, max(lo, round(math.exp(rng.uniform(math.log(lo), math.log(hi))))))


# (hidden, intermediate), (hidden, heads, kv heads, head_dim)
MLPS = [(2048, 8192), (3584, 14336), (4096, 11008), (4096, 14336)]
HEADS = [(2048, 32, 8, 64), (2048, 16, 8, 128), (4096, 32, 8, 128), (4096, 32, 32, 128)]
VOCABS = [32000, 50257, 128256, 151936, 256000]


def draw(rng):
    op = rng.choice(["glu", "rope", "rmsnorm", "ce", "flce", "mlp", "mlp", "qkv", "infer"])
    if op == "glu":
        dtype = rng.choice(["fp32", "bf16", "bf16", "fp16"])
        cols = rng.choice([5632, 9216, 11008, 14336, 24576, _log(rng, 1000, 16000)])
        return {"op": op, "act": rng.choice(["silu", "silu", "gelu_tanh", "gelu_exact"]),
                "rows": _log(rng, 32, 8192), "cols": cols, "dtype": dtype}
    if op == "rope":
        h, kv, d = rng.choice([(32, 8, 128), (32, 32, 128), (16, 8, 128), (32, 8, 64)])
        return {"op": op, "batch": rng.choice([1, 2, 4]), "seq": _log(rng, 32, 4096), "heads": h, "kv_heads": kv,
                "head_dim": d, "base": rng.choice([10000.0, 500000.0]), "dtype": rng.choice(["bf16", "bf16", "fp16", "fp32"])}
    if op == "rmsnorm":
        return {"op": op, "rows": _log(rng, 32, 16384), "cols": rng.choice([896, 2048, 2304, 3584, 4096, 4097, 8192]),
                "dtype": rng.choice(["bf16", "bf16", "fp16", "fp32"])}
    if op == "ce":
        vocab = rng.choice(VOCABS)
        dtype = rng.choice(["bf16", "bf16", "fp32", "fp16"])
        most = int(8192 * 128256 * 2 / (vocab * BYTES[dtype]))
        return {"op": op, "rows": _log(rng, 128, min(16384, most)), "vocab": vocab,
                "softcap": rng.choice([0.0, 0.0, 30.0]), "smoothing": rng.choice([0.0, 0.0, 0.1]),
                "evaluate": rng.random() < 0.25, "dtype": dtype}
    if op == "flce":
        hidden, vocab = rng.choice([(2048, 32000), (2048, 128256), (4096, 32000), (4096, 128256)])
        train = rng.random() < 0.5
        return {"op": op, "rows": _log(rng, 128, 2730 if train else 4096), "hidden": hidden, "vocab": vocab,
                "train_head": train, "dtype": "bf16"}
    if op == "mlp":
        h, i = rng.choice(MLPS)
        dtype = rng.choice(["bf16", "bf16", "bf16", "fp16"])
        return {"op": op, "act": rng.choice(["silu", "silu", "gelu_tanh"]),
                "rows": _log(rng, 128, 8192 if dtype == "bf16" else 2048), "hidden": h, "inter": i,
                "rank": rng.choice([8, 16, 32, 64]), "dtype": dtype}
    if op == "qkv":
        k, h, kv, d = rng.choice(HEADS)
        return {"op": op, "rows": _log(rng, 256, 16384), "seqs": rng.choice([1, 3, 8]), "hidden": k, "heads": h,
                "kv_heads": kv, "head_dim": d, "rank": rng.choice([16, 32, 64]), "dtype": "bf16"}
    h, i = rng.choice(MLPS)
    return {"op": op, "rows": _log(rng, 1, 512), "hidden": h, "inter": i, "dtype": "bf16"}


class _Draws:
    """Seeded tensors on the GPU (the exact values of `exact` come from the same ones)."""

    def __init__(self, case, seed):
        self.g = torch.Generator(device="cuda").manual_seed(seed)
        self.dtype = DTYPES[case["dtype"]]

    def normal(self, *shape, std=1.0):
        t = torch.empty(shape, dtype=self.dtype, device="cuda")
        return t.normal_(0.0, std, generator=self.g)

    def uniform(self, *shape, bound):
        t = torch.empty(shape, dtype=self.dtype, device="cuda")
        return t.uniform_(-bound, bound, generator=self.g)

    def targets(self, n, vocab):
        """Labels with one in twenty ignored, the first and the last kept."""
        t = torch.randint(0, vocab, (n,), device="cuda", generator=self.g)
        drop = torch.rand(n, device="cuda", generator=self.g) < 0.05
        drop[0] = drop[-1] = False
        return t.masked_fill_(drop, IGNORE)


def _cos_sin(n, head_dim, base, dtype):
    inv = 1.0 / base ** (torch.arange(0, head_dim, 2, device="cuda", dtype=torch.float32) / head_dim)
    ang = torch.arange(n, device="cuda", dtype=torch.float32).unsqueeze(1) * inv
    ang = torch.cat([ang, ang], 1)
    return ang.cos().to(dtype), ang.sin().to(dtype)


def _lengths(rows, seqs):
    """Lengths of packed sequences, from about half to one and a half of the mean."""
    cuts = [0] + [min(rows, max(1, round(rows * (i + 0.5 * math.sin(2.0 * i)) / seqs))) for i in range(1, seqs)] + [rows]
    cuts.sort()
    return [b - a for a, b in zip(cuts, cuts[1:]) if b > a]


def _inputs(case, seed):
    """Every tensor of the case, without gradients."""
    d = _Draws(case, seed)
    op = case["op"]
    if op == "glu":
        return {n: d.normal(case["rows"], case["cols"]) for n in ("gate", "up", "dout")}
    if op == "rope":
        b, s, h, kv, hd = (case[k] for k in ("batch", "seq", "heads", "kv_heads", "head_dim"))
        t = {n: d.normal(b, s, m, hd) for n, m in (("q", h), ("k", kv), ("dq", h), ("dk", kv))}
        cos, sin = _cos_sin(s, hd, case["base"], d.dtype)
        t["cos"], t["sin"] = cos.unsqueeze(0), sin.unsqueeze(0)
        return t
    if op == "rmsnorm":
        t = {n: d.normal(case["rows"], case["cols"]) for n in ("x", "dy")}
        t["weight"] = d.normal(case["cols"], std=0.1).add_(1.0)
        return t
    if op == "ce":
        return {"logits": d.normal(case["rows"], case["vocab"], std=2.0), "target": d.targets(case["rows"], case["vocab"])}
    if op == "flce":
        return {"x": d.normal(case["rows"], case["hidden"]), "weight": d.normal(case["vocab"], case["hidden"], std=0.02),
                "target": d.targets(case["rows"], case["vocab"])}
    if op in ("mlp", "infer"):
        m, h, i, r = case["rows"], case["hidden"], case["inter"], case.get("rank", 16)
        t = {"x": d.normal(1, m, h)}
        for n, out, inp in (("gate", i, h), ("up", i, h), ("down", h, i)):
            t["w_" + n] = d.normal(out, inp, std=0.02)
            t["a_" + n] = d.uniform(r, inp, bound=math.sqrt(3.0 / inp))
            t["b_" + n] = d.normal(out, r, std=0.01)
        if op == "mlp":
            t["dy"] = d.normal(1, m, h)
        return t
    m, k, r, hd = case["rows"], case["hidden"], case["rank"], case["head_dim"]
    t = {"x": d.normal(m, k)}
    for n, heads in (("q", case["heads"]), ("k", case["kv_heads"]), ("v", case["kv_heads"])):
        t["w_" + n] = d.normal(heads * hd, k, std=0.02)
        t["a_" + n] = d.uniform(r, k, bound=math.sqrt(3.0 / k))
        t["b_" + n] = d.normal(heads * hd, r, std=0.01)
        t["d" + n] = d.normal(m, heads * hd)
    lengths = _lengths(m, case["seqs"])
    t["positions"] = torch.cat([torch.arange(n, device="cuda") for n in lengths])
    t["cos"], t["sin"] = _cos_sin(max(lengths), hd, 500000.0, d.dtype)
    return t


def _trained(case):
    """The names of the inputs whose gradients the pass returns."""
    if case["op"] == "glu":
        return ["gate", "up"]
    if case["op"] == "rope":
        return ["q", "k"]
    if case["op"] == "rmsnorm":
        return ["x", "weight"]
    if case["op"] == "ce":
        return [] if case["evaluate"] else ["logits"]
    if case["op"] == "flce":
        return ["x", "weight"] if case["train_head"] else ["x"]
    if case["op"] == "mlp":
        return ["x"] + [p + n for n in ("gate", "up", "down") for p in ("a_", "b_")]
    if case["op"] == "qkv":
        return ["x"] + [p + n for n in ("q", "k", "v") for p in ("a_", "b_")]
    return []


def prepare(case, seed):
    t = _inputs(case, seed)
    if case["op"] == "infer":  # a serving program merges the adapters once and keeps the merged weights
        merged = prepare_inference_weights(*(v for n in ("gate", "up", "down")
                                             for v in (t["w_" + n], t["a_" + n], t["b_" + n], 2.0)))
        t = {"x": t["x"], "merged": merged}
    for n in _trained(case):
        t[n].requires_grad_(True)
    return case, t


def _scale(case):
    """alpha / rank with the common alpha = 2 rank."""
    return 2.0


def run(state):
    case, t = state
    op = case["op"]
    leaves = [t[n] for n in _trained(case)]
    if op == "glu":  # the program still needs gate and up (preserve_inputs)
        if case["act"] == "silu":
            out = swiglu(t["gate"], t["up"], preserve_inputs=True)
        else:
            out = geglu(t["gate"], t["up"], "tanh" if case["act"] == "gelu_tanh" else "none", preserve_inputs=True)
        return (out, *torch.autograd.grad(out, leaves, t["dout"]))
    if op == "rope":  # the projections' [B, S, H, D] memory, passed as models pass it
        q, k = t["q"].transpose(1, 2), t["k"].transpose(1, 2)
        oq, ok = apply_rope(q, k, t["cos"], t["sin"])
        return (oq, ok, *torch.autograd.grad((oq, ok), leaves, (t["dq"].transpose(1, 2), t["dk"].transpose(1, 2))))
    if op == "rmsnorm":  # dy also feeds the residual branch: not in place
        y = apply_rmsnorm_v4(t["x"], t["weight"], in_place=False)
        return (y, *torch.autograd.grad(y, leaves, t["dy"]))
    if op == "ce":
        softcap = case["softcap"] or None
        if case["evaluate"]:
            o = forge_cross_entropy(t["logits"], t["target"], softcap=softcap, label_smoothing=case["smoothing"],
                                    return_token_accuracy=True, return_predicted_tokens=True)
            return o.loss, o.token_accuracy, o.predicted_tokens
        # The gradient is written over the logits, as in training, where the next step brings new
        # ones. Passed again, the same state holds that gradient as its logits: other values, the
        # same work.
        loss = forge_cross_entropy(t["logits"], t["target"], softcap=softcap, label_smoothing=case["smoothing"])
        return (loss, *torch.autograd.grad(loss, leaves))
    if op == "flce":
        loss = forge_fused_linear_cross_entropy(t["x"], t["weight"], t["target"])
        return (loss, *torch.autograd.grad(loss, leaves))
    s = _scale(case)
    if op == "mlp":
        args = [v for n in ("gate", "up", "down") for v in (t["w_" + n], t["a_" + n], t["b_" + n], s)]
        out = LoRAMLPv6.apply(t["x"], *args) if case["act"] == "silu" else LoRAMLPGeGLU.apply(t["x"], *args)
        return (out, *torch.autograd.grad(out, leaves, t["dy"]))
    if op == "qkv":
        args = [v for n in ("q", "k", "v") for v in (t["w_" + n], t["a_" + n], t["b_" + n], s)]
        outs = lora_qkv_rope(t["x"], *args, t["cos"], t["sin"], t["positions"], case["head_dim"])
        return (*outs, *torch.autograd.grad(outs, leaves, (t["dq"], t["dk"], t["dv"])))
    with torch.no_grad():
        return lora_mlp_v5_inference(t["x"], *t["merged"])


def work(case):
    op, e = case["op"], BYTES[case["dtype"]]
    if op == "glu":  # forward: gate, up -> out; backward: dout, gate, up -> dgate, dup
        n = case["rows"] * case["cols"]
        return {"bytes": 8 * n * e, "flops": 20 * n}
    if op == "rope":  # each direction reads and writes Q and K and reads the half tables
        n = case["batch"] * case["seq"] * (case["heads"] + case["kv_heads"]) * case["head_dim"]
        return {"bytes": 2 * (2 * n * e + case["seq"] * case["head_dim"] * e), "flops": 6 * n}
    if op == "rmsnorm":  # x -> y; x, dy -> dx; the weight, its gradient and rstd
        n = case["rows"] * case["cols"]
        return {"bytes": 5 * n * e + 8 * case["rows"] + 3 * case["cols"] * e, "flops": 12 * n}
    if op == "ce":
        n = case["rows"] * case["vocab"]
        return {"bytes": n * e * (1 if case["evaluate"] else 2) + 8 * case["rows"], "flops": 6 * n}
    if op == "flce":
        m, h, v = case["rows"], case["hidden"], case["vocab"]
        k = 2 if case["train_head"] else 1
        return {"bytes": 2 * m * h * e + k * v * h * e, "flops": 2 * (k + 1) * m * h * v}
    if op == "mlp":
        m, h, i, r = case["rows"], case["hidden"], case["inter"], case["rank"]
        return {"bytes": 4 * m * h * e + 3 * h * i * e + 12 * r * (h + i) * e,
                "flops": 12 * m * h * i + 6 * m * r * (h + i) + m * r * (16 * h + 14 * i)}
    if op == "qkv":
        m, k, r = case["rows"], case["hidden"], case["rank"]
        n = (case["heads"] + 2 * case["kv_heads"]) * case["head_dim"]
        return {"bytes": 2 * m * (k + n) * e + n * k * e + 2 * r * (3 * k + n) * e,
                "flops": m * (4 * k * n + 6 * r * n + 24 * k * r)}
    m, h, i = case["rows"], case["hidden"], case["inter"]
    return {"bytes": 2 * m * h * e + 3 * h * i * e, "flops": 6 * m * h * i}


def tolerance(case):
    if case["op"] == "ce" and case["evaluate"]:  # tokens_accuracy and predictions: ties of rounded logits only
        return {"rel": {"fp32": 1e-5}.get(case["dtype"], 1e-2), "differ": 1e-3}
    return {"rel": {"fp32": 1e-5, "bf16": 1.5e-2, "fp16": 2.5e-3}[case["dtype"]]}


def _rotate(x, cos, sin):
    half = x.shape[-1] // 2
    return x * cos + torch.cat([-x[..., half:], x[..., :half]], -1) * sin


def exact(case, seed):
    t = _inputs(case, seed)
    op = case["op"]
    trained = _trained(case)
    t = {n: v.double() if v.is_floating_point() else v for n, v in t.items()}
    for n in trained:
        t[n].requires_grad_(True)
    leaves = [t[n] for n in trained]
    s = _scale(case)

    def lora(x, n):
        return x @ t["w_" + n].T + s * ((x @ t["a_" + n].T) @ t["b_" + n].T)

    if op == "glu":
        a = F.silu(t["gate"]) if case["act"] == "silu" else F.gelu(
            t["gate"], approximate="tanh" if case["act"] == "gelu_tanh" else "none")
        out = a * t["up"]
        return (out.detach(), *torch.autograd.grad(out, leaves, t["dout"]))
    if op == "rope":
        oq, ok = (_rotate(t[n].transpose(1, 2), t["cos"].unsqueeze(1), t["sin"].unsqueeze(1)) for n in ("q", "k"))
        grads = torch.autograd.grad((oq, ok), leaves, (t["dq"].transpose(1, 2), t["dk"].transpose(1, 2)))
        return (oq.detach(), ok.detach(), *grads)
    if op == "rmsnorm":
        x = t["x"]
        y = x * torch.rsqrt(x.square().mean(-1, keepdim=True) + 1e-6) * t["weight"]
        return (y.detach(), *torch.autograd.grad(y, leaves, t["dy"]))
    if op == "ce":
        z = t["logits"]
        if case["softcap"]:
            z = case["softcap"] * torch.tanh(z / case["softcap"])
        loss = F.cross_entropy(z, t["target"], ignore_index=IGNORE, label_smoothing=case["smoothing"])
        if not case["evaluate"]:
            return (loss.detach(), *torch.autograd.grad(loss, leaves))
        kept = t["target"] != IGNORE
        best = z.argmax(-1)
        return loss, (best == t["target"])[kept].double().mean(), None
    if op == "flce":
        loss = F.cross_entropy(t["x"] @ t["weight"].T, t["target"], ignore_index=IGNORE)
        return (loss.detach(), *torch.autograd.grad(loss, leaves))
    if op == "qkv":
        pos, hd = t["positions"], case["head_dim"]
        outs = [lora(t["x"], n) for n in ("q", "k", "v")]
        for j in (0, 1):
            heads = outs[j].view(outs[j].shape[0], -1, hd)
            outs[j] = _rotate(heads, t["cos"][pos].unsqueeze(1), t["sin"][pos].unsqueeze(1)).reshape(outs[j].shape)
        grads = torch.autograd.grad(outs, leaves, (t["dq"], t["dk"], t["dv"]))
        return (*(o.detach() for o in outs), *grads)
    if op == "infer":
        x = t["x"]
        return lora(F.silu(lora(x, "gate")) * lora(x, "up"), "down").detach()
    e, g = lora(t["x"], "gate"), lora(t["x"], "up")
    out = lora((F.silu(e) if case["act"] == "silu" else F.gelu(e, approximate="tanh")) * g, "down")
    return (out.detach(), *torch.autograd.grad(out, leaves, t["dy"]))
