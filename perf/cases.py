"""The work that a user of this package has it do, as cases that can be timed and compared.

A case is one call (inference) or one forward + backward (training) through the public entry points: the drop-in
``convert_linears_to_fp8`` modules, the opt-in fused blocks (``fuse_feed_forward``, ``fuse_rmsnorm``, ``fuse_qkv``) and
``matmul`` with tensor-wise amaxes.  The part of a transformer block that the package does not compute (attention, rope,
residual adds) is left out: projections are timed with their norm, the MLP with its own.

Keys of a case:
  kind     "linear"     one Fp8Linear
           "mlp"        w2(silu(w1(x)) * w3(x)) of Fp8Linear modules
           "fused_mlp"  norm + MLP with the gate fused into the casts and the norm handing over its output quantised
           "qkv"        norm + wq / wk / wv as one product
           "tensorwise" matmul(x, amax [1,1], w, amax [1,1]) with the amaxes taken from the tensors
  tokens   rows of the activation
  d_in, d_out  widths of the activation and of the output (linear, tensorwise), or model width and hidden width (mlp,
               fused_mlp), or model width and width of k and v (qkv)
  train    forward + backward (every gradient) or forward without gradients
  bias     the linear has a bias
  cached   config.cache_weight_casts: weights stay quantised between calls, as in generation and gradient accumulation
  save_fp8 config.save_fp8_input: the quantised copy of the input is kept for backward instead of the input itself
"""
import math

import torch
from torch import nn

import lingua_amd
from lingua_amd import convert_linears_to_fp8, ops
from lingua_amd.norm import fuse_rmsnorm
from lingua_amd.qkv import fuse_qkv
from lingua_amd.swiglu import fuse_feed_forward

KINDS = ("linear", "mlp", "fused_mlp", "qkv", "tensorwise")


def _case(name, kind, tokens, d_in, d_out, train=False, bias=False, cached=False, save_fp8=False):
    c = {"kind": kind, "tokens": tokens, "d_in": d_in, "d_out": d_out, "train": train, "bias": bias, "cached": cached,
         "save_fp8": save_fp8}
    if name is not None:
        c["name"] = name
    return c


def listed():
    return [
        # one sequence in generation, a 1B-sized attention projection, weights kept quantised: the smallest call there is
        _case("decode_linear_1b", "linear", 1, 2048, 2048, cached=True),
        # 32 sequences in generation through a 7B-sized MLP, weights kept quantised
        _case("decode_mlp_7b", "mlp", 32, 4096, 11008, cached=True),
        # generation with the default configuration, which quantises the weight in every call
        _case("decode_linear_7b_default", "linear", 7, 4096, 4096),
        # one prompt of no particular length through a 1B-sized MLP
        _case("prompt_mlp_1b", "mlp", 333, 2048, 8192),
        # the benchmark's single linear
        _case("linear_1b", "linear", 4096, 2048, 2048),
        # the benchmark's MLP forward, 8 x 4096 tokens: the largest inference batch
        _case("eval_mlp_1b", "mlp", 32768, 2048, 8192),
        # a short, ragged batch in training, with a bias and the quantised input kept for backward
        _case("train_linear_ragged", "linear", 1021, 2048, 2048, train=True, bias=True, save_fp8=True),
        # attention projections of the 1B-sized model's training step, 4 x 4096 tokens
        _case("train_qkv_1b", "qkv", 16384, 2048, 2048, train=True),
        # MLP of the same training step
        _case("train_fused_mlp_1b", "fused_mlp", 16384, 2048, 8192, train=True),
        # a wide hidden dimension (rows beyond what the gate kernels hold in registers), one ragged sequence
        _case("train_fused_mlp_wide", "fused_mlp", 4093, 4096, 14336, train=True),
        # tensor-wise scaling on activations with outliers
        _case("tensorwise_7b", "tensorwise", 16384, 4096, 11008),
        # the headline workload: 7B-sized MLP, forward + backward, drop-in modules
        _case("train_mlp_7b", "mlp", 16384, 4096, 11008, train=True),
    ]


_MOST_FLOPS = 18 * 16384 * 4096 * 11008  # the largest listed case


def _log_uniform(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(("linear", "linear", "mlp", "fused_mlp", "qkv", "tensorwise"))
    # widths from a small model's to the widest listed one, multiples of 16 as every linear here requires
    d_in = 16 * _log_uniform(rng, 64, 320)
    d_out = 16 * _log_uniform(rng, 64, 896)
    if kind == "fused_mlp":
        d_out = 16 * _log_uniform(rng, 128, 896)
    if kind == "qkv":
        d_out = d_in if rng.random() < 0.5 else max(256, d_in // 64 * 16)  # k and v as wide as q, or a quarter of it
    train = kind in ("fused_mlp", "qkv") or (kind != "tensorwise" and rng.random() < 0.4)
    stage = "train" if train else rng.choice(("decode", "prompt", "batch"))
    if kind == "tensorwise":
        stage = "batch"
    lo, hi = {"decode": (1, 64), "prompt": (65, 2048), "batch": (2049, 32768), "train": (256, 16384)}[stage]
    tokens = _log_uniform(rng, lo, hi)
    c = _case(None, kind, tokens, d_in, d_out, train=train, bias=kind == "linear" and rng.random() < 0.3,
              cached=stage == "decode" and rng.random() < 0.6,
              save_fp8=kind == "linear" and train and rng.random() < 0.3)
    over = work(c)["flops"] / _MOST_FLOPS
    if over > 1:
        c["tokens"] = max(1, int(c["tokens"] / over))
    return c


class RMSNorm(nn.Module):
    """What the reference's blocks have in front of their linears (lingua/transformer.py:264-292)."""

    def __init__(self, dim, eps=1e-5):
        super().__init__()
        self.eps = eps
        self.weight = nn.Parameter(torch.ones(dim))

    def forward(self, x):
        x = x.float()
        return (x * torch.rsqrt(x.pow(2).mean(-1, keepdim=True) + self.eps) * self.weight.float()).to(torch.bfloat16)


class FeedForward(nn.Module):
    def __init__(self, dim, hidden):
        super().__init__()
        self.w1 = nn.Linear(dim, hidden, bias=False)
        self.w3 = nn.Linear(dim, hidden, bias=False)
        self.w2 = nn.Linear(hidden, dim, bias=False)

    def forward(self, x):
        return self.w2(nn.functional.silu(self.w1(x)) * self.w3(x))


class NormMLP(nn.Module):
    def __init__(self, dim, hidden):
        super().__init__()
        self.ffn_norm = RMSNorm(dim)
        self.feed_forward = FeedForward(dim, hidden)

    def forward(self, x):
        return self.feed_forward(self.ffn_norm(x))


class Projections(nn.Module):
    """The three products at the head of an attention (lingua/transformer.py:357-359)."""

    def __init__(self, dim, kv):
        super().__init__()
        self.wq = nn.Linear(dim, dim, bias=False)
        self.wk = nn.Linear(dim, kv, bias=False)
        self.wv = nn.Linear(dim, kv, bias=False)

    def forward(self, x):
        return self.wq(x), self.wk(x), self.wv(x)


class NormProjections(nn.Module):
    def __init__(self, dim, kv):
        super().__init__()
        self.attention_norm = RMSNorm(dim)
        self.attention = Projections(dim, kv)

    def forward(self, x):
        return self.attention(self.attention_norm(x))


def _normal(shape, std, g):
    return torch.randn(shape, generator=g, device=g.device, dtype=torch.float32).mul_(std).to(torch.bfloat16)


def _outliers(rows, cols, g):
    """Student-t activations (3 degrees of freedom), one channel in a thousand x 100, one row in a hundred zero."""
    z = torch.randn((rows, cols), generator=g, device=g.device)
    chi = torch.zeros_like(z)
    for _ in range(3):
        chi.add_(torch.randn((rows, cols), generator=g, device=g.device).square_())
    x = z.mul_(chi.div_(3.0).rsqrt_())
    x[:, torch.randperm(cols, generator=g, device=g.device)[: max(1, cols // 1000)]] *= 100.0
    x[torch.randperm(rows, generator=g, device=g.device)[: rows // 100]] = 0.0
    return x.to(torch.bfloat16)


def prepare(case, seed):
    dev = torch.device("cuda", torch.cuda.current_device())
    g = torch.Generator(device=dev).manual_seed(seed)
    kind, t, d_in, d_out = case["kind"], case["tokens"], case["d_in"], case["d_out"]
    state = {"case": case}
    if kind == "tensorwise":
        state["x"] = _outliers(t, d_in, g)
        state["w"] = _normal((d_out, d_in), 0.02, g)
        return state
    with dev:
        if kind == "linear":
            model = nn.ModuleDict({"layer": nn.Linear(d_in, d_out, bias=case["bias"])})
        else:
            model = nn.ModuleDict({"layer": {"mlp": FeedForward, "fused_mlp": NormMLP, "qkv": NormProjections}[kind](d_in, d_out)})
    model = model.to(torch.bfloat16)
    with torch.no_grad():
        for name, p in model.named_parameters():
            if name.endswith("norm.weight"):
                p.copy_(_normal(p.shape, 0.1, g)).add_(1.0)
            else:
                p.copy_(_normal(p.shape, 0.02, g))
    model = convert_linears_to_fp8(model, "rowwise", r"^layer")
    if kind == "fused_mlp":
        fuse_feed_forward(fuse_rmsnorm(model))
    elif kind == "qkv":
        fuse_qkv(fuse_rmsnorm(model))
    state["model"] = model["layer"]
    state["params"] = dict(model["layer"].named_parameters())
    state["x"] = _normal((t, d_in), 1.0, g).requires_grad_(case["train"])
    if case["train"]:
        widths = {"linear": (d_out,), "qkv": (d_in, d_out, d_out)}.get(kind, (d_in,))
        state["grads"] = [_normal((t, n), 1e-2, g) for n in widths]
    return state


def run(state):
    case, x = state["case"], state["x"]
    config = lingua_amd.config
    config.cache_weight_casts, config.save_fp8_input = case["cached"], case["save_fp8"]
    if case["kind"] == "tensorwise":
        w = state["w"]
        amax_x, amax_w = (ops.amax_reduce(ops.cast_rowwise(t, want_q=False)[2]) for t in (x, w))
        return lingua_amd.matmul(x, amax_x, w, amax_w, None)
    model = state["model"]
    if not case["train"]:
        with torch.no_grad():
            return model(x)
    x.grad = None
    for p in state["params"].values():
        p.grad = None
    out = model(x)
    out = out if isinstance(out, tuple) else (out,)
    torch.autograd.backward(out, state["grads"])
    return {"out": [o.detach() for o in out], "dx": x.grad, "dw": {n: p.grad for n, p in state["params"].items()}}


def work(case):
    t, d_in, d_out, kind = case["tokens"], case["d_in"], case["d_out"], case["kind"]
    if kind in ("linear", "tensorwise"):
        weights, x, y = d_in * d_out, t * d_in, t * d_out
    elif kind == "qkv":
        weights, x, y = d_in * (d_in + 2 * d_out), t * d_in, t * (d_in + 2 * d_out)
    else:
        weights, x, y = 3 * d_in * d_out, t * d_in, t * d_in
    if case["train"]:  # x, weights and output gradients in; outputs and the gradients of x and the weights out
        return {"bytes": 4 * (x + weights + y), "flops": 6 * t * weights}
    return {"bytes": 2 * (x + y) + (1 if case["cached"] else 2) * weights, "flops": 2 * t * weights}


def tolerance(case):
    # About four times what the path differs by when its products are computed in 64 bits instead (measured on every
    # listed case and a few drawn ones).  A product on its own: 2.2e-4 .. 3.2e-4, an element up to one bf16 step off
    # (8e-3); 5.5e-4 with tensor-wise scales on outliers.  Sums of two or three bf16 gradients: 3e-3 when they are
    # rounded once instead of every time.  Chained products quantise a bf16 intermediate again, where a bf16 step
    # becomes an e4m3 step: 2.0e-3 .. 3.6e-3, an element up to 0.15 off.
    if case["kind"] == "linear":
        return {"rel": 1.2e-3, "max": 3.2e-2}
    if case["kind"] == "tensorwise":
        return {"rel": 2.2e-3, "max": 3.2e-2}
    if case["kind"] == "qkv":
        return {"rel": 1.2e-2, "max": 0.1}
    return {"rel": 1.2e-2, "max": 0.55}
