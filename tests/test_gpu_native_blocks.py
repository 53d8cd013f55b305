"""The host extension's form of the fused blocks' passes against the Python form: the same kernels on the same operands, so
the same bits, and the Python form wherever the extension does not take the call."""
import pytest
import torch
from torch import nn

pytestmark = pytest.mark.gpu

CALLS = ("rmsnorm_fwd", "rmsnorm_bwd", "qkv_fwd", "shared_bwd", "swiglu_fwd", "swiglu_bwd")


class RMSNorm(nn.Module):
    def __init__(self, dim, dtype):
        super().__init__()
        self.eps = 1e-5
        self.weight = nn.Parameter(torch.ones(dim, dtype=dtype))


class Block(nn.Module):
    def __init__(self, names, dim, widths, norm_dtype):
        super().__init__()
        self.norm = RMSNorm(dim, norm_dtype)
        self.inner = nn.Module()
        for name, (k, n) in zip(names, widths):
            setattr(self.inner, name, nn.Linear(k, n, bias=False, dtype=torch.bfloat16))


class Projections(nn.Module):
    def forward(self, x):
        return self.wq(x), self.wk(x), self.wv(x)


def _block(kind, dim, width, norm_dtype):
    from lingua_amd import convert_linears_to_fp8
    from lingua_amd.norm import fuse_rmsnorm
    from lingua_amd.qkv import fuse_qkv
    from lingua_amd.swiglu import fuse_feed_forward
    if kind == "qkv":
        b = Block(("wq", "wk", "wv"), dim, ((dim, dim), (dim, width), (dim, width)), norm_dtype)
        b.inner.__class__ = Projections
    else:
        b = Block(("w1", "w3", "w2"), dim, ((dim, width), (dim, width), (width, dim)), norm_dtype)
    g = torch.Generator().manual_seed(dim + width)
    with torch.no_grad():
        for name, p in b.named_parameters():
            p.copy_(torch.randn(p.shape, generator=g) * (0.1 if name == "norm.weight" else 0.03) + (1.0 if name == "norm.weight" else 0.0))
    b = convert_linears_to_fp8(b.cuda(), "rowwise", r"inner")
    fuse_rmsnorm(b, r"^norm$")
    (fuse_qkv if kind == "qkv" else fuse_feed_forward)(b, r"^inner$")
    return b


def _pass(b, x, grads, train):
    from lingua_amd import float8
    float8.clear_cast_memos()
    x = x.detach().requires_grad_(train)
    for p in b.parameters():
        p.grad = None
    with torch.set_grad_enabled(train):
        out = b.inner(b.norm(x))
    out = out if isinstance(out, tuple) else (out,)
    if train:
        torch.autograd.backward(out, grads)
    return [o.detach() for o in out] + ([x.grad] + [p.grad for p in b.parameters()] if train else [])


@pytest.mark.parametrize("train", [True, False])
@pytest.mark.parametrize("kind,rows,dim,width,norm_dtype,strided", [
    ("qkv", 1, 64, 16, torch.bfloat16, False),          # one token, the narrowest k and v
    ("qkv", 337, 208, 48, torch.float32, True),         # rows off 128-byte lines, rows of x apart
    ("qkv", 1040, 1024, 1024, torch.bfloat16, False),   # one K loop over the input gradients, one list of weight gradients' tiles
    ("mlp", 3, 48, 80, torch.float32, False),
    ("mlp", 513, 336, 1040, torch.bfloat16, True),
    ("mlp", 2049, 1024, 2048, torch.bfloat16, False),
    ("mlp", 17, 64, 16400, torch.bfloat16, False),      # wider than the gate's one-pass backward
])
def test_same_bits_as_the_python_form(monkeypatch, kind, rows, dim, width, norm_dtype, strided, train):
    from lingua_amd import _lib, float8
    native, made = _lib.native_for(0), set()

    class Counting:
        def __getattr__(self, name):
            def call(*args):
                out = getattr(native, name)(*args)
                if out is not None:
                    made.add(name)
                return out
            return call if name in CALLS else getattr(native, name)

    b = _block(kind, dim, width, norm_dtype)
    g = torch.Generator().manual_seed(rows)
    x = torch.randn((rows, dim + 16), generator=g).bfloat16().cuda()
    x = x[:, :dim] if strided else x[:, :dim].contiguous()
    widths = (dim, width, width) if kind == "qkv" else (dim,)
    grads = [(torch.randn((rows, n), generator=g) * 0.01).bfloat16().cuda() for n in widths]
    with monkeypatch.context() as m:
        m.setattr(float8, "_native_call", lambda a, algo: False)
        want = _pass(b, x, grads, train)
    with monkeypatch.context() as m:
        m.setattr(_lib, "_native", Counting())
        got = _pass(b, x, grads, train)
    float8.clear_cast_memos()
    wide = width > 16384
    expected = {"rmsnorm_fwd", "qkv_fwd" if kind == "qkv" else "swiglu_fwd"}
    if train:
        expected |= {"rmsnorm_bwd"} | ({"shared_bwd"} if kind == "qkv" else set() if wide else {"swiglu_bwd"})
    assert made == expected
    assert len(got) == len(want)
    for a, c in zip(got, want):
        assert a.shape == c.shape and a.dtype == c.dtype and torch.equal(a, c)


def test_some_gradients_take_the_python_form():
    """Frozen weights: the extension does not take the backward pass, and the gradients asked for are the same."""
    for kind, frozen in (("qkv", "inner.wk.weight"), ("mlp", "inner.w3.weight")):
        b = _block(kind, 128, 64, torch.bfloat16)
        x = torch.randn(40, 128, generator=torch.Generator().manual_seed(1)).bfloat16().cuda()
        grads = [torch.ones(40, n, device="cuda", dtype=torch.bfloat16) for n in ((128, 64, 64) if kind == "qkv" else (128,))]
        want = dict(zip([n for n, _ in b.named_parameters()], _pass(b, x, grads, True)[-len(list(b.parameters())):]))
        dict(b.named_parameters())[frozen].requires_grad_(False)
        got = dict(zip([n for n, _ in b.named_parameters()], _pass(b, x, grads, True)[-len(list(b.parameters())):]))
        assert got[frozen] is None
        for name in got:
            if name != frozen:
                rel = (got[name].float() - want[name].float()).norm() / want[name].float().norm()
                assert rel < 1e-2, name   # the input gradient's sum may be rounded per product: 2^-8 of each
