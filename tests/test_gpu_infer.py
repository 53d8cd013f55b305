"""Inference passes: no autograd node, no column amaxes, one call of the library per linear -- and the very bytes of the
training forward, whose product runs on the same kernel."""
import pytest
import torch

import oracle
from conftest import rel_l2, seeded_bf16

pytestmark = pytest.mark.gpu


def make(K, N, bias):
    from lingua_amd import Fp8Linear
    lin = Fp8Linear(K, N, bias=bias, device="cuda", dtype=torch.bfloat16)
    with torch.no_grad():
        lin.weight.copy_(seeded_bf16((N, K), 0.02, seed=N + K))
        if bias:
            lin.bias.copy_(seeded_bf16((N,), 0.5, seed=N))
    return lin


@pytest.mark.parametrize("shape", [(1, 64), (3, 5, 256), (64, 2064), (65, 272), (2, 150, 1040), (0, 32)])
@pytest.mark.parametrize("bias,cached", [(False, False), (True, True)])
def test_inference_equals_the_training_forward(shape, bias, cached):
    from lingua_amd import float8
    lin = make(shape[-1], 144, bias)
    x = seeded_bf16(shape, seed=sum(shape)).cuda()
    want = lin(x.clone().requires_grad_(True)).detach()
    old = float8.config.cache_weight_casts
    float8.config.cache_weight_casts = cached
    try:
        with torch.no_grad():
            for _ in range(2):                      # the second pass finds what the first one kept
                got = lin(x)
                assert got.shape == shape[:-1] + (144,) and not got.requires_grad
                assert torch.equal(got.view(torch.int16), want.view(torch.int16))
        with torch.inference_mode():
            assert torch.equal(lin(x).view(torch.int16), want.view(torch.int16))
        frozen = make(shape[-1], 144, bias).requires_grad_(False)
        assert torch.equal(frozen(x).view(torch.int16), want.view(torch.int16))
        if len(shape) == 2 and shape[0] > 1:        # rows of a wider tensor, columns of a taller one
            wide = torch.zeros((shape[0], shape[1] + 16), dtype=torch.bfloat16, device="cuda")
            wide[:, :shape[1]] = x
            with torch.no_grad():
                assert torch.equal(lin(wide[:, :shape[1]]).view(torch.int16), want.view(torch.int16))
                assert torch.equal(lin(x.t().contiguous().t()).view(torch.int16), want.view(torch.int16))
    finally:
        float8.config.cache_weight_casts = old
        float8.clear_cast_memos()


@pytest.mark.parametrize("M,K,N", [(8, 1040, 11008), (32, 1040, 7104), (32, 1040, 11008), (16, 4112, 9216), (48, 1040, 11008),
                                   (64, 1040, 16400), (17, 272, 36864), (64, 272, 36864)])
def test_one_result_whoever_asks(M, K, N):
    """Few tokens: with and without gradients, weight kept quantised or not, also where the product runs on another
    kernel than the few-token one.  Values over all of e4m3's exponents, so that the order of a sum shows."""
    from lingua_amd import float8
    spread = lambda n, k, s: (seeded_bf16((n, k), seed=s).float() *
                              torch.exp2(torch.randint(-7, 8, (n, k), generator=torch.Generator().manual_seed(s)).float())).to(torch.bfloat16)
    lin = make(K, N, True)
    with torch.no_grad():
        lin.weight.copy_(spread(N, K, 1))
    x = spread(M, K, 2).cuda()
    want = lin(x.clone().requires_grad_(True)).detach()
    old = float8.config.cache_weight_casts
    try:
        for float8.config.cache_weight_casts in (False, True):
            with torch.no_grad():
                assert torch.equal(lin(x).view(torch.int16), want.view(torch.int16))
    finally:
        float8.config.cache_weight_casts = old
        float8.clear_cast_memos()


def test_linears_share_an_activation_and_see_it_change():
    """Above 64 tokens w1 and w3 share one quantised copy, which a lookup from another stream does not get; a write to the
    activation in between is seen."""
    from lingua_amd import float8
    w1, w3 = make(256, 128, False), make(256, 272, False)
    for tokens in (40, 100):
        x = seeded_bf16((tokens, 256), seed=tokens).cuda()
        want = [oracle.linear_forward(x.cpu(), w.weight.detach().cpu()) for w in (w1, w3)]
        with torch.no_grad():
            assert rel_l2(w1(x), want[0]) <= 1e-3
            assert (len(float8._fwd_cast.entries) > 0) == (tokens > 64)
            assert rel_l2(w3(x), want[1]) <= 1e-3
            if tokens > 64:
                (entry,) = float8._fwd_cast.entries.values()
                assert entry[3] == {w1.weight.data_ptr(), w3.weight.data_ptr()}   # who has used it
                with torch.cuda.stream(torch.cuda.Stream()):
                    assert float8._fwd_cast.get(x, "somebody else") is None
                assert float8._fwd_cast.get(x, "somebody else") is not None
            w1(x)
            x.mul_(3.0)
            assert rel_l2(w3(x), oracle.linear_forward(x.cpu(), w3.weight.detach().cpu())) <= 1e-3
        float8.clear_cast_memos()


def test_a_linear_without_outputs_leaves_no_quantised_activation():
    """The next linear on the activation quantises it: nothing was written for the one before it."""
    from lingua_amd import float8
    none, some = make(256, 0, False), make(256, 272, False)
    x = seeded_bf16((100, 256), seed=5).cuda()
    with torch.no_grad():
        assert none(x).shape == (100, 0) and not float8._fwd_cast.entries
        assert rel_l2(some(x), oracle.linear_forward(x.cpu(), some.weight.detach().cpu())) <= 1e-3
    float8.clear_cast_memos()


def test_a_prompts_activation_is_not_kept_during_generation():
    """The memo holds the last activation alive; a call with few tokens, which shares none, lets go of it."""
    from lingua_amd import float8
    lin = make(256, 128, False)
    with torch.no_grad():
        lin(seeded_bf16((100, 256), seed=6).cuda())
        assert len(float8._fwd_cast.entries) == 1
        lin(seeded_bf16((1, 256), seed=7).cuda())
        assert not float8._fwd_cast.entries


@pytest.mark.parametrize("M", [1, 16, 17, 33, 64, 65])
@pytest.mark.parametrize("K", [16, 272, 4096, 4112, 8192, 8208, 12288, 12304])
def test_weight_quantised_inside_the_product(M, K):
    """Few tokens: the weight's row amaxes, scales and bytes are made between its only read and the product.  Rows of
    every register budget (4096, 8192, 12288 columns) and past the last; zero rows, rows with an infinity or a NaN (their
    outputs are NaN), a weight with a padded row stride; the same bits as the casts and the product one by one."""
    from lingua_amd import ops
    N = 52
    x = seeded_bf16((M, K), seed=M + K).cuda()
    w = torch.zeros((N, K + 8), dtype=torch.bfloat16)[:, :K]
    w.copy_(seeded_bf16((N, K), 0.02, seed=K))
    w[1] = 0.0
    w[7, K - 1], w[20, 0] = float("nan"), float("inf")
    bias = seeded_bf16((N,), seed=2).cuda()
    w = w.cuda()
    qx, sx, _ = ops.cast_rowwise(x)
    qw, sw, _ = ops.cast_rowwise(w)
    want = ops.gemm_nt(qx, qw, sx, sw, bias)
    got = torch.empty_like(want)
    ops.linear_fwd(x, w, bias, got)
    assert torch.equal(torch.isnan(got), torch.isnan(want)) and bool(torch.isnan(want[:, [7, 20]]).all())
    assert torch.equal(torch.nan_to_num(got.float()), torch.nan_to_num(want.float()))


@pytest.mark.parametrize("M", [1, 3, 4, 5, 8, 9])
@pytest.mark.parametrize("K", [16, 1040, 2048, 2064, 4096, 4112])
@pytest.mark.parametrize("kept", [True, False])
def test_tokens_quantised_inside_the_product(M, K, kept):
    """A handful of tokens: every workgroup quantises them for itself, the weight kept quantised or not.  Rows of both
    register budgets and past the last, padded row strides, a zero row, rows with an infinity or a NaN (NaN outputs);
    the same bits as the casts and the product one by one."""
    from lingua_amd import ops
    N = 84
    x = torch.zeros((M, K + 8), dtype=torch.bfloat16)[:, :K]
    x.copy_(seeded_bf16((M, K), seed=M + K))
    if M > 2:
        x[1] = 0.0
    if M > 4:
        x[2, K - 1], x[M - 1, 0] = float("nan"), float("-inf")
    x, w = x.cuda(), seeded_bf16((N, K), 0.02, seed=K).cuda()
    bias = seeded_bf16((N,), seed=2).cuda()
    qx, sx, _ = ops.cast_rowwise(x)
    qw, sw, _ = ops.cast_rowwise(w)
    want = ops.gemm_nt(qx, qw, sx, sw, bias)
    got = torch.empty_like(want)
    ops.linear_fwd(x, w, bias, got, w_cast=(qw, sw) if kept else None, w_ready=kept)
    assert torch.equal(torch.isnan(got), torch.isnan(want)) and (M <= 4 or bool(torch.isnan(want[[2, M - 1]]).all()))
    assert torch.equal(torch.nan_to_num(got.float()), torch.nan_to_num(want.float()))


@pytest.mark.parametrize("M,K,N", [(5, 272, 48), (40, 1040, 72), (64, 4112, 7168), (80, 272, 48), (1100, 2064, 80)])
@pytest.mark.parametrize("give_qx", [False, True])
@pytest.mark.parametrize("give_col", [False, True])
@pytest.mark.parametrize("give_qw,give_amax", [(False, False), (False, True), (True, False), (True, True)])
def test_what_the_linear_call_hands_out(M, K, N, give_qx, give_col, give_qw, give_amax):
    """The quantised operands, the activation's column amaxes and the weight's row amaxes where they are asked for, few
    tokens and many: the bits of the single entries, and the same y with or without them."""
    from lingua_amd import ops
    x, w = seeded_bf16((M, K), seed=M + K).cuda(), seeded_bf16((N, K), 0.02, seed=K).cuda()
    bias = seeded_bf16((N,), seed=2).cuda()
    want_col = torch.empty(K, device="cuda")
    wqx, wsx, _ = ops.cast_rowwise(x, col_amax=want_col)
    wqw, wsw, want_amax = ops.cast_rowwise(w)
    want = ops.gemm_nt(wqx, wqw, wsx, wsw, bias)
    fresh = lambda like: torch.full_like(like.view(torch.uint8), 0x55).view(like.dtype)
    qx, sx, qw, sw, col, amax = (fresh(t) for t in (wqx, wsx, wqw, wsw, want_col, want_amax))
    y = fresh(want)
    ops.linear_fwd(x, w, bias, y, x_cast=(qx, sx) if give_qx else None, col_amax=col if give_col else None,
                   w_cast=(qw, sw) if give_qw else None, amax_w=amax if give_amax else None)
    same = lambda a, b: torch.equal(a.view(torch.uint8), b.view(torch.uint8))
    assert same(y, want)
    assert not give_qx or same(qx, wqx) and same(sx, wsx)
    assert not give_col or same(col, want_col)
    assert not give_qw or same(qw, wqw) and same(sw, wsw)
    assert not give_amax or same(amax, want_amax)
