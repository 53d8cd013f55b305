"""The host extension's form of a linear's passes against the Python form: the same kernels on the same operands, so the
same bits, the same refusals, and the Python form wherever the extension does not take the call."""
import pytest
import torch

pytestmark = pytest.mark.gpu


@pytest.fixture
def form(monkeypatch):
    """Switches the extension off and counts the calls that it made."""
    from lingua_amd import _lib, float8

    class Switch:
        made = 0

    def counted(name, fn):
        def call(*args):
            out = fn(*args)
            Switch.made += out is not None
            return out
        return call

    native = _lib.native_for(0)

    class Counting:
        key = staticmethod(native.key)
        linear_fwd = staticmethod(counted("fwd", native.linear_fwd))
        linear_bwd = staticmethod(counted("bwd", native.linear_bwd))
        cast_colwise_transposed = staticmethod(counted("cast", native.cast_colwise_transposed))

    monkeypatch.setattr(_lib, "_native", Counting)
    asked = float8._native_call

    def use(on):
        float8.clear_cast_memos()
        Switch.made = 0
        monkeypatch.setattr(float8, "_native_call", asked if on else lambda a, algo: False)
        return Switch
    yield use
    float8.clear_cast_memos()


def _layer(K, N, bias, seed):
    from lingua_amd import Fp8Linear
    g = torch.Generator().manual_seed(seed)
    lin = Fp8Linear(K, N, bias=bias, dtype=torch.bfloat16, device="cuda")
    with torch.no_grad():
        for p in lin.parameters():
            p.copy_((torch.randn(p.shape, generator=g) * 0.05).cuda())
    return lin, g


def _input(shape, strided, g):
    x = torch.randn(shape, generator=g).to(torch.bfloat16).cuda()
    if strided:  # rows 16 elements further apart than they are long
        wide = torch.zeros((*shape[:-1], shape[-1] + 16), dtype=torch.bfloat16, device="cuda")
        wide[..., :shape[-1]] = x
        x = wide[..., :shape[-1]]
    return x


def _bits(ts):
    return [None if t is None else t.detach().contiguous().view(torch.int16) for t in ts]


def _same(a, b):
    assert len(a) == len(b)
    for u, v in zip(_bits(a), _bits(b)):
        assert (u is None) == (v is None) and (u is None or torch.equal(u, v))


@pytest.mark.parametrize("shape,K,N,strided", [((1,), 64, 48, False), ((17,), 144, 256, False), ((3, 5, 11), 256, 64, False),
                                               ((1021,), 128, 80, True), ((4, 9), 64, 64, True)])
@pytest.mark.parametrize("bias,save,cached", [(False, False, False), (True, True, False), (True, False, True)])
def test_training_pass_has_the_bits_of_the_python_form(form, monkeypatch, shape, K, N, strided, bias, save, cached):
    """Tokens that are no multiple of 16, leading dimensions, rows with a stride; the quantised input kept, weights kept
    quantised; every gradient, and the input's or the weight's alone."""
    from lingua_amd import float8
    monkeypatch.setattr(float8.config, "save_fp8_input", save)
    monkeypatch.setattr(float8.config, "cache_weight_casts", cached)
    for need_x, need_w in ((True, True), (True, False), (False, True)):
        results = []
        for on in (False, True):
            lin, g = _layer(K, N, bias, 7)
            x = _input((*shape, K), strided, g).requires_grad_(need_x)
            lin.weight.requires_grad_(need_w)
            grad = torch.randn((*shape, N), generator=g).to(torch.bfloat16).cuda()
            made = form(on)
            y = lin(x)
            y.backward(grad)
            results.append([y, x.grad, lin.weight.grad, lin.bias.grad if bias else None])
            assert (made.made > 0) == on
        _same(*results)


@pytest.mark.parametrize("tokens", [1, 8, 64, 65, 300])
@pytest.mark.parametrize("cached,lead,strided", [(False, (), False), (True, (), False), (False, (2,), False), (True, (), True), (False, (2,), True)])
def test_inference_pass_has_the_bits_of_the_python_form(form, monkeypatch, tokens, cached, lead, strided):
    """Around the number of tokens from which linears on one activation share its cast: two of them, one after the other,
    twice, and what the memo holds afterwards."""
    from lingua_amd import float8
    monkeypatch.setattr(float8.config, "cache_weight_casts", cached)
    results = []
    for on in (False, True):
        (a, g), (b, _) = _layer(256, 128, True, 3), _layer(256, 64, False, 4)
        x = _input((*lead, tokens, 256), strided, g)
        made = form(on)
        with torch.no_grad():
            out = [a(x), b(x), a(x), b(x)]
        results.append(out)
        assert (made.made > 0) == (on and not (strided and lead))   # three dimensions with gaps need a copy: the Python form
        assert (len(float8._fwd_cast.entries) > 0) == (tokens * (2 if lead else 1) > 64)
    _same(*results)


@pytest.mark.parametrize("kind", ["slice", "transposed", "bias view"])
def test_inference_on_operands_the_extension_leaves_shares_the_cast(form, monkeypatch, kind):
    """Two linears on one activation quantise it once also where the extension does not take the call: three dimensions with
    gaps (flattened without a copy, and with one: then each linear has an activation of its own), and a strided bias."""
    from lingua_amd import float8
    (a, g), (b, _) = _layer(256, 128, True, 3), _layer(256, 64, True, 4)
    x = _input((2, 80, 256), kind == "slice", g)
    if kind == "transposed":
        x = x.transpose(0, 1)
    if kind == "bias view":
        for lin in (a, b):
            wide = torch.zeros(2 * lin.bias.numel(), dtype=torch.bfloat16, device="cuda")
            wide[::2] = lin.bias.detach()
            lin.bias = torch.nn.Parameter(wide[::2])
    filed = []
    put = float8._fwd_cast.put
    monkeypatch.setattr(float8._fwd_cast, "put", lambda *args: filed.append(args) or put(*args))
    form(True)
    with torch.no_grad():
        out = [a(x), b(x)]
    assert len(filed) == (2 if kind == "transposed" else 1)
    form(False)
    with torch.no_grad():
        _same(out, [a(x), b(x)])


def test_switches_count_as_true_where_python_takes_them_so(form, monkeypatch):
    """A configuration read from a file may hold 1 for True."""
    from lingua_amd import float8
    results = []
    for yes in (True, 1):
        for name in ("share_input_casts", "fp8_wgrad"):
            monkeypatch.setattr(float8.config, name, yes)
        (a, g), (b, _) = _layer(64, 48, True, 9), _layer(64, 32, True, 10)
        x = _input((80, 64), False, g).requires_grad_(True)
        made = form(True)
        (torch.cat([a(x), b(x)], dim=1) ** 2).sum().backward()
        with torch.no_grad():
            out = [a(x), b(x)]
        assert made.made == 6
        results.append([*out, x.grad, a.weight.grad, b.weight.grad, a.bias.grad, b.bias.grad])
    _same(*results)


def test_what_the_python_form_refuses_stays_refused(form):
    lin, g = _layer(64, 48, False, 1)
    x = torch.randn(33, 64, generator=g).cuda()
    odd = torch.zeros(33 * 64 + 1, dtype=torch.bfloat16, device="cuda")[1:].view(33, 64)   # two-byte aligned
    narrow, _ = _layer(48, 64, False, 1)
    for on in (False, True):
        form(on)
        for grad in (True, False):
            with torch.set_grad_enabled(grad):
                with pytest.raises(RuntimeError, match="bf16 input and weight required"):
                    lin(x)
                with pytest.raises(RuntimeError, match="must be on the same GPU|no CPU path"):
                    lin(x.bfloat16().cpu())
                with pytest.raises(RuntimeError, match="aligned"):
                    lin(odd)
                with pytest.raises(RuntimeError, match="reduction dims differ"):
                    narrow(x.bfloat16())


def test_gradients_that_need_a_copy_take_the_python_form(form):
    """An expanded gradient (what sum() sends back) has no rows to point at; a graph of the gradients is not built here."""
    results = []
    for on in (False, True):
        lin, g = _layer(64, 48, True, 9)
        x = _input((40, 64), False, g).requires_grad_(True)
        form(on)
        lin(x).sum().backward()
        results.append([x.grad, lin.weight.grad, lin.bias.grad])
    _same(*results)


@pytest.mark.parametrize("on", [False, True])
def test_bias_gradients_of_a_batch_of_output_gradients(form, on):
    """A linear of which the bias alone learns has vectorised gradients (is_grads_batched): no kernel sees its backward pass."""
    lin, g = _layer(64, 48, True, 9)
    lin.weight.requires_grad_(False)
    x = _input((40, 64), False, g)
    form(on)
    y = lin(x)
    grads = torch.randn(3, 40, 48, generator=g).to(torch.bfloat16).cuda()
    batch, = torch.autograd.grad(y, lin.bias, grads, is_grads_batched=True)
    _same([batch], [grads.sum(dim=1)])


def test_weight_gradients_beside_such_gradients_share_the_input_cast(form, monkeypatch):
    """Two linears on one activation quantise it along its tokens once, whichever form their gradients take."""
    from lingua_amd import float8
    results = []
    for on in (False, True):
        (a, g), (b, _) = _layer(64, 48, False, 9), _layer(64, 32, False, 10)
        x = _input((40, 64), False, g).requires_grad_(True)
        form(on)
        filed = []
        with monkeypatch.context() as m:
            put = float8._bwd_cast.put
            m.setattr(float8._bwd_cast, "put", lambda *args: filed.append(args[0]) or put(*args))
            (a(x).sum() + b(x).sum()).backward()
        assert len(filed) == 1
        results.append([x.grad, a.weight.grad, b.weight.grad])
    _same(*results)


def test_key_tells_tensors_apart_as_the_tuple_did():
    from lingua_amd import _lib
    key = _lib.native_for(0).key
    t = torch.zeros(8, 16, dtype=torch.bfloat16, device="cuda")
    same = key(t)
    assert key(t) == same and key(t.view(8, 16)) == same
    for other in (t[:, :8], t.view(16, 8), t.t(), t[1:], t.view(torch.int16), t.unsqueeze(0), torch.zeros_like(t)):
        assert key(other) != same
    with torch.cuda.stream(torch.cuda.Stream()):
        assert key(t) != same
    t.add_(1)
    assert key(t) != same
