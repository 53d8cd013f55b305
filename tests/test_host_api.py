"""CPU-only checks of the host side: the C ABI exports what the header
declares, argument validation happens before any launch, and the converter /
module mirror the reference interface (lingua/float8.py:134-191)."""
import ctypes
import os
import re
import struct
import subprocess
import sys

import pytest
import torch
from torch import nn

import lingua_amd
from lingua_amd import _lib, ops
from lingua_amd.float8 import Fp8Linear, convert_linears_to_fp8, named_replace

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))


def test_library_exports_every_declared_symbol():
    header = open(os.path.join(ROOT, "include", "lingua_fp8.h")).read()
    header = re.sub(r"/\*.*?\*/", "", header, flags=re.S)
    declared = set(re.findall(r"\b(l8_\w+)\s*\(", header))
    assert {"l8_cast_rowwise", "l8_cast_tensorwise", "l8_cast_colwise_transposed", "l8_gemm_nt", "l8_col_amax",
            "l8_amax_reduce", "l8_version", "l8_last_error", "l8_device_check", "l8_cast_rowwise_workspace"} <= declared
    lib = ctypes.CDLL(_lib.LIB_PATH)
    for name in declared:
        assert hasattr(lib, name), name
    assert declared == set(_lib.SIGNATURES)
    assert _lib.load().l8_version() >= 1


def test_argument_validation_happens_before_launch():
    lib = _lib.load()
    fake = 1 << 20  # never dereferenced: every call below must be rejected on the host
    assert lib.l8_gemm_nt(fake, fake, 4, 4, 8, 16, 16, fake, 1, fake, 1, None, fake, 4, 0, None) == -1
    assert "multiple of 16" in _lib.last_error()
    assert lib.l8_gemm_nt(fake, fake, 4, 4, 16, 16, 16, fake, 7, fake, 1, None, fake, 4, 0, None) == -1
    assert lib.l8_gemm_nt(fake, fake, 4, 4, 16, 16, 16, fake, 1, fake, 1, None, fake, 4, 99, None) == -1
    assert lib.l8_gemm_nt(None, fake, 4, 4, 16, 16, 16, fake, 1, fake, 1, None, fake, 4, 0, None) == -1
    assert lib.l8_gemm_nt(fake + 1, fake, 4, 4, 16, 16, 16, fake, 1, fake, 1, None, fake, 4, 0, None) == -1
    assert lib.l8_cast_rowwise(fake, 4, 12, 12, fake, 12, fake, None, None, None, 0, None) == -1
    assert lib.l8_cast_rowwise(fake, -1, 8, 8, fake, 8, fake, None, None, None, 0, None) == -1
    assert lib.l8_cast_tensorwise(fake, 4, 8, 8, None, 0, 0, fake, 8, fake, None) == -1
    assert lib.l8_cast_colwise_transposed(fake, 4, 8, 8, None, fake, 4, fake, None) == -1
    # a tile of the transposed casts (256 rows) must stay within 1 GiB
    assert lib.l8_cast_tensorwise(fake, 4, 8, 1 << 21, fake, 0, 1, fake, 16, fake, None) == -1
    assert "row stride too large" in _lib.last_error()
    assert lib.l8_cast_colwise_transposed(fake, 4, 8, 1 << 21, fake, fake, 16, fake, None) == -1
    assert "row stride too large" in _lib.last_error()
    # empty problems are accepted and do nothing
    assert lib.l8_cast_rowwise(None, 0, 8, 8, None, 8, None, None, None, None, 0, None) == 0
    # the column-amax by-product needs the workspace the library asks for
    assert lib.l8_cast_rowwise_workspace(64, 1024) > 0
    assert lib.l8_cast_rowwise(fake, 64, 1024, 1024, fake, 1024, fake, None, fake, None, 0, None) == -1
    assert "workspace" in _lib.last_error()
    assert lib.l8_gemm_nt(None, None, 0, 4, 16, 16, 16, None, 1, None, 1, None, None, 4, 0, None) == 0


def test_column_amaxes_of_several_operands_are_refused_where_those_of_one_are():
    """Neighbours that one launch could take: a width that is no multiple of 8, pointers and strides that are.  Refused before
    anything is enqueued: on a machine without a GPU the first launch would answer with another error."""
    lib = _lib.load()
    fake = 1 << 20
    for C in (12, 2044):
        item = (fake, 8, C, (C + 15) // 16 * 16, fake, (C + 15) // 16 * 16, fake, 0, fake, fake, 1 << 30)
        assert lib.l8_cast_rowwise(*item, None) == -1 and "multiples of 8" in _lib.last_error()
        for n in (1, 2, 3):
            assert lib.l8_cast_rowwise_cols_many(struct.pack(f"{11 * n}q", *item * n), n, None) == -1
            assert f"C={C}" in _lib.last_error() and "multiples of 8" in _lib.last_error()


def test_linear_call_validates_its_arguments_on_the_host():
    """l8_linear_fwd takes a struct of eight-byte members; what it cannot serve is refused before any launch, and the
    workspace it asks for covers exactly the members that are left to it."""
    lib = _lib.load()
    fake = 1 << 20
    base = dict(x=fake, M=80, K=64, ldx=64, w=fake, N=48, ldw=64, bias=0, y=fake, ldy=48, qx=0, sx=0, col=0, x_ready=0, qw=0,
                sw=0, amax_w=0, w_ready=0, algo=0, ws=0, ws_bytes=0, stream=0)

    def pack(**kw):
        return ops._FWD.pack(*dict(base, **kw).values())

    full = lib.l8_linear_fwd_workspace(pack())
    assert full >= 80 * 64 + 80 * 4 + 48 * 64 + 48 * 4
    assert lib.l8_linear_fwd_workspace(pack(qw=fake, sw=fake, w_ready=1)) < full
    assert lib.l8_linear_fwd_workspace(pack(qx=fake, sx=fake)) < full
    assert lib.l8_linear_fwd_workspace(pack(col=fake)) > full
    # up to 64 tokens the weight is quantised inside the product, up to 8 the tokens too: nothing to put anywhere
    assert 32 * 64 + 32 * 4 <= lib.l8_linear_fwd_workspace(pack(M=32)) < lib.l8_linear_fwd_workspace(pack(M=32, amax_w=fake))
    assert lib.l8_linear_fwd_workspace(pack(M=8)) == 0 < lib.l8_linear_fwd_workspace(pack(M=9))
    # ... where the product of quantised operands is the same kernel, and with it the order of its sums
    for M, N, K in ((32, 11008, 64), (16, 9216, 4112), (48, 11008, 64), (64, 16400, 64), (17, 36864, 64)):
        assert not ops.gemm_pick(M, N, K)[1].startswith("skinny")
        assert lib.l8_linear_fwd_workspace(pack(M=M, N=N, K=K, ldx=K, ldw=K, ldy=N)) >= M * K + M * 4 + N * K + N * 4
    assert lib.l8_linear_fwd(pack()) == -1 and "workspace" in _lib.last_error()
    assert lib.l8_linear_fwd(pack(M=-1)) == -1 and lib.l8_linear_fwd_workspace(pack(M=-1)) == -1
    assert lib.l8_linear_fwd(pack(x_ready=1)) == -1 and "x_ready" in _lib.last_error()
    assert lib.l8_linear_fwd(pack(w_ready=1)) == -1 and "w_ready" in _lib.last_error()
    assert lib.l8_linear_fwd(pack(qx=fake)) == -1 and lib.l8_linear_fwd(None) == -1
    # a row stride counts where its operand is given
    assert lib.l8_linear_fwd_rows(pack(), 0, 0) == -1 and "workspace" in _lib.last_error()
    assert lib.l8_linear_fwd_rows(pack(qx=fake, sx=fake), 128, 0) == -1 and "workspace" in _lib.last_error()
    for given, ldqx, ldqw in ((dict(qx=fake, sx=fake), 48, 128), (dict(qx=fake, sx=fake), 72, 128), (dict(qw=fake, sw=fake), 128, 48)):
        assert lib.l8_linear_fwd_rows(pack(**given), ldqx, ldqw) == -1 and "ldqx" in _lib.last_error()


@pytest.mark.parametrize("change,named", [
    (dict(M=32, qx=(1 << 20) + 8, sx=1 << 20, x_ready=1), "qx"),          # few tokens: read in 16-byte pieces
    (dict(qx=(1 << 20) + 8, sx=1 << 20), "qx"), (dict(qw=(1 << 20) + 8, sw=1 << 20, w_ready=1), "qw"),
    (dict(x=(1 << 20) + 8), "x must"), (dict(w=(1 << 20) + 8), "w must"), (dict(w=0), "w must"), (dict(ldx=60), "ldx"), (dict(ldw=68), "ldw"),
    (dict(K=72, ldx=72, ldw=72), "multiple of 16"), (dict(y=0), "y is null"), (dict(ldy=40), "ldy"), (dict(algo=99), "algo")])
@pytest.mark.parametrize("M", [4, 32, 80])
def test_linear_call_is_refused_before_anything_is_enqueued(M, change, named):
    """An operand that the product cannot take is found before the casts: on a machine without a GPU the first launch
    would answer with another error."""
    lib = _lib.load()
    fake = 1 << 20
    base = dict(x=fake, M=M, K=64, ldx=64, w=fake, N=48, ldw=64, bias=0, y=fake, ldy=48, qx=0, sx=0, col=0, x_ready=0, qw=0,
                sw=0, amax_w=0, w_ready=0, algo=0, ws=fake, ws_bytes=1 << 20, stream=0)
    assert lib.l8_linear_fwd(ops._FWD.pack(*dict(base, **change).values())) == -1 and named in _lib.last_error()


@pytest.mark.parametrize("M,N,K,name", [(1, 36608, 4096, "skinny"), (1, 36864, 4096, "skinny"), (16, 128256, 4096, "skinny"),
                                        (17, 36608, 2048, "skinny"), (17, 36864, 2048, "2x2t_r5"), (32, 128256, 4096, "2x2t_r5"),
                                        (64, 36864, 4096, "2x2t_r5"), (65, 36864, 4096, "stream"), (1, 1 << 20, 64, "skinny")])
def test_few_tokens_take_no_big_tiles_however_wide_the_weight(M, N, K, name):
    """Host arithmetic (256 compute units where there is no GPU): weights on either side of the width at which one row of
    256 x 256 tiles fills the chip."""
    if torch.cuda.is_available() and torch.cuda.get_device_properties(0).multi_processor_count != 256:
        pytest.skip("the sizes are for 256 compute units")
    assert name in ops.gemm_pick(M, N, K)[1]


@pytest.fixture
def recorded_linear_calls(monkeypatch):
    """The inference call of a linear on CPU tensors, its library call recorded instead of made."""
    from lingua_amd import float8
    calls = []

    def linear_fwd(x, w, bias, y, x_cast=None, x_ready=False, w_cast=None, w_ready=False, *rest, **kw):
        calls.append({"outputs": y.shape[-1], "x_cast": x_cast, "x_ready": x_ready})

    monkeypatch.setattr(float8, "_check_operands", lambda a, b_t: None)
    monkeypatch.setattr(ops, "linear_fwd", linear_fwd)
    monkeypatch.setattr(ops, "current_stream_ptr", lambda index: 0)
    float8.clear_cast_memos()
    yield calls
    float8.clear_cast_memos()


def test_only_a_written_activation_cast_is_shared(recorded_linear_calls):
    """Above 64 tokens linears share the quantised activation -- but not the memory that a linear without outputs, for
    which the library has nothing to do, never wrote."""
    from lingua_amd import float8
    x = torch.zeros(80, 32, dtype=torch.bfloat16)
    for outputs in (0, 48, 64):
        float8.linear_infer(x, torch.zeros(outputs, 32, dtype=torch.bfloat16), None)
    assert [(c["outputs"], c["x_ready"]) for c in recorded_linear_calls] == [(0, False), (48, False), (64, True)]


class _RecordedLibrary:
    """Stands in for the library: notes which entry is called, and between which devices' brackets."""

    def __init__(self, monkeypatch):
        self.calls, self.inside = [], None
        outer = self

        class timed:
            def __init__(self, name, work, dev):
                self.name, self.dev = name, dev

            def __enter__(self):
                outer.inside = (self.name, self.dev)

            def __exit__(self, *exc):
                outer.inside = None

        monkeypatch.setattr(ops, "_timed", timed)
        monkeypatch.setattr(ops, "_prep", lambda t, what: 0)
        monkeypatch.setattr(_lib, "load", lambda: self)
        monkeypatch.setattr(_lib, "check", lambda code, what: None)

    def __getattr__(self, name):
        if not name.startswith("l8_"):
            raise AttributeError(name)
        return lambda *args: self.calls.append((name, self.inside)) or 0


def test_products_in_one_launch_run_on_their_operands_device(monkeypatch):
    """The library launches on the current device and counts its compute units: like every launch, this one is made
    with the tensors' device current."""
    rec = _RecordedLibrary(monkeypatch)
    qa, s = torch.zeros(16, 32, dtype=torch.float8_e4m3fn), torch.ones(16, 1)
    ops.gemm_nt_multi((qa, qa), qa, (s, s), s)
    assert rec.calls == [("l8_gemm_nt_multi", ("gemm_nt_multi", qa.device))]


def test_linear_call_asks_its_workspace_of_the_operands_device(monkeypatch):
    """How much the call needs depends on the compute units of the device that it runs on."""
    rec = _RecordedLibrary(monkeypatch)
    monkeypatch.setattr(torch._C, "_cuda_getDevice", lambda: 0, raising=False)   # the operands' index is None: another one

    x, w, y = (torch.zeros(s, dtype=torch.bfloat16) for s in ((80, 32), (48, 32), (80, 48)))
    ops.linear_fwd(x, w, None, y)
    assert rec.calls == [(name, ("linear_fwd", x.device)) for name in ("l8_linear_fwd_workspace", "l8_linear_fwd")]


@pytest.mark.parametrize("names,singly", [({"swiglu_cast_rowwise"}, False), ({"gemm_nt_multi", "cast_rowwise_many", "linear_fwd"}, False),
                                          ({"gemm_nt", "cast_rowwise"}, True), (["gemm_nt", "cast_rowwise"], True), (None, True)])
def test_a_kernel_timer_changes_only_what_it_asks_for(monkeypatch, recorded_linear_calls, names, singly):
    """Calls that run several kernels in one launch take them one by one under a timer for those kernels, and as ever
    under a timer for others."""
    from lingua_amd import float8
    rec = _RecordedLibrary(monkeypatch)
    monkeypatch.setattr(ops, "kernel_timer", [])
    monkeypatch.setattr(ops, "kernel_timer_names", names)
    x, w = torch.zeros(80, 32, dtype=torch.bfloat16), torch.zeros(48, 32, dtype=torch.bfloat16)
    qa, s = torch.zeros(16, 32, dtype=torch.float8_e4m3fn), torch.ones(16, 1)
    ops.gemm_nt_multi((qa, qa), qa, (s, s), s)
    ops.cast_rowwise_many((x, w))
    assert [name for name, _ in rec.calls] == (["l8_gemm_nt_ws"] * 2 + ["l8_cast_rowwise"] * 2 if singly else
                                               ["l8_gemm_nt_multi", "l8_cast_rowwise_many"])
    float8.linear_infer(x, w, None)
    assert len(recorded_linear_calls) == (0 if singly else 1)


def test_package_imports_where_pytorch_has_no_gpu_support():
    """Such a build lacks the private call that hands out raw streams; only a call on a GPU tensor may need it."""
    code = ("import torch; del torch._C._cuda_getCurrentRawStream; import lingua_amd\n"
            "try: lingua_amd.ops.cast_rowwise(torch.zeros(4, 16, dtype=torch.bfloat16))\n"
            "except RuntimeError as e: print(e)")
    done = subprocess.run([sys.executable, "-c", code], cwd=ROOT, capture_output=True, text=True, timeout=300)
    assert done.returncode == 0 and "no CPU path" in done.stdout, done.stderr


def test_no_cpu_path():
    x = torch.zeros(4, 16, dtype=torch.bfloat16)
    with pytest.raises(RuntimeError, match="no CPU path"):
        ops.cast_rowwise(x)
    lin = Fp8Linear(16, 8, bias=False, dtype=torch.bfloat16)
    with pytest.raises(RuntimeError):
        lin(x)


class Block(nn.Module):
    def __init__(self):
        super().__init__()
        self.w1 = nn.Linear(8, 16, bias=False)
        self.w2 = nn.Linear(16, 8, bias=True)
        self.norm = nn.LayerNorm(8)


class Model(nn.Module):
    def __init__(self):
        super().__init__()
        self.tok_embeddings = nn.Embedding(10, 8)
        self.layers = nn.ModuleList([Block(), Block()])
        self.output = nn.Linear(8, 10, bias=False)


def test_unknown_recipe_raises_runtime_error():
    with pytest.raises(RuntimeError, match="Unknown float8 recipe 'tensorwise'"):
        convert_linears_to_fp8(Model(), "tensorwise", r"layers\.[0-9]+\.")


def test_converter_filter_identity_and_state_dict():
    with torch.device("meta"):
        m = Model()
    params_before = dict(m.named_parameters())
    keys_before = list(m.state_dict().keys())
    out = convert_linears_to_fp8(m, "rowwise", r"layers\.[0-9]+\.")
    assert out is m
    for i in range(2):
        for name in ("w1", "w2"):
            lin = getattr(m.layers[i], name)
            assert type(lin) is Fp8Linear and isinstance(lin, nn.Linear)
            assert lin.weight is params_before[f"layers.{i}.{name}.weight"]
            assert lin.weight.device.type == "meta"
        assert m.layers[i].w2.bias is params_before[f"layers.{i}.w2.bias"]
        assert m.layers[i].w1.bias is None
        assert type(m.layers[i].norm) is nn.LayerNorm
    assert type(m.output) is nn.Linear                       # excluded by the default filter
    assert type(m.tok_embeddings) is nn.Embedding
    assert list(m.state_dict().keys()) == keys_before
    assert {id(p) for p in m.parameters()} == {id(p) for p in params_before.values()}


def test_converting_twice_or_a_subclass_asserts():
    m = convert_linears_to_fp8(Model(), "rowwise", r"layers\.")
    with pytest.raises(AssertionError):
        convert_linears_to_fp8(m, "rowwise", r"layers\.")

    class MyLinear(nn.Linear):
        pass

    m2 = nn.Sequential(MyLinear(4, 4))
    with pytest.raises(AssertionError, match="MyLinear"):
        convert_linears_to_fp8(m2, "rowwise", "")
    # a subclass that the filter does not match is left alone
    assert convert_linears_to_fp8(m2, "rowwise", "nomatch") is m2


def test_root_linear_is_replaced_and_returned():
    lin = nn.Linear(8, 4, bias=True, dtype=torch.bfloat16)
    out = convert_linears_to_fp8(lin, "rowwise", "")
    assert type(out) is Fp8Linear and out is not lin
    assert out.weight is lin.weight and out.bias is lin.bias
    assert out.weight.dtype == torch.bfloat16 and (out.in_features, out.out_features) == (8, 4)


def test_named_replace_is_post_order_with_dotted_names():
    seen = []

    def fn(mod, name):
        seen.append(name)
        return mod

    m = Model()
    assert named_replace(fn, m) is m
    assert seen[-1] == ""
    assert seen.index("layers.0.w1") < seen.index("layers.0") < seen.index("layers")
    assert "layers.1.norm" in seen and "output" in seen


def test_public_names_match_reference_module():
    for name in ("EPS", "scale", "matmul", "Fp8LinearFn", "Fp8Linear", "named_replace", "convert_linears_to_fp8"):
        assert hasattr(lingua_amd, name)
    assert lingua_amd.EPS == 1e-12


def test_custom_op_fake_kernels_on_meta_tensors():
    """lingua_amd.custom_ops: shape-only implementations (what torch.compile traces with) need no GPU."""
    import torch
    from lingua_amd import custom_ops  # noqa: F401  (registers the operators)
    a = torch.empty((32, 64), dtype=torch.bfloat16, device="meta")
    w = torch.empty((48, 64), dtype=torch.bfloat16, device="meta")
    bias = torch.empty((48,), dtype=torch.bfloat16, device="meta")
    out, amax_w, col = torch.ops.lingua_amd.fp8_linear_fwd(a, w, bias, True, 0)
    assert out.shape == (32, 48) and out.dtype == torch.bfloat16
    assert amax_w.shape == (48, 1) and amax_w.dtype == torch.bfloat16
    assert col.shape == (64,) and col.dtype == torch.float32
    assert torch.ops.lingua_amd.fp8_linear_fwd(a, w, None, False, 0)[2].numel() == 0
    ga, gb, gbias = torch.ops.lingua_amd.fp8_linear_bwd(out, a, w, amax_w, col, True, True, True, True, 0)
    assert ga.shape == a.shape and gb.shape == w.shape and gbias.shape == (48,)
    ga, gb, gbias = torch.ops.lingua_amd.fp8_linear_bwd(out, a, w, amax_w, col, False, True, False, True, 0)
    assert ga.numel() == 0 and gb.shape == w.shape and gbias.numel() == 0


def test_which_problems_share_the_k_range_of_their_last_round():
    """Host-side decision of tile configuration 15 (no GPU needed): the K range of the last round's tiles is shared
    out only where the exchange of partial sums pays, and the split the rule describes covers every (tile, K tile)
    of the tail exactly once with every owner waiting only for a workgroup with a lower number."""
    lib = _lib.load()
    cus = 256
    # the step's three products on 256 compute units: only the K = 16384 one (688 tiles, 2.69 rounds) splits
    assert lib.l8_gemm_shares_k(11008, 4096, 16384, cus) == 8
    assert lib.l8_gemm_shares_k(4096, 11008, 16384, cus) == 8
    assert lib.l8_gemm_shares_k(16384, 11008, 4096, cus) == 0      # K loop too short to pay for the exchange
    assert lib.l8_gemm_shares_k(16384, 4096, 11008, cus) == 0      # 1024 tiles: four full rounds
    assert lib.l8_gemm_shares_k(4096, 6656, 8192, cus) == 8
    assert lib.l8_gemm_shares_k(3300, 5096, 6128, cus) == 4        # four XCDs have a tail tile, four have none
    assert lib.l8_gemm_shares_k(1024, 1024, 16384, cus) == 0       # less than one round: nothing to share
    assert lib.l8_gemm_shares_k(16384, 4096, 11008, 4) < 0         # bad argument

    def split(cnt, W, KT, write=8, fix=4, least=16):
        rounds, r = divmod(cnt, W)
        if rounds == 0 or r == 0:
            return None
        helpers = W - r
        m = (r + helpers - 1) // helpers
        piece = (KT + fix - m * write) // (m + 1)
        return None if piece < least else (r, helpers, KT - piece)

    for W in (1, 2, 5, 16, 32, 38):
        for cnt in range(1, 3 * W + 1):
            for KT in (1, 20, 47, 48, 64, 100, 128, 500):
                s = split(cnt, W, KT)
                got = lib.l8_gemm_shares_k(256 * 8 * cnt, 256, 128 * KT, 8 * W)
                assert got == (8 if s else 0), (cnt, W, KT)
                if not s:
                    continue
                r, helpers, cut = s
                assert 0 < cut < KT
                cover = {}
                for loc in range(W):
                    if loc < helpers:                      # helper: K tiles cut.. of tiles loc, loc + helpers, ...
                        for tt in range(loc, r, helpers):
                            for k in range(cut, KT):
                                assert (tt, k) not in cover
                                cover[(tt, k)] = loc
                    else:                                  # owner of tile loc - helpers: K tiles 0..cut-1
                        for k in range(cut):
                            assert (loc - helpers, k) not in cover
                            cover[(loc - helpers, k)] = loc
                assert len(cover) == r * KT
                assert all(cover[(tt, KT - 1)] < cover[(tt, 0)] for tt in range(r))


def test_build_refuses_a_persistent_gemm_kernel_that_uses_scratch():
    from lingua_amd import build
    ok = {"_ZN2l821gemm_nt_stream_kernelILi4ELb0ELb0EEEvNS_8GemmArgsE": {"VGPRs": 158, "AGPRs": 256, "ScratchSize": 0, "VGPRs Spill": 0},
          "_ZN2l814gemm_nt_kernelILi2ELi2ELi4ELi4ELi5ELi8ELi0EEEvNS_8GemmArgsE": {"ScratchSize": 36, "VGPRs Spill": 8}}
    build._check_usage(ok)   # the one-workgroup-per-tile kernels may spill outside their K loop
    for field in ("ScratchSize", "VGPRs Spill"):
        bad = {k: dict(v) for k, v in ok.items()}
        bad["_ZN2l821gemm_nt_stream_kernelILi4ELb0ELb0EEEvNS_8GemmArgsE"][field] = 12
        with pytest.raises(RuntimeError):
            build._check_usage(bad)
    # the memory-streaming kernels (casts, gate, norm) must not use scratch memory either
    spilled = {k: dict(v) for k, v in ok.items()}
    spilled["_ZN2l822cast_rowwise_wg_kernelILi6ELb1EEEvPKtlilPhlPfPtS5_i"] = {"VGPRs": 128, "ScratchSize": 8, "VGPRs Spill": 1}
    with pytest.raises(RuntimeError, match="streaming"):
        build._check_usage(spilled)
    # a check that finds nothing to check must fail too: no remark parsed at all, or one without the figures
    with pytest.raises(RuntimeError):
        build._check_usage({})
    with pytest.raises(RuntimeError):
        build._check_usage({"_ZN2l821gemm_nt_stream_kernelILi4ELb0ELb0EEEvNS_8GemmArgsE": {"VGPRs": 158, "AGPRs": 256}})
    # and the shipped build's record lists every instantiation of the persistent kernel
    usage_file = os.path.join(os.path.dirname(build.LIB_PATH), "build", "resource_usage.txt")
    if os.path.exists(usage_file):
        text = open(usage_file).read()
        for inst in ("ILi4ELb0ELb0E", "ILi4ELb1ELb0E", "ILi4ELb0ELb1E", "ILi8ELb0ELb0E", "ILi2ELb0ELb0E", "ILi16ELb0ELb0E"):
            assert "gemm_nt_stream_kernel" + inst in text, inst


@pytest.mark.parametrize("variant", [False, True])
@pytest.mark.parametrize("there", [False, True])
@pytest.mark.parametrize("compiles", [False, True])
def test_build_links_the_library_whatever_becomes_of_the_host_extension(monkeypatch, tmp_path, variant, there, compiles):
    """The library needs hipcc alone.  The extension is compiled with every build of the shipped library and, where it is
    missing, with a tuning variant's; that it cannot be is an error, but one that leaves the library linked."""
    from lingua_amd import build
    ran = []

    def run(cmd, verbose):
        ran.append("native" if "native.cpp" in cmd[-1] else "link" if "-shared" in cmd else "object")
        if ran[-1] == "native" and not compiles:
            raise RuntimeError("g++ failed")
        return {}

    monkeypatch.setattr(build, "_run", run)
    monkeypatch.setattr(build, "_native_cmd", lambda: ["g++", "native.cpp"])
    monkeypatch.setattr(build, "_check_usage", lambda usage: None)
    monkeypatch.setattr(build, "OBJ_DIR", str(tmp_path))
    monkeypatch.setattr(build, "NATIVE_PATH", str(tmp_path / "_native.so"))
    if there:
        (tmp_path / "_native.so").touch()
    if variant:
        monkeypatch.setenv("LINGUA_FP8_LIB", str(tmp_path / "variant.so"))
    else:
        monkeypatch.delenv("LINGUA_FP8_LIB", raising=False)
    tried = not (variant and there)
    if tried and not compiles:
        with pytest.raises(RuntimeError, match="failed"):
            build.build()
    else:
        build.build()
    assert ran.count("link") == 1 and ran.count("native") == tried


def test_converter_drops_compiled_code_like_the_reference():
    """lingua/float8.py:187 resets the dynamo code caches after the swap ("force re-compile everything"): a
    module compiled before the conversion is traced again by its next call.  Runs on the CPU with a filter that
    matches nothing, so no Fp8Linear (GPU only) is executed."""
    import torch
    from lingua_amd import convert_linears_to_fp8
    traces = []

    def backend(gm, example_inputs):
        traces.append(len(traces))
        return gm.forward

    torch._dynamo.reset()
    model = torch.nn.Sequential(torch.nn.Linear(8, 8), torch.nn.ReLU())
    compiled = torch.compile(model, backend=backend)
    x = torch.randn(2, 8)
    compiled(x)
    compiled(x)
    assert len(traces) == 1                    # second call served from the code cache
    assert convert_linears_to_fp8(model, "rowwise", r"layers\.[0-9]+\.") is model
    compiled(x)
    assert len(traces) == 2                    # traced afresh after the conversion
    torch._dynamo.reset()


def test_scale_rule_switch_is_host_state_with_a_checked_argument():
    """l8_set_scale_rule / l8_get_scale_rule: host-only state, default = the correctly rounded quotient, unknown rules
    rejected with a message; the Python switch drops the quantised copies it holds."""
    import lingua_amd
    from lingua_amd import _lib, ops
    lib = _lib.load()
    assert lib.l8_get_scale_rule() == 0 and ops.get_scale_rule() == "divide"
    assert lib.l8_set_scale_rule(7) != 0 and b"unknown rule" in lib.l8_last_error()
    assert lib.l8_get_scale_rule() == 0
    try:
        lingua_amd.set_scale_rule("times_inverse")
        assert lib.l8_get_scale_rule() == 1 and lingua_amd.get_scale_rule() == "times_inverse"
        with pytest.raises(RuntimeError, match="unknown scale rule"):
            lingua_amd.set_scale_rule("fast")
        assert lingua_amd.get_scale_rule() == "times_inverse"
    finally:
        lingua_amd.set_scale_rule("divide")
    assert lib.l8_get_scale_rule() == 0


def test_linear_refuses_operands_it_cannot_serve_before_any_gpu_work():
    """No CPU path, bf16 only, feature counts in multiples of 16 (the reference gets the last one from
    torch._scaled_mm at lingua/float8.py:65): RuntimeError with the reason, raised before anything is launched."""
    from lingua_amd.float8 import Fp8LinearFn
    x = torch.zeros(8, 32, dtype=torch.bfloat16)
    w = torch.zeros(48, 32, dtype=torch.bfloat16)
    with pytest.raises(RuntimeError, match="no CPU path"):
        Fp8LinearFn.apply(x, w, None)
    with pytest.raises(RuntimeError, match="bf16 input and weight required"):
        Fp8LinearFn.apply(x.float(), w, None)
    meta_x = torch.zeros(8, 40, dtype=torch.bfloat16, device="meta")
    with pytest.raises(RuntimeError):
        Fp8LinearFn.apply(meta_x, torch.zeros(48, 40, dtype=torch.bfloat16, device="meta"), None)


def test_transforms_and_tracers_still_see_the_autograd_function(monkeypatch):
    """A forward without gradients takes one bare library call, whose result has no tangent, no batch dimension and no
    place in a trace: forward-mode AD and functorch are refused as before, a trace holds the function and not its result."""
    from lingua_amd import float8
    lin = Fp8Linear(32, 48, bias=False, dtype=torch.bfloat16).requires_grad_(False)
    x = torch.randn(8, 32).to(torch.bfloat16)
    bare = []
    monkeypatch.setattr(float8, "linear_infer", lambda a, w, b: bare.append(1) or a @ w.t())
    monkeypatch.setattr(float8, "linear_forward", lambda a, w, *rest: (a @ w.t(), w.abs().amax(1, keepdim=True), None))
    lin(x)
    assert bare == [1]
    with torch.autograd.forward_ad.dual_level(), pytest.raises(NotImplementedError, match="jvp"):
        lin(torch.autograd.forward_ad.make_dual(x, x))
    for transform in (torch.func.vmap(lin), torch.func.grad(lambda t: lin(t).sum())):
        with pytest.raises(RuntimeError, match="functorch"):
            transform(x.unsqueeze(0))
    traced = torch.jit.trace(lin, x, check_trace=False)
    assert torch.equal(traced(2 * x), 2 * (x @ lin.weight.t()))
    assert bare == [1]


def test_a_named_library_that_is_not_there_fails_loudly():
    """LINGUA_FP8_LIB points lingua_amd at another build of the library (a tuning variant); a path that does not exist
    is an error that names the path, never a silent return to the shipped library."""
    import subprocess
    import sys
    code = ("import lingua_amd._lib as L\n"
            "try:\n    L.load()\nexcept RuntimeError as e:\n    print('RuntimeError', str(e))\n")
    env = dict(os.environ, LINGUA_FP8_LIB="/nonexistent/libl8_variant.so", PYTHONPATH=os.path.dirname(os.path.dirname(os.path.abspath(__file__))))
    out = subprocess.run([sys.executable, "-c", code], env=env, capture_output=True, text=True, timeout=120)
    assert "RuntimeError" in out.stdout and "/nonexistent/libl8_variant.so" in out.stdout, out.stdout + out.stderr


def test_rows_too_far_apart_for_whole_tiles_stay_refused():
    """256 rows 8 MiB apart pass the 32-bit offsets of a tile; 192 do not, but a large problem is refused whichever of the two its
    size chooses (host checks only: nothing is enqueued)."""
    lib = _lib.load()
    fake, far = 1 << 20, 1 << 23
    if not torch.cuda.is_available():
        assert lib.l8_gemm_pick(3000, 3600, 4096) == 25
    for M, N in ((3000, 3600), (4096, 4096)):
        assert lib.l8_gemm_nt(fake, fake, M, N, 4096, far, 4096, fake, 1, fake, 1, None, fake, N, 0, None) == -1
        assert "leading dimension" in _lib.last_error()
