"""GPU parity of the cast kernels against the CPU oracle: e4m3 bytes, fp32
scales and bf16 amaxes must be bit-identical (NaN codes compare equal
irrespective of sign, see golden_util.fp8_equal_mod_nan_sign)."""
import pytest
import torch

import oracle
from conftest import seeded_bf16
from golden_util import bits_equal, fp8_equal_mod_nan_sign, load_golden

pytestmark = pytest.mark.gpu


def _lib_handle():
    from lingua_amd import _lib
    return _lib.load()


def dev(t):
    return t.to("cuda")


def check_rowwise(x, with_col=False):
    from lingua_amd import ops
    col = torch.full((x.shape[1],), 7e29, dtype=torch.float32, device="cuda") if with_col else None   # stale contents
    q, s, a = ops.cast_rowwise(dev(x), col_amax=col)
    qo, so, ao = oracle.cast_rowwise(x)
    assert torch.equal(q.cpu().view(torch.uint8), qo), "bytes differ"
    assert bits_equal(s.cpu().reshape(-1), so), "scales differ"
    assert bits_equal(a.cpu().reshape(-1), ao), "amax differ"
    if with_col:
        assert bits_equal(col.cpu(), oracle.col_amax(x).float()), "column amax differ"
    return q, s


def test_golden_vectors():
    from lingua_amd import ops
    g = load_golden()
    for name, t in (("x", g["x"]), ("w", g["w"]), ("g", g["go"])):
        q, s, a = ops.cast_rowwise(dev(t))
        assert torch.equal(q.cpu().view(torch.uint8), g["q_" + name]), name
        assert bits_equal(s.cpu().reshape(-1), g["s_" + name]), name
    assert bits_equal(ops.cast_rowwise(dev(g["x"]))[2].cpu().reshape(-1), g["amax_x"])
    w = dev(g["w"])
    _, _, amax_w = ops.cast_rowwise(w, want_q=False)
    qwt, swt = ops.cast_tensorwise(w, ops.amax_reduce(amax_w), transpose=True)
    assert torch.equal(qwt.cpu().view(torch.uint8), g["q_wt"])
    assert bits_equal(swt.cpu().reshape(-1).expand(g["s_wt"].shape).contiguous(), g["s_wt"])
    for name, t in (("gt", g["go"]), ("xt", g["x"])):
        td = dev(t)
        q, s = ops.cast_colwise_transposed(td, ops.col_amax(td))
        assert torch.equal(q.cpu().view(torch.uint8), g["q_" + name]), name
        assert bits_equal(s.cpu().reshape(-1), g["s_" + name]), name
    x = dev(g["x"])
    q, s = ops.cast_tensorwise(x, ops.amax_reduce(ops.cast_rowwise(x, want_q=False)[2]))
    assert torch.equal(q.cpu().view(torch.uint8), g["q_x_tw"]) and bits_equal(s.cpu().reshape(-1), g["s_x_tw"])


@pytest.mark.parametrize("shape", [(1, 8), (3, 16), (7, 520), (5, 4096), (300, 2048), (33, 11008), (9, 12288),
                                   (1027, 1024), (3, 16384), (2, 40000)])
@pytest.mark.parametrize("with_col", [False, True])
def test_rowwise_shapes(shape, with_col):
    x = seeded_bf16(shape, seed=shape[0] * 131 + shape[1])
    x[0, 0] = 0.0
    if shape[0] > 2:
        x[2] = 0.0
    check_rowwise(x, with_col)


@pytest.mark.parametrize("shape", [(2, 4096), (3, 4104), (2, 6144), (1600, 4616), (3, 6152), (2, 8192), (1030, 8200)])
@pytest.mark.parametrize("with_col", [False, True])
def test_rowwise_either_side_of_the_layout_lines(shape, with_col):
    """A wavefront per row up to 4096 columns, then a workgroup per row with three, four, six ... chunks per lane; more
    rows than one pass of the grid."""
    check_rowwise(seeded_bf16(shape, seed=shape[0] + shape[1]), with_col)


def test_rowwise_config1_inputs():
    check_rowwise(seeded_bf16((4096, 2048), 1.0, seed=0), with_col=True)
    check_rowwise(seeded_bf16((2048, 2048), 0.02, seed=1))


def test_rowwise_strided_input_and_col_amax_overwritten():
    from lingua_amd import ops
    big = seeded_bf16((64, 1536), seed=9)
    x = big[:, 256:256 + 1024]              # row stride 1536, offset 512 bytes
    xd = dev(big)[:, 256:256 + 1024]
    col = torch.full((1024,), 1e30, dtype=torch.float32, device="cuda")     # stale contents must not survive
    q, s, a = ops.cast_rowwise(xd, col_amax=col)
    qo, so, ao = oracle.cast_rowwise(x.contiguous())
    assert torch.equal(q.cpu().view(torch.uint8), qo) and bits_equal(s.cpu().reshape(-1), so)
    assert bits_equal(col.cpu(), oracle.col_amax(x.contiguous()).float())
    # the stand-alone column amax and the two-pass kernel for very long rows overwrite as well
    lib = _lib_handle()
    col2 = torch.full((1024,), 1e30, dtype=torch.float32, device="cuda")
    assert lib.l8_col_amax(xd.data_ptr(), 64, 1024, 1536, col2.data_ptr(), torch.cuda.current_stream().cuda_stream) == 0
    assert bits_equal(col2.cpu(), oracle.col_amax(x.contiguous()).float())
    wide = seeded_bf16((3, 40960), seed=10)
    col3 = torch.full((40960,), 1e30, dtype=torch.float32, device="cuda")
    q3, s3, _ = ops.cast_rowwise(dev(wide), col_amax=col3)
    assert torch.equal(q3.cpu().view(torch.uint8), oracle.cast_rowwise(wide)[0])
    assert bits_equal(col3.cpu(), oracle.col_amax(wide).float())


def test_rowwise_nonfinite_rows():
    from lingua_amd import ops
    x = seeded_bf16((6, 1024), seed=4)
    x[1, 3] = float("inf")
    x[2, 5] = float("nan")
    x[3, 7] = float("-inf")
    x[3, 9] = float("nan")
    q, s, a = ops.cast_rowwise(dev(x))
    qo, so, ao = oracle.cast_rowwise(x)
    assert fp8_equal_mod_nan_sign(q, qo)
    s, a = s.cpu().reshape(-1), a.cpu().reshape(-1)
    assert torch.equal(s.isnan(), so.isnan()) and torch.equal(s.isinf(), so.isinf())
    fin = so.isfinite()
    assert bits_equal(s[fin], so[fin])
    assert torch.equal(a.isnan(), ao.isnan()) and bits_equal(a[~ao.isnan()], ao[~ao.isnan()])


@pytest.mark.parametrize("amax", [448.0, 1.0, 0.0123, 3.3895e38, 1e-30, 240.0, 5.5e-13, 7.0])
def test_every_bf16_pattern_through_the_hardware_converter(amax):
    # one row per 4096 patterns; each row's amax is forced to `amax`, larger magnitudes and NaNs are zeroed
    bits = torch.arange(0, 65536, dtype=torch.int32).to(torch.int16)
    x = bits.view(torch.bfloat16).clone().reshape(16, 4096)
    a = torch.tensor(amax).to(torch.bfloat16)
    bad = ~(x.float().abs() <= a.float())
    x[bad] = 0.0
    x[:, 0] = a
    check_rowwise(x)
    # same patterns as one long row (two-pass kernel) and through the transposed kernels
    from lingua_amd import ops
    long_row = x.reshape(1, -1)
    check_rowwise(long_row)
    xd = dev(x)
    qt, st = ops.cast_colwise_transposed(xd, ops.col_amax(xd))
    qo, so = oracle.cast_colwise_transposed(x)
    assert torch.equal(qt.cpu().view(torch.uint8), qo) and bits_equal(st.cpu().reshape(-1), so)
    qw, sw = ops.cast_tensorwise(xd, dev(a.reshape(1, 1)))
    qwo, swo = oracle.cast_tensorwise(x, a)
    assert torch.equal(qw.cpu().view(torch.uint8), qwo) and bits_equal(sw.cpu().reshape(-1), swo)


@pytest.mark.parametrize("shape", [(1, 8), (4, 8), (128, 64), (129, 72), (100, 200), (257, 1000), (2048, 512),
                                   (50, 11008), (1030, 136)])
def test_transposed_kernels_shapes(shape):
    from lingua_amd import ops
    x = seeded_bf16(shape, seed=shape[0] * 7 + shape[1])
    x[0, 0] = 0.0
    if shape[1] > 16:
        x[:, 11] = 0.0  # an all-zero column: scale floor
    xd = dev(x)
    ca = ops.col_amax(xd)
    assert bits_equal(ca.cpu(), oracle.col_amax(x).float())
    q, s = ops.cast_colwise_transposed(xd, ca)
    qo, so = oracle.cast_colwise_transposed(x)
    R = shape[0]
    assert q.shape[1] % 16 == 0 and q.shape[1] - R < 16
    assert torch.equal(q.cpu().view(torch.uint8)[:, :R], qo) and bits_equal(s.cpu().reshape(-1), so)
    assert (q.cpu().view(torch.uint8)[:, R:] == 0).all()      # reduction padding is e4m3 zero
    amax = ops.amax_reduce(ops.cast_rowwise(xd, want_q=False)[2])
    assert bits_equal(amax.cpu().reshape(()), oracle.amax_of_amaxes(oracle.row_amax(x)))
    for tr in (False, True):
        q, s = ops.cast_tensorwise(xd, amax, transpose=tr)
        qo, so = oracle.cast_tensorwise(x, transpose=tr)
        assert torch.equal(q.cpu().view(torch.uint8), qo), tr
        assert bits_equal(s.cpu().reshape(-1), so), tr


def test_colwise_nonfinite_columns():
    from lingua_amd import ops
    x = seeded_bf16((40, 64), seed=6)
    x[3, 5] = float("inf")
    x[7, 9] = float("nan")
    xd = dev(x)
    q, s = ops.cast_colwise_transposed(xd, ops.col_amax(xd))
    qo, so = oracle.cast_colwise_transposed(x)
    assert fp8_equal_mod_nan_sign(q[:, :40], qo)
    s = s.cpu().reshape(-1)
    assert s[5].isinf() and s[9].isnan()
    fin = so.isfinite()
    assert bits_equal(s[fin], so[fin])


@pytest.mark.parametrize("bad", [float("inf"), float("nan")])
@pytest.mark.parametrize("amax_dtype", [torch.bfloat16, torch.float32])
def test_transposed_casts_with_a_nonfinite_amax_over_several_tiles(bad, amax_dtype):
    """The transposed kernels redo a column (or, tensor-wise, everything) whose amax is not finite with the
    integer conversion: ragged shape, more than one tile in both directions, both halves of a tile's rows."""
    from lingua_amd import ops
    x = seeded_bf16((300, 136), seed=11)
    x[1, 3] = bad
    x[140, 70] = bad
    x[299, 135] = bad
    xd = dev(x)
    amax = torch.tensor([[bad]], dtype=amax_dtype)
    for tr in (False, True):
        q, s = ops.cast_tensorwise(xd, dev(amax), transpose=tr)
        qo, so = oracle.cast_tensorwise(x, amax, transpose=tr)
        assert fp8_equal_mod_nan_sign(q.cpu().view(torch.uint8), qo), tr
        s = s.cpu().reshape(-1)
        assert torch.equal(s.isnan(), so.isnan()) and torch.equal(s.isinf(), so.isinf()), tr
    if amax_dtype == torch.float32:
        q, s = ops.cast_colwise_transposed(xd, ops.col_amax(xd))
        qo, so = oracle.cast_colwise_transposed(x)
        assert fp8_equal_mod_nan_sign(q[:, :300].cpu().view(torch.uint8), qo)
        s = s.cpu().reshape(-1)
        fin = so.isfinite()
        assert not fin[3] and not fin[70] and not fin[135] and int(fin.sum()) == 133
        assert bits_equal(s[fin], so[fin])


@pytest.mark.parametrize("ldq_pad", [0, 7])
def test_transposed_casts_with_ragged_edges_on_the_large_tile(ldq_pad):
    """Tensors with at least four 128 x 128 tiles per compute unit take the 128 x 128 tile (smaller ones a 64 x 128
    tile, which the random-shape sweep covers): rows and columns that are not multiples of the tile, a padded input
    row stride, an output row stride that rules out 16-byte stores, and one column with a non-finite amax."""
    from lingua_amd import _lib
    lib = _lib.load()
    R, C, ldx = 4100, 4104, 4112
    g = torch.Generator().manual_seed(21)
    xb = torch.randn(R, ldx, generator=g).to(torch.bfloat16)
    xb[:, C:] = 3.0e38                      # padding columns must not be read
    xb[17, 130] = float("inf")
    x = xb.cuda()
    xc = xb[:, :C].contiguous()
    ldq = (R + 15) // 16 * 16 + ldq_pad
    st = torch.cuda.current_stream().cuda_stream
    col = torch.zeros(C, dtype=torch.float32, device="cuda")
    _lib.check(lib.l8_col_amax(x.data_ptr(), R, C, ldx, col.data_ptr(), st), "l8_col_amax")
    q = torch.full((C, ldq), 0x55, dtype=torch.uint8, device="cuda")
    s = torch.empty(C, dtype=torch.float32, device="cuda")
    _lib.check(lib.l8_cast_colwise_transposed(x.data_ptr(), R, C, ldx, col.data_ptr(), q.data_ptr(), ldq, s.data_ptr(), st),
               "l8_cast_colwise_transposed")
    wq, ws = oracle.cast_colwise_transposed(xc)
    assert fp8_equal_mod_nan_sign(q.cpu()[:, :R], wq)
    assert (q.cpu()[:, R:] == 0x55).all()
    fin = ws.isfinite()
    assert int((~fin).sum()) == 1 and not fin[130] and bits_equal(s.cpu()[fin], ws[fin])
    amax = oracle.amax_of_amaxes(oracle.row_amax(xc[:, :128]))      # a finite amax that does not bound the tensor
    q = torch.full((C, ldq), 0x55, dtype=torch.uint8, device="cuda")
    s1 = torch.empty(1, dtype=torch.float32, device="cuda")
    xfin = xb.clone()
    xfin[17, 130] = 1.0
    xfin[:, :C] = xfin[:, :C].clamp(-float(amax.float()), float(amax.float()))
    _lib.check(lib.l8_cast_tensorwise(xfin.cuda().data_ptr(), R, C, ldx, amax.cuda().data_ptr(), 0, 1, q.data_ptr(), ldq,
                                      s1.data_ptr(), st), "l8_cast_tensorwise")
    wq, ws = oracle.cast_tensorwise(xfin[:, :C].contiguous(), amax, transpose=True)
    assert torch.equal(q.cpu()[:, :R], wq) and (q.cpu()[:, R:] == 0x55).all() and bits_equal(s1.cpu(), ws.reshape(-1))


def test_transposed_casts_with_ragged_edges_on_the_tall_tile():
    """Tensors of at least 16384 rows and 8192 columns take a 128 x 256 tile: same edge cases as for the other tiles,
    the whole output against the C oracle."""
    from lingua_amd import _lib
    lib = _lib.load()
    R, C, ldx = 16390, 8200, 8208
    g = torch.Generator().manual_seed(22)
    xb = torch.randn(R, ldx, generator=g).to(torch.bfloat16)
    xb[:, C:] = 3.0e38                      # padding columns must not be read
    xb[16389, 8199] = float("nan")
    x = xb.cuda()
    xc = xb[:, :C].contiguous()
    st = torch.cuda.current_stream().cuda_stream
    col = torch.zeros(C, dtype=torch.float32, device="cuda")
    _lib.check(lib.l8_col_amax(x.data_ptr(), R, C, ldx, col.data_ptr(), st), "l8_col_amax")
    for ldq in (16400, 16391):              # 16-byte stores, byte stores
        q = torch.full((C, ldq), 0x55, dtype=torch.uint8, device="cuda")
        s = torch.empty(C, dtype=torch.float32, device="cuda")
        _lib.check(lib.l8_cast_colwise_transposed(x.data_ptr(), R, C, ldx, col.data_ptr(), q.data_ptr(), ldq, s.data_ptr(), st),
                   "l8_cast_colwise_transposed")
        wq, ws = oracle.cast_colwise_transposed(xc)
        assert fp8_equal_mod_nan_sign(q[:, :R].cpu(), wq), ldq
        assert bool((q[:, R:] == 0x55).all()), ldq
        fin = ws.isfinite()
        assert int((~fin).sum()) == 1 and not fin[8199] and bits_equal(s.cpu()[fin], ws[fin]), ldq


from bench_workloads import outlier_stress_input  # noqa: E402


def test_outlier_stress_full_size_rowwise_tensorwise_colwise():
    from lingua_amd import ops
    x, ch, zr = outlier_stress_input()
    xd = dev(x)
    col = torch.zeros(x.shape[1], dtype=torch.float32, device="cuda")
    q, s, a = ops.cast_rowwise(xd, col_amax=col)
    qo, so, ao = oracle.cast_rowwise(x)
    assert torch.equal(q.cpu().view(torch.uint8), qo)
    assert bits_equal(s.cpu().reshape(-1), so) and bits_equal(a.cpu().reshape(-1), ao)
    assert (s.cpu().reshape(-1)[zr].view(torch.int32) == 0x2720D7C5).all()
    assert (q.cpu().view(torch.uint8)[zr] == 0).all()
    assert bits_equal(col.cpu(), oracle.col_amax(x).float())
    amax = ops.amax_reduce(a)
    qt, st = ops.cast_tensorwise(xd, amax)
    qto, sto = oracle.cast_tensorwise(x)
    assert torch.equal(qt.cpu().view(torch.uint8), qto) and bits_equal(st.cpu().reshape(-1), sto)
    qc, sc = ops.cast_colwise_transposed(xd, col)
    qco, sco = oracle.cast_colwise_transposed(x)
    assert torch.equal(qc.cpu().view(torch.uint8), qco) and bits_equal(sc.cpu().reshape(-1), sco)
    # row-wise scaling keeps far more of the signal than one scale for the whole tensor
    xf = x.float()
    deq_r = q.cpu().float() * s.cpu()
    deq_t = qt.cpu().float() * st.cpu()
    err_r = (deq_r - xf).norm() / xf.norm()
    err_t = (deq_t - xf).norm() / xf.norm()
    assert err_r < err_t


def test_ffn_hidden_shape_properties_full_size():
    # [16384, 11008]: too large for a full oracle pass to be cheap; checked through properties and a row sample
    from lingua_amd import ops
    g = torch.Generator(device="cuda").manual_seed(0)
    h = torch.randn(16384, 11008, generator=g, device="cuda", dtype=torch.float32).to(torch.bfloat16)
    col = torch.zeros(11008, dtype=torch.float32, device="cuda")
    q, s, a = ops.cast_rowwise(h, col_amax=col)
    qb = q.view(torch.uint8)
    assert ((qb & 0x7F).amax(dim=1) == 0x7E).all()          # every row reaches +-448
    assert torch.equal(a.reshape(-1), h.abs().amax(dim=1))
    assert torch.equal(col, h.abs().amax(dim=0).float())
    rows = torch.arange(0, 16384, 257)
    qo, so, _ = oracle.cast_rowwise(h[rows.cuda()].cpu())
    assert torch.equal(qb[rows.cuda()].cpu(), qo) and bits_equal(s.reshape(-1)[rows.cuda()].cpu(), so)
    # transposed cast == row-wise cast of the transpose, both on the GPU
    qt, st = ops.cast_colwise_transposed(h, col)
    ht = h.t().contiguous()
    q2, s2, _ = ops.cast_rowwise(ht)
    assert torch.equal(qt.view(torch.uint8), q2.view(torch.uint8)) and torch.equal(st, s2)


def test_every_finite_amax_lands_on_448_in_the_hardware_converter():
    """One row (and one column) per finite positive bf16 amax, bit patterns 0x0001 .. 0x7F7F: element 0 is the amax,
    so `amax * (1 / scale)` -- which may exceed 448 by an ulp or two -- goes through the hardware converter for
    every amax there is, in the row-wise kernel and in the transposed one (lingua/float8.py:43-47); the other
    elements are random magnitudes below it."""
    from lingua_amd import ops
    n = 0x7F7F
    g = torch.Generator().manual_seed(77)
    amax_bits = torch.arange(1, n + 1, dtype=torch.int32)
    C = 16
    frac = torch.rand(n, C, generator=g)
    mag = (frac * (amax_bits.reshape(n, 1) + 1).float()).to(torch.int32).clamp_(max=amax_bits.reshape(n, 1))
    sign = torch.randint(0, 2, (n, C), generator=g, dtype=torch.int32) << 15
    bits = mag | sign
    bits[:, 0] = amax_bits
    x = bits.to(torch.int16).view(torch.bfloat16)
    rows = torch.zeros(n + 1, C, dtype=torch.bfloat16)   # + one zero row: a multiple of 8 columns once transposed
    rows[:n] = x
    q, s = check_rowwise(rows)
    above_floor = rows[:n, 0].float() >= 1e-12                       # smaller amaxes are lifted to the floor of the scale
    assert bool((q.cpu().view(torch.uint8)[:n, 0][above_floor] == 0x7E).all())   # every other amax quantises to +448
    # the same values with one amax per column, through the transposed kernel
    xt = rows.t().contiguous()                                       # [16, 32640]
    xd = dev(xt)
    col = ops.col_amax(xd)
    assert bits_equal(col.cpu(), oracle.col_amax(xt).float())
    qt, st = ops.cast_colwise_transposed(xd, col)
    qo, so = oracle.cast_colwise_transposed(xt)
    assert torch.equal(qt.cpu().view(torch.uint8), qo) and bits_equal(st.cpu().reshape(-1), so)
    assert torch.equal(qt.cpu().view(torch.uint8), q.cpu().view(torch.uint8))  # same bytes either way


def test_pytorchs_gpu_division_by_a_scalar_is_the_product_with_the_inverse():
    """What `torch.clamp(amax_t.float(), min=EPS) / FP8_MAX` (lingua/float8.py:44) gives on this GPU, for every
    non-negative bf16 amax: PyTorch's GPU kernel multiplies by fp32(1/448), its CPU kernel divides, and the two differ
    in the last bit for a good third of the amaxes.  This pins the oracle's "times_inverse" rule against PyTorch's own
    kernel; the default rule is pinned against the CPU kernel in tests/test_oracle_cast.py."""
    bits = torch.arange(0, 0x7F81, dtype=torch.int32).to(torch.int16).view(torch.bfloat16)
    on_gpu = (torch.clamp(bits.cuda().float(), min=1e-12) / 448.0).cpu()
    on_cpu = torch.clamp(bits.float(), min=1e-12) / 448.0
    assert bits_equal(oracle.scale_from_amax(bits), on_cpu)
    with oracle.scale_rule("times_inverse"):
        assert bits_equal(oracle.scale_from_amax(bits), on_gpu)
    differ = (on_gpu.view(torch.int32) != on_cpu.view(torch.int32)).float().mean().item()
    assert 0.2 < differ < 0.6


@pytest.mark.parametrize("shape", [(4096, 2048), (777, 1000), (64, 11008), (3, 8)])
def test_casts_under_the_gpu_division_rule_equal_pytorchs_own_gpu_ops(shape, gpu_division_rule):
    """With `lingua_amd.set_scale_rule("times_inverse")` every layout's bytes and scales equal, bit for bit, what the
    reference's op chain (oracle.recipe_torch issues it op for op) gives when PyTorch runs it on this GPU -- and the
    oracle under the same rule."""
    from oracle import recipe_torch as rt
    from lingua_amd import ops
    x = seeded_bf16(shape, 1.0, seed=shape[0] + shape[1])
    x[0, 0] = 0
    if shape[0] > 2:
        x[1] = 0                      # a zero row: the floor of the clamp under this rule
    xd = x.cuda()
    # row-wise
    q, s, a = ops.cast_rowwise(xd)
    q_t, s_t = rt.scale(xd, rt.row_amax(xd))
    assert bits_equal(q.view(torch.uint8), q_t.view(torch.uint8)) and bits_equal(s.reshape(-1), s_t.reshape(-1))
    q_o, s_o, _ = oracle.cast_rowwise(x)
    assert torch.equal(q.cpu().view(torch.uint8), q_o) and bits_equal(s.cpu().reshape(-1), s_o)
    # an amax of the caller's, fp32
    amax32 = rt.row_amax(xd).float() * 1.5
    q, s = ops.cast_rowwise_given_amax(xd, amax32)
    q_t, s_t = rt.scale(xd, amax32)
    assert bits_equal(q.view(torch.uint8), q_t.view(torch.uint8)) and bits_equal(s.reshape(-1), s_t.reshape(-1))
    # column-wise, transposed (the wgrad operands)
    col = torch.zeros(shape[1], dtype=torch.float32, device="cuda")
    ops.cast_rowwise(xd, col_amax=col)
    q, s = ops.cast_colwise_transposed(xd, col)
    xt = xd.t().contiguous()
    q_t, s_t = rt.scale(xt, rt.row_amax(xt))
    assert bits_equal(q[:, :shape[0]].contiguous().view(torch.uint8), q_t.view(torch.uint8)) and bits_equal(s.reshape(-1), s_t.reshape(-1))
    # one scale for the tensor, both layouts
    amax = xd.abs().amax().reshape(1, 1)
    for transpose in (False, True):
        q, s = ops.cast_tensorwise(xd, amax, transpose=transpose)
        q_t, s_t = rt.scale(xt if transpose else xd, amax)
        cols = shape[0] if transpose else shape[1]
        assert bits_equal(q[:, :cols].contiguous().view(torch.uint8), q_t.view(torch.uint8)) and bits_equal(s.reshape(-1), s_t.reshape(-1))


@pytest.mark.parametrize("N,K", [(8, 16), (16, 272), (2048, 72), (2056, 2048), (8192, 136), (8200, 64), (16384, 8), (16392, 64)])
def test_transposed_cast_finds_the_amax_among_the_row_amaxes(N, K):
    """The dgrad weight quantised straight from its row amaxes: lists of one to eight loads per thread and past the last
    length, the largest amax in the first and last row, an infinity and a NaN; the bytes of reduction + cast."""
    from lingua_amd import ops
    w = seeded_bf16((N, K), 0.02, seed=N).cuda()
    for row, value in ((0, 3.0), (N - 1, -5.0), (N // 2, float("inf")), (N - 3, float("nan"))):
        w[row, K - 1] = value
        amax = ops.cast_rowwise(w, want_q=False)[2]
        q, s = ops.cast_tensorwise_t_rows(w, amax)
        wq, ws = ops.cast_tensorwise(w, ops.amax_reduce(amax), transpose=True)
        assert torch.equal(q.view(torch.uint8), wq.view(torch.uint8)), (N, K, value)
        assert torch.equal(s.view(torch.int32), ws.view(torch.int32)), (N, K, value)


@pytest.mark.parametrize("R", [1, 15, 16, 17, 63, 65, 127, 129, 1021])
@pytest.mark.parametrize("pad_to", [16, 48, 512])
def test_transposed_cast_pads_with_zeros(R, pad_to):
    """Columns beyond the rows of x are zeros -- also under a column whose amax is infinite or NaN, and in tiles that hold
    nothing else -- and the rest is what the unpadded cast writes."""
    from lingua_amd import ops
    for C in (8, 200):
        x = seeded_bf16((R, C), seed=R + C)
        x[R - 1, 3], x[0, C - 1] = float("inf"), float("nan")
        xd = x.cuda()
        torch.full((C * (R + pad_to),), 0x55, dtype=torch.uint8, device="cuda")  # what the allocator hands out next is not zero
        q, s = ops.cast_colwise_transposed(xd, ops.col_amax(xd), pad_to=pad_to)
        wq, ws = oracle.cast_colwise_transposed(x)
        assert q.shape == (C, (R + pad_to - 1) // pad_to * pad_to)
        assert torch.equal(q.cpu().view(torch.uint8)[:, :R], wq) and not q.view(torch.uint8)[:, R:].any()
        assert torch.equal(s.cpu().reshape(-1).view(torch.int32), ws.reshape(-1).view(torch.int32))


@pytest.mark.parametrize("C", [16, 520, 2048, 2056, 4104, 8192, 8200, 16384, 16392])
@pytest.mark.parametrize("rows", [(1, 1), (3, 4097), (70, 1, 9), (4100, 2, 5), (5, 6, 7, 8), (3, 0, 2)])
def test_several_operands_in_one_launch(C, rows):
    """Rows of every kernel, the first and last row of an operand next to each other in the list, more operands than a
    launch takes, an empty one, a padded row stride, zero rows and rows with an infinity or a NaN: the bytes, scales and
    amaxes of one call per operand."""
    from lingua_amd import ops
    if max(rows) * C > 1 << 25:
        rows = tuple(min(n, 600) for n in rows)
    xs = []
    for i, n in enumerate(rows):
        x = torch.zeros((n, C + 8), dtype=torch.bfloat16, device="cuda")[:, :C]
        x.copy_(torch.randn(n, C, generator=torch.Generator(device="cuda").manual_seed(i), device="cuda") * 10.0 ** (i - 1))
        if n > 2:
            x[n - 1] = 0.0
            x[0, C - 1], x[1, 0] = float("inf"), float("nan")
        xs.append(x)
    want = [ops.cast_rowwise(x) for x in xs]
    out = (torch.full((sum(rows), C), 0x55, dtype=torch.uint8, device="cuda").view(torch.float8_e4m3fn),
           torch.zeros((sum(rows), 1), device="cuda"))
    for got in (ops.cast_rowwise_many(xs), ops.cast_rowwise_many(xs, out=out)):
        for (q, s, a), (wq, ws, wa) in zip(got, want):
            assert torch.equal(q.view(torch.uint8), wq.view(torch.uint8))
            assert torch.equal(s.view(torch.int32), ws.view(torch.int32)) and torch.equal(a.view(torch.int16), wa.view(torch.int16))
    assert torch.equal(out[0].view(torch.uint8), torch.cat([w[0].view(torch.uint8) for w in want]))


@pytest.mark.parametrize("R,C", [(33, 144), (1, 16), (130, 1040), (48, 256), (257, 4112)])
def test_rows_on_lines_hold_what_dense_rows_hold(R, C):
    """on_lines moves the rows of a quantised operand to 128-byte lines, nothing else: every cast's bytes and scales, and the
    products that read them (one, several with one operand, a linear's forward in one call)."""
    from lingua_amd import ops
    x, w, h = (seeded_bf16((n, C), seed=n + C).cuda() for n in (R, 48, R))
    amax, col = ops.cast_rowwise(x)[2], ops.col_amax(x)
    wmax = ops.cast_rowwise(w)[2]
    norm_w = torch.rand(C, device="cuda").to(torch.bfloat16)

    def bits(t):
        return t.contiguous().view({1: torch.uint8, 2: torch.int16, 4: torch.int32}[t.element_size()])

    calls = [lambda on: ops.cast_rowwise(x, on_lines=on), lambda on: ops.cast_rowwise_given_amax(x, amax, on_lines=on),
             lambda on: ops.cast_tensorwise(x, amax[:1], on_lines=on), lambda on: ops.cast_tensorwise(x, amax[:1], transpose=True, on_lines=on),
             lambda on: ops.cast_tensorwise_t_rows(w, wmax, on_lines=on), lambda on: ops.cast_colwise_transposed(x, col, on_lines=on),
             lambda on: [t for trio in ops.cast_rowwise_many((x, w), on_lines=on) for t in trio],
             lambda on: ops.swiglu_cast_rowwise(x, h, on_lines=on), lambda on: ops.swiglu_bwd_cast_rowwise(x, x, h, on_lines=on),
             lambda on: ops.rmsnorm_cast_rowwise(x, norm_w, 1e-5, on_lines=on) if C <= 8192 else ()]
    for i, call in enumerate(calls):
        for a, b in zip(call(False), call(True)):
            assert a.shape == b.shape and torch.equal(bits(a), bits(b)), i
            if b.dtype == torch.float8_e4m3fn and b.shape[0] > 1:
                assert b.stride(0) % 128 == 0 and b.data_ptr() % 128 == 0 or i == 2
    (q, s, _), (qw, sw, _) = ops.cast_rowwise(x), ops.cast_rowwise(w)
    (ql, _, _), (qwl, _, _) = ops.cast_rowwise(x, on_lines=True), ops.cast_rowwise(w, on_lines=True)
    want = ops.gemm_nt(q, qw, s, sw)
    assert torch.equal(bits(ops.gemm_nt(ql, qwl, s, sw)), bits(want))
    for a, b in zip(ops.gemm_nt_multi((q, q), qw, (s, s), sw), ops.gemm_nt_multi((ql, ql), qwl, (s, s), sw)):
        assert torch.equal(bits(a), bits(b))
    for x_cast, w_cast in (((ql, s), (qwl, sw)), ((ql, s), (qw, sw)), ((q, s), (qwl, sw))):
        y = torch.empty_like(want)
        ops.linear_fwd(x, w, None, y, x_cast=x_cast, x_ready=True, w_cast=w_cast, w_ready=True)
        assert torch.equal(bits(y), bits(want))


def _many_inputs(shapes, seed):
    """Odd sizes, one with a row stride, one with an infinity and a NaN."""
    xs = []
    for i, (R, C) in enumerate(shapes):
        wide = seeded_bf16((R, C + 8), seed=seed + i).cuda()
        xs.append(wide[:, :C] if i == 1 else wide[:, :C].contiguous())
    xs[0][0, 0], xs[0][-1, -1] = float("inf"), float("nan")
    return xs


@pytest.mark.parametrize("shapes", [[(33, 144), (257, 16), (1, 8)], [(130, 2056), (130, 520), (130, 520), (130, 2056)],
                                    [(1021, 1040)] * 5, [(520, 4112), (516, 8200)], [(16400, 8200), (16384, 8192)]])
def test_several_transposed_casts_in_one_launch_equal_single_ones(shapes):
    """Column-wise ones of several widths and heights (more than a launch takes; small, ordinary and large tiles), then
    tensor-wise ones with their row amaxes, then both kinds mixed; bytes, scales and the zero padding."""
    from lingua_amd import ops
    xs = _many_inputs(shapes, 31)
    cols = [ops.col_amax(x) for x in xs]

    def compare(casts, want):
        for (q, s), (wq, ws) in zip(ops.cast_transposed_many(casts), want):
            assert torch.equal(q.view(torch.uint8), wq.view(torch.uint8)) and torch.equal(s.view(torch.int32), ws.view(torch.int32))

    compare(list(zip(xs, cols)), [ops.cast_colwise_transposed(x, c) for x, c in zip(xs, cols)])
    ws = [x[:x.shape[0] // 8 * 8] for x in xs if x.shape[0] >= 8]
    amaxes = [ops.cast_rowwise(w)[2] for w in ws]
    compare(list(zip(ws, amaxes)), [ops.cast_tensorwise_t_rows(w, a) for w, a in zip(ws, amaxes)])
    compare([(xs[0], cols[0]), (ws[0], amaxes[0]), (ws[-1], amaxes[-1]), (xs[1], cols[1])],
            [ops.cast_colwise_transposed(xs[0], cols[0]), ops.cast_tensorwise_t_rows(ws[0], amaxes[0]),
             ops.cast_tensorwise_t_rows(ws[-1], amaxes[-1]), ops.cast_colwise_transposed(xs[1], cols[1])])


@pytest.mark.parametrize("shapes", [[(33, 144), (257, 16)], [(1, 8), (2, 2048), (700, 2056), (64, 4104)], [(40, 33024), (3, 64), (5, 24)]])
def test_several_row_casts_with_column_amaxes_equal_single_ones(shapes):
    """Folds of different widths and lengths in one launch, more than a launch takes, and rows that leave nothing to fold."""
    from lingua_amd import ops
    xs = _many_inputs(shapes, 47)
    for x, (q, s, col) in zip(xs, ops.cast_rowwise_cols_many(xs)):
        want = torch.full((x.shape[1],), -1.0, device="cuda")
        wq, ws, _ = ops.cast_rowwise(x, col_amax=want)
        assert torch.equal(q.view(torch.uint8), wq.view(torch.uint8)) and torch.equal(s.view(torch.int32), ws.view(torch.int32))
        assert torch.equal(col.view(torch.int32), want.view(torch.int32))


@pytest.fixture
def new_memory_is_nan():
    """Memory that PyTorch hands out unwritten holds NaNs instead of whatever was there."""
    torch.use_deterministic_algorithms(True)
    assert torch.utils.deterministic.fill_uninitialized_memory
    yield
    torch.use_deterministic_algorithms(False)


def test_column_amaxes_of_nothing_are_zeros(new_memory_is_nan):
    """Operands without rows: every kernel that reports column amaxes writes them (the scales that are made of them multiply
    the zeros of an empty sum), alone and beside an operand that has rows."""
    from lingua_amd import _lib, ops
    C = 272
    x = torch.empty((0, C), dtype=torch.bfloat16, device="cuda")
    one = torch.ones((1, C), dtype=torch.bfloat16, device="cuda")
    got = [torch.empty(C, device="cuda") for _ in range(6)]
    assert bool(torch.isnan(torch.stack(got)).all())
    ops.cast_rowwise(x, col_amax=got[0])
    ops.swiglu_cast_rowwise(x, x, col_amax=got[1])
    ops.swiglu_bwd_cast_rowwise(x, x, x, got[2], got[3])
    ops.rmsnorm_cast_rowwise(x, one[0], 1e-5, col_amax=got[4])
    stream = torch.cuda.current_stream().cuda_stream
    _lib.check(_lib.load().l8_cast_rowwise_noalloc(0, 0, C, C, 0, C, 0, 0, got[5].data_ptr(), stream), "l8_cast_rowwise_noalloc")
    got.append(ops.col_amax(x))
    many = [col for _, _, col in ops.cast_rowwise_cols_many([x, one, x])]
    assert bool((torch.stack(got + [many[0], many[2]]) == 0).all()) and bool((many[1] == 1).all())


@pytest.mark.parametrize("fused", [False, True])
def test_weight_gradients_of_an_empty_batch_are_zeros(new_memory_is_nan, fused):
    """No tokens through linears on one activation, each for itself and as one product."""
    from lingua_amd import convert_linears_to_fp8, float8
    from lingua_amd.qkv import fuse_qkv

    class Block(torch.nn.Module):
        def __init__(self):
            super().__init__()
            self.wq, self.wk, self.wv = (torch.nn.Linear(64, n, bias=False, device="cuda", dtype=torch.bfloat16) for n in (64, 32, 32))
            for p in self.parameters():
                torch.nn.init.constant_(p, 0.5)

    float8.clear_cast_memos()
    block = convert_linears_to_fp8(Block(), "rowwise", "w[qkv]")
    if fused:
        block = fuse_qkv(block, "^$")
    x = torch.zeros((0, 64), dtype=torch.bfloat16, device="cuda", requires_grad=True)
    sum(y.sum() for y in (block.wq(x), block.wk(x), block.wv(x))).backward()
    assert x.grad.shape == x.shape
    assert all(bool((w.weight.grad == 0).all()) for w in (block.wq, block.wk, block.wv))


@pytest.mark.parametrize("R,C", [(0, 16), (1, 8), (127, 72), (128, 64), (129, 2048), (1021, 2048), (1024, 136), (1025, 136), (4100, 520), (20000, 48)])
@pytest.mark.parametrize("strided", [False, True])
def test_column_sums(R, C, strided):
    """One slab and several, the last one short, columns that do not fill a workgroup, a row stride.  Integers of magnitude up
    to 8: sums below 2^24 are exact in fp32, whatever their order, so the result is the exact sum rounded once; then normal
    values against the sum in 64 bits: at most R roundings of fp32 on top of the one to bf16; an infinity and a NaN stay."""
    from lingua_amd import ops
    g = torch.Generator().manual_seed(R + C)
    wide = torch.randint(-8, 9, (R, C + 8), generator=g).to(torch.bfloat16).cuda()
    x = wide[:, :C] if strided else wide[:, :C].contiguous()
    assert torch.equal(ops.col_sum(x), x.double().sum(0).to(torch.bfloat16))
    x = torch.randn(R, C, generator=g).to(torch.bfloat16).cuda()
    want, mag = x.double().sum(0), x.double().abs().sum(0)
    assert bool(((ops.col_sum(x).double() - want).abs() <= want.abs() * 2.0 ** -8 + mag * R * 2.0 ** -24).all())
    if R > 1:
        x[0, 0], x[R - 1, 1] = float("inf"), float("nan")
        got = ops.col_sum(x)
        assert bool(torch.isinf(got[0])) and bool(torch.isnan(got[1])) and bool(torch.isfinite(got[2:]).all())


@pytest.mark.parametrize("shift", [0, 1, 4])
def test_bias_gradient_of_rows_off_16_byte_lines(shift):
    """Only the bias learns, and the gradient's rows start off 16-byte lines, or not at all on a common one."""
    from lingua_amd.float8 import linear_backward
    g = torch.Generator().manual_seed(3)
    wide = torch.randint(-8, 9, (130, 64 + shift), generator=g).to(torch.bfloat16).cuda()
    got = linear_backward(wide[:, shift:], None, torch.zeros(64, 32, dtype=torch.bfloat16, device="cuda"),
                          torch.zeros(64, dtype=torch.bfloat16, device="cuda"), None, False, False, True, False, 0)
    assert got[0] is None and got[1] is None and torch.equal(got[2], wide[:, shift:].double().sum(0).to(torch.bfloat16))


@pytest.mark.parametrize("rows,C", [((1, 3, 5), 8), ((600, 2, 4093), 520), ((1021, 1021), 2048), ((33, 700, 5), 2056), ((4, 2100), 4096), ((9, 40), 4104)])
@pytest.mark.parametrize("poison", [False, True])
def test_column_amaxes_of_several_operands_in_one_launch(rows, C, poison):
    """Operands that share a launch (and, of other widths, those that do not): bytes, scales and column amaxes of the casts one
    by one, each with workgroups of its own whatever its share of the rows."""
    from lingua_amd import ops
    xs = [seeded_bf16((r, C + 8 * i), std=10.0 ** (i - 1), seed=r + i).cuda()[:, :C] for i, r in enumerate(rows)]
    if poison:
        xs[0][0, C // 2] = float("inf")
        xs[1][rows[1] - 1, C - 1] = float("nan")
    xs.append(seeded_bf16((5, 16), seed=3).cuda())
    for x, (q, s, col) in zip(xs, ops.cast_rowwise_cols_many(xs)):
        col0 = torch.empty_like(col)
        q0, s0, _ = ops.cast_rowwise(x, col_amax=col0)
        assert torch.equal(q.view(torch.uint8), q0.view(torch.uint8)) and bits_equal(s.cpu(), s0.cpu()) and bits_equal(col.cpu(), col0.cpu())


@pytest.mark.parametrize("M,N,K", [(1, 16, 16), (5, 72, 200), (127, 64, 128), (129, 528, 48), (1021, 2048, 2048), (1024, 256, 2048), (256, 8192, 1024)])
@pytest.mark.parametrize("poison", [False, True])
def test_casts_of_a_backward_pass_in_two_launches(M, N, K, poison):
    """l8_linear_bwd_casts against the casts one by one: up to 256 rows of partial column maxima are read by the workgroups of the
    transposed cast, each of its three operands at tile edges, with rows apart, with column amaxes that are not finite."""
    import struct
    from lingua_amd import _lib, ops
    lib = _lib.load()
    assert lib.l8_linear_bwd_casts_pays(M, N, K) and not lib.l8_linear_bwd_casts_pays(1025, N, K)
    g, a, w = (seeded_bf16((r, c + 8), std=s, seed=r + c).cuda()[:, :c] for r, c, s in ((M, N, 1e-2), (M, K, 1.0), (N, K, 0.02)))
    if poison:
        g[M // 2, N // 2] = float("inf")
        g[M - 1, 0] = float("nan")
        a[0, K - 1] = float("nan")
    Mp = (M + 15) // 16 * 16
    g_col, a_col = (torch.empty(c, dtype=torch.float32, device="cuda") for c in (N, K))
    qg0, sg0, _ = ops.cast_rowwise(g, col_amax=g_col)
    ops.cast_rowwise(a, col_amax=a_col)
    _, _, amax_w = ops.cast_rowwise(w)
    want = [(qg0, sg0), ops.cast_colwise_transposed(g, g_col), ops.cast_colwise_transposed(a, a_col),
            ops.cast_tensorwise(w, ops.amax_reduce(amax_w), transpose=True)]
    for parts in (3, 2, 1):     # gradient, activation and weight; the weight or the activation ready
        got = [(torch.full((r, c + 16), 0x55, dtype=torch.uint8, device="cuda")[:, :c], torch.empty(n, dtype=torch.float32, device="cuda"))
               for r, c, n in ((M, N, M), (N, Mp, N), (K, Mp, K), (K, N, 1))]
        need = lib.l8_cast_rowwise_workspace(M, N)
        ws = torch.empty(need + 16, dtype=torch.uint8, device="cuda")
        p = [t.data_ptr() for pair in got for t in pair]
        ld = [q.stride(0) for q, _ in got]
        with_a, with_w = parts != 1, parts != 2
        args = [g.data_ptr(), M, N, g.stride(0), p[0], ld[0], p[1], p[2], ld[1], p[3], Mp,
                a.data_ptr(), K, a.stride(0), a_col.data_ptr(), p[4] if with_a else 0, ld[2], p[5],
                w.data_ptr(), w.stride(0), amax_w.data_ptr(), p[6] if with_w else 0, ld[3], p[7],
                ws.data_ptr(), need, torch.cuda.current_stream().cuda_stream]
        _lib.check(lib.l8_linear_bwd_casts(struct.pack("27q", *args)), "l8_linear_bwd_casts")
        for i, ((q, s), (q0, s0)) in enumerate(zip(got, want)):
            if (i == 2 and not with_a) or (i == 3 and not with_w):
                assert (q == 0x55).all()
                continue
            assert torch.equal(q, q0.view(torch.uint8)), i
            assert bits_equal(s.cpu(), s0.cpu().reshape(-1)), i


@pytest.mark.parametrize("n", [1, 7, 8, 9, 1023, 8191, 8192, 32769, 65537])
@pytest.mark.parametrize("offset", [0, 1])
def test_amax_reduce_edges(n, offset):
    """Lists around one load per lane and one round of loads, on and off 16-byte lines, the maximum in each end; a NaN wins."""
    from lingua_amd import ops
    v = torch.rand(n + offset, generator=torch.Generator().manual_seed(n)).bfloat16()
    for at, value in ((offset, -3.0), (n + offset - 1, 5.0), (offset + n // 2, float("nan"))):
        v[at] = value
        got = ops.amax_reduce(v.cuda()[offset:])
        assert torch.equal(got.cpu().reshape(()), v[offset:].abs().max()) or (value != value and bool(got.isnan()))


@pytest.mark.parametrize("R,C", [(255, 32), (256, 40), (257, 24), (2047, 264), (2048, 40), (2049, 40), (2100, 264)])
def test_column_sums_around_the_one_launch(R, C):
    """Rows around one per thread and around the last that one launch takes, columns that end inside a workgroup's 32."""
    test_column_sums(R, C, False)
    test_column_sums(R, C, True)


@pytest.mark.parametrize("M,N,K", [(1, 16, 16), (63, 32, 128), (65, 40, 48), (257, 72, 64), (1021, 2048, 2048), (1024, 264, 2048)])
def test_bias_gradient_beside_the_casts_of_a_backward_pass(M, N, K):
    """l8_linear_bwd_casts_bias: the bits of l8_col_sum, rows around one per thread and columns that end inside a workgroup's,
    and the casts' bits with and without it."""
    import struct
    from lingua_amd import _lib, ops
    lib = _lib.load()
    g, a, w = (seeded_bf16((r, c + 8), std=s, seed=r + c).cuda()[:, :c] for r, c, s in ((M, N, 1e-2), (M, K, 1.0), (N, K, 0.02)))
    Mp, need = (M + 15) // 16 * 16, lib.l8_cast_rowwise_workspace(M, N)
    a_col, amax_w = ops.col_amax(a), ops.cast_rowwise(w)[2]
    results = []
    for wanted in (False, True):
        q = [torch.full((r, c), 0x55, dtype=torch.uint8, device="cuda") for r, c in ((M, N), (N, Mp), (K, Mp), (K, N))]
        s = [torch.zeros(n, device="cuda") for n in (M, N, K, 1)]
        ws = torch.empty(need + 16, dtype=torch.uint8, device="cuda")
        sums = torch.full((N,), 7.0, dtype=torch.bfloat16, device="cuda")
        args = [g.data_ptr(), M, N, g.stride(0), q[0].data_ptr(), N, s[0].data_ptr(), q[1].data_ptr(), Mp, s[1].data_ptr(), Mp,
                a.data_ptr(), K, a.stride(0), a_col.data_ptr(), q[2].data_ptr(), Mp, s[2].data_ptr(),
                w.data_ptr(), w.stride(0), amax_w.data_ptr(), q[3].data_ptr(), N, s[3].data_ptr(),
                ws.data_ptr(), need, torch.cuda.current_stream().cuda_stream]
        _lib.check(lib.l8_linear_bwd_casts_bias(struct.pack("27q", *args), sums.data_ptr() if wanted else None), "l8_linear_bwd_casts_bias")
        assert torch.equal(sums, ops.col_sum(g) if wanted else torch.full_like(sums, 7.0))
        results.append(q + s)
    assert all(torch.equal(x, y) for x, y in zip(*results))


@pytest.mark.parametrize("C", [512, 520, 1024, 2048, 2056, 4096, 4104])
@pytest.mark.parametrize("R", [1, 3, 512, 513])
def test_few_rows_have_the_bits_of_many(R, C):
    """The kernels for up to 512 rows and for more, around the widths where the loads per lane change, with and without the
    bytes: the rows of a small cast are those of a large one."""
    from lingua_amd import ops
    x = seeded_bf16((600, C + 8), std=1.0, seed=C).cuda()[:, :C]
    x[R - 1, C - 1], x[0, 0] = float("inf"), 300.0
    if R > 2:
        x[1, C // 2] = float("nan")
        x[2] = 0.0
    q0, s0, a0 = ops.cast_rowwise(x)
    q, s, a = ops.cast_rowwise(x[:R])
    assert torch.equal(q.view(torch.uint8), q0.view(torch.uint8)[:R])
    assert bits_equal(s.cpu(), s0[:R].cpu()) and bits_equal(a.cpu(), a0[:R].cpu())
    assert bits_equal(ops.cast_rowwise(x[:R], want_q=False)[2].cpu(), a.cpu())
