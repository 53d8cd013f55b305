"""GPU parity of the fp8 NT GEMM: exact on integer-valued operands (pins the
matrix-core lane layout, tile edges and K tails), within rel-L2 <= 1e-3 of the
oracle's bf16(fp32-accumulated dequantised product) on random operands."""
import pytest
import torch

import oracle
from conftest import rel_l2, seeded_bf16

pytestmark = pytest.mark.gpu

TOL = 1e-3  # rel-L2 of bf16 outputs, from the benchmark specification


def n_algos():
    from lingua_amd import ops
    return len(ops.gemm_algos())


def fp8(t):
    return t.to(torch.float8_e4m3fn)


ALGOS = list(range(0, 17))
SHAPES_EXACT = [(1, 1, 16), (32, 32, 64), (256, 256, 128), (256, 256, 256), (300, 200, 144), (257, 513, 272),
                (64, 1000, 48), (1000, 24, 208), (512, 768, 240)]


@pytest.mark.parametrize("algo", ALGOS)
def test_exact_small_integer_operands(algo):
    from lingua_amd import ops
    if algo > n_algos():
        pytest.skip("no such tile configuration")
    g = torch.Generator().manual_seed(100 + algo)
    for (M, N, K) in SHAPES_EXACT:
        A = torch.randint(-1, 2, (M, K), generator=g).float()
        B = torch.randint(-1, 2, (N, K), generator=g).float()
        sa = torch.tensor([2.0 ** (i % 5 - 2) for i in range(M)]).reshape(M, 1)
        sb = torch.tensor([2.0 ** (i % 3) for i in range(N)]).reshape(N, 1)
        out = ops.gemm_nt(fp8(A).cuda(), fp8(B).cuda(), sa.cuda(), sb.cuda(), algo=algo)
        want = (A.double() @ B.double().t()) * sa.double() * sb.double().t()
        assert torch.equal(out.cpu().double(), want), (algo, M, N, K)


@pytest.mark.parametrize("K", [16, 128, 144, 256, 272, 400, 528, 1152])
@pytest.mark.parametrize("with_bias,scalar", [(False, False), (False, True), (True, False)])
@pytest.mark.parametrize("algo", [12, 23, 24])
def test_persistent_kernel_carries_its_fragments_from_tile_to_tile(algo, K, with_bias, scalar):
    """One to nine K tiles per output tile (even and odd numbers of them leave the next tile's fragments in one or the other
    register set, the last K tile short or whole) and 289 whole or 561 half tiles, so that workgroups have one, two or three;
    ragged last tiles.
    Integers in -1 .. 1 and powers of two for scales: the fp32 sums are exact, so is the one rounding to bf16."""
    from lingua_amd import ops
    g = torch.Generator().manual_seed(170 + K)
    M, N = 4101, 4104
    A, B = (torch.randint(-1, 2, (n, K), generator=g).float() for n in (M, N))
    sa = torch.tensor([2.0 ** (i % 5 - 2) for i in range(M)]).reshape(M, 1).cuda()
    sb = torch.tensor([2.0 ** (i % 3) for i in range(1 if scalar else N)]).reshape(-1, 1).cuda()
    bias = torch.randint(-8, 9, (N,), generator=g).to(torch.bfloat16).cuda() if with_bias else None
    out = ops.gemm_nt(fp8(A).cuda(), fp8(B).cuda(), sa, sb, bias, algo=algo)
    want = (A.cuda() @ B.cuda().t()) * sa * sb.t() + (0 if bias is None else bias.float())   # fp32: exact here
    assert torch.equal(out, want.to(torch.bfloat16))


@pytest.mark.parametrize("M", [1, 15, 16, 17, 32, 33, 48, 49, 64])
def test_few_tokens_exact_on_integers_and_within_tolerance_of_the_oracle(M):
    """At most 64 tokens (the default's choice; 65 take a tile kernel): token tiles of 16 full and ragged, weight rows
    that do not fill a tile of 16, reductions shorter than one step of 128, ragged, and longer than the eight waves'
    first round of steps; scalar scales and a bias.  Integers in -1 .. 1 sum exactly whatever the order."""
    from lingua_amd import ops
    assert ops.gemm_pick(M, 2048, 2048)[1].startswith("skinny") and not ops.gemm_pick(65, 2048, 2048)[1].startswith("skinny")
    g = torch.Generator().manual_seed(700 + M)
    for (N, K) in [(1, 16), (16, 128), (17, 144), (33, 1040), (100, 2064), (520, 4112)]:
        A = torch.randint(-1, 2, (M, K), generator=g).float()
        B = torch.randint(-1, 2, (N, K), generator=g).float()
        sa = torch.tensor([2.0 ** (i % 5 - 2) for i in range(M)]).reshape(M, 1)
        sb = torch.tensor([2.0 ** (i % 3) for i in range(N)]).reshape(N, 1)
        out = ops.gemm_nt(fp8(A).cuda(), fp8(B).cuda(), sa.cuda(), sb.cuda())
        assert torch.equal(out.cpu().double(), (A.double() @ B.double().t()) * sa.double() * sb.double().t()), (M, N, K)
        qa, qb = random_fp8_bytes((M, K), g), random_fp8_bytes((N, K), g)
        bias = (torch.randn(N, generator=g) * 50).to(torch.bfloat16)
        for sa_, sb_, b_ in ((sa, sb, bias), (sa[:1], sb, None), (sa, sb[:1], bias)):
            out = ops.gemm_nt(qa.cuda().view(torch.float8_e4m3fn), qb.cuda().view(torch.float8_e4m3fn), sa_.cuda(), sb_.cuda(),
                              b_.cuda() if b_ is not None else None)
            # about 3 % of the products of random bytes round to the other neighbour (the matrix instruction's own sum,
            # whatever the kernel); where one of few outputs dominates the norm, its step is up to 2^-8 of it
            assert rel_l2(out, oracle.gemm_nt(qa, qb, sa_, sb_, b_)) <= (TOL if M * N >= 5000 else 2.0 ** -8), (M, N, K)


@pytest.mark.parametrize("algo,tile", [(18, (128, 128)), (19, (64, 128)), (20, (128, 64)), (21, (64, 64)), (22, (32, 64)), (23, (256, 128)),
                                       (24, (128, 256))])
def test_small_tiles_exact_on_integers_at_their_edges(algo, tile):
    """The configurations for problems of at most one workgroup per compute unit: tiles full, one short and one over,
    reductions from a ring that is never filled (K = 16; a second group of waves without a K tile) to one that wraps
    several times."""
    from lingua_amd import ops
    g = torch.Generator().manual_seed(800 + algo)
    bm, bn = tile
    for (M, N, K) in [(bm, bn, 16), (bm - 1, bn + 1, 128), (bm + 1, bn - 1, 400), (3 * bm, 2 * bn, 1152), (2 * bm + 5, bn + 8, 2064)]:
        A = torch.randint(-1, 2, (M, K), generator=g).float()
        B = torch.randint(-1, 2, (N, K), generator=g).float()
        sa = torch.tensor([2.0 ** (i % 5 - 2) for i in range(M)]).reshape(M, 1)
        bias = torch.randint(-8, 9, (N,), generator=g).to(torch.bfloat16)
        out = ops.gemm_nt(fp8(A).cuda(), fp8(B).cuda(), sa.cuda(), torch.ones(1, 1).cuda(), bias.cuda(), algo=algo)
        want = ((A.double() @ B.double().t()) * sa.double() + bias.double()).to(torch.bfloat16)
        assert torch.equal(out.cpu(), want), (algo, M, N, K)


@pytest.mark.parametrize("mnk,name", [((200, 4096, 4096), "1x1t"), ((1021, 2048, 2048), "1x2t"), ((512, 4096, 4096), "1x2t"),
                                      ((2176, 960, 256), "2x1t"), ((2048, 2048, 4096), "2x2t_r9"), ((1500, 3008, 1440), "2x2t_r5"),
                                      ((64, 11008, 4096), "mt2x2w_1x1t"), ((32, 11008, 4096), "mt1x2w_1x1t"), ((16, 11008, 4096), "skinny"),
                                      ((9, 9216, 5120), "mt1x2w_1x1t"), ((8, 9216, 5120), "skinny"), ((32, 16448, 4096), "skinny"), ((16384, 2048, 2048), "stream"),
                                      ((4096, 2048, 2048), "mt4x1w_2x4t"), ((4165, 1920, 2832), "mt4x1w_2x4t"), ((3115, 2752, 2336), "mt2x2w_4x4t"),
                                      ((1566, 9904, 1136), "mt2x2w_2x4t"), ((5561, 9104, 1664), "mt4x1w_2x4t"), ((5561, 9104, 4096), "mt2x2w_4x4t"),
                                      ((64, 36864, 4096), "2x2t_r5"), ((65, 36864, 4096), "mt2x2w_2x4t")])
def test_tile_chosen_by_how_many_workgroups_it_makes(mnk, name):
    from lingua_amd import ops
    if torch.cuda.get_device_properties(0).multi_processor_count != 256:
        pytest.skip("the sizes are for 256 compute units")
    assert name in ops.gemm_pick(*mnk)[1]


@pytest.mark.parametrize("rows,N,K,together", [((2008, 2048, 520), 2048, 272, True), ((2500, 2500), 2056, 16, True), ((1536, 1500), 2048, 400, True),
                                               ((2817, 2900, 3070), 2200, 1040, True), ((256, 8), 512, 144, False),
                                               ((1536, 1500), 2048, 4112, False),
                                               ((2048, 2048, 2048), 2052, 128, None), ((2048, 0, 2048), 2048, 128, None)])
def test_products_with_one_operand_in_one_launch(rows, N, K, together):
    """Every product has the bits it has alone -- in one launch those of the big tiles, which add up K in order, in several
    those of the kernel that its own size picks: last tile rows that are short, of different
    lengths, one row alone in a tile; short column tiles; K tiles that are short, fewer than the ring; a workgroup's second
    tile in another product than its first; outputs (N % 8) and lists (an empty product) that cannot go together."""
    import struct
    from lingua_amd import _lib, ops
    if together is not None and torch.cuda.get_device_properties(0).multi_processor_count == 256:
        parts = [v for m in rows for v in (0, m, 0, 0)]
        assert _lib.load().l8_gemm_multi_pays(struct.pack(f"{len(parts)}q", *parts), len(rows), N, K) == together
    g = torch.Generator().manual_seed(950 + N)
    qb = random_fp8_bytes((N, K), g).cuda().view(torch.float8_e4m3fn)
    sb = (torch.rand(N, 1, generator=g) + 0.5).cuda()
    qas = [random_fp8_bytes((m, K), g).cuda().view(torch.float8_e4m3fn) for m in rows]
    sas = [(torch.rand(m, 1, generator=g) + 0.5).cuda() for m in rows]
    for qa, sa, out in zip(qas, sas, ops.gemm_nt_multi(qas, qb, sas, sb)):
        want = ops.gemm_nt(qa, qb, sa, sb, algo=12 if together else 0)
        assert out.shape == want.shape and torch.equal(out.view(torch.int16), want.view(torch.int16))


def spread(q, ld):
    """q with its rows `ld` bytes apart and NaN codes between them."""
    wide = torch.full((q.shape[0], ld), 0x7f, dtype=torch.uint8, device="cuda")
    wide[:, :q.shape[1]] = q.view(torch.uint8)
    return wide.view(torch.float8_e4m3fn)[:, :q.shape[1]]


@pytest.mark.parametrize("rows,N,K", [((2008, 2048, 520), 2048, 272), ((1536, 1500), 2048, 400), ((2817, 2900, 3070), 2200, 1040)])
def test_products_in_one_launch_with_rows_apart(rows, N, K):
    """Operands whose rows are further apart than they are long, one distance for A and another for B, have the bits of dense
    ones and no byte from between the rows; operands of different distances go one by one."""
    import struct
    from lingua_amd import _lib, ops
    if torch.cuda.get_device_properties(0).multi_processor_count == 256:
        parts = [v for m in rows for v in (0, m, 0, 0)]
        assert _lib.load().l8_gemm_multi_pays(struct.pack(f"{len(parts)}q", *parts), len(rows), N, K)
    g = torch.Generator().manual_seed(970 + N)
    qb = random_fp8_bytes((N, K), g).cuda().view(torch.float8_e4m3fn)
    sb = (torch.rand(N, 1, generator=g) + 0.5).cuda()
    qas = [random_fp8_bytes((m, K), g).cuda().view(torch.float8_e4m3fn) for m in rows]
    sas = [(torch.rand(m, 1, generator=g) + 0.5).cuda() for m in rows]
    lines = (K + 127) // 128 * 128
    want = ops.gemm_nt_multi(qas, qb, sas, sb)
    for ldas, ldb in (([lines] * len(rows), lines), ([lines + 16] * len(rows), K), ([K] * len(rows), lines)):
        got = ops.gemm_nt_multi([spread(q, ld) for q, ld in zip(qas, ldas)], spread(qb, ldb), sas, sb)
        assert all(torch.equal(a.view(torch.int16), b.view(torch.int16)) for a, b in zip(got, want))
    got = ops.gemm_nt_multi([spread(q, lines + 16 * i) for i, q in enumerate(qas)], spread(qb, lines), sas, sb)
    for qa, sa, out in zip(qas, sas, got):
        assert torch.equal(out.view(torch.int16), ops.gemm_nt(qa, qb, sa, sb).view(torch.int16))


@pytest.mark.parametrize("algo,mnk", [(0, (40, 52, 272)), (2, (130, 200, 144)), (2, (256, 256, 128)), (12, (256, 256, 128)),
                                      (12, (300, 520, 400)), (12, (4136, 4104, 272)), (11, (520, 264, 144)), (17, (33, 50, 1040)),
                                      (18, (128, 128, 256)), (21, (65, 70, 128)), (22, (32, 64, 400)), (14, (520, 264, 144)),
                                      (23, (256, 128, 128)), (23, (300, 520, 400)), (23, (4136, 4104, 272)), (23, (4136, 4104, 128)),
                                      (24, (128, 256, 128)), (24, (300, 520, 400)), (24, (4136, 4104, 272)), (24, (4136, 4104, 128))])
def test_product_added_to_what_the_output_holds(algo, mnk):
    """add=True leaves the bits of out.add_(product): every kernel's epilogue (interior and ragged tiles, a workgroup's
    second tile, a configuration without an add of its own), an output with a row stride, nothing written beside it."""
    from lingua_amd import ops
    M, N, K = mnk
    g = torch.Generator().manual_seed(900 + algo + M)
    qa, qb = (random_fp8_bytes(s, g).cuda().view(torch.float8_e4m3fn) for s in ((M, K), (N, K)))
    sa, sb = (torch.rand(M, 1, generator=g) + 0.5).cuda(), (torch.rand(1, 1, generator=g) + 0.5).cuda()
    for sb_ in (sb, sb.expand(N, 1).contiguous()):
        buf = (torch.randn(M, N + 16, generator=g) * 1e4).to(torch.bfloat16).cuda()
        want = buf.clone()
        want[:, 8:8 + N] += ops.gemm_nt(qa, qb, sa, sb_, algo=algo)
        ops.gemm_nt(qa, qb, sa, sb_, algo=algo, out=buf[:, 8:8 + N], add=True)
        assert torch.equal(buf.view(torch.int16), want.view(torch.int16))
    with pytest.raises(RuntimeError, match="add needs out"):
        ops.gemm_nt(qa, qb, sa, sb, algo=algo, add=True)


def sum_of_products(terms):
    from lingua_amd import ops
    return ops.gemm_nt_sum(*zip(*terms))


def one_by_one(terms):
    from lingua_amd import ops
    out = None
    for qa, qb, sa, sb in terms:
        out = ops.gemm_nt(qa, qb, sa, sb, out=out, add=out is not None)
    return out


# (two tiles per workgroup and one, K tiles even and odd in number, whole and short, rows on lines and apart)
@pytest.mark.parametrize("M,N,Ks", [(4093, 8184, (512, 512)), (4093, 8184, (528, 1152, 656)), (3590, 3592, (640, 2064)), (3590, 3592, (1040, 512, 768))])
def test_sum_of_products_is_rounded_once(M, N, Ks):
    """Integers in -1 .. 1 and powers of two for scales: the fp32 sums are exact, whichever product's scale they are counted in,
    so the result is the one rounding to bf16 of the exact sum."""
    from lingua_amd import _lib
    assert _lib.load().l8_gemm_pick(M, N, sum(Ks)) == 12
    g = torch.Generator().manual_seed(M + len(Ks))
    terms, want = [], 0
    for i, K in enumerate(Ks):
        A, B = (torch.randint(-1, 2, (n, K), generator=g).float().cuda() for n in (M, N))
        sa = torch.tensor([2.0 ** ((r * (i + 3)) % 5 - 2) for r in range(M)]).reshape(M, 1).cuda()
        sb = torch.tensor([[2.0 ** (1 - i)]]).cuda()
        want = want + (A.double() @ B.double().t()) * sa.double() * sb.double()
        terms.append((spread(fp8(A).view(torch.uint8), K + 16 * i).view(torch.float8_e4m3fn), fp8(B), sa, sb))
    assert torch.equal(sum_of_products(terms).view(torch.int16), want.float().to(torch.bfloat16).view(torch.int16))


def test_sum_of_products_whose_scales_lie_far_apart():
    """Rows whose products differ by up to 2^150 in scale, rows of zeros with the smallest scale, rows whose scale is infinite or
    NaN: what adding one product to the other gives, but for its roundings to bf16 (2^-9 of either product and of the sum)."""
    M, N, K = 3590, 3592, 528
    g = torch.Generator().manual_seed(77)
    qs = [random_fp8_bytes(s, g).cuda().view(torch.float8_e4m3fn) for s in ((M, K), (N, K), (M, K), (N, K))]
    s0, s1 = (torch.rand(M, 1, generator=g) + 0.5 for _ in range(2))
    tiny = 1e-12 / 448
    for r, (a, b) in enumerate([(1e20, 1e-25), (1e-25, 1e20), (1.0, tiny), (tiny, 1.0), (1.0, float("inf")), (float("nan"), 1.0),
                                (1.0, float("nan")), (float("inf"), 1.0), (1e20, 1.0), (tiny, tiny)]):
        s0[r * 131], s1[r * 131] = a, b
    # the casts give such a scale to rows that hold an infinity or a NaN, whose bytes are NaN codes: the whole row of results is NaN
    for q, rows in ((qs[0], (5, 7)), (qs[2], (4, 6))):
        for r in rows:
            q.view(torch.uint8)[r * 131, 9] = 0x7f
    qs[2].view(torch.uint8)[2 * 131] = 0
    qs[0].view(torch.uint8)[3 * 131] = 0
    terms = [(qs[0], qs[1], s0.cuda(), torch.tensor([[0.25]]).cuda()), (qs[2], qs[3], s1.cuda(), torch.tensor([[3.0]]).cuda())]
    got, want = sum_of_products(terms).float().cpu(), one_by_one(terms).float().cpu()
    assert torch.equal(torch.isnan(got), torch.isnan(want)) and torch.equal(torch.isinf(got), torch.isinf(want))
    parts = sum(one_by_one([t]).float().abs().cpu() for t in terms)
    fine = torch.isfinite(want)
    bound = parts * 2.0 ** -7
    # (a sum of cancelling terms in fp32: K * 2^-24 of the largest term that a row can hold)
    floor = torch.maximum(s0 * 0.25, s1 * 3.0) * (448.0 ** 2 * K * K * 2.0 ** -24)
    assert ((got - want).abs()[fine] <= (bound + floor.expand_as(bound))[fine]).all()


@pytest.mark.parametrize("M,N,Ks,algo", [(3590, 3592, (528, 656), 12), (3590, 3592, (528, 1040, 656), 12), (4093, 8184, (512, 528, 1152), 12), (2990, 3592, (528, 656, 784), 25)])
def test_sum_of_products_in_rows_that_no_one_scale_serves(M, N, Ks, algo):
    """Rows in which the products' scales fall or rise by 2^60 and more, once or twice, pass fp32's range on either side or are
    zero or negative, columns in which the coarse product is exactly zero: such rows have the bits of the products added one by
    one, all others those that they have without such rows beside them."""
    from lingua_amd import _lib
    assert _lib.load().l8_gemm_pick(M, N, sum(Ks)) == algo
    g = torch.Generator().manual_seed(M + len(Ks))
    qs = [tuple(random_fp8_bytes((n, K), g).cuda() for n in (M, N)) for K in Ks]
    scales = [torch.rand(M, 1, generator=g) + 0.5 for _ in Ks]
    plain = [s.clone() for s in scales]
    odd = [(1e20, 1.0, 1e-25), (1.0, 2.0 ** -60, 2.0 ** -120), (2.0 ** 45, 1e-12 / 448, 1e-12 / 448 / 4096), (1e-25, 1.0, 1e20), (1e20, 1e-25, 1e20),
           (1e-25, 1e20, 1e-25), (1e35, 1e-5, 1.0), (1e-38, 1e-38, 1e-38), (0.0, 1.0, 1.0), (1.0, 0.0, 0.0), (0.0, 0.0, 0.0), (-1e20, 1.0, 1e-25)]
    rows = [min(i * (M // len(odd)) + 17 * (i % 4), M - 1) for i in range(len(odd) - 1)] + [M - 1]
    for r, values in zip(rows, odd):
        for s, v in zip(scales, values):
            s[r] = v
    qs[0][1][5::37] = 0  # columns in which the first product is zero, and of these every second one in which the second is
    qs[1][1][5::74] = 0
    qs[0][0][rows[0]] = 0

    def terms(sas):
        return [(spread(a, a.shape[1] + 32 * i), b.view(torch.float8_e4m3fn), s.cuda(), torch.tensor([[0.75 + i]]).cuda()) for i, ((a, b), s) in enumerate(zip(qs, sas))]
    got, want, beside = sum_of_products(terms(scales)), one_by_one(terms(scales)), sum_of_products(terms(plain))
    assert torch.equal(got[rows].view(torch.int16), want[rows].view(torch.int16))
    assert torch.isfinite(got[rows[0]]).all()
    got[rows] = 0
    beside[rows] = 0
    assert torch.equal(got.view(torch.int16), beside.view(torch.int16))


def test_sum_of_products_that_one_loop_does_not_serve():
    """Sizes for smaller tiles, reductions too short or too long, a tile configuration asked for: added one by one, the same bits."""
    from lingua_amd import ops
    for M, N, Ks, algo in ((150, 256, (512, 528), 0), (3590, 3592, (512, 496), 0), (2304, 4096, (16384, 512), 0), (3590, 3592, (512, 512), 12)):
        g = torch.Generator().manual_seed(M + N)
        terms = []
        for K in Ks:
            qa, qb = (random_fp8_bytes((n, K), g).cuda().view(torch.float8_e4m3fn) for n in (M, N))
            terms.append((qa, qb, (torch.rand(M, 1, generator=g) + 0.5).cuda(), (torch.rand(1, 1, generator=g) + 0.5).cuda()))
        want = None
        for t in terms:
            want = ops.gemm_nt(*t, algo=algo, out=want, add=want is not None)
        assert torch.equal(ops.gemm_nt_sum(*zip(*terms), algo=algo).view(torch.int16), want.view(torch.int16))


@pytest.mark.parametrize("algo", [0, 1, 2, 3, 11, 15])
def test_k_indexing_with_one_hot_operands(algo):
    # B[n] is one-hot at k = pi(n): C[m,n] = A[m, pi(n)] exactly, for any K (tails included)
    from lingua_amd import ops
    g = torch.Generator().manual_seed(5)
    for (M, N, K) in [(96, 400, 400), (130, 1040, 1040), (64, 2064, 2064), (300, 4096, 4096)]:
        A = torch.randint(-8, 9, (M, K), generator=g).float()
        pi = torch.randperm(K, generator=g)[:N]
        B = torch.zeros(N, K)
        B[torch.arange(N), pi] = 1.0
        one = torch.ones(1, 1)
        out = ops.gemm_nt(fp8(A).cuda(), fp8(B).cuda(), one.cuda(), one.cuda(), algo=algo)
        assert torch.equal(out.cpu().float(), A[:, pi]), (M, N, K)
        # and the mirrored case: one-hot A picks rows of B
        out2 = ops.gemm_nt(fp8(B).cuda(), fp8(A).cuda(), one.cuda(), one.cuda(), algo=algo)
        assert torch.equal(out2.cpu().float(), A[:, pi].t()), (M, N, K)


def random_fp8_bytes(shape, g):
    q = torch.randint(0, 256, shape, generator=g, dtype=torch.int32).to(torch.uint8)
    q[(q & 0x7F) == 0x7F] = 0x38
    return q


@pytest.mark.parametrize("algo", ALGOS)
def test_random_operands_vs_oracle(algo):
    from lingua_amd import ops
    if algo > n_algos():
        pytest.skip("no such tile configuration")
    g = torch.Generator().manual_seed(200 + algo)
    for (M, N, K) in [(384, 320, 512), (100, 72, 80), (513, 260, 1040)]:
        qa, qb = random_fp8_bytes((M, K), g), random_fp8_bytes((N, K), g)
        sa = torch.rand(M, 1, generator=g) + 0.5
        sb = torch.rand(N, 1, generator=g) + 0.5
        bias = (torch.randn(N, generator=g) * 50).to(torch.bfloat16)
        A, B = qa.cuda().view(torch.float8_e4m3fn), qb.cuda().view(torch.float8_e4m3fn)
        for sa_, sb_, b_ in ((sa, sb, None), (sa, sb, bias), (sa, sb[:1], None), (sa[:1], sb[:1], bias)):
            out = ops.gemm_nt(A, B, sa_.cuda(), sb_.cuda(), b_.cuda() if b_ is not None else None, algo=algo)
            want = oracle.gemm_nt(qa, qb, sa_, sb_, b_)
            assert rel_l2(out, want) <= TOL, (algo, M, N, K)


def test_rows_so_far_apart_that_only_the_smaller_tiles_can_address_them():
    """256 rows of A 8 MiB apart pass the 32-bit offsets of a tile, 128 do not: a problem whose choice may fall on taller tiles
    is computed all the same, on the smaller ones.  Integers of magnitude up to 4: the sums are exact."""
    from lingua_amd import _lib, ops
    M, N, K, lda = 130, 16640, 2064, 1 << 23
    g = torch.Generator().manual_seed(3)
    qa = torch.randint(-4, 5, (M, K), generator=g).float().cuda().to(torch.float8_e4m3fn)
    qb = torch.randint(-4, 5, (N, K), generator=g).float().cuda().to(torch.float8_e4m3fn)
    sa, sb = torch.ones(M, 1, device="cuda"), torch.ones(N, 1, device="cuda")
    assert _lib.load().l8_gemm_pick(M, N, K) in (23, 24)
    far = torch.empty_strided((M, K), (lda, 1), dtype=torch.float8_e4m3fn, device="cuda")
    far.view(torch.uint8).copy_(qa.view(torch.uint8))
    assert torch.equal(ops.gemm_nt(far, qb, sa, sb), ops.gemm_nt(qa, qb, sa, sb))


def test_output_leading_dimension_and_unaligned_n():
    from lingua_amd import ops
    g = torch.Generator().manual_seed(9)
    M, N, K = 70, 52, 96
    qa, qb = random_fp8_bytes((M, K), g), random_fp8_bytes((N, K), g)
    sa, sb = torch.ones(M, 1), torch.ones(N, 1)
    buf = torch.full((M, 64), 7.0, dtype=torch.bfloat16, device="cuda")
    out = buf[:, 4:4 + N]
    ops.gemm_nt(qa.cuda().view(torch.float8_e4m3fn), qb.cuda().view(torch.float8_e4m3fn), sa.cuda(), sb.cuda(), out=out)
    want = oracle.gemm_nt(qa, qb, sa, sb)
    assert rel_l2(out, want) <= TOL
    assert (buf[:, :4] == 7.0).all() and (buf[:, 4 + N:] == 7.0).all()  # nothing written outside the view


def test_config1_forward_product_full_vs_oracle():
    from lingua_amd import ops
    x = seeded_bf16((4096, 2048), 1.0, seed=0)
    w = seeded_bf16((2048, 2048), 0.02, seed=1)
    qx, sx, _ = ops.cast_rowwise(x.cuda())
    qw, sw, _ = ops.cast_rowwise(w.cuda())
    out = ops.gemm_nt(qx, qw, sx, sw)
    want = oracle.gemm_nt(qx.cpu().view(torch.uint8), qw.cpu().view(torch.uint8), sx.cpu(), sw.cpu())
    assert rel_l2(out, want) <= TOL


@pytest.mark.parametrize("mnk", [(16384, 11008, 4096), (16384, 4096, 11008), (11008, 4096, 16384)])
def test_7b_shapes_vs_library_matmul_and_oracle_rows(mnk):
    # full size: against torch's fp32 GPU matmul of the dequantised operands (an independent library routine),
    # and a sample of rows against the CPU oracle
    from lingua_amd import ops
    M, N, K = mnk
    g = torch.Generator(device="cuda").manual_seed(M + N)
    a = torch.randn(M, K, generator=g, device="cuda").to(torch.bfloat16)
    b = (torch.randn(N, K, generator=g, device="cuda") * 0.02).to(torch.bfloat16)
    qa, sa, _ = ops.cast_rowwise(a)
    qb, sb, _ = ops.cast_rowwise(b)
    out = ops.gemm_nt(qa, qb, sa, sb)
    torch.backends.cuda.matmul.allow_tf32 = False
    ref = ((qa.float() * sa) @ (qb.float() * sb).t()).to(torch.bfloat16)
    assert rel_l2(out, ref) <= TOL
    rows = torch.arange(0, M, max(1, M // 48), device="cuda")[:48]
    want = oracle.gemm_nt(qa[rows].cpu().view(torch.uint8), qb.cpu().view(torch.uint8), sa[rows].cpu(), sb.cpu())
    assert rel_l2(out[rows], want) <= TOL


# Shapes for which tile configuration 15 shares the K range of the last round's tiles out between workgroups (long K, tile
# count a little above a multiple of the compute units; 256 compute units assumed, on other parts the same shapes
# may run unsplit and the assertions hold all the same): 16 x 26 tiles with 64 K tiles (every XCD splits: 20 tail
# tiles, 12 helpers with one or two pieces each), and 13 x 20 ragged tiles with 48 K tiles and a K tail (four XCDs
# have one tail tile and split it, four have none).
SHAPES_SHARED_K = [(4096, 6656, 8192), (3300, 5096, 6128)]
SHAPES_SHARED_K_RANDOM = SHAPES_SHARED_K + [(11008, 4096, 16384)]  # + a 7B wgrad shape: three pieces per helper


@pytest.mark.parametrize("mnk", SHAPES_SHARED_K)
def test_shared_k_range_exact_and_repeatable(mnk):
    # {-1, 0, 1} operands and power-of-two scales: every partial sum is exact in fp32, so the split product must
    # equal the unsplit one and the true one bit for bit; two calls must agree bit for bit as well
    from lingua_amd import _lib, ops
    M, N, K = mnk
    g = torch.Generator(device="cuda").manual_seed(K)
    A = torch.randint(-1, 2, (M, K), generator=g, device="cuda").float()
    B = torch.randint(-1, 2, (N, K), generator=g, device="cuda").float()
    sa = torch.tensor([2.0 ** (i % 5 - 2) for i in range(M)], device="cuda").reshape(M, 1)
    sb = torch.tensor([2.0 ** (i % 3) for i in range(N)], device="cuda").reshape(N, 1)
    qa, qb = fp8(A), fp8(B)
    out = ops.gemm_nt(qa, qb, sa, sb, algo=ops.GEMM_ALGO_SHARED_K)
    torch.backends.cuda.matmul.allow_tf32 = False
    want = ((A @ B.t()) * sa * sb.t()).to(torch.bfloat16)  # integer sums below 2^24: exact in fp32
    assert torch.equal(out, want)
    again = ops.gemm_nt(qa, qb, sa, sb, algo=ops.GEMM_ALGO_SHARED_K)
    assert torch.equal(out, again)
    # the entry point without a workspace never splits
    plain = torch.empty_like(out)
    code = _lib.load().l8_gemm_nt(qa.data_ptr(), qb.data_ptr(), M, N, K, K, K, sa.data_ptr(), ops.SCALE_ROW, sb.data_ptr(),
                                  ops.SCALE_ROW, None, plain.data_ptr(), N, 0, torch.cuda.current_stream().cuda_stream)
    _lib.check(code, "l8_gemm_nt")
    assert torch.equal(out, plain)


@pytest.mark.parametrize("mnk", SHAPES_SHARED_K_RANDOM)
def test_shared_k_range_random_operands(mnk):
    from lingua_amd import ops
    M, N, K = mnk
    g = torch.Generator().manual_seed(M)
    qa, qb = random_fp8_bytes((M, K), g).cuda(), random_fp8_bytes((N, K), g).cuda()
    sa = (torch.rand(M, 1, generator=g) + 0.5).cuda()
    sb = (torch.rand(1, 1, generator=g) + 0.5).cuda()   # scalar scale on the B side, as in dgrad
    A, B = qa.view(torch.float8_e4m3fn), qb.view(torch.float8_e4m3fn)
    out = ops.gemm_nt(A, B, sa, sb, algo=ops.GEMM_ALGO_SHARED_K)
    torch.backends.cuda.matmul.allow_tf32 = False
    ref = ((A.float() * sa) @ (B.float() * sb).t()).to(torch.bfloat16)
    assert rel_l2(out, ref) <= TOL
    rows = torch.arange(0, M, M // 24, device="cuda")[:24]
    want = oracle.gemm_nt(qa[rows].cpu(), qb.cpu(), sa[rows].cpu(), sb.cpu())
    assert rel_l2(out[rows], want) <= TOL
    assert torch.equal(out, ops.gemm_nt(A, B, sa, sb, algo=ops.GEMM_ALGO_SHARED_K))  # fixed order of the partial sums: repeatable bit for bit


def test_shared_k_range_gives_up_instead_of_hanging():
    # With a wait limit of zero polls an owner never sees its helper's partial sums: its tile must come out as
    # NaN (never as a wrong number), the kernel must still finish, and the next call with the normal limit is right.
    from lingua_amd import _lib, ops
    M, N, K = SHAPES_SHARED_K[0]
    g = torch.Generator(device="cuda").manual_seed(3)
    A = torch.randint(-1, 2, (M, K), generator=g, device="cuda").float()
    B = torch.randint(-1, 2, (N, K), generator=g, device="cuda").float()
    one = torch.ones(1, 1, device="cuda")
    qa, qb = fp8(A), fp8(B)
    want = (A @ B.t()).to(torch.bfloat16)
    lib = _lib.load()
    ops.gemm_nt(qa, qb, one, one, algo=ops.GEMM_ALGO_SHARED_K)   # makes the workspace if this is its first use
    before = ops.shared_k_tiles_given_up()
    _lib.check(lib.l8_gemm_set_wait_limit(0), "l8_gemm_set_wait_limit")
    try:
        out = ops.gemm_nt(qa, qb, one, one, algo=ops.GEMM_ALGO_SHARED_K)
        torch.cuda.synchronize()
    finally:
        _lib.check(lib.l8_gemm_set_wait_limit(1 << 18), "l8_gemm_set_wait_limit")
    bad = torch.isnan(out)
    gave_up = ops.shared_k_tiles_given_up() - before
    assert gave_up == int(bad.reshape(M // 256, 256, N // 256, 256).permute(0, 2, 1, 3).reshape(-1, 256 * 256).any(dim=1).sum())
    assert torch.equal(out[~bad], want[~bad])           # what is not poisoned is right
    if torch.cuda.get_device_properties(0).multi_processor_count == 256:
        tiles = bad.reshape(M // 256, 256, N // 256, 256).permute(0, 2, 1, 3).reshape(-1, 256 * 256)
        n_bad = int(tiles.all(dim=1).sum())
        assert n_bad == int(tiles.any(dim=1).sum())      # whole tiles, nothing partial
        assert n_bad == 8 * 20                           # the 20 tail tiles of each XCD
    assert torch.equal(ops.gemm_nt(qa, qb, one, one, algo=ops.GEMM_ALGO_SHARED_K), want)
    assert ops.shared_k_tiles_given_up() - before == gave_up      # the healthy call adds nothing


# The persistent kernel with a bias, on problems where a workgroup computes several tiles (scales and bias are
# requested afresh per tile while the stores of the tile before are still in flight): ragged edges in both
# directions, a K tail, 17 x 18 and 33 x 34 tiles.
SHAPES_BIAS_PERSISTENT = [(4100, 4360, 1040), (8200, 8456, 1040)]


@pytest.mark.parametrize("algo", [0, 12])
@pytest.mark.parametrize("mnk", SHAPES_BIAS_PERSISTENT)
def test_persistent_kernel_with_bias_exact_integer_operands(algo, mnk):
    from lingua_amd import ops
    M, N, K = mnk
    g = torch.Generator(device="cuda").manual_seed(M + algo)
    A = torch.randint(-1, 2, (M, K), generator=g, device="cuda").float()
    B = torch.randint(-1, 2, (N, K), generator=g, device="cuda").float()
    sa = torch.tensor([2.0 ** (i % 5 - 2) for i in range(M)], device="cuda").reshape(M, 1)
    sb = torch.tensor([2.0 ** (i % 3) for i in range(N)], device="cuda").reshape(N, 1)
    bias = torch.randint(-64, 65, (N,), generator=g, device="cuda").to(torch.bfloat16)  # integers: exact sums
    torch.backends.cuda.matmul.allow_tf32 = False
    prod = A @ B.t()  # integer sums below 2^24: exact in fp32
    for sa_, sb_ in ((sa, sb), (sa[:1], sb[:1]), (sa, sb[:1])):
        out = ops.gemm_nt(fp8(A), fp8(B), sa_, sb_, bias, algo=algo)
        want = (prod * sa_ * sb_.t() + bias.float()).to(torch.bfloat16)
        assert torch.equal(out, want), (algo, mnk, sa_.numel(), sb_.numel())
        # and the same bits as the plain one-workgroup-per-tile kernel
        assert torch.equal(out, ops.gemm_nt(fp8(A), fp8(B), sa_, sb_, bias, algo=5))


@pytest.mark.parametrize("algo", [0, 12])
def test_persistent_kernel_with_bias_random_operands_vs_oracle_rows(algo):
    from lingua_amd import ops
    for (M, N, K) in SHAPES_BIAS_PERSISTENT + [(16384, 4096, 4096)]:
        g = torch.Generator().manual_seed(M + N)
        qa, qb = random_fp8_bytes((M, K), g), random_fp8_bytes((N, K), g)
        sa = torch.rand(M, 1, generator=g) + 0.5
        sb = torch.rand(N, 1, generator=g) + 0.5
        bias = (torch.randn(N, generator=g) * 5e4).to(torch.bfloat16)   # the size of the products: it must show
        A, B = qa.cuda().view(torch.float8_e4m3fn), qb.cuda().view(torch.float8_e4m3fn)
        rows = torch.cat([torch.arange(0, M, max(1, M // 40))[:40], torch.arange(M - 6, M)])
        for sa_, sb_ in ((sa, sb), (sa[:1], sb[:1])):
            out = ops.gemm_nt(A, B, sa_.cuda(), sb_.cuda(), bias.cuda(), algo=algo)
            want = oracle.gemm_nt(qa[rows], qb, sa_[rows] if sa_.numel() == M else sa_, sb_, bias)
            assert rel_l2(out[rows.cuda()], want) <= TOL, (algo, M, N, K)
            plain = ops.gemm_nt(A, B, sa_.cuda(), sb_.cuda(), bias.cuda(), algo=5)
            assert rel_l2(out, plain) <= 1e-4, (algo, M, N, K)  # the whole matrix, against the plain kernel


def _scaled_mm_rowwise(qa, qb, sa, sb, bias=None):
    """The call of lingua/float8.py:65-73 (use_fast_accum=True branch): row-wise scales, bias, bf16 out."""
    return torch._scaled_mm(qa, qb.t(), scale_a=sa.reshape(-1, 1), scale_b=sb.reshape(1, -1), bias=bias,
                            out_dtype=torch.bfloat16, use_fast_accum=True)


@pytest.mark.parametrize("mnk", [(4096, 2048, 2048), (2048, 8192, 2048), (4100, 4368, 1040), (16384, 4096, 4096)])
def test_against_the_scaled_mm_call_the_reference_makes(mnk):
    """`torch._scaled_mm` with row-wise scales is what the reference's matmul() calls (lingua/float8.py:65-73); on this
    GPU it is the vendor library's kernel, an independent implementation on the same matrix instructions.  On the same
    quantised operands the two bf16 results must agree far inside the benchmark's tolerance.  Both deviate from the
    correctly rounded product in about 1 % of the elements, K = 128 or K = 16384 alike: the fp8 matrix instruction sums
    its 64 products with roughly 12 bits below the largest of them, which no kernel above it can change -- that, not
    the order of accumulation, is why rel-L2 against the fp32 oracle sits near 2e-4 on every shape."""
    from lingua_amd import ops
    M, N, K = mnk
    x = seeded_bf16((M, K), 1.0, seed=M)
    w = seeded_bf16((N, K), 0.02, seed=N + 1)
    bias = seeded_bf16((N,), 1.0, seed=3).cuda()
    qa, sa, _ = ops.cast_rowwise(x.cuda())
    qb, sb, _ = ops.cast_rowwise(w.cuda())
    try:
        ref = _scaled_mm_rowwise(qa, qb, sa, sb)
        ref_b = _scaled_mm_rowwise(qa, qb, sa, sb, bias)
    except (RuntimeError, NotImplementedError) as e:   # a PyTorch build without row-wise scaling on this GPU
        pytest.skip(f"torch._scaled_mm with row-wise scales is not available here: {e}")
    for algo in (0, 5):
        out = ops.gemm_nt(qa, qb, sa, sb, algo=algo)
        assert rel_l2(out, ref) <= 1e-4, (algo, mnk)
        assert (out != ref).float().mean().item() <= 5e-4, (algo, mnk)   # measured: 5e-6 of the elements
        out_b = ops.gemm_nt(qa, qb, sa, sb, bias, algo=algo)
        assert rel_l2(out_b, ref_b) <= 1e-4, (algo, mnk)
    # the deviation both share: against the fp32 oracle on a sample of rows
    rows = torch.arange(0, M, max(1, M // 32))[:32]
    want = oracle.gemm_nt(qa[rows.cuda()].cpu().view(torch.uint8), qb.cpu().view(torch.uint8), sa[rows.cuda()].cpu(), sb.cpu())
    assert rel_l2(ref[rows.cuda()], want) <= TOL and rel_l2(out[rows.cuda()], want) <= TOL


@pytest.mark.parametrize("M,extra,K", [(1, 16, 2048), (8, 21, 3072), (9, 5, 16), (16, 16, 4096), (17, 40, 272), (32, 1, 9008), (33, 16, 1040),
                                       (48, 37, 2064), (49, 16, 128), (64, 100, 4112), (64, 16, 9008)])
@pytest.mark.parametrize("mode", ["plain", "bias", "add"])
def test_two_tiles_of_weight_rows_per_workgroup(M, extra, K, mode):
    """Just beyond one tile of 16 weight rows per compute unit, where the skinny kernels take 32 rows per workgroup: bit by bit
    what they give for the two halves of the weight (16 rows per workgroup), the last workgroup short of rows or not."""
    from lingua_amd import ops
    g = torch.Generator().manual_seed(M * K + extra)
    N = 16 * torch.cuda.get_device_properties(0).multi_processor_count + extra
    half = N // 2 // 16 * 16
    qa, qb = (torch.randint(-8, 9, (r, K), generator=g).float().cuda().to(torch.float8_e4m3fn) for r in (M, N))
    sa, sb = (torch.rand(r, 1, generator=g).cuda() + 0.5 for r in (M, N))
    bias = torch.randn(N, generator=g).bfloat16().cuda() if mode == "bias" else None
    out = torch.randn(M, N, generator=g).bfloat16().cuda()
    parts = [out[:, :half].contiguous(), out[:, half:].contiguous()]
    y = ops.gemm_nt(qa, qb, sa, sb, bias, algo=17, out=out, add=mode == "add")
    for part, rows in zip(parts, (slice(0, half), slice(half, N))):
        want = ops.gemm_nt(qa, qb[rows], sa, sb[rows], bias[rows].contiguous() if bias is not None else None, algo=17, out=part, add=mode == "add")
        assert torch.equal(y[:, rows], want)
    if mode == "plain":   # products of integers up to 8 add up exactly in fp32
        want = qa.double() @ qb.double().t() * sa.double() * sb.double().t()
        assert bool(((y.double() - want).abs() <= want.abs() * (2.0 ** -8 + 2.0 ** -20)).all())


@pytest.mark.parametrize("K", [16, 128, 144, 256, 400, 1152])
@pytest.mark.parametrize("with_bias,scalar", [(False, False), (False, True), (True, False)])
def test_three_quarter_tiles_carry_their_fragments(K, with_bias, scalar):
    """Tiles of 192 rows (22 x 17 of them here, the last row of tiles short): one to nine K tiles, one or two tiles per workgroup."""
    test_persistent_kernel_carries_its_fragments_from_tile_to_tile(25, K, with_bias, scalar)


@pytest.mark.parametrize("M,N,K", [(1, 8, 16), (95, 256, 128), (97, 264, 144), (192, 128, 4096), (193, 520, 272), (575, 1000, 528)])
def test_three_quarter_tiles_at_their_edges(M, N, K):
    """Rows around a wave's 96 and a tile's 192, columns off 256, a C with rows apart, and a sum added to C: exact integers."""
    from lingua_amd import ops
    g = torch.Generator().manual_seed(M + N)
    A, B = (torch.randint(-1, 2, (n, K), generator=g).float() for n in (M, N))
    sa = torch.tensor([2.0 ** (i % 5 - 2) for i in range(M)]).reshape(M, 1)
    sb = torch.tensor([2.0 ** (i % 3) for i in range(N)]).reshape(N, 1)
    want = ((A.double() @ B.double().t()) * sa.double() * sb.double().t()).to(torch.bfloat16)
    for add in (False, True):
        wide = torch.full((M, N + 8), 1.0, dtype=torch.bfloat16, device="cuda")
        ops.gemm_nt(fp8(A).cuda(), fp8(B).cuda(), sa.cuda(), sb.cuda(), algo=25, out=wide[:, :N], add=add)
        assert torch.equal(wide[:, :N].cpu(), (want.float() + 1.0).to(torch.bfloat16) if add else want)
        assert bool((wide[:, N:] == 1.0).all())


@pytest.mark.parametrize("Ks", [(512, 512), (528, 1152, 656)])
def test_sum_of_products_on_three_quarter_tiles(Ks):
    """As on whole tiles: exact sums, one rounding, whichever product's scale they are counted in."""
    from lingua_amd import _lib, ops
    M, N = 2990, 3592
    assert _lib.load().l8_gemm_pick(M, N, sum(Ks)) == 25
    g = torch.Generator().manual_seed(len(Ks))
    terms, want = [], 0
    for i, K in enumerate(Ks):
        A, B = (torch.randint(-1, 2, (n, K), generator=g).float().cuda() for n in (M, N))
        sa = torch.tensor([2.0 ** ((r * (i + 3)) % 5 - 2) for r in range(M)]).reshape(M, 1).cuda()
        sb = torch.tensor([[2.0 ** (1 - i)]]).cuda()
        want = want + (A.double() @ B.double().t()) * sa.double() * sb.double()
        terms.append((fp8(A), fp8(B), sa, sb))
    got = ops.gemm_nt_sum(*zip(*terms))
    assert torch.equal(got.view(torch.int16), want.float().to(torch.bfloat16).view(torch.int16))


@pytest.mark.parametrize("K", [16, 272, 1152])
@pytest.mark.parametrize("rows,N,tile_rows", [((2000, 500, 500), 3600, 192), ((1930, 960), 3600, 192), ((200, 2400, 390), 3600, 256), ((200, 2400, 390), 3328, 192)])
def test_list_of_products_on_three_quarter_tiles(rows, N, tile_rows, K):
    """Products with one B whose tiles of 192 rows start where the one before ends, the last tile of each short, the first one
    barely longer than a tile; and a list that these would give a second round.  Exact integers."""
    import struct
    from lingua_amd import _lib, ops
    if torch.cuda.get_device_properties(0).multi_processor_count == 256:
        parts = struct.pack(f"{4 * len(rows)}q", *(v for m in rows for v in (0, m, 0, 0)))
        assert _lib.load().l8_gemm_multi_pays(parts, len(rows), N, K) and _lib.load().l8_gemm_multi_tile_rows(parts, len(rows), N) == tile_rows
    g = torch.Generator().manual_seed(K)
    B = torch.randint(-1, 2, (N, K), generator=g).float().cuda()
    sb = torch.tensor([2.0 ** (i % 3) for i in range(N)]).reshape(N, 1).cuda()
    As = [torch.randint(-1, 2, (m, K), generator=g).float().cuda() for m in rows]
    sas = [torch.tensor([2.0 ** (i % 5 - 2) for i in range(m)]).reshape(m, 1).cuda() for m in rows]
    got = ops.gemm_nt_multi([fp8(A) for A in As], fp8(B), sas, sb)
    for A, sa, y in zip(As, sas, got):
        assert torch.equal(y, ((A.double() @ B.double().t()) * sa.double() * sb.double().t()).to(torch.bfloat16))


@pytest.mark.parametrize("algo", [0, 25])
def test_outputs_that_three_quarter_tiles_cannot_store(algo):
    """N off 8 columns, and a C whose rows start off 16 bytes: computed by the plain kernel.  Exact integers."""
    from lingua_amd import ops
    g = torch.Generator().manual_seed(9)
    for M, N, pad in ((2990, 3593, 0), (2990, 3592, 4)):
        A, B = (torch.randint(-1, 2, (n, 144), generator=g).float().cuda() for n in (M, N))
        one = torch.ones(1, 1, device="cuda")
        wide = torch.zeros((M, N + pad), dtype=torch.bfloat16, device="cuda")
        ops.gemm_nt(fp8(A), fp8(B), one, one, algo=algo, out=wide[:, :N])
        assert torch.equal(wide[:, :N].float(), A @ B.t()) and not bool(wide[:, N:].any())
