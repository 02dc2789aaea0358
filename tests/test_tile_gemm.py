"""Dense products of long steps on wave-tiled weights (csrc/tile_gemm.hip, ops.linear_tile / linear_long / tile_plan)."""
import random

import pytest
import torch

from kafka_llm_service_amd import ops


def test_plans_are_launches():
    """Every plan is one that the kernel takes: at least two units of 64 of K a split, whole gate, up pairs a wave, slabs within
    their bound; what it cannot take has no plan."""
    rng = random.Random(3)
    for _ in range(300):
        M, N, K = rng.randint(1, 9000), 32 * rng.randint(1, 900), 64 * rng.randint(2, 230)
        form = rng.choice(["slabs", "bf16", "glu", "relu2"])
        plan = ops.tile_plan(M, N, K, form, library=False)
        if form == "glu" and N % 64:
            assert plan is None
            continue
        mt, nt, s = plan
        assert (mt, nt) in ops.TILES and K // 64 >= 2 * s and (form != "glu" or nt % 4 == 0)
        assert s == 1 or form != "relu2" and 4 * s * M * N <= ops.TILE_SLAB_BYTES
    assert ops.tile_plan(300, 4100, 4096) is None and ops.tile_plan(300, 4096, 64) is None and ops.tile_plan(300, 4096, 4112) is None
    assert ops.tile_plan(0, 4096, 4096) is None and ops.tile_plan(300, 32800, 65536, library=False) is None   # 4 GB of weights
    for M, N, form, taken in ((2561, 6176, "bf16", True), (8448, 6176, "slabs", True), (8449, 6176, "bf16", False),   # ragged columns
                              (2561, 6144, "bf16", True), (5600, 9216, "bf16", False), (2700, 28672, "bf16", False),   # whole ones: a fifth less
                              (4096, 4064, "bf16", False), (2816, 5920, "bf16", True),      # one round of 256 x 256 tiles, and a bit more
                              (2561, 28672, "glu", True), (3600, 28672, "glu", True), (3601, 28672, "glu", False),
                              (2561, 14336, "relu2", True), (3601, 14336, "relu2", False), (2816, 11776, "relu2", False),
                              (2816, 11776, "glu", False)):                             # two rounds
        assert (ops.tile_plan(M, N, 4096, form) is not None) == taken, (M, N, form)
    assert ops.tile_plan(300, 28672, 4096) is None and ops.tile_plan(300, 28672, 4096, "glu") is not None


def test_lengths_share_a_search():
    """A prompt of a length that had none before asks for a plan once per 64 rows, not once per length, and gets the plan that its own length
    would or one behind by no more than the rows between."""
    ops._tile_best.cache_clear()
    for M in range(1985, 2049):
        for form in ("slabs", "glu"):
            assert ops.tile_plan(M, 6144, 1984, form, library=False) is not None
    assert ops._tile_best.cache_info().misses == 2
    rng = random.Random(5)
    for _ in range(400):
        M, N, K = rng.randint(129, 9000), 64 * rng.randint(1, 450), 64 * rng.randint(2, 230)
        form = rng.choice(["slabs", "bf16", "glu", "relu2"])
        own, up = ops._tile_best(M, N, K, form), ops._tile_best(-(-M // 64) * 64, N, K, form)
        assert own[0] <= up[0]
        if own[1] != up[1]:
            assert up[0] <= own[0] * (1 + 64 / M)


def test_long_products_on_the_cpu():
    """Without a GPU linear_long is the plain product, from either weight, whatever the strides of x."""
    w = torch.randn(96, 128)
    wt = ops.tile_weight(w)
    for x in (torch.randn(150, 128), torch.randn(128, 150).t(), torch.randn(150, 256)[:, ::2], torch.randn(1, 128).expand(150, 128)):
        for y in (ops.linear_long(x, w, wt, slabs=True), ops.linear_long(x, None, wt), ops.linear_long(x, w, None)):
            torch.testing.assert_close(y, x @ w.t())
    assert ops.linear_relu2_long(torch.randn(150, 128), wt) is None
    assert ops.linear_glu_long(torch.randn(150, 128), ops.tile_weight(torch.randn(128, 128), glu=True)) is None


def _gelu(z):
    return torch.nn.functional.gelu(z, approximate="tanh")


def _close(got, want, K):
    # sums of K terms of size ~ 1 / sqrt(K) in fp32 (errors of 1e-6 of them) rounded to bf16, 2^-9 of a value
    assert ((got.float() - want).abs() <= 2 ** -8 * want.abs() + 1e-3).all()


@pytest.mark.gpu
@pytest.mark.parametrize("mt,nt", sorted(ops.TILES))
def test_tiles_against_fp32(mt, nt):
    """Rows and columns that end inside, at and past a tile, one row, one 32-column tile, more than a group of row tiles; K of two and
    three units a split (four and six stages; the ring holds four) and of uneven splits; wide rows of x; both outputs of either order
    of weights. Rows of a padded output stay as they were."""
    g = torch.Generator().manual_seed(mt * 10 + nt)
    bm, bn = 32 * mt, 32 * nt
    for M, N, K, s in ((1, 32, 128, 1), (bm - 1, bn, 192, 1), (bm, bn + 32, 256, 2), (bm + 1, 3 * bn - 32, 448, 3), (2100, 64, 320, 2),
                       (200, 2 * bn + 64, 1088, 8), (65, 192, 1024, 8)):
        x = torch.randn(M, K + 24, generator=g).to(torch.bfloat16).cuda()[:, 8:8 + K]
        w = (torch.randn(N, K, generator=g) / K ** 0.5).to(torch.bfloat16).cuda()
        want = x.float() @ w.float().t()
        wt = ops.tile_weight(w)
        assert ops.tile_ok(x, wt)
        ext = ops.ext()
        y = torch.full((M + 1, N + 8), 7.0, dtype=torch.bfloat16, device="cuda")
        ext.tile_gemm(x, wt, y[:M, :N], None, mt, nt, 1, False)
        _close(y[:M, :N], want, K)
        assert (y[M:] == 7).all() and (y[:, N:] == 7).all()
        _close(ops.linear_tile(x, wt, (mt, nt, 1), relu2=True), want.relu() ** 2, K)
        if s > 1:
            p = ops.linear_tile(x, wt, (mt, nt, s))
            assert p.shape == (s, M, N) and ((p.sum(0) - want).abs() <= 1e-4).all()
        if N % 64 == 0 and nt % 4 == 0:
            gt, F = ops.tile_weight(w, glu=True), N // 2
            _close(ops.linear_tile(x, gt, (mt, nt, 1), glu=True), torch.nn.functional.silu(want[:, :F]) * want[:, F:], K)
            _close(ops.linear_tile(x, gt, (mt, nt, 1), glu=True, act="gelu"), _gelu(want[:, :F]) * want[:, F:], K)
            if s > 1:
                assert ((ops.linear_tile(x, gt, (mt, nt, s), glu=True).sum(0) - want).abs() <= 1e-4).all()


@pytest.mark.gpu
@pytest.mark.parametrize("M", [1, 31, 64, 65, 128, 129, 300])
def test_gelu_gated_products(M):
    """The same activation in the weight-streaming kernel's epilogue (one split), over its slabs, and of steps beyond it."""
    g = torch.Generator().manual_seed(M)
    for N, K in ((256, 256), (96 * 64, 512), (448 * 64, 256)):
        w = (torch.randn(N, K, generator=g) / K ** 0.5).to(torch.bfloat16).cuda()
        x, wt, F = (torch.randn(M, K, generator=g) * 2).to(torch.bfloat16).cuda(), ops.tile_weight(w, glu=True), N // 2
        want = x.float() @ w.float().t()
        want = _gelu(want[:, :F]) * want[:, F:]
        if M <= ops.STREAM_MAX_M:
            _close(ops.linear_glu(x, wt, act="gelu"), want, K)
            _close(ops.linear_glu(x, wt, 1, act="gelu"), want, K)
        a = ops.linear_glu_long(x, wt, act="gelu")
        if a is not None:
            _close(a, want, K)
        _close(ops.silu_mul((x.float() @ w.float().t()).expand(2, M, N).contiguous() / 2, act="gelu"), want, K)


@pytest.mark.gpu
@pytest.mark.parametrize("mt,nt", [t for t in sorted(ops.TILES) if t[1] % 4])
def test_gates_need_whole_pairs_in_a_wave(mt, nt):
    """Tiles whose waves hold three 32-column tiles cannot activate gate, up pairs: refused; their slabs are in gate | up order."""
    x, w = torch.randn(65, 128).to(torch.bfloat16).cuda(), torch.randn(384, 128).to(torch.bfloat16).cuda() / 12
    wt = ops.tile_weight(w, glu=True)
    for act in ("silu", "gelu"):
        with pytest.raises(RuntimeError):
            ops.linear_tile(x, wt, (mt, nt, 1), glu=True, act=act)
    p = torch.empty(1, 65, 384, device="cuda")
    ops.ext().tile_gemm(x, wt, None, p, mt, nt, 1, True)
    assert ((p[0] - x.float() @ w.float().t()).abs() <= 1e-4).all()


@pytest.mark.gpu
def test_relu_squared_of_what_is_not_finite():
    """NaN stays, minus infinity is zero, plus infinity infinite."""
    x = torch.ones(200, 128, dtype=torch.bfloat16, device="cuda")
    x[0, 0], x[1, 0], x[2, 0] = float("nan"), float("inf"), float("-inf")
    y = ops.linear_tile(x, ops.tile_weight(torch.ones(64, 128, dtype=torch.bfloat16, device="cuda")), (4, 4, 1), relu2=True)
    assert y[0].isnan().all() and (y[1] == float("inf")).all() and (y[2] == 0).all() and (y[3:] == 128 ** 2).all()


@pytest.mark.gpu
def test_long_products_by_their_plans():
    """linear_long, linear_relu2_long and linear_glu_long over sizes of every route (tiles with and without splits, the library) and forms of x that the
    kernel leaves to the library (odd strides, a shifted start)."""
    g = torch.Generator().manual_seed(0)
    for M, N, K in ((131, 2048, 2048), (300, 4096, 1024), (700, 96, 4096), (1300, 6176, 512), (257, 24608, 128), (3000, 1024, 256),
                    (2561, 6176, 256), (2600, 6144, 512)):
        w = (torch.randn(N, K, generator=g) / K ** 0.5).to(torch.bfloat16).cuda()
        wt = ops.tile_weight(w)
        base = torch.randn(M, K + 16, generator=g).to(torch.bfloat16).cuda()
        for x in (base[:, :K].contiguous(), base[:, 8:8 + K], base[:, 1:1 + K], base[:, :K].t().contiguous().t()):
            want = x.float() @ w.float().t()
            for y in (ops.linear_long(x, w, wt), ops.linear_long(x, None, wt), ops.linear_long(x, w, wt, slabs=True)):
                _close(y.sum(0) if ops.is_slab(y) else y, want, K)
            a = ops.linear_relu2_long(x, wt)
            if a is not None:
                _close(a, want.relu() ** 2, K)
            if N % 64 == 0:
                a = ops.linear_glu_long(x, ops.tile_weight(w, glu=True))
                if a is not None:
                    _close(a, torch.nn.functional.silu(want[:, :N // 2]) * want[:, N // 2:], K)


def test_long_plans_take_more_from_the_library():
    """Past one round of the library's tiles a product with an activation is the tile kernel's, a plain one where the figures say so; all that
    tile_plan takes stays as it is, so do shapes that the kernel does not take and products within a round."""
    rng = random.Random(11)
    for _ in range(400):
        M, N, K = rng.randint(129, 12000), 32 * rng.randint(1, 900), 64 * rng.randint(2, 230)
        form = rng.choice(["slabs", "bf16", "glu", "relu2"])
        had, plan, own = ops.tile_plan(M, N, K, form), ops.long_plan(M, N, K, form), ops.tile_plan(M, N, K, form, library=False)
        assert ops.long_plan(M, N, K, form, library=False) == own and plan in (had, own) and (had is None or plan == had)
        past = -(-M // 256) * -(-N // 256) > 256
        if form in ("glu", "relu2") and M > 768 and past:
            assert plan == own
        if had is None and (M <= 768 or not past or form in ("slabs", "bf16") and (M <= 1024 or ops.dense_cut(M, N, K))):
            assert plan is None
    assert ops.long_plan(4099, 28672, 4096, "glu") is not None and ops.long_plan(4099, 4096, 4096) is None
    assert ops.long_plan(5600, 9216, 4096) is not None and ops.long_plan(5600, 9216 + 16, 4096) is None


def test_plans_of_deep_loops_and_of_full_rounds():
    """Loops of 6144 and more of K on tiles of 128 columns are priced as they run, so that two splits on 256 columns take them; plain products whose library
    tiles fill whole rounds are the library's, one row tile less is not."""
    for M, N, K, form in ((1100, 4096, 14336, "bf16"), (1270, 4096, 14336, "bf16"), (1560, 4096, 14336, "slabs"), (1790, 4096, 14336, "slabs"),
                          (2227, 2048, 7168, "slabs")):
        assert ops.long_plan(M, N, K, form)[1:] == (8, 2), (M, N, K)
    assert ops.long_plan(1100, 4096, 4096)[2] == 1 and ops.long_plan(1700, 4096, 4096, "slabs")[2] == 1
    for M, N, K in ((8192, 4096, 14336), (7990, 14336, 2048), (8192, 6144, 4096), (8192, 28672, 4096), (4000, 28672, 4096)):
        assert ops.long_plan(M, N, K) is None and ops.long_plan(M, N, K, library=False) is not None and ops.long_plan(M, N, K, "glu") is not None
    assert ops.long_plan(5600, 9216, 4096) is not None and ops.long_plan(7900, 28672, 4096) is not None


@pytest.mark.gpu
@pytest.mark.parametrize("mt,nt", sorted(ops.TILES))
def test_low_last_row_tiles_and_short_loops(mt, nt):
    """A last row tile on both sides of the low one's height, behind one and several whole ones, columns past the last tile, K from two units
    (fewer than the ring holds) to more than twice what it holds, even and uneven splits; rows beyond stay as they were."""
    g = torch.Generator().manual_seed(mt * 100 + nt)
    bm = 32 * mt
    for M, N, K, s in ((bm + 1, 64, 128, 1), (bm + 63, 32 * nt + 32, 192, 1), (2 * bm + 64, 96, 256, 2), (2 * bm + 65, 64, 320, 1), (bm + 64, 64, 384, 3),
                       (9 * bm + 3, 32, 448, 1), (bm + 17, 64 * nt, 640, 2), (bm + 33, 64, 704, 1), (bm + 2, 128, 832, 5)):
        x = torch.randn(M, K, generator=g).to(torch.bfloat16).cuda()
        w = (torch.randn(N, K, generator=g) / K ** 0.5).to(torch.bfloat16).cuda()
        want, wt = x.float() @ w.float().t(), ops.tile_weight(w)
        y = torch.full((M + 70, N), 7.0, dtype=torch.bfloat16, device="cuda")
        ops.ext().tile_gemm(x, wt, y[:M], None, mt, nt, 1, False)
        _close(y[:M], want, K)
        assert (y[M:] == 7).all()
        if s > 1:
            assert ((ops.linear_tile(x, wt, (mt, nt, s)).sum(0) - want).abs() <= 1e-4).all()


@pytest.mark.gpu
@pytest.mark.parametrize("act", ["silu", "gelu"])
def test_gates_against_64_bits(act):
    """Gates over all that the exponential has normal numbers for, and far past it on both sides, of the element-wise launch and of the products' epilogues
    (each sum is one term, so exact). The result is bf16 (8 bits: half a unit is up to 2^-8 of it), the gate's fp32 error at most 88 times a few 2^-24 (the
    argument of the gelu form); beyond s = -88.7 the result may be 0, as may what is not a normal number."""
    v = torch.arange(-90, 90.25, 0.25)
    v = torch.cat([v, v / 8, torch.tensor([-3e38, -1e30, -1e4, -100.0, -10.06, 100.0, 1e4, 3e38, -0.0])]).to(torch.bfloat16)
    g = v.double()
    s = g if act == "silu" else 1.5957691216057308 * (g + 0.044715 * g ** 3)
    want = torch.where(s < -700, torch.zeros_like(g), g / (1 + torch.exp(-s.clamp(min=-700))))
    bound = (2 ** -8 + 2 ** -15) * want.abs() + torch.where((s < -88.7) & (s > -700), g.abs() * 3e-39, torch.zeros_like(g)) + 1.2e-38

    def check(y):
        off = (y.cpu().double() - want).abs() > bound
        assert not off.any(), (g[off], want[off], y.cpu()[off])

    n = len(v)
    x = torch.ones(n, 16, dtype=torch.bfloat16)
    x[:, :8] = v[:, None]
    check(ops.silu_mul(x.cuda(), act=act)[:, 3])
    check(ops.silu_mul(x.float().cuda().view(1, n, 16), act=act)[:, 3])
    edge = torch.tensor([[float("inf")] * 8 + [1.0] * 8, [-float("inf")] * 8 + [1.0] * 8, [float("nan")] * 8 + [1.0] * 8]).to(torch.bfloat16).cuda()
    y = ops.silu_mul(edge, act=act)
    assert (y[0] == float("inf")).all() and y[1:].isnan().all()
    K, F = 256, 128
    w, x = torch.zeros(2 * F, K), torch.zeros(n, K, dtype=torch.bfloat16)
    w[:F, 0] = w[F:, 1] = 1
    x[:, 0], x[:, 1] = v, 1
    wt, x = ops.tile_weight(w.to(torch.bfloat16).cuda(), glu=True), x.cuda()
    for mt, nt in ((4, 4), (8, 8)):
        check(ops.linear_tile(x, wt, (mt, nt, 1), glu=True, act=act)[:, 5])
    rows = ops.STREAM_MAX_M
    check(torch.cat([ops.linear_glu(x[i:i + rows], wt, 1, act=act) for i in range(0, n, rows)])[:, 5])


@pytest.mark.gpu
@pytest.mark.parametrize("M,N,K", [(128, 96 * 128, 2048), (97, 128 * 128 - 32, 2112), (130, 48 * 128, 2048), (257, 85 * 128, 2176), (300, 32 * 128 - 64, 2048),
                                   (2048, 16 * 128, 2048), (129, 128 * 128, 2368), (2049, 16 * 128, 2048), (257, 31 * 128, 2048), (500, 24 * 128, 1984)])
def test_small_tiles_alone_on_a_cu(M, N, K):
    """128 x 128 tiles by themselves on a CU and, beyond the rule's lines, two to a CU: one row tile, ragged rows and columns, odd numbers of units."""
    g = torch.Generator().manual_seed(M + N + K)
    x = torch.randn(M, K, generator=g).to(torch.bfloat16).cuda()
    w = (torch.randn(N, K, generator=g) / K ** 0.5).to(torch.bfloat16).cuda()
    y = torch.full((M + 30, N), 7.0, dtype=torch.bfloat16, device="cuda")
    ops.ext().tile_gemm(x, ops.tile_weight(w), y[:M], None, 4, 4, 1, False)
    _close(y[:M], x.float() @ w.float().t(), K)
    assert (y[M:] == 7).all()
