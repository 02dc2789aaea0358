"""Small products (csrc/small_gemm.hip, ops.linear_small, hybrid.linear_f32, the heads' products of latent attention)."""
import pytest
import torch

from kafka_llm_service_amd import ops
from kafka_llm_service_amd.models.budurax import head_product
from kafka_llm_service_amd.ops import hybrid as hops


def _close(got, want):
    # sums of K terms of size ~ 1 / sqrt(K) in fp32 (errors of 1e-6 of them) rounded to bf16, 2^-9 of a value
    assert ((got.float() - want).abs() <= 2 ** -8 * want.abs() + 1e-4).all()


def test_on_the_cpu():
    """Without a GPU the plain products, whatever the strides."""
    x, w = torch.randn(5, 24)[:, ::2], torch.randn(7, 12)
    torch.testing.assert_close(ops.linear_small(x, w), x @ w.t())
    a, h = torch.randn(6, 3, 8), torch.randn(3, 10, 8)
    for n in (h, None):
        torch.testing.assert_close(head_product(a.transpose(0, 1), n, h.transpose(1, 2)), torch.einsum("tha,hna->htn", a, h))


@pytest.mark.gpu
@pytest.mark.parametrize("K", [8, 16, 40, 64, 128, 256, 264, 1016, 1024, 1032, 4096])
def test_against_fp32(K):
    """Rows and columns that end inside, at and past the 16 of a tile; K that ends inside a step of 32, of one step and of shares that
    differ by one; rows and results in wider buffers (what lies beside them stays); fp32 results and their bias."""
    g = torch.Generator().manual_seed(K)
    for M, N in ((1, 4), (15, 8), (16, 16), (17, 64), (33, 68), (200, 260)):
        x = torch.randn(M, K + 16, generator=g).to(torch.bfloat16).cuda()[:, 8:8 + K]
        w = (torch.randn(N, K + 8, generator=g) / K ** 0.5).to(torch.bfloat16).cuda()[:, :K]
        b = torch.randn(N, generator=g).cuda()
        want = x.float() @ w.float().t()
        y = torch.full((M + 1, N + 4), 7.0, dtype=torch.bfloat16, device="cuda")
        ops.ext().small_gemm(x, w, y[:M, :N])
        _close(y[:M, :N], want)
        assert (y[M:] == 7).all() and (y[:, N:] == 7).all()
        f = torch.empty(M, N, device="cuda")
        ops.ext().small_gemm(x, w, f)
        assert ((f - want).abs() <= 2e-5).all()
        ops.ext().small_gemm(x, w, f, b)
        assert ((f - want - b).abs() <= 2e-5).all()
        assert ((hops.linear_f32(x, w.contiguous(), b) - want - b).abs() <= 2e-5).all()
        o = torch.randn(N + 1, generator=g).cuda()[1:]      # (a bias that starts between two 16-byte pieces)
        assert ((hops.linear_f32(x, w.contiguous(), o) - want - o).abs() <= 2e-5).all()
        _close(ops.linear_small(x, w), want)


@pytest.mark.gpu
@pytest.mark.parametrize("K", [1032, 2056])
def test_biases_of_other_forms(K):
    """Rows that the kernel for few weight rows does not take (K in steps of 8) have taken any bias that adds to the result: bf16, every second
    element, one for all columns, one a row."""
    g = torch.Generator().manual_seed(K)
    for M, N in ((3, 16), (40, 64)):
        x = torch.randn(M, K, generator=g).to(torch.bfloat16).cuda()
        w = (torch.randn(N, K, generator=g) / K ** 0.5).to(torch.bfloat16).cuda()
        want, b = x.float() @ w.float().t(), torch.randn(2 * N, generator=g).cuda()
        for bias in (b[:N].to(torch.bfloat16), b[::2], b[:1], b[:N].expand(M, N), b[:M, None] if M <= 2 * N else b[:1, None]):
            assert ((hops.linear_f32(x, w, bias) - want - bias).abs() <= 2e-5).all()


@pytest.mark.gpu
def test_rows_beyond_and_forms_of_the_library():
    """One row past each limit, and operands that the kernel does not take (odd columns, odd strides, a shifted start)."""
    g = torch.Generator().manual_seed(1)
    for N, K in ((64, 1024), (68, 1024), (32, 1024), (16, 1024), (32, 16), (512, 128)):
        n = ops.small_rows(N, K)
        for M in (n, n + 1):
            x, w = torch.randn(max(M, 1), K, generator=g).to(torch.bfloat16).cuda(), (torch.randn(N, K, generator=g) / K ** 0.5).to(torch.bfloat16).cuda()
            assert ops.small_ok(x, w, n) == (0 < M <= n)
            _close(ops.linear_small(x, w), x.float() @ w.float().t())
    x = torch.randn(20, 72, generator=g).to(torch.bfloat16).cuda()
    w = torch.randn(18, 64, generator=g).to(torch.bfloat16).cuda() / 8
    for a, b in ((x[:, :64], w), (x[:, 1:65], w[:16]), (x[:, :64].t().contiguous().t(), w[:16]), (x[:, :60], w[:16, :60])):
        assert not ops.small_ok(a, b, 4096)
        _close(ops.linear_small(a, b), a.float() @ b.float().t())


@pytest.mark.gpu
def test_extents_beyond_the_kernels_grid():
    """Columns, depth and heads that its launch refuses, and the last ones that it takes: the library's or the kernel's, the same product."""
    for M, N, K in ((2, 4, 1 << 20), (2, 4, (1 << 20) - 8), (2, 1 << 20, 8), (2, 1 << 19, 8), (2, (1 << 19) - 4, 8)):
        x, w = torch.ones(M, K, dtype=torch.bfloat16, device="cuda"), torch.ones(N, K, dtype=torch.bfloat16, device="cuda")
        w[-1] = 2
        y = ops.linear_small(x, w).float()
        assert (y[:, :-1] == x[:1].float().sum().to(torch.bfloat16).float()).all() and (y[:, -1] == 2 * y[:, 0]).all()
    for H in ((1 << 16) - 1, 1 << 16):
        x, w = torch.ones(H, 1, 8, dtype=torch.bfloat16, device="cuda"), torch.ones(H, 4, 8, dtype=torch.bfloat16, device="cuda")
        w[-1] = 2
        y = head_product(x, w, w.transpose(1, 2).contiguous())
        assert (y[:-1] == 8).all() and (y[-1] == 16).all()


@pytest.mark.gpu
@pytest.mark.parametrize("n", [1, 16, 63, 64, 65])
def test_heads(n):
    """Products per head into the head's columns of a wider row and into rows of their own, queries as slices of a fused row."""
    g = torch.Generator().manual_seed(n)
    H, D, R = 6, 128, 192
    q = torch.randn(n, H, D + 64, generator=g).to(torch.bfloat16).cuda()[:, :, :D]
    uk = (torch.randn(H, D, R, generator=g) / D ** 0.5).to(torch.bfloat16).cuda()
    want = torch.stack([q[:, h].float() @ uk[h].float() for h in range(H)])
    _close(head_product(q.transpose(0, 1), uk.transpose(1, 2).contiguous(), uk), want)
    o = torch.randn(H, n, R, generator=g).to(torch.bfloat16).cuda()
    uv = (torch.randn(H, D, R, generator=g) / R ** 0.5).to(torch.bfloat16).cuda()
    ao = torch.empty(n, H * D, dtype=torch.bfloat16, device="cuda")
    head_product(o, uv, uv.transpose(1, 2).contiguous(), ao.view(n, H, D).transpose(0, 1))
    for h in range(H):
        _close(ao[:, h * D:(h + 1) * D], o[h].float() @ uv[h].float().t())


@pytest.mark.gpu
@pytest.mark.parametrize("E,K,gate", [(8, 1024, False), (8, 1024, True), (63, 2048, True), (64, 96, False), (65, 1024, False)])
def test_router_logits_of_long_steps(E, K, gate):
    """Choices other than the plain one, whose logits come from the kernels for small products where the weights are exact in bf16:
    against the same with fp32 weights (sums of K products of size 1 in another order, far below the scores' distances)."""
    g = torch.Generator().manual_seed(E)
    w = torch.randn(E + gate, K, generator=g).to(torch.bfloat16).cuda() / 8
    for T in (1, 1030, 2049):
        h = torch.randn(T, K, generator=g).to(torch.bfloat16).cuda()
        got, want = (hops.moe_router_grouped(h, w.float(), None, 2, 1, 1, extra_gate=gate, score="sigmoid", norm=False, w_act=a) for a in (w, None))
        assert (got[1] == want[1]).float().mean() >= 0.999
        same = got[1] == want[1]
        assert ((got[0] - want[0]).abs()[same] <= 1e-4).all()
        if gate:
            assert ((got[2] - want[2]).abs() <= 1e-4).all()


@pytest.mark.gpu
def test_logits_in_fp32():
    """The weight-streaming kernel's sums as they are (fp32 sums of K terms of size 1 / sqrt(K)), rows and columns that end inside its
    tiles; None for what it would split or not take."""
    g = torch.Generator().manual_seed(7)
    for N, K in ((32000, 256), (24608, 512)):
        w = (torch.randn(N, K, generator=g) / K ** 0.5).to(torch.bfloat16).cuda()
        wt = ops.tile_weight(w)
        for M in (1, 31, 33, 64, 100, 128):
            x = torch.randn(M, K + 8, generator=g).to(torch.bfloat16).cuda()[:, :K]
            y = ops.stream_logits(x, wt, 128)
            assert y.dtype == torch.float32 and ((y - x.float() @ w.float().t()).abs() <= 2e-5).all()
    assert ops.stream_logits(x, wt, 127) is None and ops.stream_logits(x, None, 128) is None and ops.stream_logits(x.cpu(), wt, 128) is None
    assert ops.stream_logits(x[:, ::2], wt, 128) is None and ops.stream_logits(x.float(), wt, 128) is None
    few = ops.tile_weight(torch.zeros(64, 4096, dtype=torch.bfloat16, device="cuda"))
    x = torch.zeros(4, 4096, dtype=torch.bfloat16, device="cuda")
    assert ops.stream_plan(4, 64, 4096)[2] > 1 and ops.stream_logits(x, few, 128) is None


@pytest.mark.parametrize("device", ["cpu", pytest.param("cuda", marks=pytest.mark.gpu)])
def test_gate_times_token_rows(device):
    """gelu(product) times the tokens' rows: in the product's kernel and, for short or too many rows, apart (the product rounded to bf16
    between, 2^-8 of it more), columns from the middle of the table."""
    g = torch.Generator().manual_seed(9)
    for M, N, K in ((1, 4, 1024), (17, 64, 2048), (40, 64, 512), (1030, 64, 1024)):
        x, w = torch.randn(M, K + 8, generator=g).to(torch.bfloat16)[:, :K], (torch.randn(N, K, generator=g) / K ** 0.5).to(torch.bfloat16)
        emb, tok = torch.randn(11, 3 * N, generator=g).to(torch.bfloat16), torch.randint(0, 11, (M,), generator=g)
        got = hops.side_gate_product(x.to(device), w.to(device), tok.to(device), emb.to(device), N).float().cpu()
        z = x.float() @ w.float().t()
        e = emb[tok, N:2 * N].float()
        # (the slope of gelu is below 1.13)
        assert ((got - torch.nn.functional.gelu(z, approximate="tanh") * e).abs() <= 2 ** -8 * (got.abs() + 1.2 * z.abs() * e.abs()) + 1e-3).all()
    if device == "cuda":
        tok = torch.tensor([3, -1, 11, 0], device=device)
        y = hops.side_gate_product(torch.ones(4, 1024, dtype=torch.bfloat16, device=device), torch.ones(8, 1024, dtype=torch.bfloat16, device=device),
                                   tok, emb.to(device), 0)
        assert y[1:3].isnan().all() and y[[0, 3]].isfinite().all()


@pytest.mark.gpu
@pytest.mark.parametrize("M,N,K", [(1025, 64, 1024), (2048, 64, 4096), (2047, 36, 1096), (1366, 48, 2048), (2048, 32, 1024), (2048, 4, 1024)])
def test_gate_of_long_steps(M, N, K):
    """One launch up to 2048 rows, of 32 columns a workgroup past 256 workgroups of 16: the same bound as above, fp32 sums of K terms beside it."""
    from unittest import mock

    g = torch.Generator().manual_seed(M + N)
    x, w = torch.randn(M, K, generator=g).to(torch.bfloat16), (torch.randn(N, K, generator=g) / K ** 0.5).to(torch.bfloat16)
    emb, tok = torch.randn(7, 3 * N, generator=g).to(torch.bfloat16), torch.randint(-1, 8, (M,), generator=g)
    with mock.patch.object(ops, "linear_small", side_effect=AssertionError("two launches")):
        got = hops.side_gate_product(x.cuda(), w.cuda(), tok.cuda(), emb.cuda(), N).double().cpu()
    known = (tok >= 0) & (tok < 7)
    assert got[~known].isnan().all()
    z, mag = x[known].double() @ w.double().t(), x[known].double().abs() @ w.double().abs().t()
    e = emb[tok[known], N:2 * N].double()
    want = torch.nn.functional.gelu(z, approximate="tanh") * e
    assert ((got[known] - want).abs() <= 2 ** -8 * want.abs() + 1.13 * K * 2.0 ** -24 * mag * e.abs() + 1e-5 * e.abs()).all()


@pytest.mark.gpu
@pytest.mark.parametrize("K", [64, 120, 512, 1024])
@pytest.mark.parametrize("M,N", [(1, 128), (17, 36), (64, 128), (65, 64)])
def test_heads_with_a_sigmoid_gate(K, M, N):
    """The gate in the product's epilogue is the product and the gate's launch, to the last bit; a gate that the kernel does not read goes the
    other way."""
    H, g = 3, torch.Generator().manual_seed(K + M)
    x, w = (torch.randn(H, n, K, generator=g).to(torch.bfloat16).cuda() for n in (M, N))
    wt = w.transpose(1, 2).contiguous()
    wide = (4 * torch.randn(M, 8 + H * N + 1, generator=g)).to(torch.bfloat16).cuda()
    wide[0, 9:11] = torch.tensor([float("inf"), -float("inf")])
    for gate in (wide[:, 8:8 + H * N].contiguous(), torch.nn.functional.pad(wide, (0, -(8 + H * N + 1) % 4))[:, 8:8 + H * N], wide[:, 9:]):
        want = torch.empty(M, H * N, dtype=torch.bfloat16, device="cuda")
        hops.sigmoid_mul(head_product(x, w, wt), gate, want)
        got = torch.full_like(want, float("nan"))
        head_product(x, w, wt, got.view(M, H, N).transpose(0, 1), gate)
        if gate.stride(0) % 4 == 0 and gate.data_ptr() % 8 == 0:
            assert torch.equal(got, want)
        else:   # (the library's sums in another order: a bf16 step of the product)
            assert (got.float() - want.float()).norm() < 2e-3 * want.float().norm()
