"""Row kernels of short steps: norms with a piece a thread, routing with an expert a lane."""
import pytest
import torch

from kafka_llm_service_amd.ops import hybrid as hops

pytestmark = pytest.mark.gpu
EPS = 2.0 ** -24


@pytest.mark.parametrize("T,d,off", [(1, 4, 0), (3, 1020, 0), (3, 4096, 0), (512, 4092, 0), (513, 4096, 0), (2, 4100, 0), (5, 7, 0), (3, 1024, 1)])
@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
def test_rms_norm(T, d, off, dtype):
    """Against 64-bit sums: a row's mean square is a sum of d squares in fp32, its root and the two products round once each."""
    torch.manual_seed(T + d)
    x, w = torch.randn(T, d + 4, device="cuda")[:, off:off + d], torch.randn(d, device="cuda").to(dtype)
    out = torch.full((T, d + 4), 7.0, dtype=dtype, device="cuda")
    hops.rms_norm(x, w, 1e-5, out[:, off:off + d])
    want = x.double() / (x.double().pow(2).mean(1, keepdim=True) + 1e-5).sqrt() * w.double()
    unit = 2.0 ** -8 if dtype == torch.bfloat16 else 0.0
    assert ((out[:, off:off + d].double() - want).abs() <= (unit + (d + 8) * EPS) * want.abs()).all()
    assert (out[:, :off] == 7).all() and (out[:, off + d:] == 7).all()


@pytest.mark.parametrize("T,d", [(3, 1028), (512, 2048), (2, 4096), (513, 4092), (3, 4104), (4, 1024)])   # 256 and 1024 threads a row
@pytest.mark.parametrize("S", [0, 1, 2, 4, 8])
def test_norm_add(T, d, S):
    torch.manual_seed(T + d + S)
    x, w = torch.randn(T, d, device="cuda"), torch.randn(d, device="cuda")
    y1 = torch.randn(S, T, d, device="cuda") if S else torch.randn(T, d, device="cuda").bfloat16()
    y2 = torch.randn(T, d, device="cuda").bfloat16() if S in (0, 2) else None
    y = (y1.double().sum(0) if S else y1.double()) + (y2.double() if y2 is not None else 0.0)
    mag = (y1.double().abs().sum(0) if S else y1.double().abs()) + (y2.double().abs() if y2 is not None else 0.0)
    r = 1 / (y.pow(2).mean(1, keepdim=True) + 1e-5).sqrt()
    want = x.double() + y * r * w.double()
    out = torch.empty(T, d, dtype=torch.bfloat16, device="cuda")
    hops.norm_add(x, y1, y2, w, 1e-5, out)
    bound = EPS * (12 * mag * r * w.double().abs() + (d + 8) * (y * r * w.double()).abs() + 2 * want.abs())
    # (a row's scale carries the elements' errors as their mean, less than their largest)
    bound = bound + 12 * EPS * (mag.amax(1, keepdim=True) * r) * (y * r * w.double()).abs()
    assert ((x.double() - want).abs() <= bound).all()
    assert ((out.double() - x.double()).abs() <= 2.0 ** -8 * x.double().abs()).all()


@pytest.mark.parametrize("E,k,groups,keep", [(4, 2, 1, 1), (8, 3, 4, 2), (63, 6, 9, 4), (64, 8, 8, 3), (66, 6, 6, 2), (128, 4, 64, 7), (512, 8, 8, 4)])
@pytest.mark.parametrize("score,group_score", [("softmax", "max"), ("sigmoid", "top2")])
def test_router_choice(E, k, groups, keep, score, group_score):
    """One and eight experts a lane, against the choice on the CPU: weights to the few roundings of an exponential and a sum of E, the same
    experts (random scores, no ties)."""
    torch.manual_seed(E + k)
    T, d = 37, 64
    h, w = torch.randn(T, d).bfloat16(), torch.randn(E, d).bfloat16()
    corr = torch.rand(E) / 4
    args = dict(score=score, group_score=group_score, scale=1.5)
    a = hops.moe_router_grouped(h, w.float(), corr, k, groups, keep, **args)
    b = hops.moe_router_grouped(h.cuda(), w.float().cuda(), corr.cuda(), k, groups, keep, **args)
    assert torch.equal(a[1], b[1].cpu())
    assert ((a[0] - b[0].cpu()).abs() <= (E + 40) * 4 * EPS * a[0].abs()).all()


@pytest.mark.parametrize("K", [32, 64, 96, 160, 544, 1024, 2080, 4096, 8224])   # runs of steps that end inside, at and past a wave's share
def test_narrow_products_by_whole_lines(K):
    """Rows and columns at the edges of 16, in buffers whose neighbours are not numbers: sums of K products of bf16, each rounded in fp32."""
    torch.manual_seed(K)
    for T, N in ((1, 1), (15, 16), (16, 17), (17, 33), (33, 48), (40, 64)):
        x = torch.full((T, K + 16), float("nan"), device="cuda", dtype=torch.bfloat16)
        x[:, 8:8 + K] = torch.randn(T, K, device="cuda").bfloat16()
        x = x[:, 8:8 + K]
        w = torch.randn(N, K, device="cuda").bfloat16()
        want, size = x.double() @ w.double().t(), x.double().abs() @ w.double().abs().t()
        z = torch.empty(T, N, device="cuda")
        hops.ext().narrow_linear(x, w, None, z)
        assert ((z.double() - want).abs() <= (K + 16) * EPS * size).all(), (T, N)
        if N % 4 == 0:
            s = torch.empty(T, N, device="cuda")
            hops.ext().small_gemm(x, w, s)
            assert ((s.double() - want).abs() <= (K + 16) * EPS * size).all(), (T, N)


@pytest.mark.parametrize("T", [1, 512, 635])   # as many workgroups for the queries as they fill, and fewer
@pytest.mark.parametrize("H,dim,rd,dims,R", [(32, 64, 64, 64, 512), (3, 16, 64, 32, 40), (33, 8, 8, 4, 64), (130, 8, 128, 128, 64), (4, 16, 0, 0, 64)])
def test_latent_prep(T, H, dim, rd, dims, R):
    """Against the same in fp32 on the CPU: two products and a sum an element, the norm a sum of R squares; every fourth row without
    a slot, and queries alone."""
    g = torch.Generator().manual_seed(T + H)
    off, page, cap = H * (dim + rd), 16, 640
    row = torch.randn(T, off + R + rd + 8, generator=g)
    w, cs = torch.rand(R, generator=g), torch.randn(700, max(dims, 1), generator=g)
    pos, slots = torch.randint(0, 700, (T,), generator=g), torch.randperm(cap, generator=g)[:T]
    slots[3::4] = -1
    for o in (off, -1):
        got = []
        for dev in ("cpu", "cuda"):
            c, ct = torch.full((cap // page, page, R + rd), 7.0, device=dev), torch.full((cap // page, R, page), 7.0, device=dev)
            q = torch.full((T, H, rd), 7.0, device=dev)
            hops.latent_prep(row.to(dev), H, dim, rd, R, o, w.to(dev), 1e-5, pos.to(dev), cs.to(dev) if dims else None, dims, c, slots.to(dev), q, ct)
            got.append([t.cpu() for t in (c, ct, q)])
        big = 8 * (row.abs().max() * cs.abs().max()).item()
        for a, b in zip(*got):
            assert ((a - b).abs() <= (R + 8) * EPS * a.abs() + 4 * EPS * big).all()
