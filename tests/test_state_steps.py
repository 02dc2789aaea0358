"""One token per segment: the recurrences' states moved once, against 64-bit sums of the same values."""
import pytest
import torch

from kafka_llm_service_amd.ops import hybrid as hops

pytestmark = pytest.mark.gpu
EPS = 2.0 ** -24


def segments(R):
    # decoded tokens in slots out of order, every third the first of its sequence, one longer segment that has its own kernel
    segs, at = [], 0
    for i in range(R):
        n = 3 if i == 3 else 1
        segs.append((at, n, 0 if i % 3 == 1 else 9, R - i))
        at += n
    return segs, at


def close(got, want, bound):
    bad = ~((got.double().cpu() - want).abs() <= bound)
    assert not bad.any(), (got.double().cpu() - want).abs().max()


@pytest.mark.parametrize("P,N,offset", [
    (4, 1, 0), (4, 300, 0),            # 256 row groups, more rows than one piece of them
    (8, 7, 0), (12, 128, 0),           # columns that do not divide the workgroup
    (64, 128, 0), (64, 129, 0), (64, 257, 0),   # one piece, one row more, two and one row
    (64, 16, 0), (64, 17, 0), (64, 32, 0), (64, 33, 0), (64, 64, 0), (64, 65, 0),   # one, two, up to four rows a thread, and one more
    (252, 5, 0), (256, 32, 0), (256, 33, 0),    # the widest head
    (64, 128, 1), (30, 20, 0), (255, 9, 0)])    # a state off 16 bytes, odd columns: the kernel of single columns
@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
def test_scan_step(P, N, offset, dtype):
    torch.manual_seed(P * 1000 + N)
    H, G, R = 4, 2, 7
    segs, T = segments(R)
    xbc = (torch.randn(T, H * P + 2 * G * N) / 2).to(dtype)
    proj = torch.randn(T, H + 3).to(dtype)
    bias, A, D = torch.randn(H), torch.randn(H), torch.randn(H)
    state = torch.randn(R + 1, H, N, P)
    for _, _, p0, slot in segs:
        if p0 == 0:
            state[slot] = float("nan")     # (written, not read)
    buf = torch.empty(state.numel() + offset, device="cuda")
    gs = buf[offset:].view(state.shape)
    gs.copy_(state)
    seg = torch.tensor(segs, dtype=torch.int32).cuda()
    tok = torch.cat([torch.full((n,), i, dtype=torch.int32) for i, (_, n, _, _) in enumerate(segs)]).cuda()
    y = torch.full((T, H * P), 7.0, device="cuda")
    hops.ssm_scan(xbc.cuda(), proj.cuda(), 3, bias.cuda(), A.cuda(), D.cuda(), H, P, N, G, tok, seg, gs, y, rows=(1, 1))
    for t, n, p0, slot in segs:
        if n != 1:   # left alone
            assert (y[t:t + n] == 7).all() and torch.equal(gs[slot].cpu(), state[slot])
            continue
        x = xbc[t].double()
        xv = x[:H * P].view(H, P)
        B, C = (x[H * P + a * G * N:H * P + (a + 1) * G * N].view(G, N).repeat_interleave(H // G, 0) for a in (0, 1))
        dt = torch.nn.functional.softplus(proj[t, 3:].double() + bias.double())
        S0 = state[slot].double() if p0 else torch.zeros(H, N, P, dtype=torch.float64)
        old = torch.exp(-torch.exp(A.double()) * dt)[:, None, None] * S0
        new = B[:, :, None] * (dt[:, None] * xv)[:, None]
        # the step size and the decay are functions of rounded arguments: exp(-e^A dt) is off by up to e^A dt of them more
        rel = 16 * EPS * (1 + (torch.exp(A.double()) * dt))[:, None, None]
        close(gs[slot], old + new, rel * (old.abs() + new.abs()) + 1e-37)
        parts = (old.abs() + new.abs()) * C[:, :, None].abs()
        want = ((old + new) * C[:, :, None]).sum(1) + D.double()[:, None] * xv
        close(y[t].view(H, P), want, (rel * parts).sum(1) + (N + 4) * EPS * (parts.sum(1) + (D.double()[:, None] * xv).abs()))
    assert torch.equal(gs[0].cpu(), state[0])   # (no segment's)


@pytest.mark.parametrize("D,Dv", [(1, 4), (7, 20), (256, 32), (128, 64), (129, 64), (128, 128), (129, 128), (64, 256), (256, 256),
                                  (256, 260), (33, 516), (16, 1028)])   # 4, 8 and 16 waves, one and several pieces
@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
def test_memory_step(D, Dv, dtype):
    torch.manual_seed(D * 1000 + Dv)
    H, R, cap = 2, 7, 6.0
    segs, T = segments(R)
    qkv, gates = torch.randn(T, H * (2 * D + Dv)).to(dtype), 4 * torch.randn(T, 2 * H)
    S, nrm, mx = torch.randn(R + 1, H, D, Dv), torch.randn(R + 1, H, D), torch.randn(R + 1, H)
    for _, _, p0, slot in segs:
        if p0 == 0:
            S[slot], nrm[slot], mx[slot] = float("nan"), float("nan"), float("nan")
    gS, gn, gm = S.cuda(), nrm.cuda(), mx.cuda()
    seg = torch.tensor(segs, dtype=torch.int32).cuda()
    tok = torch.cat([torch.full((n,), i, dtype=torch.int32) for i, (_, n, _, _) in enumerate(segs)]).cuda()
    out = torch.full((T, H * Dv), 7.0, device="cuda")
    hops.mlstm_scan(qkv.cuda(), gates.cuda(), H, D, Dv, cap, tok, seg, gS, gn, gm, out, rows=(1, 1))
    for t, n, p0, slot in segs:
        if n != 1:
            assert (out[t:t + n] == 7).all() and torch.equal(gS[slot].cpu(), S[slot])
            continue
        x = qkv[t].double()
        q, k, v = x[:H * D].view(H, D) * D ** -0.5, x[H * D:2 * H * D].view(H, D), x[2 * H * D:].view(H, Dv)
        c = cap * torch.tanh(gates[t].double() / cap)
        ig, fg = c[:H], torch.nn.functional.logsigmoid(c[H:])
        m0, S0, n0 = ((a[slot].double() if p0 else torch.zeros_like(a[slot]).double()) for a in (mx, S, nrm))
        m = torch.maximum(fg + m0, ig)
        dec, gain = torch.exp(fg + m0 - m), torch.exp(ig - m)
        # (exponents of up to 4 cap whose parts carry a few roundings of the tanh each)
        rel = 16 * EPS * 4 * cap
        old, new = dec[:, None, None] * S0, gain[:, None, None] * k[:, :, None] * v[:, None]
        close(gS[slot], old + new, rel * (old.abs() + new.abs()) + 1e-37)
        on, nn = dec[:, None] * n0, gain[:, None] * k
        close(gn[slot], on + nn, rel * (on.abs() + nn.abs()) + 1e-37)
        close(gm[slot], m, rel * (1 + m.abs()))
        den = torch.maximum(((on + nn) * q).sum(1).abs(), torch.exp(-m)) + 1e-6
        dd = rel * ((on.abs() + nn.abs()) * q.abs()).sum(1) + D * EPS * ((on.abs() + nn.abs()) * q.abs()).sum(1) + rel * torch.exp(-m)
        num = ((old + new) * q[:, :, None]).sum(1)
        dn = (rel + (D + 4) * EPS) * ((old.abs() + new.abs()) * q.abs()[:, :, None]).sum(1)
        close(out[t].view(H, Dv), num / den[:, None], 1.01 * (dn / den[:, None] + (num / den[:, None]).abs() * (dd / den)[:, None]) +
              8 * EPS * (num / den[:, None]).abs())
    assert torch.equal(gS[0].cpu(), S[0])


@pytest.mark.parametrize("n,p0", [(128 * 4 + 1, 0), (128 * 9 + 5, 7), (128 * 12, 3)])   # chunks that the carry asks for in one, three and three goes
def test_chunks_carried(n, p0):
    """Segments of more chunks than the carry keeps in flight, against 64-bit sums. A result is a sum of at most 128 rows, 128 channels
    and one entry state per chunk in fp32: as many roundings of the sum of its parts' magnitudes, and a few for each decay."""
    torch.manual_seed(n)
    H, P, N, D, Dv, cap, dev = 2, 24, 32, 32, 40, 6.0, "cuda:0"
    seg, tok = torch.tensor([(0, n, p0, 1)], dtype=torch.int32), torch.zeros(n, dtype=torch.int32, device=dev)
    bound = (128 + 128 + n // 128 + 40) * EPS

    xbc, proj = (torch.randn(n, H * P + 2 * N) / 2).bfloat16(), torch.randn(n, H).bfloat16()
    bias, A, Dp = torch.randn(H) - 4, torch.rand(H) - 2, torch.randn(H)
    state, y = torch.randn(2, H, N, P), torch.empty(n, H * P, device=dev)
    gs = state.cuda()
    tabs = tuple(torch.from_numpy(t).to(dev) for t in hops.chunk_tables(seg.numpy(), hops.SSD_CHUNK, hops.SSD_CHUNK_MIN))
    hops.ssm_scan(xbc.cuda(), proj.cuda(), 0, bias.cuda(), A.cuda(), Dp.cuda(), H, P, N, 1, tok, seg.cuda(), gs, y, chunks=tabs, rows=None)
    S = state[1].double() * (p0 > 0)
    mag = S.abs()
    want, most = [], []
    for t in range(n):
        x = xbc[t].double()
        xv, B, C = x[:H * P].view(H, P), x[H * P:H * P + N], x[H * P + N:]
        dt = torch.nn.functional.softplus(proj[t].double() + bias.double())
        dec, new = torch.exp(-torch.exp(A.double()) * dt)[:, None, None], B[None, :, None] * (dt[:, None] * xv)[:, None]
        S, mag = dec * S + new, dec * mag + new.abs()
        want.append((S * C[:, None]).sum(1) + Dp.double()[:, None] * xv)
        most.append((mag * C.abs()[:, None]).sum(1) + (Dp.double()[:, None] * xv).abs())
    close(y.view(n, H, P), torch.stack(want), bound * torch.stack(most))
    close(gs[1], S, bound * mag)

    qkv, gates = torch.randn(n, H * (2 * D + Dv)).bfloat16(), 4 * torch.randn(n, 2 * H)
    M, nrm, mx = torch.randn(2, H, D, Dv), torch.randn(2, H, D), torch.randn(2, H)
    gM, gn, gm, out = M.cuda(), nrm.cuda(), mx.cuda(), torch.empty(n, H * Dv, device=dev)
    tabs = tuple(torch.from_numpy(t).to(dev) for t in hops.chunk_tables(seg.numpy(), hops.MLSTM_CHUNK, hops.MLSTM_CHUNK_MIN))
    hops.mlstm_scan(qkv.cuda(), gates.cuda(), H, D, Dv, cap, tok, seg.cuda(), gM, gn, gm, out, chunks=tabs, rows=None)
    S, v0, m = (a[1].double() * (p0 > 0) for a in (M, nrm, mx))
    magS, magn = S.abs(), v0.abs()
    want, most = [], []
    for t in range(n):
        x = qkv[t].double()
        q, k, v = x[:H * D].view(H, D) * D ** -0.5, x[H * D:2 * H * D].view(H, D), x[2 * H * D:].view(H, Dv)
        c = cap * torch.tanh(gates[t].double() / cap)
        ig, fg = c[:H], torch.nn.functional.logsigmoid(c[H:])
        m1 = torch.maximum(fg + m, ig)
        dec, gain, m = torch.exp(fg + m - m1), torch.exp(ig - m1), m1
        kv = gain[:, None, None] * k[:, :, None] * v[:, None]
        S, magS = dec[:, None, None] * S + kv, dec[:, None, None] * magS + kv.abs()
        v0, magn = dec[:, None] * v0 + gain[:, None] * k, dec[:, None] * magn + gain[:, None] * k.abs()
        den = torch.maximum((v0 * q).sum(1).abs(), torch.exp(-m)) + 1e-6
        o = (S * q[:, :, None]).sum(1) / den[:, None]
        want.append(o)
        # (a log gate's roundings, a few of cap, enter as an exponent's; running sums of 128 of them as 128)
        most.append(((magS * q.abs()[:, :, None]).sum(1) + o.abs() * (magn * q.abs()).sum(1)[:, None]) / den[:, None] + o.abs())
    gate = bound + 128 * 2 * cap * EPS
    close(out.view(n, H, Dv), torch.stack(want), gate * torch.stack(most))
    close(gM[1], S, gate * magS)
    close(gn[1], v0, gate * magn)


@pytest.mark.parametrize("T,d,off", [(1, 64, 0), (5, 1024, 0), (5, 1028, 0), (64, 4096, 0), (3, 4100, 0), (5, 7, 0), (5, 1030, 0), (5, 1024, 1),
                                     (600, 4096, 0)])   # threads and pieces a row, single elements, a width and rows that the registers do not take
@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
def test_layer_end_with_the_next_norm(T, d, off, dtype):
    """One launch of a layer's end and the next one's shifted norm against the two: the same operations on the same values, whose products
    and sums may be contracted differently (2 roundings of a value of the row's scale), and in bf16 half a unit of the result."""
    torch.manual_seed(T + d)
    dev, layer = "cuda:0", 1
    segs = [(t, 1, 0 if t % 3 == 1 else 4, T - t) for t in range(T)]
    seg, tok = torch.tensor(segs, dtype=torch.int32, device=dev), torch.arange(T, dtype=torch.int32, device=dev)
    x, y, stack = torch.randn(T, d, device=dev), torch.randn(T, d, device=dev).to(dtype), torch.randn(3, T, d, device=dev)
    w, b, mu, sw = (torch.randn(d, device=dev).to(dtype) for _ in range(4))
    dwa = torch.rand(layer + 2, device=dev)
    state = torch.randn(T + 1, d, device=dev)
    for _, _, p0, slot in segs:
        if p0 == 0:
            state[slot] = float("nan")   # (not read)
    for yy, ss, dd in ((y, stack, dwa), (y, None, None), (None, stack, dwa), (y, stack, None)):
        res = []
        for joined in (False, True):
            xs, st, sk = x.clone(), state.clone(), ss.clone() if ss is not None else None
            out = torch.full((T, d + 8), 7.0, dtype=dtype, device=dev)
            rows = out[:, off:off + d]
            nxt = (w, b, 1e-5, rows, mu, tok, seg, st)
            hops.side_dwa(xs, yy, sw if yy is not None else None, 1e-6, sk, layer, dd, nxt if joined else None)
            if not joined:
                hops.ln_shift(xs, *nxt)
            assert (out[:, :off] == 7).all() and (out[:, off + d:] == 7).all()
            res.append((xs, rows.float(), st, sk))
        for k, (a, c) in enumerate(zip(*res)):
            if a is not None:
                assert torch.equal(a.isnan(), c.isnan())
                a, c = a.nan_to_num(), c.nan_to_num()
                unit = 2.0 ** -8 if k == 1 and dtype == torch.bfloat16 else 0.0
                assert ((a - c).abs() <= unit * a.abs() + 8 * EPS * a.abs().amax()).all(), k
        assert torch.equal(res[1][2][0], state[0])   # (no segment's slot)
