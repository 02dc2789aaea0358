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
