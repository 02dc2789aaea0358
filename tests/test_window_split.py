"""Windowed attention of decoded tokens: an item's keys over the four waves of a workgroup, and over several workgroups."""
import pytest
import torch

from kafka_llm_service_amd.ops import hybrid as hops

pytestmark = pytest.mark.gpu
CONTEXTS = [1, 31, 32, 33, 64, 97, 128, 129, 255, 300, 513, 1024, 1025]   # blocks that leave waves, or whole ranges, without keys


@pytest.mark.parametrize("H,G,D,Dv,window,sink", [
    (8, 2, 128, 128, 0, True), (32, 1, 64, 64, 0, False), (8, 8, 16, 20, 100, True), (6, 3, 192, 72, 33, False),
    (4, 2, 256, 256, 0, True), (4, 4, 96, 130, 1, False), (16, 2, 48, 256, 500, True)])
def test_decoded_tokens(H, G, D, Dv, window, sink):
    torch.manual_seed(H * D + Dv)
    dev, R = "cuda:0", len(CONTEXTS)
    pages = [-(-n // 16) for n in CONTEXTS]
    order = torch.randperm(sum(pages) + 1)[1:]          # (page 0 is nobody's)
    bt, at = torch.zeros(R, max(pages), dtype=torch.int32), 0
    kc = torch.zeros(sum(pages) + 1, 16, G * D, dtype=torch.bfloat16)
    vt = torch.zeros(sum(pages) + 1, G * Dv, 16, dtype=torch.bfloat16)
    q = (2 * torch.randn(R, H, D)).bfloat16()
    snk = torch.randn(H) if sink else None
    want, bound = torch.empty(R, H, Dv, dtype=torch.float64), torch.empty(R, H, Dv, dtype=torch.float64)
    for r, n in enumerate(CONTEXTS):
        ids = order[at:at + pages[r]]
        at += pages[r]
        bt[r, :pages[r]] = ids.int()
        k, v = torch.randn(pages[r] * 16, G, D).bfloat16(), torch.randn(pages[r] * 16, G, Dv).bfloat16()   # (rows past n: another's)
        kc[ids] = k.view(pages[r], 16, G * D)
        vt[ids] = v.view(pages[r], 16, G * Dv).transpose(1, 2)
        lo = max(0, n - window) if window else 0
        kk, vv = (x[lo:n].double().repeat_interleave(H // G, 1) for x in (k, v))
        s = torch.einsum("hd,jhd->hj", q[r].double(), kk) * D ** -0.5
        top = s.amax(1, keepdim=True)
        p = torch.exp(s - top)
        den = p.sum(1) + (torch.exp(snk.double() - top[:, 0]) if sink else 0.0)
        p = p / den[:, None]
        want[r] = torch.einsum("hj,jhv->hv", p, vv)
        # weights and the result are bf16 (8 bits: half a unit is up to 2^-8 of the value); a score of D products in fp32 moves its weight by as many 2^-24 of them
        scale = 2.0 ** -24 * D * torch.einsum("hd,jhd->hj", q[r].double().abs(), kk.abs()).amax(1) * D ** -0.5
        bound[r] = (2.0 ** -8 + 4 * scale[:, None] + 1e-5) * torch.einsum("hj,jhv->hv", p, vv.abs()) + 2.0 ** -8 * want[r].abs() + 1e-30
    bound *= 1.02
    tiles = torch.tensor([(r, 1, r, 0) for r in range(R)], dtype=torch.int32, device=dev)
    args = (kc.to(dev), vt.to(dev), bt.to(dev), None, torch.tensor([n - 1 for n in CONTEXTS], device=dev), H, G, D ** -0.5, window,
            snk.to(dev) if sink else None)
    outs = []
    for max_keys, target in ((0, 256), (max(CONTEXTS), 256), (max(CONTEXTS), 4096)):   # one range, as chosen, as many as there can be
        out = torch.full((R, H * Dv), float("nan"), dtype=torch.bfloat16, device=dev)
        old, hops.WINDOW_SPLIT_WGS = hops.WINDOW_SPLIT_WGS, target
        try:
            hops.window_attn(q.view(R, H * D).to(dev), *args, out, tiles, max_keys, kinds=(True, False))
        finally:
            hops.WINDOW_SPLIT_WGS = old
        err = (out.cpu().double().view(R, H, Dv) - want).abs()
        assert (err <= bound).all(), (max_keys, target, (err / bound).max())
        outs.append(out)
    assert 0 < window < 512 or not torch.equal(outs[0], outs[2])   # (the ranges did differ)


def test_splits():
    for wgs in (1, 2, 16, 85, 128, 129, 256, 100000):
        for keys in (0, 1, 128, 300, 512, 8000, 10 ** 6):
            ns = hops.window_splits(wgs, keys)
            assert 1 <= ns <= 64 and (ns == 1 or (ns * wgs <= hops.WINDOW_SPLIT_WGS and keys > (2 * ns - 1) * 128))
