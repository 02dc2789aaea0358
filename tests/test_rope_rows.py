"""Rotation and paged store of long steps (csrc/rope_kv.hip, a wave per row) and of bf16 rows with values in columns of their own
(csrc/hybrid_parallel.hip), against the plain functions."""
import pytest
import torch

from kafka_llm_service_amd import ops
from kafka_llm_service_amd.ops import hybrid as hops
from kafka_llm_service_amd.ops import ref


def _slots(g, T, pages):
    """Rows in places of their own, then runs: whole pages, a page's end and its beginning apart, a page with two rows exchanged, a
    page that begins before the rows do (and ends after them)."""
    s = torch.randperm(pages * 16, generator=g)[:T]
    if T >= 256:
        p = torch.randperm(pages, generator=g).repeat_interleave(16) * 16 + torch.arange(16).repeat(pages)
        s = p[5:T + 5].clone()
        s[48:50] = s[48:50].flip(0)
        s[100:107] = -1
        s[207:223] = s[207:223].roll(3)
    s[T // 3] = -1                 # rows without a place in the cache
    s[T - 1] = -1
    return s


def _close(got, want):
    # two products and a sum in fp32 (contracted or not: 2^-22 of the products, which are up to 6 x 6) rounded to bf16: half a step, 2^-8 of a
    # value that is a power of two; against a value that is rounded too a whole one, 2^-7
    part = 2 ** -7 if want.dtype == torch.bfloat16 else 2 ** -8
    assert ((got.float().cpu() - want.float()).abs() <= part * want.float().abs() + 1e-4).all()


@pytest.mark.gpu
@pytest.mark.parametrize("Hq,Hkv,D", [(32, 8, 128), (8, 1, 128), (5, 5, 128), (40, 10, 128), (32, 8, 64), (3, 1, 64), (28, 17, 64)])
def test_long_steps(Hq, Hkv, D):
    """Around the rows from which a wave takes a row, heads that end inside and past a batch of five (or two of values), rows of a
    wider projection, rows without a slot."""
    g = torch.Generator().manual_seed(Hq + D)
    for T in (383, 384, 1027):
        qkv = torch.randn(T, (Hq + 2 * Hkv) * D + 8, generator=g).to(torch.bfloat16)[:, :(Hq + 2 * Hkv) * D]
        pos, cs, nb = torch.randint(0, 300, (T,), generator=g), torch.randn(300, D, generator=g), T // 16 + 2
        slots = _slots(g, T, nb)
        out = []
        for dev in ("cuda", "cpu"):
            q = torch.zeros(T, Hq, D, dtype=torch.bfloat16, device=dev)
            k = torch.zeros(nb, Hkv, D // 8, 16, 8, dtype=torch.bfloat16, device=dev).view(nb, Hkv, 16, D)
            v = torch.zeros(nb, Hkv, D, 16, dtype=torch.bfloat16, device=dev)
            src = torch.empty(T, qkv.shape[1] + 8, dtype=torch.bfloat16, device=dev)[:, :qkv.shape[1]].copy_(qkv)
            (ops if dev == "cuda" else ref).rope_kv_write(src, pos.to(dev), cs.to(dev), q, k, v, slots.to(dev), Hq, Hkv)
            out.append((q, k, v))
        for a, b in zip(out[0][:2], out[1][:2]):
            _close(a, b)
        assert torch.equal(out[0][2].cpu(), out[1][2])


@pytest.mark.gpu
@pytest.mark.parametrize("H,G,D,dims,norm,v", [(8, 2, 128, 64, False, 0), (8, 2, 128, 128, True, 0), (3, 3, 64, 16, True, 0), (5, 1, 8, 0, False, 0),
                                               (2, 2, 512, 512, True, 0), (4, 2, 16, 16, False, 8), (6, 3, 256, 96, True, 24),
                                               (4, 2, 128, 64, False, 3), (4, 4, 32, 32, True, -1)])
def test_values_of_their_own(H, G, D, dims, norm, v):
    """Rows of a step whose lanes take one head each and of one that takes four and stores values by pages, values after the keys, further on (whole pieces or not) and
    the keys themselves, no rotation, rotation of a part and of all, rows without a slot."""
    g = torch.Generator().manual_seed(H * D + dims)
    off = H * D if v < 0 else (H + G) * D + v
    for T in (1, 37, 2 ** 19 // ((H + G) * D // 8) + 5):
        rows = torch.randn(T, (H + 2 * G) * D + 32, generator=g).to(torch.bfloat16)
        pos, nb = torch.randint(0, 300, (T,), generator=g), T // 16 + 2
        cs = torch.randn(300, dims, generator=g) if dims else None
        w = [torch.rand(D, generator=g) + 0.5 if norm else None for _ in range(2)]
        slots = _slots(g, T, nb)
        out = []
        for dev, dt in (("cuda", torch.bfloat16), ("cpu", torch.float32)):
            kc, vt = torch.zeros(nb, 16, G * D, dtype=dt, device=dev), torch.zeros(nb, G * D, 16, dtype=dt, device=dev)
            q = torch.zeros(T, H * D, dtype=dt, device=dev)
            hops.rope_kv_store(rows.to(dev, dt), H, G, D, D, pos.to(dev), None if cs is None else cs.to(dev), dims, False, None, kc, vt,
                               slots.to(dev), q, *(None if x is None else x.to(dev) for x in w), 1e-5, v_off=off)
            out.append((q, kc, vt))
        for a, b in zip(out[0][:2], out[1][:2]):
            _close(a, b)
        assert torch.equal(out[0][2].cpu().float(), out[1][2])
