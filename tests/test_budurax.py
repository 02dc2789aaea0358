"""Budurax in the serving engine against the plain whole-sequence implementation of tests/budurax_plain.py.

Small configurations of odd sizes (nothing a multiple of 64, a rotary part wider than its rotated dimensions, one
state-space group, a layer without feed-forward, a model without shift / depth average / token input) with random
weights made here. Each test runs on the CPU reference ops and, marked ``gpu``, on the HIP kernels.
"""
import copy
import math

import pytest
import torch

import budurax_plain as plain
from kafka_llm_service_amd.engine.engine import EngineConfig, LLMEngine
from kafka_llm_service_amd.engine.sequence import SamplingParams
from kafka_llm_service_amd.models import budurax as bx
from kafka_llm_service_amd.ops import hybrid as hops

DEVICES = ["cpu", pytest.param("cuda:0", marks=pytest.mark.gpu)]


def _attn(heads=3, dim=24, rot_dim=16, dims=8, vdim=20, rank=40, scaling=True, kv_from=None, scale=None):
    rot = {"base": 10000.0, "dims": dims}
    if scaling:
        rot["scaling"] = {"factor": 4.0, "original": 64, "fast": 16.0, "slow": 2.0}
    m = {"heads": heads, "dim": dim, "rot_dim": rot_dim, "vdim": vdim, "kv_rank": rank, "rot": rot,
         "scale": scale if scale is not None else (dim + rot_dim) ** -0.5}
    if kv_from is not None:
        m["kv_from"] = kv_from
    return m


def _mamba(heads=4, vdim=12, state=20, groups=2, norm_groups=4, conv=3):
    return {"heads": heads, "vdim": vdim, "state": state, "groups": groups, "norm_groups": norm_groups, "conv": conv}


def cfg_a(scale=None):
    ff = {"kind": "dense", "ff": 72}
    return {"architecture": "Budurax", "vocab": 211, "width": 88, "norm": {"eps": 1e-5}, "token_side": {"dim": 6},
            "layers": [{"type": "mamba2", "mixer": _mamba(), "mlp": ff},
                       {"type": "latent_attention", "mixer": _attn(scale=scale), "mlp": ff},
                       {"type": "latent_attention", "mixer": _attn(kv_from=1, scale=scale), "mlp": None},
                       {"type": "mamba2", "mixer": _mamba(heads=2, vdim=40, state=9, groups=1, norm_groups=1, conv=5),
                        "mlp": ff}]}


def cfg_b():
    """Ones and equal values: one head, one group, two taps, rot.dims = rot_dim, no scaling, no extras."""
    ff = {"kind": "dense", "ff": 40}
    return {"architecture": "Budurax", "vocab": 97, "width": 48, "norm": {"eps": 1e-6},
            "layers": [{"type": "latent_attention", "mixer": _attn(1, 16, 8, 8, 16, 16, scaling=False), "mlp": ff},
                       {"type": "mamba2", "mixer": _mamba(1, 16, 16, 1, 1, 2), "mlp": ff}]}


class Bench:
    """A config, its random weights and engines over them."""

    def __init__(self, cfg: dict, seed=0, extras=True, sharpen=1.0):
        self.cfg = cfg
        self.mc = bx.BuduraxConfig.from_dict(cfg, name="test")
        self.W = bx.random_tensors(self.mc, seed, shift=extras, dwa=extras)
        if sharpen != 1.0:  # peaky softmax: single keys carry the result
            for k in self.W:
                if k.endswith("mix.q"):
                    self.W[k] = (self.W[k].float() * sharpen).to(torch.bfloat16)
        self._oracle = {}

    def engine(self, device, dtype="float32", blocks=64, seqs=4, **kw):
        model = bx.BuduraxLM(self.mc, device, dtype=getattr(torch, dtype), max_positions=1024).load_tensors(self.W)
        return LLMEngine(EngineConfig(model="test", device=device, num_kv_blocks=blocks, max_num_seqs=seqs,
                                      max_model_len=1024, dtype=dtype, **kw), model_cfg=self.mc, model=model)

    def oracle(self, tokens):
        key = tuple(tokens)
        if key not in self._oracle:
            self._oracle[key] = plain.forward(self.cfg, self.W, list(tokens)).float()
        return self._oracle[key]


def toks(n, vocab, seed):
    g = torch.Generator().manual_seed(seed)
    return torch.randint(0, vocab, (n,), generator=g).tolist()


def rel_err(got, want):
    """Per row: rms of the mean-free difference over the rms of the mean-free expectation."""
    d = got.double().cpu() - want.double()
    d = d - d.mean(-1, keepdim=True)
    w = want.double() - want.double().mean(-1, keepdim=True)
    return (d.pow(2).mean(-1).sqrt() / w.pow(2).mean(-1).sqrt()).max().item()


TOL = {"float32": 2e-4, "bfloat16": 0.08}


def feed_all(eng, rid, tokens, cuts):
    """Feed ``tokens`` in portions of the given sizes (the last size repeats), all positions wanted."""
    rows, at, i = [], 0, 0
    while at < len(tokens):
        n = min(cuts[min(i, len(cuts) - 1)], len(tokens) - at)
        last = at + n == len(tokens)
        rows.append(eng.feed([(rid, tokens[at:at + n], list(range(n)))], [rid] if last else []))
        at += n
        i += 1
    return torch.cat(rows)


@pytest.fixture(scope="module")
def bench_a():
    return Bench(cfg_a())


@pytest.fixture(scope="module")
def bench_sharp():
    return Bench(cfg_a(scale=1.2), seed=3, sharpen=3.0)


# ---- mechanisms alone ----------------------------------------------------------------------------------------------
def _seg(device, runs):
    """runs: (rows, first position, slot) -> seg, tok_seg"""
    seg, ts, r = [], [], 0
    for j, (n, p0, slot) in enumerate(runs):
        seg.append((r, n, p0, slot))
        ts += [j] * n
        r += n
    return (torch.tensor(seg, dtype=torch.int32, device=device), torch.tensor(ts, dtype=torch.int32, device=device))


@pytest.mark.parametrize("device", DEVICES)
def test_rotary_table(device):
    for rot in (_attn()["rot"], _attn(scaling=False)["rot"], {"base": 250.0, "dims": 6,
                                                               "scaling": {"factor": 16.0, "original": 32, "fast": 4.0,
                                                                           "slow": 0.5}}):
        t = bx.rotary_table(300, rot, device).cpu().double()
        cos, sin = plain.rotary_tables(300, rot)
        half = rot["dims"] // 2
        assert torch.allclose(t[:, :half], cos, atol=3e-5) and torch.allclose(t[:, half:], sin, atol=3e-5)


@pytest.mark.parametrize("device", DEVICES)
@pytest.mark.parametrize("d", [70, 2500, 4200])   # (the kernels keep rows of up to 1024 / 4096 values in registers)
def test_norm_and_shift(device, d):
    torch.manual_seed(0)
    T = 9
    x = torch.randn(T, d) * 3 + 1
    w, b, mu = torch.randn(d), torch.randn(d), torch.rand(d)
    want = plain.token_shift(plain.layer_norm(x.double(), w.double(), b.double(), 1e-5), mu.double())
    # the same rows as two runs of one sequence (5 + 4 rows) and, between them in the batch, another sequence's run
    other = torch.randn(3, d)
    state = torch.full((3, d), float("nan"), device=device)
    out1 = torch.empty(5, d, device=device)
    last = torch.empty(2, d, device=device)
    seg, ts = _seg(device, [(5, 0, 2)])
    hops.ln_shift(x[:5].to(device), w.to(device), b.to(device), 1e-5, out1, mu.to(device), ts, seg, state, last)
    hops.scatter_rows(state, seg, last)
    xb = torch.cat([other, x[5:]]).to(device)
    seg, ts = _seg(device, [(3, 0, 0), (4, 5, 2)])
    out2 = torch.empty(7, d, device=device)
    hops.ln_shift(xb, w.to(device), b.to(device), 1e-5, out2, mu.to(device), ts, seg, state, last)
    got = torch.cat([out1, out2[3:]]).cpu().double()
    assert torch.allclose(got, want, atol=2e-5)
    want_o = plain.token_shift(plain.layer_norm(other.double(), w.double(), b.double(), 1e-5), mu.double())
    assert torch.allclose(out2[:3].cpu().double(), want_o, atol=2e-5)
    # plain norm (no shift), bf16 output
    o = torch.empty(T, d, dtype=torch.bfloat16, device=device)
    hops.ln_shift(x.to(device), w.bfloat16().to(device), b.bfloat16().to(device), 1e-5, o)
    ref = plain.layer_norm(x.double(), w.bfloat16().double(), b.bfloat16().double(), 1e-5)
    assert torch.allclose(o.cpu().double(), ref, atol=0.05, rtol=0.01)


@pytest.mark.parametrize("device", DEVICES)
@pytest.mark.parametrize("d", [52, 2500, 4200])
def test_add_norm_gelu_side_depth(device, d):
    torch.manual_seed(1)
    T, F, sd, V = 6, 30, 5, 40
    x, y = torch.randn(T, d), torch.randn(T, d) * 2
    w, b, w2, b2 = (torch.randn(d) for _ in range(4))
    xd = x.clone().to(device)
    h2 = torch.empty(T, d, device=device)
    hops.add_ln(xd, y.to(device), w.to(device), b.to(device), 1e-6, h2, w2.to(device), b2.to(device))
    x1 = x.double() + plain.layer_norm(y.double(), w.double(), b.double(), 1e-6)
    assert torch.allclose(xd.cpu().double(), x1, atol=1e-5)
    assert torch.allclose(h2.cpu().double(), plain.layer_norm(x1, w2.double(), b2.double(), 1e-6), atol=2e-5)
    xc = x.clone().to(device)
    hops.add_ln(xc, y.to(device), w.to(device), b.to(device), 1e-6, h2)
    assert torch.allclose(h2.cpu(), xc.cpu()) and torch.allclose(xc.cpu().double(), x1, atol=1e-5)
    gu = torch.randn(T, 2 * F) * 2
    a = torch.empty(T, F, device=device)
    hops.gelu_mul(gu.to(device), a)
    assert torch.allclose(a.cpu().double(), plain.gelu_tanh(gu[:, :F].double()) * gu[:, F:].double(), atol=1e-5)
    # token input + depth average over a stack of three earlier results
    tokens = torch.randint(0, V, (T,))
    emb, sgate = torch.randn(V, 3 * sd), torch.randn(T, sd)
    g = torch.empty(T, sd, device=device)
    hops.side_gate(sgate.to(device), tokens.to(device), emb.to(device), sd, g)
    want_g = plain.gelu_tanh(sgate.double()) * emb[tokens][:, sd:2 * sd].double()
    assert torch.allclose(g.cpu().double(), want_g, atol=1e-5)
    stack = torch.randn(5, T, d)
    sw, dwa = torch.randn(d), torch.rand(4)
    sd_dev = stack.clone().to(device)
    xs = x.clone().to(device)
    hops.side_dwa(xs, y.to(device), sw.to(device), 1e-6, sd_dev, 2, dwa.to(device))
    x2 = x.double() + plain.rms_unit(y.double(), 1e-6) * sw.double()
    want = sum(dwa[j].double() * stack[j].double() for j in range(3)) + dwa[3].double() * x2
    assert torch.allclose(sd_dev[3].cpu().double(), x2, atol=1e-5)
    assert torch.allclose(xs.cpu().double(), want, atol=1e-5)


def _paged(device, rows, page=16, n_pages=12, order=(7, 2, 9, 4, 0, 11)):
    """rows [n, w] scattered into a page pool through a shuffled page list."""
    cache = torch.full((n_pages, page, rows.shape[1]), float("nan"), device=device)
    need = -(-rows.shape[0] // page)
    bt = torch.tensor([list(order[:need]) + [0] * (8 - need)], dtype=torch.int32, device=device)
    flat = cache.view(-1, rows.shape[1])
    for j in range(rows.shape[0]):
        flat[order[j // page] * page + j % page] = rows[j].to(device)
    flat[torch.isnan(flat)] = 1e4  # rows beyond the sequence: finite garbage that must never be attended
    return cache, bt


@pytest.mark.parametrize("device", DEVICES)
@pytest.mark.parametrize("R,rd,H", [(40, 16, 3), (72, 8, 5), (200, 24, 2), (448, 64, 9)])
def test_latent_attention_single_keys(device, R, rd, H):
    """One key is made to dominate each row's softmax: the output must be that key's latent, wherever the key lies
    (the first keys, both sides of every page border, the row's own position) - and a key one past the row's position
    must never be seen."""
    torch.manual_seed(2)
    n = 70
    kv = torch.randn(n, R + rd)
    kv = kv / kv.norm(dim=-1, keepdim=True)
    cache, bt = _paged(device, kv)
    targets = [0, 1, 15, 16, 17, 31, 32, 47, 48, 63, 64, 69]
    pos = [69, 69, 15, 16, 17, 31, 32, 47, 48, 63, 64, 69]   # the target is the row's own position from 15 on
    T = len(targets)
    q = torch.stack([kv[j] for j in targets]) * 60.0         # score 60 for the target, < 60 elsewhere
    q_lat = q[:, :R][None].repeat(H, 1, 1).contiguous()
    q_rot = q[:, R:][:, None].repeat(1, H, 1).contiguous()
    out = torch.empty(H, T, R, device=device)
    seg, ts = _seg(device, [(T, 0, 0)])
    positions = torch.tensor(pos, device=device)
    hops.latent_attn(q_lat.to(device), q_rot.to(device), cache, bt, ts, seg, positions, 1.0, out)
    for i, j in enumerate(targets):
        assert torch.allclose(out[:, i].cpu(), kv[j, :R].expand(H, R), atol=2e-3), (i, j)
    # the same queries one position short of their target: the target is outside and must not win
    short = torch.tensor([max(p - 1, 0) if t == p else p for t, p in zip(targets, pos)], device=device)
    hops.latent_attn(q_lat.to(device), q_rot.to(device), cache, bt, ts, seg, short, 1.0, out)
    for i, (j, p) in enumerate(zip(targets, pos)):
        if j == p and p > 0:
            assert (out[:, i].cpu() - kv[j, :R]).abs().max() > 0.05, (i, j)
    # against the plain softmax over all visible keys, diffuse scores, per head different queries
    q_lat, q_rot = torch.randn(H, T, R), torch.randn(T, H, rd)
    hops.latent_attn(q_lat.to(device), q_rot.to(device), cache, bt, ts, seg, positions, 0.3, out)
    for i, p in enumerate(pos):
        s = (q_lat[:, i].double() @ kv[:p + 1, :R].double().T + q_rot[i].double() @ kv[:p + 1, R:].double().T) * 0.3
        want = torch.softmax(s, -1) @ kv[:p + 1, :R].double()
        assert torch.allclose(out[:, i].cpu().double(), want, atol=1e-5), i


@pytest.mark.gpu
@pytest.mark.parametrize("R,rd,H", [(64, 16, 3), (128, 32, 6), (256, 16, 32), (512, 64, 40), (96, 16, 1), (32, 48, 9)])
def test_latent_attention_matrix_cores(R, rd, H):
    """The bf16 matrix-core kernel: a 40-token portion of a 150-token sequence beside another sequence's single
    token. Every row's query singles out one key - the first keys, both sides of page and 128-key block borders, the
    row's own position and the one before - and must return that key's latent; then diffuse queries against the plain
    softmax."""
    device = "cuda:0"
    torch.manual_seed(5)
    nA, nB, page = 150, 37, 16
    kvA = torch.nn.functional.normalize(torch.randn(nA, R + rd), dim=-1).bfloat16()
    kvB = torch.nn.functional.normalize(torch.randn(nB, R + rd), dim=-1).bfloat16()
    cache = torch.zeros(24, page, R + rd, dtype=torch.bfloat16, device=device)
    orderA, orderB = [7, 2, 9, 4, 0, 11, 20, 13, 5, 16], [3, 21, 8]
    bt = torch.zeros(2, 16, dtype=torch.int32, device=device)
    bt[0, :len(orderA)] = torch.tensor(orderA)
    bt[1, :len(orderB)] = torch.tensor(orderB)
    flat = cache.view(-1, R + rd)
    for kv, order in ((kvA, orderA), (kvB, orderB)):
        for j in range(kv.shape[0]):
            flat[order[j // page] * page + j % page] = kv[j].to(device)
    cache_t = cache[:, :, :R].transpose(1, 2).contiguous()
    posA = list(range(110, 150))
    pos = posA + [nB - 1]
    T = len(pos)
    cands = [0, 1, 15, 16, 17, 31, 32, 111, 112, 127, 128, 129]
    targets = [[c for c in cands + [p - 1, p] if c <= p][(i * 5) % len([c for c in cands + [p - 1, p] if c <= p])]
               for i, p in enumerate(posA)] + [nB - 1]
    kvs = [kvA] * len(posA) + [kvB]
    tt = hops.tile_tokens(H)
    tiles = [(a, min(tt, 40 - a), 0, 0) for a in range(0, 40, tt)] + [(40, 1, 1, 0)]
    tiles = torch.tensor(tiles, dtype=torch.int32, device=device)
    seg, ts = _seg(device, [(40, 110, 0), (1, nB - 1, 1)])
    positions = torch.tensor(pos, device=device)
    q = torch.stack([kvs[i][j].float() for i, j in enumerate(targets)]) * 80.0
    q_lat = q[:, :R][None].repeat(H, 1, 1).bfloat16().contiguous().to(device)
    q_rot = q[:, R:][:, None].repeat(1, H, 1).bfloat16().contiguous().to(device)
    out = torch.empty(H, T, R, dtype=torch.bfloat16, device=device)
    hops.latent_attn(q_lat, q_rot, cache, bt, ts, seg, positions, 1.0, out, cache_t, tiles)
    for i, j in enumerate(targets):
        assert torch.allclose(out[:, i].float().cpu(), kvs[i][j, :R].float().expand(H, R), atol=6e-3), (i, pos[i], j)
    q_lat = torch.randn(H, T, R).bfloat16()
    q_rot = torch.randn(T, H, rd).bfloat16()
    hops.latent_attn(q_lat.to(device), q_rot.to(device), cache, bt, ts, seg, positions, 0.4, out, cache_t, tiles)
    ref = torch.empty(H, T, R, dtype=torch.bfloat16, device=device)
    hops.latent_attn(q_lat.to(device), q_rot.to(device), cache, bt, ts, seg, positions, 0.4, ref)  # vector kernel
    for i, p in enumerate(pos):
        kv = kvs[i][:p + 1].double()
        s = (q_lat[:, i].double() @ kv[:, :R].T + q_rot[i].double() @ kv[:, R:].T) * 0.4
        want = torch.softmax(s, -1) @ kv[:, :R]
        assert torch.allclose(out[:, i].double().cpu(), want, atol=3e-3), (i, p)
        assert torch.allclose(ref[:, i].double().cpu(), want, atol=3e-3), (i, p)


@pytest.mark.gpu
@pytest.mark.parametrize("R,rd,H", [(64, 16, 3), (512, 64, 40)])
def test_latent_attention_split_key_ranges(R, rd, H):
    """A decode step of three sequences (1100, 300 and 5 cached keys): the launch deals each tile's key blocks over
    several workgroups and merges them; sequences shorter than a split's range leave it empty."""
    device = "cuda:0"
    torch.manual_seed(7)
    lens, page = [1100, 300, 5], 16
    cache = torch.zeros(100, page, R + rd, dtype=torch.bfloat16, device=device)
    perm = torch.randperm(100).tolist()
    bt = torch.zeros(3, 80, dtype=torch.int32, device=device)
    kvs, at = [], 0
    for r, n in enumerate(lens):
        kv = torch.nn.functional.normalize(torch.randn(n, R + rd), dim=-1).bfloat16()
        kvs.append(kv)
        need = -(-n // page)
        pages = perm[at:at + need]
        at += need
        bt[r, :need] = torch.tensor(pages)
        flat = cache.view(-1, R + rd)
        for j in range(n):
            flat[pages[j // page] * page + j % page] = kv[j].to(device)
    cache_t = cache[:, :, :R].transpose(1, 2).contiguous()
    seg, ts = _seg(device, [(1, n - 1, r) for r, n in enumerate(lens)])
    positions = torch.tensor([n - 1 for n in lens], device=device)
    tiles = torch.tensor([(r, 1, r, 0) for r in range(3)], dtype=torch.int32, device=device)
    assert hops.attn_splits(3, H, max(lens)) > 1
    q_lat, q_rot = torch.randn(H, 3, R).bfloat16(), torch.randn(3, H, rd).bfloat16()
    out = torch.empty(H, 3, R, dtype=torch.bfloat16, device=device)
    hops.latent_attn(q_lat.to(device), q_rot.to(device), cache, bt, ts, seg, positions, 0.5, out, cache_t, tiles,
                     max_keys=max(lens))
    for i, n in enumerate(lens):
        kv = kvs[i].double()
        sc = (q_lat[:, i].double() @ kv[:, :R].T + q_rot[i].double() @ kv[:, R:].T) * 0.5
        want = torch.softmax(sc, -1) @ kv[:, :R]
        assert torch.allclose(out[:, i].double().cpu(), want, atol=3e-3), i
    # single dominant keys in the first, a middle and the last split
    for j in (0, 640, 1099):
        q = kvs[0][j].float() * 80.0
        ql = q[:R][None, None].repeat(H, 3, 1).bfloat16().contiguous().to(device)
        qr = q[R:][None, None].repeat(3, H, 1).bfloat16().contiguous().to(device)
        hops.latent_attn(ql, qr, cache, bt, ts, seg, positions, 1.0, out, cache_t, tiles, max_keys=max(lens))
        assert torch.allclose(out[:, 0].float().cpu(), kvs[0][j, :R].float().expand(H, R), atol=6e-3), j


@pytest.mark.gpu
@pytest.mark.parametrize("H,rd", [(32, 64), (16, 0), (40, 64), (1, 0)])
@pytest.mark.parametrize("window,sink", [(0, False), (70, True)])
def test_latent_decode_block_edges(H, rd, window, sink):
    """kv_rank 512: contexts around the edges of pages and 64-key blocks, a tile of two tokens where the heads allow, several
    splits (some empty), windows and sinks; what lies in the pages behind the last position is NaN. Latents of unit length: the
    scores are up to 4.5 in bf16 products (relative 2^-9 each way, 0.02), weights rounded to bf16 (2^-9), outputs below 1."""
    device, R, page = "cuda:0", 512, 16
    torch.manual_seed(11)
    lens = [1, 2, 16, 17, 63, 64, 65, 80, 127, 128, 129, 193, 300]
    new = 2 if H <= 16 else 1
    pages = [-(-(n + new - 1) // page) for n in lens]
    cache = torch.full((sum(pages), page, R + rd), float("nan"), dtype=torch.bfloat16, device=device)
    perm, at, kvs = torch.randperm(sum(pages)).tolist(), 0, []
    bt = torch.zeros(len(lens), max(pages), dtype=torch.int32, device=device)
    pos, tiles = [], []
    for r, n in enumerate(lens):
        kv = torch.nn.functional.normalize(torch.randn(n + new - 1, R + rd), dim=-1).bfloat16()
        kvs.append(kv)
        ids = perm[at:at + pages[r]]
        at += pages[r]
        bt[r, :pages[r]] = torch.tensor(ids)
        for j in range(0, len(kv), page):
            cache[ids[j // page], :len(kv[j:j + page])] = kv[j:j + page].to(device)
        tiles.append((len(pos), new, r, 0))
        pos += [n - 1 + i for i in range(new)]
    T = len(pos)
    q_lat, q_rot = torch.randn(H, T, R).bfloat16(), torch.randn(T, H, rd).bfloat16()
    sk = torch.randn(H) if sink else None
    cache_t = cache[:, :, :R].transpose(1, 2).contiguous()
    g = [t.to(device) for t in (q_lat, q_rot)]
    tt, ps = torch.tensor(tiles, dtype=torch.int32, device=device), torch.tensor(pos, device=device)
    for ns in (1, 3):
        out = torch.empty(T, H, R, dtype=torch.bfloat16, device=device).transpose(0, 1)
        po, pml = (torch.empty(ns, H, T, w, device=device) for w in (R, 2))
        hops.ext().hy_latent_attn_mfma(*g, cache, cache_t, bt, tt, hops.tile_tokens(H), ps, 0.3, out, ns,
                                       po if ns > 1 else None, pml if ns > 1 else None, window,
                                       sk.to(device) if sink else None)
        for i, p in enumerate(pos):
            lo = max(0, p - window + 1) if window else 0
            kv = kvs[i // new][lo:p + 1].double()
            s = (q_lat[:, i].double() @ kv[:, :R].T + q_rot[i].double() @ kv[:, R:].T) * 0.3
            if sink:
                s = torch.cat([s, sk.double()[:, None]], 1)
            want = torch.softmax(s, -1)[:, :len(kv)] @ kv[:, :R]
            assert torch.allclose(out[:, i].double().cpu(), want, atol=3e-3), (ns, i, p)


def cfg_m():
    """Sizes the matrix-core attention kernel takes (latent 64, rotary part 16), two attention layers sharing a cache."""
    ff = {"kind": "dense", "ff": 96}
    return {"architecture": "Budurax", "vocab": 173, "width": 80, "norm": {"eps": 1e-5}, "token_side": {"dim": 4},
            "layers": [{"type": "latent_attention", "mixer": _attn(5, 16, 16, 16, 24, 64), "mlp": ff},
                       {"type": "mamba2", "mixer": _mamba(2, 16, 8, 1, 2, 4), "mlp": ff},
                       {"type": "latent_attention", "mixer": _attn(5, 16, 16, 16, 24, 64, kv_from=0), "mlp": ff}]}


@pytest.mark.gpu
def test_matrix_core_attention_in_the_engine():
    """bf16 on the GPU with an eligible latent size: whole prompt, portions, single tokens and a mixed batch through
    the matrix-core kernel against the plain model, and against the same engine in fp32 (vector kernel)."""
    b = Bench(cfg_m(), seed=11, sharpen=2.0)
    t, u = toks(300, 173, 1), toks(41, 173, 2)
    eng = b.engine("cuda:0", "bfloat16", blocks=40)
    assert any(p is not None for p in eng.model.pages_t)
    assert rel_err(feed_all(eng, "w", t, [300]), b.oracle(t)) < TOL["bfloat16"]
    assert rel_err(feed_all(eng, "c", t, [130, 2, 61, 1, 1, 1, 40, 1]), b.oracle(t)) < TOL["bfloat16"]
    got_t, got_u = [], []
    got_t.append(eng.feed([("t", t[:200], list(range(200)))]))
    out = eng.feed([("u", u[:40], list(range(40))), ("t", t[200:201], [0])])
    got_u.append(out[:40])
    got_t.append(out[40:])
    out = eng.feed([("t", t[201:], list(range(99))), ("u", u[40:], [0])], ["t", "u"])
    got_t.append(out[:99])
    got_u.append(out[99:])
    assert rel_err(torch.cat(got_t), b.oracle(t)) < TOL["bfloat16"]
    assert rel_err(torch.cat(got_u), b.oracle(u)) < TOL["bfloat16"]
    assert eng.kvm.num_free() == 40


@pytest.mark.gpu
def test_chunk_parallel_scan():
    """Long segments scanned in chunks (zero-state scan, ordered rebuild of the entry states, second scan) against the
    token-by-token reference: a fresh 700-row segment, a 3-row one and a 600-row one that continue stored states."""
    from kafka_llm_service_amd.ops import hybrid_reference as href

    device = "cuda:0"
    torch.manual_seed(6)
    Hh, P, N, G = 6, 24, 40, 2
    inner, C = Hh * P, Hh * P + 2 * G * N
    runs = [(700, 0, 1), (3, 5, 0), (600, 40, 2)]
    T = sum(r[0] for r in runs)
    xbc, proj = torch.randn(T, C) / 2, torch.randn(T, inner + C + Hh)
    dt_bias, A_log, D = torch.randn(Hh) / 2 - 2.0, torch.rand(Hh), torch.randn(Hh)
    state0 = torch.randn(3, Hh, N, P)
    seg, ts = _seg("cpu", runs)
    want_state, want_y = state0.clone(), torch.empty(T, inner)
    href.ssm_scan(xbc, proj, inner + C, dt_bias, A_log, D, Hh, P, N, G, ts, seg, want_state, want_y)
    plan = hops.scan_chunks(seg.numpy(), Hh)
    assert plan is not None and plan[3] == 3 and plan[0].shape[0] == 3 + 1 + 3
    dplan = tuple(torch.from_numpy(a).to(device) for a in plan[:3]) + (plan[3],)
    state, y = state0.clone().to(device), torch.empty(T, inner, device=device)
    hops.ssm_scan_chunked(xbc.to(device), proj.to(device), inner + C, dt_bias.to(device), A_log.to(device),
                          D.to(device), Hh, P, N, G, dplan, state, y)
    assert torch.allclose(y.cpu(), want_y, atol=2e-4, rtol=2e-4)
    assert torch.allclose(state.cpu(), want_state, atol=2e-4, rtol=2e-4)
    assert hops.scan_chunks(_seg("cpu", [(100, 0, 0)])[0].numpy(), Hh) is None      # short: plain scan
    assert hops.scan_chunks(_seg("cpu", [(600, 0, 0)])[0].numpy(), 4096) is None    # enough workgroups already


@pytest.mark.gpu
def test_long_prompt_in_the_engine():
    """A 900-token prompt in one step, and in portions of 600 + 300 (chunk-parallel scan in both), beside a short
    request, against the plain model (fp32)."""
    b = Bench(cfg_a(), seed=13)
    t, u = toks(900, 211, 4), toks(30, 211, 5)
    eng = b.engine("cuda:0", "float32", blocks=80)
    assert rel_err(feed_all(eng, "w", t, [900]), b.oracle(t)) < TOL["float32"]
    got = [eng.feed([("t", t[:600], list(range(600))), ("u", u[:29], list(range(29)))])]
    got.append(eng.feed([("u", u[29:], [0]), ("t", t[600:], list(range(300)))], ["t", "u"]))
    got_t = torch.cat([got[0][:600], got[1][1:]])
    got_u = torch.cat([got[0][600:], got[1][:1]])
    assert rel_err(got_t, b.oracle(t)) < TOL["float32"]
    assert rel_err(got_u, b.oracle(u)) < TOL["float32"]


@pytest.mark.gpu
def test_streamed_projections():
    """Decode-sized steps run the projections on the weight-streaming GEMM when their shapes fit it (width 256 here):
    single tokens and a 100-token portion (streamed) against the plain model, and the same steps with streaming off."""
    ff = {"kind": "dense", "ff": 512}
    cfg = {"architecture": "Budurax", "vocab": 320, "width": 256, "norm": {"eps": 1e-5}, "token_side": {"dim": 8},
           "layers": [{"type": "latent_attention", "mixer": _attn(4, 32, 32, 32, 64, 64), "mlp": ff},
                      {"type": "mamba2", "mixer": _mamba(8, 32, 16, 2, 2, 4), "mlp": ff}]}
    b = Bench(cfg, seed=12)
    t = toks(140, 320, 3)
    outs = []
    for mode in ("stream", "blas"):
        eng = b.engine("cuda:0", "bfloat16", decode_gemm=mode)
        assert eng.model.stream == (mode == "stream")
        outs.append(feed_all(eng, "r", t, [100, 1]))
        assert rel_err(outs[-1], b.oracle(t)) < TOL["bfloat16"]
    assert rel_err(outs[0], outs[1].float().cpu()) < TOL["bfloat16"]


@pytest.mark.parametrize("device", DEVICES)
def test_conv_and_scan_portions(device):
    """Convolution tail and state-space state carried over portions of 1, 2, 3 and 7 rows, with another sequence's run
    in the same launch, against the plain whole-sequence functions; the slot starts out holding NaN."""
    torch.manual_seed(3)
    Hh, P, N, G, taps, T = 4, 12, 20, 2, 4, 23
    inner, C = Hh * P, Hh * P + 2 * G * N
    proj = torch.randn(T, inner + C + Hh)
    w, b = torch.randn(C, taps) / 2, torch.randn(C) / 4
    dt_bias, A_log, D = torch.randn(Hh) / 2, torch.rand(Hh), torch.randn(Hh)
    xbc_want = plain.silu(plain.causal_conv(proj[:, inner:inner + C].double(), w.double(), b.double()))
    # the recurrence, written out once more for this test
    S = torch.zeros(Hh, N, P, dtype=torch.float64)
    y_want = torch.zeros(T, inner, dtype=torch.float64)
    grp = torch.arange(Hh) // (Hh // G)
    for t in range(T):
        x = xbc_want[t, :inner].view(Hh, P)
        B, Cc = xbc_want[t, inner:inner + G * N].view(G, N)[grp], xbc_want[t, inner + G * N:].view(G, N)[grp]
        dt = torch.log1p(torch.exp(proj[t, inner + C:].double() + dt_bias.double()))
        S = torch.exp(-torch.exp(A_log.double()) * dt)[:, None, None] * S + dt[:, None, None] * B[:, :, None] * x[:, None]
        y_want[t] = (torch.einsum("hnp,hn->hp", S, Cc) + D.double()[:, None] * x).reshape(-1)
    conv_state = torch.full((3, taps - 1, C), float("nan"), device=device)
    ssm_state = torch.full((3, Hh, N, P), float("nan"), device=device)
    other = torch.randn(2, inner + C + Hh)
    got_x, got_y, at = [], [], 0
    for n in (1, 2, 3, 7, 1, 9):
        rows = torch.cat([other, proj[at:at + n]]).to(device)
        seg, ts = _seg(device, [(2, 0, 0), (n, at, 2)])
        xbc = torch.empty(2 + n, C, device=device)
        hops.conv_silu(rows, inner, w.to(device), b.to(device), ts, seg, conv_state, xbc)
        y = torch.empty(2 + n, inner, device=device)
        hops.ssm_scan(xbc, rows, inner + C, dt_bias.to(device), A_log.to(device), D.to(device), Hh, P, N, G, ts, seg,
                      ssm_state, y)
        got_x.append(xbc[2:].cpu())
        got_y.append(y[2:].cpu())
        at += n
    assert at == T
    assert torch.allclose(torch.cat(got_x).double(), xbc_want, atol=1e-5)
    assert torch.allclose(torch.cat(got_y).double(), y_want, atol=1e-4, rtol=1e-4)
    assert torch.allclose(ssm_state[2].cpu().double(), S, atol=1e-4, rtol=1e-4)
    # gate + grouped norm
    yv, z, nw = torch.randn(5, inner), torch.randn(5, inner + 3), torch.randn(inner)
    out = torch.empty(5, inner, device=device)
    hops.gated_norm(yv.to(device), z.to(device), nw.to(device), 4, 1e-5, out)
    v = (yv.double() * plain.silu(z[:, :inner].double())).view(5, 4, inner // 4)
    want = plain.rms_unit(v, 1e-5).reshape(5, inner) * nw.double()
    assert torch.allclose(out.cpu().double(), want, atol=1e-5)


@pytest.mark.parametrize("device", DEVICES)
@pytest.mark.parametrize("P,N", [(64, 128), (32, 32), (40, 9), (128, 64)])
def test_scan_state_sizes(device, P, N):
    torch.manual_seed(4)
    Hh, G, T = 2, 1, 11
    inner, C = Hh * P, Hh * P + 2 * G * N
    xbc, proj = torch.randn(T, C) / 2, torch.randn(T, Hh)
    dt_bias, A_log, D = torch.zeros(Hh), torch.rand(Hh), torch.ones(Hh)
    state = torch.zeros(1, Hh, N, P, device=device)
    y = torch.empty(T, inner, device=device)
    seg, ts = _seg(device, [(T, 0, 0)])
    hops.ssm_scan(xbc.to(device), proj.to(device), 0, dt_bias.to(device), A_log.to(device), D.to(device), Hh, P, N, G,
                  ts, seg, state, y)
    S = torch.zeros(Hh, N, P, dtype=torch.float64)
    for t in range(T):
        x = xbc[t, :inner].double().view(Hh, P)
        B, Cc = xbc[t, inner:inner + N].double(), xbc[t, inner + N:].double()
        dt = torch.log1p(torch.exp(proj[t].double()))
        S = torch.exp(-torch.exp(A_log.double()) * dt)[:, None, None] * S + dt[:, None, None] * B[None, :, None] * x[:, None]
        want = (torch.einsum("hnp,n->hp", S, Cc) + x).reshape(-1)
        assert torch.allclose(y[t].cpu().double(), want, atol=1e-4, rtol=1e-4), t
    # a step of single tokens (the decode kernel): the same sequence goes on, beside another one's first token in a
    # slot that holds NaN
    state = torch.cat([state, torch.full_like(state, float("nan"))])
    xb2, pr2 = torch.randn(2, C) / 2, torch.randn(2, Hh)
    seg, ts = _seg(device, [(1, T, 0), (1, 0, 1)])
    y2 = torch.empty(2, inner, device=device)
    hops.ssm_scan(xb2.to(device), pr2.to(device), 0, dt_bias.to(device), A_log.to(device), D.to(device), Hh, P, N, G,
                  ts, seg, state, y2)
    for r, S0 in ((0, S), (1, torch.zeros_like(S))):
        x = xb2[r, :inner].double().view(Hh, P)
        B, Cc = xb2[r, inner:inner + N].double(), xb2[r, inner + N:].double()
        dt = torch.log1p(torch.exp(pr2[r].double()))
        S1 = torch.exp(-torch.exp(A_log.double()) * dt)[:, None, None] * S0 + dt[:, None, None] * B[None, :, None] * x[:, None]
        want = (torch.einsum("hnp,n->hp", S1, Cc) + x).reshape(-1)
        assert torch.allclose(y2[r].cpu().double(), want, atol=1e-4, rtol=1e-4), r
        assert torch.allclose(state[r].cpu().double(), S1, atol=1e-4, rtol=1e-4), r


# ---- the model in the engine ---------------------------------------------------------------------------------------
@pytest.mark.parametrize("device", DEVICES)
@pytest.mark.parametrize("dtype", ["float32", "bfloat16"])
def test_whole_prompt_and_layers(bench_a, device, dtype):
    t = toks(45, 211, 1)
    eng = bench_a.engine(device, dtype)
    lay = []
    got = eng.feed([("a", t, list(range(len(t))))], ["a"], layers_out=lay)
    assert rel_err(got, bench_a.oracle(t)) < TOL[dtype]
    if dtype == "float32":
        _, want_l = plain.forward(bench_a.cfg, bench_a.W, t, return_layers=True)
        for i, x in enumerate(lay):
            assert torch.allclose(x.cpu().double(), want_l[i], atol=2e-3, rtol=1e-4), f"layer {i}"


@pytest.mark.parametrize("device", DEVICES)
def test_other_sizes_and_no_extras(device):
    for b in (Bench(cfg_b(), seed=5, extras=False), Bench(cfg_b(), seed=6)):
        t = toks(37, 97, 2)
        eng = b.engine(device)
        assert rel_err(feed_all(eng, "w", t, [len(t)]), b.oracle(t)) < TOL["float32"]
        assert rel_err(feed_all(eng, "c", t, [2, 3, 16, 1, 1, 5]), b.oracle(t)) < TOL["float32"]


@pytest.mark.parametrize("device", DEVICES)
def test_models_of_one_layer_kind(device):
    """Only Mamba-2 layers (the page pool stays unused), only attention layers (no recurrent matrices), one tap."""
    ff = {"kind": "dense", "ff": 56}
    only_m = {"architecture": "Budurax", "vocab": 131, "width": 40, "norm": {"eps": 1e-6},
              "layers": [{"type": "mamba2", "mixer": _mamba(2, 10, 6, 2, 1, 1), "mlp": ff},
                         {"type": "mamba2", "mixer": _mamba(4, 5, 3, 1, 2, 8), "mlp": None}]}
    only_a = {"architecture": "Budurax", "vocab": 131, "width": 40, "norm": {"eps": 1e-6}, "token_side": {"dim": 3},
              "layers": [{"type": "latent_attention", "mixer": _attn(2, 8, 4, 4, 6, 12), "mlp": None},
                         {"type": "latent_attention", "mixer": _attn(7, 4, 4, 4, 3, 12, kv_from=0), "mlp": ff}]}
    for cfg in (only_m, only_a):
        b = Bench(cfg, seed=21)
        t = toks(50, 131, 8)
        eng = b.engine(device)
        assert rel_err(feed_all(eng, "w", t, [50]), b.oracle(t)) < TOL["float32"]
        assert rel_err(feed_all(eng, "c", t, [7, 2, 20, 1]), b.oracle(t)) < TOL["float32"]


@pytest.mark.parametrize("device", DEVICES)
@pytest.mark.parametrize("cuts", [[1], [2], [3, 2], [16], [17, 15, 1, 2], [31, 1, 1, 1, 33], [64, 2]])
def test_portions_and_decoding(bench_sharp, device, cuts):
    """Prompt portions of several sizes (down to two tokens, [1] = everything decoded token by token: 100 steps) give
    the whole prompt's logits at every position; the softmax is peaky, so a key lost at a page or portion border
    shows."""
    t = toks(100, 211, 7)
    eng = bench_sharp.engine(device)
    assert rel_err(feed_all(eng, "r", t, cuts), bench_sharp.oracle(t)) < TOL["float32"]


@pytest.mark.parametrize("device", DEVICES)
@pytest.mark.parametrize("dtype", ["float32", "bfloat16"])
def test_mixed_batches_and_reuse(bench_sharp, device, dtype):
    """Four unequal requests interleaved in shared steps (portions beside single tokens, a request sitting out a
    step), then more requests through the same two slots and a pool of few pages: every request's logits equal the
    request alone."""
    b = bench_sharp
    reqs = {k: toks(n, 211, 10 + i) for i, (k, n) in enumerate([("a", 70), ("b", 1), ("c", 33), ("d", 18),
                                                                ("e", 50), ("f", 40)])}
    eng = b.engine(device, dtype, blocks=10, seqs=2)   # 160 cached tokens, two slots
    got = {k: [] for k in reqs}
    at = {k: 0 for k in reqs}

    def step(parts):
        entries, end = [], []
        for k, n in parts:
            entries.append((k, reqs[k][at[k]:at[k] + n], list(range(n))))
            at[k] += n
            if at[k] == len(reqs[k]):
                end.append(k)
        out = eng.feed(entries, end)
        r = 0
        for k, n in parts:
            got[k].append(out[r:r + n])
            r += n

    step([("a", 17), ("b", 1)])          # b ends: its slot and page go back
    step([("a", 2), ("c", 30)])          # c takes b's slot; a crosses a page border inside a portion
    step([("c", 1), ("a", 13)])
    step([("a", 1)])                     # c sits out
    step([("c", 1), ("a", 36)])
    step([("a", 1), ("c", 1)])           # both end here: a at 70, c at 33
    assert at["a"] == 70 and at["c"] == 33
    step([("d", 18), ("e", 2)])          # reused slots and pages, fresh state
    step([("e", 47)])
    step([("e", 1), ("f", 40)])
    assert eng.kvm.num_free() == 10 and eng.slots.num_free() == 2
    for k, t in reqs.items():
        assert rel_err(torch.cat(got[k]), b.oracle(t)) < TOL[dtype], k
    st = eng.slots.stats()
    assert st["acquired_total"] == 6


@pytest.mark.parametrize("device", DEVICES)
def test_long_decoding_and_dirty_state(bench_a, device):
    """A short prompt, then 150 single-token steps (the rotary positions pass the YaRN original context, the scan state
    and convolution tail are carried 150 times); the state tensors start out as NaN: a sequence's first portion must
    not read its slot."""
    t = toks(160, 211, 20)
    eng = bench_a.engine(device)
    for group in (eng.v_cache.shift, eng.v_cache.conv, eng.v_cache.ssm):
        for s in group:
            if s is not None:
                s.fill_(float("nan"))
    got = feed_all(eng, "r", t, [10, 1])
    assert torch.isfinite(got).all()
    assert rel_err(got, bench_a.oracle(t)) < TOL["float32"]


@pytest.mark.parametrize("device", DEVICES)
def test_greedy_generation_through_scheduler(bench_a, device):
    """engine.generate: the engine's scheduler, chunked prefill (8-token chunks), slot-limited admission (3 prompts,
    2 slots), sampling kernel; every generated token is the plain model's argmax up to a rounding-sized gap."""
    eng = bench_a.engine(device, seqs=2, max_prefill_chunk=8, max_num_batched_tokens=24)
    prompts = [toks(n, 211, 30 + n) for n in (21, 9, 34)]
    outs = eng.generate(prompts, SamplingParams(temperature=0.0, max_tokens=7, ignore_eos=True))
    assert all(len(o) == 7 for o in outs)
    for p, o in zip(prompts, outs):
        lg = bench_a.oracle(p + o)
        for i, tok in enumerate(o):
            row = lg[len(p) - 1 + i]
            assert (row.max() - row[tok]).item() < 1e-3 * row.abs().max().item(), i
    assert eng.slots.num_free() == 2 and eng.kvm.num_free() == eng.num_blocks


def test_config_registry_and_checkpoint(tmp_path):
    from kafka_llm_service_amd.models.config import get_config

    b = Bench(cfg_b(), seed=8)
    bx.save_checkpoint(b.mc, b.W, tmp_path / "m")
    mc = get_config(str(tmp_path / "m"))
    assert mc.arch == "budurax" and mc.num_layers == 2 and mc.vocab_size == 97
    eng = LLMEngine(EngineConfig(model=str(tmp_path / "m"), weights=str(tmp_path / "m"), device="cpu",
                                 num_kv_blocks=8, max_num_seqs=2, max_model_len=128, dtype="float32"))
    t = toks(20, 97, 9)
    assert rel_err(feed_all(eng, "x", t, [20]), b.oracle(t)) < TOL["float32"]
    bad = copy.deepcopy(b.W)
    bad["l0.mix.q"] = bad["l0.mix.q"][:-1]
    with pytest.raises(ValueError):
        bx.BuduraxLM(b.mc, "cpu").load_tensors(bad)
    assert get_config("budurax-tiny").arch == "budurax"
    assert math.isclose(get_config("budurax-tiny").norm_eps, 1e-6)


def test_trace_runner_command_line(tmp_path):
    """bin/trace_run as a program (reference ops on the CPU): a checkpoint folder, three steps on standard input - a
    new request, two requests in one step, a step in which nothing is wanted - then the logits files, the "done"
    lines and the exit code."""
    import json
    import subprocess
    import sys
    from pathlib import Path

    import numpy as np

    root = Path(__file__).resolve().parents[1]
    b = Bench(cfg_b(), seed=14)
    bx.save_checkpoint(b.mc, b.W, tmp_path / "m")
    t, u = toks(21, 97, 1), toks(6, 97, 2)
    steps = [{"step": 0, "entries": [{"id": "a", "tokens": t[:9], "want": [0, 8]}], "end": []},
             {"step": 1, "entries": [{"id": "b", "tokens": u, "want": [5]}, {"id": "a", "tokens": t[9:20], "want": []}],
              "end": ["b"]},
             {"step": 2, "entries": [{"id": "a", "tokens": t[20:], "want": [0]}], "end": ["a"]}]
    out = subprocess.run([sys.executable, str(root / "bin/trace_run"), "--model", str(tmp_path / "m"), "--dtype",
                          "float32", "--out", str(tmp_path / "o"), "--max-tokens", "64", "--device", "cpu"],
                         input="".join(json.dumps(x) + "\n" for x in steps), capture_output=True, text=True,
                         timeout=300)
    assert out.returncode == 0, out.stderr[-2000:]
    assert [ln for ln in out.stdout.splitlines() if ln.startswith("done")] == ["done 0", "done 1", "done 2"]
    got = {n: torch.from_numpy(np.fromfile(tmp_path / "o" / f"{n}.f32", dtype="<f4").reshape(-1, 97)) for n in range(3)}
    assert rel_err(got[0], b.oracle(t)[[0, 8]]) < TOL["float32"]
    assert rel_err(got[1], b.oracle(u)[[5]]) < TOL["float32"]
    assert rel_err(got[2], b.oracle(t)[[20]]) < TOL["float32"]


def _ssm_want(xbc, raw, dt_bias, A_log, D, Hh, P, N, G, S):
    """The recurrence in float64 over one sequence from state S [Hh, N, P]: (rows [T, Hh P], last state)."""
    grp, rows = torch.arange(Hh) // (Hh // G), []
    x, B, C = (t.double() for t in xbc.split([Hh * P, G * N, G * N], 1))
    dt = torch.nn.functional.softplus(raw.double() + dt_bias.double(), threshold=1e9)
    for t in range(xbc.shape[0]):
        Bt, Ct, xt = B[t].view(G, N)[grp], C[t].view(G, N)[grp], x[t].view(Hh, P)
        S = torch.exp(-torch.exp(A_log.double()) * dt[t])[:, None, None] * S + dt[t][:, None, None] * Bt[:, :, None] * xt[:, None]
        rows.append((torch.einsum("hnp,hn->hp", S, Ct) + D.double()[:, None] * xt).reshape(-1))
    return torch.stack(rows), S


@pytest.mark.gpu
@pytest.mark.parametrize("Hh,P,N,G", [(4, 64, 128, 2), (2, 8, 16, 1), (6, 72, 144, 3), (2, 40, 256, 2), (3, 136, 80, 1)])
@pytest.mark.parametrize("fast", [False, True])
def test_scan_in_matrix_core_chunks(Hh, P, N, G, fast):
    """Segments of 1 .. 300 rows, fresh in slots of NaN and from stored states, in one launch: those of at least
    SSD_CHUNK_MIN rows in chunks on the matrix cores, the others token by token. ``fast``: decays of up to e^-40 a token, a
    chunk's running sum in the thousands. The fp32 factors of the products keep all their bits, so a row's error is bounded by
    the fp32 additions of up to 300 terms: 300 * 2^-24 = 1.8e-5 of the row's largest partial sum, which the bound 2e-5 of the
    head's largest value stands for - and it is no larger than twice the token-by-token kernel's (plus 1e-6)."""
    device = "cuda:0"
    torch.manual_seed(P + N)
    runs = [(300, 0, 0), (1, 0, 1), (hops.SSD_CHUNK_MIN, 0, 2), (hops.SSD_CHUNK_MIN - 1, 7, 3), (128, 3, 4), (129, 0, 5),
            (127, 9, 6), (1, 5, 7)]
    T, inner = sum(r[0] for r in runs), Hh * P
    xbc = (torch.randn(T, inner + 2 * G * N) / 2).bfloat16()
    proj = torch.randn(T, Hh + 3).bfloat16()
    A_log, D = torch.rand(Hh) * 2 + (1.5 if fast else -1.0), torch.randn(Hh)
    dt_bias = torch.randn(Hh) / 2 + (0.0 if fast else -3.0)
    state0 = torch.full((8, Hh, N, P), float("nan"))
    for _, p0, slot in runs:
        if p0:
            state0[slot] = torch.randn(Hh, N, P)
    seg, ts = _seg("cpu", runs)
    want_y, want_S, at = [], [], 0
    for n, p0, slot in runs:
        S = state0[slot].double() if p0 else torch.zeros(Hh, N, P, dtype=torch.float64)
        y, S = _ssm_want(xbc[at:at + n], proj[at:at + n, 3:], dt_bias, A_log, D, Hh, P, N, G, S)
        want_y.append(y)
        want_S.append(S)
        at += n
    want_y = torch.cat(want_y).view(T, Hh, P)
    tabs = tuple(torch.from_numpy(t).to(device) for t in hops.chunk_tables(seg.numpy(), hops.SSD_CHUNK, hops.SSD_CHUNK_MIN))
    xg = xbc.to(device)
    assert hops.ssd_ok(xg, Hh, P, N, G)
    errs = []
    for chunks, rows in ((tabs, (1, hops.SSD_CHUNK_MIN - 1)), (None, (1, 1 << 30))):
        state, y = state0.clone().to(device), torch.full((T, inner), float("nan"), device=device)
        hops.ssm_scan(xg, proj.to(device), 3, dt_bias.to(device), A_log.to(device), D.to(device), Hh, P, N, G, ts.to(device),
                      seg.to(device), state, y, chunks, rows)
        d = (y.cpu().double().view(T, Hh, P) - want_y).abs().amax(-1) / want_y.abs().amax((0, 2))
        ds = max(((state[slot].cpu().double() - S).abs().amax() / S.abs().amax()).item()
                 for (_, _, slot), S in zip(runs, want_S))
        errs.append((d.max().item(), ds))
        assert not torch.isnan(y).any()
    print(errs)
    assert errs[0][0] < 2e-5 and errs[0][1] < 2e-5
    assert errs[0][0] < 2 * errs[1][0] + 1e-6 and errs[0][1] < 2 * errs[1][1] + 1e-6


def test_short_portions_are_scanned_token_by_token():
    """A few dozen rows beside decoded tokens make a step that waits for the host: no chunk tables, no launches for them."""
    for runs, chunks in (([(1, 9, 0), (45, 800, 1)], 0), ([(1, 9, 0), (25, 0, 1), (63, 7, 2)], 0), ([(64, 0, 0)], 1),
                         ([(1, 3, 0), (300, 5, 1), (40, 0, 2)], 3)):
        t = hops.chunk_tables(_seg("cpu", runs)[0].numpy(), hops.SSD_CHUNK, hops.SSD_CHUNK_MIN)
        assert (0 if t is None else len(t[0])) == chunks


@pytest.mark.gpu
@pytest.mark.parametrize("P,N", [(64, 32), (72, 144), (8, 256)])
def test_chunked_scan_of_rates_and_rows_without_bound(P, N):
    """The chunked scan where A_log is past the largest exponent (A = -inf: the state of a token is gone with the next one), and
    with a row whose x is infinite and one whose x is NaN: whatever stands before such a row comes out as it does without it
    (portions that end inside a chunk of 128 and a tile of 32 rows; the same error bound as above)."""
    device = "cuda:0"
    torch.manual_seed(9)
    Hh, G, n = 4, 2, 173
    inner = Hh * P
    xbc = (torch.randn(n, inner + 2 * G * N) / 2).bfloat16()
    proj = torch.randn(n, Hh).bfloat16()
    A_log = torch.tensor([0.3, 89.0, 200.0, 1.0])
    dt_bias, D = torch.randn(Hh) / 2, torch.randn(Hh)
    seg, ts = _seg("cpu", [(n, 0, 0)])
    tabs = tuple(torch.from_numpy(t).to(device) for t in hops.chunk_tables(seg.numpy(), hops.SSD_CHUNK, hops.SSD_CHUNK_MIN))

    def scan(xb):
        state, y = torch.full((1, Hh, N, P), float("nan"), device=device), torch.full((n, inner), float("nan"), device=device)
        hops.ssm_scan(xb.to(device), proj.to(device), 0, dt_bias.to(device), A_log.to(device), D.to(device), Hh, P, N, G,
                      ts.to(device), seg.to(device), state, y, tabs, None)
        return y.cpu().view(n, Hh, P), state.cpu()

    want, S = _ssm_want(xbc, proj, dt_bias, A_log, D, Hh, P, N, G, torch.zeros(Hh, N, P, dtype=torch.float64))
    want = want.view(n, Hh, P)
    y, state = scan(xbc)
    assert ((y.double() - want).abs().amax((0, 2)) < 2e-5 * want.abs().amax((0, 2))).all()
    assert ((state[0].double() - S).abs().amax((1, 2)) < 2e-5 * S.abs().amax((1, 2))).all()
    for row, bad in ((5, float("inf")), (63, float("nan")), (130, float("-inf")), (172, float("nan"))):
        xb = xbc.clone()
        xb[row, 0:3] = bad                  # three channels of the first head ...
        xb[row, inner - 1] = bad            # ... and one of the last
        y, _ = scan(xb)
        assert ((y[:row].double() - want[:row]).abs().amax((0, 2)) < 2e-5 * want.abs().amax((0, 2))).all()
        assert not torch.isfinite(y[row, 0, :3]).any() and torch.isfinite(y[row, 1:3]).all()


def test_portion_tables():
    """Which rows attend on expanded keys: none without a portion of LATENT_ROWS_MIN rows, else everything behind the leading
    single tokens; blocks of 64 gathered rows per portion, tiles of 128 rows with the most keys first."""
    seg = _seg("cpu", [(1, 5, 0), (1, 9, 1), (200, 0, 2), (3, 1000, 3), (1, 77, 4)])[0].numpy()
    first, M, px, blocks, tiles = hops.portion_tables(seg, 0)
    assert (first, M) == (2, 64 * (4 + 16 + 2))
    assert px.tolist() == [[2, 200, 0, 0, 0, 2, 200, 0], [202, 3, 1000, 0, 256, 3, 1003, 0], [205, 1, 77, 0, 1280, 4, 78, 0]]
    assert blocks.tolist() == [0] * 4 + [1] * 16 + [2] * 2
    assert tiles.tolist() == [[1, 0, 0, 0], [0, 128, 0, 0], [0, 0, 0, 0], [2, 0, 0, 0]]
    first, M, px, blocks, tiles = hops.portion_tables(seg, 100)
    assert px[:, 3].tolist() == [0, 896, 0] and M == 64 * (4 + 2 + 2) and tiles[0].tolist() == [0, 128, 0, 0]
    short = _seg("cpu", [(1, 5, 0), (hops.LATENT_ROWS_MIN - 1, 0, 1)])[0].numpy()
    assert hops.portion_tables(short, 0) is None and hops.portion_tables(seg[:2], 0) is None
    assert hops.portion_tables(None, 0) is None
    # a few rows behind a long history beside it: the whole step stays in the latent space
    far = hops.LATENT_ROWS_CHAIN
    for p0, none in ((far - 3, False), (far - 2, True)):
        seg = _seg("cpu", [(hops.LATENT_ROWS_MIN, 0, 0), (3, p0, 1)])[0].numpy()
        assert (hops.portion_tables(seg, 0) is None) == none and hops.portion_tables(seg, 50) is not None
    assert hops.portion_tables(_seg("cpu", [(hops.LATENT_ROWS_MIN, far, 0), (3, far, 1)])[0].numpy(), 0) is not None


def test_key_ranges_by_size():
    """Key ranges of single tokens' latent attention at measured points: whole where a merge costs what it saves, as many as fill the
    chip otherwise, of at least 128 keys; launches without tiles too."""
    for n, heads, keys, rank, rot, want in ((1, 32, 130, 512, 64, 1), (1, 32, 256, 512, 0, 1), (1, 32, 512, 512, 64, 4),
                                            (1, 32, 1706, 512, 64, 14), (1, 32, 8000, 512, 64, 32), (16, 32, 8000, 512, 64, 16),
                                            (64, 32, 2048, 512, 64, 4), (100, 32, 1200, 512, 64, 2), (200, 32, 8000, 512, 64, 1),
                                            (64, 64, 2048, 512, 64, 2), (128, 32, 1000, 256, 32, 2), (1, 32, 130, 256, 32, 1),
                                            (1, 32, 256, 256, 32, 2), (64, 32, 1000, 384, 64, 4), (48, 16, 1706, 512, 32, 5),
                                            (0, 32, 8000, 512, 64, 32), (0, 32, 100, 256, 0, 1)):
        assert hops.attn_splits(n, heads, keys, rank, rot) == want, (n, heads, keys, rank, rot)


def cfg_direct():
    """kv_rank 512 with 64 rotated channels and heads of 128: the sizes whose kernels read the cached rows alone."""
    ff = {"kind": "dense", "ff": 96}
    return {"architecture": "Budurax", "vocab": 173, "width": 80, "norm": {"eps": 1e-5}, "token_side": {"dim": 4},
            "layers": [{"type": "latent_attention", "mixer": _attn(3, 128, 64, 64, 128, 512), "mlp": ff},
                       {"type": "mamba2", "mixer": _mamba(2, 16, 8, 1, 2, 4), "mlp": ff},
                       {"type": "latent_attention", "mixer": _attn(3, 128, 64, 64, 128, 512), "mlp": ff}]}


def test_channels_of_latent_pages():
    """What a cached token takes: the row, and a transposed copy except in bf16 on the GPU at the sizes that do without."""
    for R, rd, dtype, dev, want in ((512, 64, torch.bfloat16, "cuda", 576), (512, 0, torch.bfloat16, "cuda:0", 512),
                                    (512, 32, torch.bfloat16, "cuda", 1056), (256, 64, torch.bfloat16, "cuda", 576),
                                    (512, 64, torch.float32, "cuda", 1088), (512, 64, torch.bfloat16, "cpu", 1088)):
        assert hops.latent_page_channels(R, rd, dtype, dev) == want, (R, rd, dtype, dev)


@pytest.mark.gpu
def test_latent_rows_are_cached_once():
    """kv_rank 512 in the engine: no transposed copy is allocated or charged, and portions, single tokens and a mixed step agree
    with the plain model; an output that the row kernel cannot write goes the vector kernel's way."""
    b = Bench(cfg_direct(), seed=11)
    t, u = toks(200, 173, 1), toks(41, 173, 2)
    eng = b.engine("cuda:0", "bfloat16", blocks=40)
    assert all(p is None or p.shape == (0, 512, 16) for p in eng.model.pages_t) and eng.model.pages_t[0] is not None
    assert eng.model.page_bytes() == 2 * 16 * 576 * 2
    assert rel_err(feed_all(eng, "c", t, [130, 2, 61, 1]), b.oracle(t)) < TOL["bfloat16"]
    got = [eng.feed([("u", u[:40], list(range(40)))])]
    got.append(eng.feed([("u", u[40:], [0]), ("v", t[:50], list(range(50)))], ["u", "v"]))
    assert rel_err(torch.cat([got[0], got[1][:1]]), b.oracle(u)) < TOL["bfloat16"]
    # 40 keys, a row of the output one element off its 8 bytes
    dev = "cuda:0"
    cache = torch.randn(3, 16, 576, device=dev).bfloat16()
    bt, pos = torch.tensor([[2, 0, 1]], dtype=torch.int32, device=dev), torch.tensor([39], device=dev)
    seg, ts = _seg(dev, [(1, 39, 0)])
    q, qr = torch.randn(4, 1, 512, device=dev).bfloat16(), torch.randn(1, 4, 64, device=dev).bfloat16()
    tiles = torch.tensor([(0, 1, 0, 0)], dtype=torch.int32, device=dev)
    outs = []
    for off in (0, 1):
        out = torch.empty(4, 1, 516, device=dev, dtype=torch.bfloat16)[:, :, off:off + 512]
        hops.latent_attn(q, qr, cache, bt, ts, seg, pos, 0.05, out, torch.empty(0, 512, 16, dtype=torch.bfloat16, device=dev),
                         tiles, 40)
        outs.append(out.float())
    # weights and results in bf16 on one side only: 2^-8 of the largest value
    assert (outs[0] - outs[1]).abs().max().item() <= 2 ** -8 * 1.1 * cache.float().abs().max().item()


def test_where_expanded_keys_pay():
    """The choice between the latent space and expanded keys and values at measured points of both sides (us in the latent space /
    expanded), and its effect on a step's tables."""
    for H, R, rd, hist, rows, window, latent, expanded in (
            (8, 512, 64, 0, 512, 0, 53, 80), (16, 512, 64, 8000, 512, 0, 457, 595), (32, 512, 64, 0, 128, 0, 44, 62),
            (32, 512, 64, 0, 512, 0, 91, 86), (32, 512, 64, 2000, 256, 0, 155, 197), (32, 512, 64, 2000, 384, 0, 280, 223),
            (32, 512, 64, 8000, 128, 0, 249, 591), (32, 512, 64, 8000, 512, 0, 868, 658), (32, 512, 0, 4000, 384, 1024, 158, 96),
            (64, 512, 64, 2000, 128, 0, 147, 261), (64, 512, 64, 8000, 192, 0, 831, 732), (32, 256, 64, 2000, 192, 0, 231, 195),
            (32, 256, 64, 2000, 96, 0, 137, 178), (16, 256, 0, 4000, 192, 1024, 91, 68), (32, 128, 64, 2000, 512, 0, 273, 189)):
        assert hops.expanded_pays([(rows, hist)], window, H, R, rd) == (expanded < latent), (H, R, rd, hist, rows, window)
    # many portions fill the chip together
    assert not hops.expanded_pays([(120, 500)], 0, 32, 512, 64) and hops.expanded_pays([(120, 500)] * 8, 0, 32, 512, 64)
    seg = _seg("cpu", [(1, 5, 0), (200, 2000, 1)])[0].numpy()
    assert hops.portion_tables(seg, 0) is not None and hops.portion_tables(seg, 0, 32, 512, 64) is None
    assert hops.portion_tables(seg, 0, 64, 512, 64)[:2] == (1, 64 * 35)


@pytest.mark.gpu
@pytest.mark.parametrize("H,rd,window,extras", [(8, 64, 0, True), (3, 0, 0, False), (16, 0, 70, True), (5, 64, 200, False),
                                                (8, 0, 1, False)])
def test_attention_of_portions_on_expanded_keys(H, rd, window, extras):
    """Portions whose rows and keys end inside, at and one past a tile (128 rows) and a block (64 keys), fresh and behind
    histories, scattered pages, beside single tokens that must stay untouched; with a sink and a gate. Against float64 on the
    same bf16 keys and values: the weights' and the output's rounding to bf16 move a value by at most 2^-9 of the largest |v|
    each (a gate shrinks both), the fp32 sums by far less."""
    device, R, D, Dv = "cuda:0", 96, 128, 128
    torch.manual_seed(H + window)
    runs = [(1, 40, 0), (129, 0, 1), (64, 0, 2), (33, 95, 3), (128, 64, 4), (1, 130, 5), (300, 37, 6)]
    T = sum(r[0] for r in runs)
    seg, _ = _seg("cpu", runs)
    W = -(-max(n + p for n, p, _ in runs) // 16)
    bt = torch.randperm(len(runs) * W).view(len(runs), W).int()
    cache = torch.full((len(runs) * W, 16, R + rd), float("nan"), dtype=torch.bfloat16)
    rows = []
    for j, (n, p0, _) in enumerate(runs):
        c = torch.randn(p0 + n, R + rd).bfloat16()
        c[-1] *= 3
        rows.append(c)
        for i in range(p0 + n):
            cache[bt[j, i // 16], i % 16] = c[i]
    q, q_rot = torch.randn(T, H, D).bfloat16(), torch.randn(T, H, rd).bfloat16()
    w_k, w_v = (torch.randn(H * D, R) / R ** 0.5).bfloat16(), (torch.randn(H * Dv, R) / R ** 0.5).bfloat16()
    sink = torch.randn(H) * 3 if extras else None
    gate = torch.randn(T, H * Dv + 8).bfloat16() if extras else None
    scale = (D + rd) ** -0.5
    want, vmax, at = torch.zeros(T, H, Dv, dtype=torch.float64), 0.0, 0
    for j, (n, p0, _) in enumerate(runs):
        c = rows[j][:, :R].to(device)
        k = torch.nn.functional.linear(c, w_k.to(device)).cpu().double().view(-1, H, D)
        v = torch.nn.functional.linear(c, w_v.to(device)).cpu().double().view(-1, H, Dv)
        kr = rows[j][:, R:].double()
        s = torch.einsum("thd,shd->hts", q[at:at + n].double(), k) + torch.einsum("thd,sd->hts", q_rot[at:at + n].double(), kr)
        dist = torch.arange(p0, p0 + n)[:, None] - torch.arange(p0 + n)
        s = (s * scale).masked_fill((dist < 0) | (dist >= window if window else dist < 0), float("-inf"))
        if sink is not None:
            s = torch.cat([s, sink.double()[:, None, None].expand(H, n, 1)], 2)
            v = torch.cat([v, torch.zeros(1, H, Dv, dtype=torch.float64)])
        want[at:at + n] = torch.einsum("hts,shd->thd", torch.softmax(s, -1), v)
        vmax = max(vmax, v.abs().max().item())
        at += n
    if gate is not None:
        want = want * torch.sigmoid(gate[:, :H * Dv].double()).view(T, H, Dv)
    t = hops.portion_tables(seg.numpy(), window)
    tabs = t[:2] + tuple(torch.from_numpy(x).to(device) for x in t[2:])
    assert t[0] == 1
    out = torch.full((T, H * Dv), 7.0, dtype=torch.bfloat16, device=device)
    qg, qr = q.to(device), q_rot.to(device)
    assert hops.latent_rows_ok(qg, qr, cache.to(device), Dv)
    hops.latent_attn_portions(qg, qr, cache.to(device), w_k.to(device), w_v.to(device), tabs, bt.to(device), scale, out,
                              window, sink.to(device) if extras else None, gate.to(device)[:, :H * Dv] if extras else None)
    got = out.cpu().double().view(T, H, Dv)
    assert (got[:1] == 7).all()
    assert (got[1:] - want[1:]).abs().max().item() < 1.1 * 2 ** -8 * vmax


@pytest.mark.gpu
@pytest.mark.parametrize("H", [48, 7])
def test_expanded_keys_by_groups_of_heads(H, monkeypatch):
    """Expanded keys and values past LATENT_BYTES: groups of heads one after the other give what one group gives (library
    products of other widths: keys and values a bf16 rounding apart, 2^-8 of the largest value at most in an average of values
    and again in the weights' exponents), and no more memory is held than the bound, the gathered rows and the allocator's
    rounding to 2 MiB."""
    device, R, rd, D, n, p0 = "cuda:0", 256, 64, 128, 150, 3000
    torch.manual_seed(H)
    W = -(-(n + p0) // 16)
    bt = torch.randperm(W, device=device).view(1, W).int()
    cache = torch.randn(W, 16, R + rd, device=device).bfloat16()
    q, q_rot = (torch.randn(n, H, d, device=device).bfloat16() for d in (D, rd))
    w_k, w_v = ((torch.randn(H * D, R, device=device) / R ** 0.5).bfloat16() for _ in range(2))
    sink, gate = torch.randn(H, device=device), torch.randn(n, H * D, device=device).bfloat16()
    t = hops.portion_tables(_seg("cpu", [(n, p0, 0)])[0].numpy(), 0)
    tabs = t[:2] + tuple(torch.from_numpy(x).to(device) for x in t[2:])
    outs, peaks, M = [], [], t[1]
    for most in (1 << 29, M * 2 * D * 2 * 20):
        monkeypatch.setattr(hops, "LATENT_BYTES", most)
        out = torch.full((n, H * D), float("nan"), dtype=torch.bfloat16, device=device)
        torch.cuda.reset_peak_memory_stats()
        held = torch.cuda.memory_allocated()
        hops.latent_attn_portions(q, q_rot, cache, w_k, w_v, tabs, bt, 192 ** -0.5, out, 0, sink, gate)
        peaks.append(torch.cuda.max_memory_allocated() - held)
        outs.append(out.float())
    top = (cache[:, :, :R].float().reshape(-1, R) @ w_v.float().t()).abs().max().item()
    assert (outs[0] - outs[1]).abs().max().item() <= 2 ** -7 * top
    if H > 20:
        assert peaks[1] <= M * 2 * D * 2 * 20 + M * (R + rd) * 2 + (8 << 20) < peaks[0]


@pytest.mark.gpu
def test_decoded_tokens_beside_expanded_portions(monkeypatch):
    """A step of two decoded tokens, a portion of 130 rows and one of 7 in the engine, the portions on expanded keys and values and the
    single tokens in the latent space beside them, into the same rows; histories behind all of them, against the plain model."""
    b = Bench(cfg_direct(), seed=5)
    eng = b.engine("cuda:0", "bfloat16", blocks=60, seqs=4)
    t = {k: toks(n, 173, i) for i, (k, n) in enumerate((("a", 71), ("b", 34), ("p", 200), ("s", 27)))}
    cut = {"a": 70, "b": 33, "p": 70, "s": 20}
    got = {k: [eng.feed([(k, t[k][:n], list(range(n)))])] for k, n in cut.items()}
    monkeypatch.setattr(hops, "expanded_pays", lambda *a: True)
    calls, orig = [], hops.latent_attn_portions

    def spy(*a):
        calls.append(a[5][0])      # the rows in front of the portions
        return orig(*a)

    monkeypatch.setattr(hops, "latent_attn_portions", spy)
    order = ["a", "b", "p", "s"]
    out = eng.feed([(k, t[k][cut[k]:], list(range(len(t[k]) - cut[k]))) for k in order], order)
    assert calls == [2, 2]         # (two layers)
    at = 0
    for k in order:
        n = len(t[k]) - cut[k]
        assert rel_err(torch.cat([got[k][0], out[at:at + n]]), b.oracle(t[k])) < TOL["bfloat16"], k
        at += n


@pytest.mark.gpu
def test_single_token_behind_more_pages_than_a_run():
    """kv_rank 512, one range over 16400 keys: page ids are kept for 16384 keys at a time. Single keys on both sides of that line, the
    first and the last carry the result (queries of 80 times a unit key: every other key's score is at least 40 lower), and a flat
    softmax over all of them: an average of unit vectors, weights in bf16 (2^-9 of it)."""
    device, H, R, rd, n = "cuda:0", 4, 512, 64, 16400
    torch.manual_seed(3)
    kv = torch.nn.functional.normalize(torch.randn(n, R + rd, device=device), dim=-1).bfloat16()
    perm = torch.randperm(n // 16, device=device)
    cache = torch.empty(n // 16, 16, R + rd, dtype=torch.bfloat16, device=device)
    cache[perm] = kv.view(-1, 16, R + rd)
    bt, pos = perm.int()[None].contiguous(), torch.tensor([n - 1], device=device)
    tiles = torch.tensor([(0, 1, 0, 0)], dtype=torch.int32, device=device)
    cache_t = torch.empty(0, R, 16, dtype=torch.bfloat16, device=device)

    def attend(q, scale):
        out = torch.empty(H, 1, R, dtype=torch.bfloat16, device=device)
        hops.ext().hy_latent_attn_mfma(q[:R].expand(H, 1, R).contiguous(), q[R:].expand(1, H, rd).contiguous(), cache, cache_t, bt,
                                       tiles, hops.tile_tokens(H), pos, scale, out, 1, None, None, 0, None)
        return out[:, 0].float()

    for j in (0, 16351, 16383, 16384, 16399):
        got = attend((kv[j].float() * 80).bfloat16(), 1.0)
        assert (got - kv[j, :R].float()).abs().max().item() < 2 ** -8
    flat = attend(torch.zeros(R + rd, dtype=torch.bfloat16, device=device), 1.0)
    want = kv[:, :R].double().mean(0)
    assert (flat.double() - want).abs().max().item() < 2 ** -8 * want.abs().max().item() + 1e-6


@pytest.mark.parametrize("device", DEVICES)
@pytest.mark.parametrize("d,T", [(4, 3), (1022, 3), (1028, 513), (1030, 5), (4096, 7), (4096, 520), (4100, 3)])
def test_add_norm_of_slabs(device, d, T):
    """A projection's split-K slabs in place of its rows: the forms of the row kernels, slab counts with loops of their own and
    without, against 64 bits: fp32 sums (d * 2^-24 of a value's size), results in bf16 (half a step, 2^-8), and the
    widths beyond the register kernels and the CPU, where the sum is rounded to bf16 first (2^-8 of a y of up to 5 sizes)."""
    g = torch.Generator().manual_seed(d + T)
    w, b, w2, b2 = ((torch.randn(d, generator=g)).to(torch.bfloat16) for _ in range(4))
    for S in (1, 2, 3, 4, 8):
        x, y = torch.randn(T, d, generator=g), torch.randn(S, T, d, generator=g)
        x1 = x.double() + plain.layer_norm(y.double().sum(0), w.double(), b.double(), 1e-5)
        low = device == "cpu" or d > 4096
        for second in (None, (w2, b2)):
            xd, o = x.clone().to(device), torch.empty(T, d, dtype=torch.bfloat16, device=device)
            hops.add_ln(xd, y.to(device), w.to(device), b.to(device), 1e-5, o, *(t.to(device) for t in second or ()))
            tol = d * 2.0 ** -24 + 1e-5 + (2 ** -7 * 5 if low else 0)
            size = w.double().abs() + x1.abs() + 1
            assert ((xd.cpu().double() - x1).abs() <= tol * size).all()
            want = xd.cpu().double()
            if second:
                want = plain.layer_norm(want, w2.double(), b2.double(), 1e-5)
            assert ((o.cpu().double() - want).abs() <= (2 ** -8 + d * 2.0 ** -24 + 1e-5) * (want.abs() + 1)).all()


@pytest.mark.parametrize("device", DEVICES)
@pytest.mark.parametrize("d", [4104, 8192])
def test_add_norm_of_wide_slabs_reduces_them_in_one_pass(device, d, monkeypatch):
    """Rows wider than the kernel takes slabs of: the reduction that a projection's own output goes through, not a sum and a conversion."""
    from kafka_llm_service_amd import ops

    calls, orig = [], ops.slab_reduce
    monkeypatch.setattr(ops, "slab_reduce", lambda y: calls.append(y.shape) or orig(y))
    test_add_norm_of_slabs(device, d, 3)
    assert calls == [(S, 3, d) for S in (1, 2, 3, 4, 8) for _ in range(2)]


@pytest.mark.gpu
@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("d,T", [(4, 3), (1024, 3), (1028, 5), (1030, 5), (4096, 7), (4096, 600), (4100, 3), (1022, 2)])
def test_row_kernels_over_widths(dtype, d, T):
    """Layer norm with the token shift, add + norm, token input + depth average and the grouped gated norm at the widths
    where their forms change (pieces of four elements or single ones, 256 or 1024 threads, registers or not), and views whose
    rows are not in 16-byte pieces, against the CPU functions: fp32 sums in another order (d * 2^-24 of the row's size, 2.4e-4
    at 4096), results rounded to the activation type: two fp32 values on either side of a boundary end one bf16 step apart, at
    most 2^-7 of the value."""
    from kafka_llm_service_amd.ops import hybrid_reference as href

    dev = "cuda:0"
    g = torch.Generator().manual_seed(d + T)

    def rn(*s):
        return torch.randn(*s, generator=g)

    def same(got, want, acc=d * 2.0 ** -24 + 1e-5):
        got, want = got.float().cpu(), want.float()
        tol = acc + (2 ** -7 if dtype == torch.bfloat16 else 0)
        assert ((got - want).abs() <= tol * (want.abs() + 1)).all(), (got - want).abs().max()

    for off in (0, 1):   # rows of a wider buffer, from its first or its second column on
        wide = rn(T, d + 8)
        x, w, b, mu = wide[:, off:off + d], rn(d).to(dtype), rn(d).to(dtype), torch.rand(d, generator=g).to(dtype)
        xd = wide.to(dev)[:, off:off + d]
        seg, ts = _seg("cpu", [(1, 5, 2), (T - 1, 0, 0)])
        state = rn(3, d)
        for direct in (False, True):
            want, out = torch.empty(T, d, dtype=dtype), torch.empty(T, d, dtype=dtype, device=dev)
            s0, s1 = state.clone(), state.to(dev)
            last = None if direct else torch.empty(2, d)
            hops.ln_shift(x, w, b, 1e-5, want, mu, ts, seg, s0, last)
            ld = None if direct else torch.empty(2, d, device=dev)
            hops.ln_shift(xd, w.to(dev), b.to(dev), 1e-5, out, mu.to(dev), ts.to(dev), seg.to(dev), s1, ld)
            same(out, want)
            same(s1, s0)
            if not direct:
                same(ld, last)
        out = torch.empty(T, d, dtype=dtype, device=dev)
        hops.ln_shift(xd, w.to(dev), b.to(dev), 1e-5, out)
        href.ln_shift(x, w, b, 1e-5, want)
        same(out, want)
        y = rn(T, d).to(dtype)
        for w2 in (None, w):
            x0, x1 = x.clone(), wide.to(dev)[:, off:off + d]
            o0, o1 = torch.empty(T, d, dtype=dtype), torch.empty(T, d, dtype=dtype, device=dev)
            b2 = None if w2 is None else b
            hops.add_ln(x0, y, w, b, 1e-5, o0, w2, b2)
            hops.add_ln(x1, y.to(dev), w.to(dev), b.to(dev), 1e-5, o1, None if w2 is None else w2.to(dev),
                        None if b2 is None else b2.to(dev))
            same(x1, x0)
            same(o1, o0)
    x = rn(T, d)
    stack = rn(4, T, d)
    for layer in (0, 2):
        dwa = torch.rand(layer + 2, generator=g)
        x0, x1, s0, s1 = x.clone(), x.to(dev), stack.clone(), stack.to(dev)
        hops.side_dwa(x0, y, w, 1e-5, s0, layer, dwa)
        hops.side_dwa(x1, y.to(dev), w.to(dev), 1e-5, s1, layer, dwa.to(dev))
        same(x1, x0)
        same(s1, s0)
    for groups in (1, 2):
        yv, z, o0 = rn(T, d), rn(T, d + 4).to(dtype), torch.empty(T, d, dtype=dtype)
        o1 = torch.empty(T, d, dtype=dtype, device=dev)
        hops.gated_norm(yv, z, w, groups, 1e-5, o0)
        hops.gated_norm(yv.to(dev), z.to(dev), w.to(dev), groups, 1e-5, o1)
        same(o1, o0)
    gu = (rn(T, 2 * d) * 3).to(dtype)
    o0, o1 = torch.empty(T, d, dtype=dtype), torch.empty(T, d, dtype=dtype, device=dev)
    hops.gelu_mul(gu, o0)
    hops.gelu_mul(gu.to(dev), o1)
    same(o1, o0)


@pytest.mark.gpu
@pytest.mark.parametrize("taps", [2, 3, 4])
def test_conv_of_single_tokens(taps):
    """A step of single tokens (fresh ones in slots of NaN, others going on): one kernel for the rows and the slots' tails,
    against the CPU function; bf16 results of fp32 sums of up to four products: at most one bf16 step (2^-7) apart."""
    g = torch.Generator().manual_seed(taps)
    C, R = 40, 7
    proj = torch.randn(R, C + 8, generator=g).bfloat16()
    w, b = torch.randn(C, taps, generator=g).bfloat16(), torch.randn(C, generator=g).bfloat16()
    seg, ts = _seg("cpu", [(1, 0 if r % 3 == 0 else r, R - 1 - r) for r in range(R)])
    state = torch.randn(R, taps - 1, C, generator=g).bfloat16()
    for r in range(0, R, 3):
        state[R - 1 - r] = float("nan")
    s0, s1 = state.clone(), state.to("cuda:0")
    o0, o1 = torch.empty(R, C, dtype=torch.bfloat16), torch.empty(R, C, dtype=torch.bfloat16, device="cuda:0")
    hops.conv_silu(proj, 8, w, b, ts, seg, s0, o0)
    hops.conv_silu(proj.cuda(), 8, w.cuda(), b.cuda(), ts.cuda(), seg.cuda(), s1, o1)
    assert torch.equal(s1.cpu(), s0)
    assert ((o1.cpu().float() - o0.float()).abs() <= 2 ** -7 * o0.float().abs() + 1e-5).all()
