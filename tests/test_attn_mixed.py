"""Prefix tiles and decode pieces in one launch (``ops.attn_mixed``): rows against fp32 attention over their whole context, and the
engine's plans for it."""
import dataclasses
import math
import os
import sys

from types import SimpleNamespace

import numpy as np
import pytest
import torch

from kafka_llm_service_amd import ops
from kafka_llm_service_amd.engine import model_runner as mr
from kafka_llm_service_amd.engine.model_runner import decode_items
from kafka_llm_service_amd.models.attention import paged_attention
from kafka_llm_service_amd.ops import reference as ref

sys.path.insert(0, os.path.dirname(__file__))


def _case(groups, own, hkv, G, seed, dev, loose=0, alt=0):
    """Rows of ``groups`` ((rows, prefix pages, prefix parts) each), then ``loose`` rows without one; ``own`` keys behind the
    prefix per row, in order; ``alt`` new tokens behind the first group's prefix."""
    g = torch.Generator().manual_seed(seed)
    B = sum(n for n, _, _ in groups) + loose
    pages = sum(p for _, p, _ in groups) + sum(-(-n // 16) for n in own) + 4 + alt // 16
    W = max([p for _, p, _ in groups] + [0]) + max(-(-n // 16) for n in own) + 4 + alt // 16
    perm = torch.randperm(pages, generator=g).tolist()
    bt = torch.zeros(B + 1, W, dtype=torch.int32)
    kv0, npre, items, at, r0 = np.zeros(B, np.int64), np.zeros(B, np.int64), [], 0, 0
    tile = 128 // G
    for gi, (n, p, nc) in enumerate(groups):
        shared = perm[at:at + p]
        at += p
        ck = -(-p * 16 // (nc * 32)) * 32
        nc = -(-p * 16 // ck)
        for c in range(nc):
            rows = [(r, min(tile, r0 + n - r), 0) for r in range(r0, r0 + n, tile)]
            if gi == 0:
                rows += [(B + t, min(tile, alt - t), 1) for t in range(0, alt, tile)]
            items += [(r, k, r0, c * ck, min(p * 16, (c + 1) * ck), c, a, nc) for r, k, a in rows]
        for r in list(range(r0, r0 + n)) + ([B] if gi == 0 else []):
            bt[r, :p] = torch.tensor(shared, dtype=torch.int32)
        kv0[r0:r0 + n], npre[r0:r0 + n] = p * 16, nc
        r0 += n
    for b in range(B):
        p, k = int(kv0[b]) // 16, -(-own[b] // 16)
        bt[b, p:p + k] = torch.tensor(perm[at:at + k], dtype=torch.int32)
        at += k
    k = torch.randn(pages, hkv, 16, 128, generator=g).to(torch.bfloat16)
    v = torch.randn(pages, hkv, 128, 16, generator=g).to(torch.bfloat16)
    q = torch.randn(B + alt, hkv * G, 128, generator=g).to(torch.bfloat16)
    lens = kv0 + np.asarray(own)
    lim = torch.tensor(list(lens - 1) + [int(groups[0][1]) * 16 + 5] * alt, dtype=torch.int32)
    return dict(B=B, q=q.to(dev), k=k.to(dev), v=v.to(dev), bt=bt.to(dev), lens=lens, kv0=kv0, npre=npre, lim=lim.to(dev),
                items=torch.tensor(items, dtype=torch.int32).reshape(-1, 8).to(dev))


def _run(c, target=1344, dec=None, edit=None, **kw):
    dev, B, Hq = c["q"].device, c["B"], c["q"].shape[1]
    if dec is None:
        dec = decode_items(c["lens"], c["kv0"], c["npre"], c["k"].shape[1], target)
    S = int((dec[:, 4] + dec[:, 5]).max())
    part = torch.full((B, Hq, S, 128), float("nan"), device=dev)
    lse = torch.full((B, Hq, S), float("nan"), device=dev)
    pre = torch.full((B, Hq, S, 128), float("nan"), device=dev, dtype=torch.bfloat16)
    T = c["q"].shape[0]
    out = torch.full((T, Hq, 128), float("nan"), device=dev, dtype=torch.bfloat16)
    parts = torch.zeros(T, dtype=torch.int32)
    for b, _, _, _, n, npre, _, _ in dec.tolist():
        parts[b] = n + npre | npre << 16
    parts[B:] = int(c["npre"][0])
    alt = (torch.zeros(T - B, Hq, S, 128, device=dev), torch.full((T - B, Hq, S), float("-inf"), device=dev)) if T > B else ()
    if edit:
        edit(parts)
    ops.attn_mixed(c["items"], torch.tensor(dec, device=dev), c["q"], c["k"], c["v"], c["bt"], c["lim"], part, lse, pre, parts.to(dev),
                   128 ** -0.5, out, *alt, **kw)
    return out


def _whole(c, b, n):
    """fp32 attention of row b over its first n keys."""
    hkv = c["k"].shape[1]
    kk, vv = ref.gather_kv(c["k"].cpu(), c["v"].cpu(), c["bt"][min(b, c["B"])].cpu(), n)
    q = c["q"][b].float().cpu().view(hkv, -1, 128)
    s = torch.einsum("hgd,nhd->hgn", q, kk.float()) / math.sqrt(128)
    return torch.einsum("hgn,nhd->hgd", s.softmax(-1), vv.float()).reshape(-1, 128)


def _check(c, out):
    # bf16 probabilities, prefix partials and rows: each 2^-9 of values of about sqrt(1/n), so 3 * 2^-9 of the largest; taken twice
    tol = 6 * 2.0 ** -9
    for b in list(range(c["B"])) + [r for r in (c["B"], c["B"] + 37, out.shape[0] - 1) if c["B"] <= r < out.shape[0]]:
        want = _whole(c, b, int(c["lens"][b] if b < c["B"] else c["kv0"][0]))
        assert (out[b].float().cpu() - want).abs().max() <= tol * max(1e-3, want.abs().max()), b


#: (groups, own keys by row, kv heads, G, loose rows, new tokens): whole and ragged row tiles, one row of a tile, one prefix part,
#: several groups, rows without a group, pieces of one row, every G
CASES = [([(5, 40, 3)], [1, 17, 33, 500, 64], 2, 4, 0, 0), ([(33, 34, 2)], [20 + 7 * i for i in range(33)], 2, 4, 0, 0),
         ([(2, 32, 1), (3, 64, 4)], [300, 5, 31, 32, 1200], 2, 8, 0, 0), ([(2, 40, 5)], [600, 40, 900, 16], 1, 2, 2, 0),
         ([(3, 48, 2)], [90, 1, 700], 3, 1, 0, 0), ([(4, 130, 32)], [50, 9000, 3, 77], 2, 4, 0, 70)]


@pytest.mark.parametrize("groups,own,hkv,G,loose,alt", CASES)
def test_rows_equal_whole_attention_cpu(groups, own, hkv, G, loose, alt):
    c = _case(groups, own, hkv, G, 3, "cpu", loose, alt)
    _check(c, _run(c))


@pytest.mark.gpu
@pytest.mark.parametrize("groups,own,hkv,G,loose,alt", CASES + [([(64, 70, 8)], [40 + 11 * i for i in range(64)], 8, 4, 0, 130)])
def test_rows_equal_whole_attention(cuda, groups, own, hkv, G, loose, alt):
    """... and again: the counters are back at zero; pieces of other lengths (many of a row, one of each)."""
    c = _case(groups, own, hkv, G, 3, cuda, loose, alt)
    _check(c, _run(c))
    for target in (1344, 1344, 64, 8):
        _check(c, _run(c, target))
    stream = torch.cuda.current_stream(cuda).cuda_stream
    assert not ops._TICKETS[(c["q"].device, f"mixed {stream}")].any()


@pytest.mark.gpu
def test_keys_that_are_no_numbers_reach_their_rows_only(cuda):
    c = _case([(6, 40, 3)], [50, 60, 700, 80, 90, 100], 2, 4, 5, cuda)
    want = _run(c)
    c["k"][c["bt"][2, 41]] = float("nan")          # a page of row 2's own keys
    out = _run(c)
    rest = [0, 1, 3, 4, 5]
    assert torch.equal(out[rest], want[rest])
    c["v"][c["bt"][0, 3]] = float("nan")           # a page that all share
    out = _run(c)
    assert out.isnan().any(-1).all()


def _more(row, n):
    def edit(parts):
        parts[row] += n
    return edit


@pytest.mark.gpu
def test_rows_whose_parts_do_not_come_are_no_numbers_and_stay_alone(cuda):
    """More parts than a merge reads (nothing waits for them), one part more than comes (after a bounded wait): that row is not a number, in this
    launch and in the next ones on its counters, and no other row is touched; on clear counters all is as before."""
    c = _case([(6, 40, 3)], [50, 60, 900, 80, 90, 100], 2, 4, 5, cuda)
    want, rest = _run(c), [0, 1, 3, 4, 5]
    assert not want.isnan().any()
    for row, n in ((2, 70), (1, 1)):
        rest = [r for r in range(6) if r != row]
        counters = torch.zeros(6 * 2, dtype=torch.int32, device=cuda)
        for edit in (_more(row, n), None, None):
            out = _run(c, edit=edit, counters=counters, polls=1 << 16)
            assert torch.equal(out[rest], want[rest]) and out[row].isnan().all()
            lost = counters.view(6, 2)
            assert (lost[row] < -(1 << 29)).all() and not lost[rest].any()
        assert torch.equal(_run(c, edit=_more(row, n), polls=1 << 16)[rest], want[rest])
        assert torch.equal(_run(c), want)          # (the stream's counters, cleared before each launch)
        assert torch.equal(_run(c, counters=counters.zero_()), want) and not counters.any()


def test_rows_of_more_parts_than_a_merge_reads_are_no_numbers():
    c = _case([(6, 40, 3)], [50, 60, 700, 80, 90, 100], 2, 4, 5, "cpu")
    want, out = _run(c), _run(c, edit=_more(2, 70))
    assert out[2].isnan().all() and torch.equal(out[[0, 1, 3, 4, 5]], want[[0, 1, 3, 4, 5]])


def test_plans_of_a_cascade_step_cover_every_key_once():
    """The engine's plan for one launch: every key of every row in exactly one tile or piece, at most 128 query rows a tile, and a
    prefix tile names as many parts as its rows' pieces do."""
    from kafka_llm_service_amd.engine.engine import EngineConfig, LLMEngine
    from kafka_llm_service_amd.engine.sequence import SamplingParams, Sequence

    eng = LLMEngine(EngineConfig(model="tiny-llama", device="cpu", num_kv_blocks=700, max_num_seqs=48, max_model_len=2400))
    r = eng.runner
    if not r.mixed_attn:                           # (the small preset's head size: the plan alone)
        r.mixed_attn, r.mixed_tile = True, 128 // r.G
    shared = list(range(1, 1 + 64 * 16))
    seqs = [Sequence(f"r{i}", shared + [5 + i] * (3 + 29 * i % 400), SamplingParams(max_tokens=4)) for i in range(41)]
    first = Sequence("shared", list(shared), SamplingParams(max_tokens=1))
    for s in [first] + seqs:                       # (the pages that the rest of them share)
        batch = eng.sched.replay([(s, s.total_len)])
        for x, _, b in batch.prefill:
            x.num_computed = b
            eng.kvm.commit(x.seq_id, b)
        for x in batch.decode:
            x.num_computed = x.total_len
    for s in seqs:
        s.prompt_ids.append(7)
        eng.kvm.append_tokens(s.seq_id, [7])
    new = seqs[-1]
    for t in range(90):
        new.prompt_ids.append(9)
    eng.kvm.append_tokens(new.seq_id, [9] * 90)
    host, _ = r.build_host(eng.sched.replay([(s, s.total_len - s.num_computed) for s in seqs]))
    assert host.mixed and host.n_prefix_items and host.B == 40 and host.prefix_joined
    o = host.nbt * host.bt_w + host.T
    dec = host.i32[o:o + 8 * host.n_dec_items].reshape(-1, 8)
    pre = host.i32[o + 8 * host.n_dec_items:][:8 * host.n_prefix_items].reshape(-1, 8)
    assert (pre[:, 1] * r.G <= 128).all()
    seen = {b: [] for b in range(host.T)}
    for b, lo, hi, split, n, npre, _, _ in dec:
        seen[b].append((lo, hi, npre + split))
        assert all(t[7] == npre for t in pre if t[0] <= b < t[0] + t[1] and not t[6])
    for q0, cnt, _, lo, hi, split, alt, _ in pre:
        for t in range(q0, q0 + cnt):
            seen[t].append((lo, hi, split))
            assert bool(alt) == (t >= host.B)
    limit = host.i32[host.nbt * host.bt_w:][:host.T]
    parts = host.i32[o + 8 * (host.n_dec_items + host.n_prefix_items):][:host.mixed]
    assert host.mixed == host.T and not host.n_merge and host.prefill_splits
    for b, spans in seen.items():
        spans.sort()
        assert [a[0] for a in spans] == [0] + [a[1] for a in spans[:-1]] and spans[-1][1] > limit[b]
        assert {a[2] for a in spans} == set(range(len(spans))) and parts[b] & 0xffff == len(spans)
        assert parts[b] >> 16 == (sum(a[1] <= 1024 for a in spans) if b < host.B else 0)


class _Tables:
    """The pages of a step's sequences, as a plan asks for them."""

    def __init__(self):
        self.pages, self.n = {}, 0

    def sequence(self, sid, prefix, own):
        k = -(-own // 16)
        self.pages[sid] = np.concatenate([np.arange(prefix), np.arange(self.n, self.n + k)])
        self.n += k
        return SimpleNamespace(seq_id=sid, total_len=prefix * 16 + own, token_at=lambda p: 1, tokens_range=lambda a, b: [1] * (b - a))

    def fill_block_tables(self, ids, bt):
        for row, sid in zip(bt, ids):
            row[:len(self.pages[sid])] = self.pages[sid][:len(row)]

    def fill_slots(self, sid, a, b, slots, at):
        slots[at:at + b - a] = 0


def _planned(hkv, G, shared, rows, own, portions, dev="cpu"):
    """(runner, plan) of a step: ``rows`` decoding sequences of ``own`` keys behind ``shared`` ones, beside ``portions`` (new tokens, own
    history) behind the same prefix, history None: a prompt with nothing in common."""
    t = _Tables()
    t.n = shared // 16
    r = mr.ModelRunner.__new__(mr.ModelRunner)
    r.device, r.kvm, r.model, r.G = torch.device(dev), t, SimpleNamespace(hkv=hkv, hq=hkv * G, D=128, scale=128 ** -0.5), G
    r.segments = r.pad_rows = r.fixed_decode_items = False
    r.graphs, r.variant, r.tile, r.mixed_tile, r.max_blocks, r.target_wgs, r.prefill_kv_chunk = None, 3, 256 // G, 128 // G, 16384, 256, 256
    r.cascade_bf16 = r.mixed_attn = r.use_cascade = r.join_suffix = r.retile_joins = True
    r.cascade_min_prefix, r.stager = 512, mr._Stager(torch.device(dev))
    dec = [t.sequence(f"d{i}", shared // 16, max(1, own - 7 * i)) for i in range(rows)]
    pre = []
    for j, (n, hist) in enumerate(portions):
        first = 0 if hist is None else shared // 16 * 16 + hist
        pre.append((t.sequence(f"p{j}", 0 if hist is None else shared // 16, n + (hist or 0)), first, first + n))
    return r, r.build_host(SimpleNamespace(decode=dec, prefill=pre))[0]


def _check_plan(r, h):
    """Every key of every row in one part, the parts of a row in slots of their own from 0 on, no more than one launch merges, and within
    the buffers that the step makes."""
    o = h.nbt * h.bt_w
    limit, B = h.i32[o:o + h.T], h.B
    o += h.T
    dec = h.i32[o:o + 8 * h.n_dec_items].reshape(-1, 8)
    o += dec.size
    pre = h.i32[o:o + 8 * h.n_prefix_items].reshape(-1, 8)
    o += pre.size
    parts = h.i32[o:o + h.mixed]
    meta = r.views(torch.zeros(3 * h.T + h.n_rows, dtype=torch.int64), torch.from_numpy(h.i32), h).attn
    seen = [[] for _ in range(h.T)]
    for b, lo, hi, split, _, npre, _, _ in dec.tolist():
        assert npre + split < meta.part.shape[2] and meta.part.numel() * 4 < 1 << 31
        seen[b].append((lo, hi, npre + split))
    for q0, n, _, lo, hi, slot, alt, _ in pre.tolist():
        assert 1 <= n <= r.mixed_tile and hi - lo <= mr.MAX_ITEM_KEYS
        for t in range(q0, q0 + n):
            assert bool(alt) == (t >= B)
            seen[t].append((lo, hi, slot))
    joined = [t for t in range(B, h.T) if seen[t]]
    assert not meta.counters.any() and meta.counters.numel() == h.mixed * r.model.hkv
    at = meta.counters.storage_offset()            # (in cache lines of their own)
    assert at % 64 == 0 and at >= o + h.mixed and not h.i32[at:at + -(-h.mixed * r.model.hkv // 64) * 64].any()
    if joined:                                     # (their partials lie in a buffer of their rows)
        assert meta.alt_off == joined[0] and meta.alt_part.shape[0] == joined[-1] + 1 - joined[0] and h.mixed == joined[-1] + 1
        assert max(a[2] for t in joined for a in seen[t]) < meta.alt_part.shape[2] and meta.alt_part.numel() * 4 <= 1 << 30
    for t, spans in enumerate(seen[:h.mixed]):
        assert len(spans) == parts[t] & 0xffff and len(spans) <= mr.MAX_PARTIALS
        if spans:
            spans.sort()
            assert [a[0] for a in spans] == [0] + [a[1] for a in spans[:-1]] and spans[-1][1] > limit[t]
            assert [a[2] for a in spans] == list(range(len(spans)))
    assert not any(seen[h.mixed:])
    if meta.prefill_items is not None:             # rows of no joined turn: launches of their own
        for q0, n, *_ in meta.prefill_items.tolist():
            assert not any(seen[B + q0:B + q0 + n])


@pytest.mark.parametrize("hkv,G", [(8, 4), (4, 8), (2, 4), (1, 8), (8, 1)])
def test_new_turns_behind_long_histories_have_as_many_parts_as_one_launch_merges(hkv, G):
    longest = 0
    for shared in (512, 1024, 2048, 18000):
        for rows, own in ((2, 300), (30, 1344)):
            for n, hist in ((90, 500), (90, 6000), (33, 16500), (83, 30000), (500, 9000), (5, 120000), (1, 60000)):
                r, h = _planned(hkv, G, shared, rows, own, [(n, hist)])
                assert h.mixed
                _check_plan(r, h)
                longest = max(longest, h.prefill_splits)
    assert longest > 20 and (hkv > 2 or longest == mr.MAX_PARTIALS)     # (the bound is met where few heads share the launch)


@pytest.mark.parametrize("hkv,G", [(8, 4), (1, 8), (8, 1)])
@pytest.mark.parametrize("rows,portions", [
    (12, [(6000, None), (90, 6000)]), (4, [(5000, None), (90, 9000)]), (8, [(7000, None), (100, 6000)]), (8, [(8000, None), (100, 8000)]),
    (8, [(6000, None), (2000, 4000)]), (8, [(90, 6000), (300, None), (41, 3000)]), (4, [(90, 30000), (7000, None), (90, 30000)]), (30, [(2048, 60000)])])
def test_partials_of_new_turns_beside_cold_prompts(rows, portions, hkv, G):
    """Rows that are not the launch's take no part in its buffers, which stay within what its merge addresses; what would not is two launches."""
    one = 0
    for shared in (1024, 6000):
        r, h = _planned(hkv, G, shared, rows, 300, portions)
        between = len(portions) == 3 and portions[1][0] > 1000
        assert h.mixed or between and hkv * G > 8
        if h.mixed:
            one += 1
            _check_plan(r, h)
        assert bool(h.prefix_joined)
    assert one or between


def test_partials_past_what_one_launch_addresses_are_two_launches(monkeypatch):
    batch = (8, 4, 1024, 40, 300, [(90, 3000)])
    h = _planned(*batch)[1]
    assert h.mixed and h.alt_slots
    row, alt = 32 * 128 * 4, (h.mixed - h.B - h.alt_lo) * h.alt_slots
    for name, n in (("MIXED_ALT_BYTES", alt * row - 1), ("MIXED_PART_BYTES", h.B * h.s_total * row)):
        with monkeypatch.context() as m:
            m.setattr(mr, name, n)
            two = _planned(*batch)[1]
        assert not two.mixed and two.n_merge and two.prefix_joined and not two.alt_slots
    with monkeypatch.context() as m:
        m.setattr(mr, "MIXED_ALT_BYTES", alt * row)
        m.setattr(mr, "MIXED_PART_BYTES", h.B * h.s_total * row + 1)
        assert _planned(*batch)[1].mixed


@pytest.mark.parametrize("hkv,G,shared,rows,own,one", [
    (8, 4, 8192, 8, 900, True), (8, 4, 8224, 8, 900, False), (8, 4, 9000, 2, 2600, False), (8, 4, 18000, 28, 900, False),   # one row tile in 32 parts
    (8, 4, 9000, 32, 1344, True), (8, 4, 9000, 33, 300, True), (8, 8, 9000, 16, 900, False), (8, 8, 9000, 17, 900, True),   # ... beside enough pieces; two
    (4, 8, 9000, 8, 900, True), (16, 2, 9000, 8, 900, True), (2, 4, 18000, 8, 900, True),   # parts that leave CUs idle, or are fewer
    (8, 4, 18000, 40, 500, False), (8, 4, 18000, 40, 700, True), (8, 4, 9000, 40, 400, True), (8, 4, 18000, 96, 60, True)])
def test_few_rows_behind_long_prefixes_take_two_launches(hkv, G, shared, rows, own, one):
    r, h = _planned(hkv, G, shared, rows, own, [])
    assert bool(h.mixed) == one and h.n_prefix_items
    if one:
        _check_plan(r, h)


def test_plans_of_one_launch_travel_whole():
    h = _planned(8, 4, 1024, 5, 200, [(90, 6000), (300, None), (41, 3000)])[1]
    z = np.zeros(0, np.float32)
    got, _ = mr.unpack_plan(*mr.pack_plan(h, mr.SampleParams(z, z, z.astype(np.int32), z.astype(np.int64), None, True)))
    assert h.mixed and h.alt_slots
    assert all(getattr(got, f) == getattr(h, f) for f in mr._PLAN_SCALARS)
    assert np.array_equal(got.i32, h.i32) and np.array_equal(got.i64, h.i64)


#: (kv heads, G, shared, decode rows, their own keys, portions, parts of the longest row): as many parts as a launch merges; a turn's tile cut
#: into several, some of whose pieces lie past the first ones' limits; a cold prompt between and before joined turns, both kinds of splits
#: beside each other; whole tiles of one head
STEPS = [(1, 8, 512, 2, 300, [(33, 60000)], 64), (2, 4, 640, 3, 100, [(70, 20)], 2), (2, 4, 1024, 5, 200, [(90, 6000), (300, None), (41, 3000)], 20),
         (2, 4, 1024, 5, 200, [(2000, None), (90, 6000)], 20), (8, 1, 1024, 4, 90, [(150, 1200)], 4)]


def _steps(hkv, G, shared, rows, own, portions, parts, dev):
    r, h = _planned(hkv, G, shared, rows, own, portions, dev)
    assert h.mixed and max(h.alt_slots, h.tile_splits) >= parts
    g = torch.Generator().manual_seed(5)
    n = r.kvm.n
    k = torch.randn(n, hkv, 16, 128, generator=g).to(torch.bfloat16)
    v = torch.randn(n, hkv, 128, 16, generator=g).to(torch.bfloat16)
    q = torch.randn(h.T, hkv * G, 128, generator=g).to(torch.bfloat16)
    meta = r.to_device(h).attn
    out = torch.full(q.shape, float("nan"), dtype=torch.bfloat16, device=dev)
    paged_attention(q.to(dev), k.to(dev), v.to(dev), meta, out)
    if dev != "cpu":
        first = out.clone()
        paged_attention(q.to(dev), k.to(dev), v.to(dev), meta, out)
        assert torch.equal(first, out) and not meta.counters.any()
    assert not out.isnan().any()
    alone = torch.full_like(out, float("nan"))     # (without the cold prompts' launch: their rows, between the joined ones too, are left alone)
    paged_attention(q.to(dev), k.to(dev), v.to(dev), dataclasses.replace(meta, prefill_items=None, prefill_merge=[]), alone)
    mine = torch.zeros(h.T, dtype=torch.bool)
    mine[:h.mixed] = meta.row_parts.cpu() > 0
    assert mine[:h.B].all() and torch.equal(alone[mine], out[mine]) and alone[~mine].isnan().all()
    o, starts = h.nbt * h.bt_w, [h.B]
    bt, limit = torch.from_numpy(h.i32[:o].reshape(h.nbt, -1)), h.i32[o:o + h.T]
    for m, _ in portions:
        starts.append(starts[-1] + m)
    picks = {b: b for b in range(h.B)}
    for j, (a, b) in enumerate(zip(starts, starts[1:])):
        picks.update({t: h.B + j for t in (a, a + 31, a + 33, a + 64, (a + b) // 2, b - 1) if a <= t < b})
    for t, row in picks.items():                   # (as _check: 3 roundings of 2^-9, taken twice)
        kk, vv = ref.gather_kv(k, v, bt[row], int(limit[t]) + 1)
        s = torch.einsum("hgd,nhd->hgn", q[t].float().view(hkv, G, 128), kk.float()) / math.sqrt(128)
        want = torch.einsum("hgn,nhd->hgd", s.softmax(-1), vv.float()).reshape(-1, 128)
        assert (out[t].float().cpu() - want).abs().max() <= 6 * 2.0 ** -9 * want.abs().max(), t


@pytest.mark.parametrize("step", STEPS)
def test_steps_with_new_turns_equal_whole_attention_cpu(step):
    _steps(*step, "cpu")


@pytest.mark.gpu
@pytest.mark.parametrize("step", STEPS)
def test_steps_with_new_turns_equal_whole_attention(cuda, step):
    _steps(*step, cuda)
