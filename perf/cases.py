"""What this framework is timed on: engine steps of served models.

A pass is one step of ``LLMEngine`` as the server's loop launches it: the step plan that the host has made while the step
before was on the GPU (``ModelRunner.build_host``) is uploaded, the model runs over the paged caches and state slots, and the
logits of the rows that need them come back on the device (``ModelRunner.forward_logits``). Engine, weights, the sequences'
histories in the caches and the plan are what a server holds before the step; they are made by ``prepare``. The step writes
its keys, values and states into the engine's caches, so a pass repeated on the same state does the same work again (the
recurrent families' decode steps move their states on, as decoding does).

Models are few layers of the real widths (the layer kinds in the proportions of the families' presets), because a step is the
same layers over and over: Llama-3-8B's and Mixtral-8x7B's layer sizes with the smaller of their two vocabularies, and three
of the segment-planned families at the width of ``bench.py --arch-compare``, which between them hold the latent attention, the
windowed and plain grouped-query attention of prompt portions and single tokens, the state-space scan, both linear-attention
scans, the matrix memory, dense and routed feed-forwards. bf16 weights and activations; the caches bf16 or, for Llama, fp8.

Weights are drawn here, so that ``exact`` needs nothing of the package. Routed models get a vocabulary whose tokens lean
towards a few experts each, as trained ones do: the choice of the experts is then no matter of the last bit.
"""
from __future__ import annotations

import dataclasses
import math

import torch

from kafka_llm_service_amd.engine.engine import EngineConfig, LLMEngine
from kafka_llm_service_amd.engine.sequence import SamplingParams, Sequence
from kafka_llm_service_amd.models.budurax import BuduraxConfig, BuduraxLM
from kafka_llm_service_amd.models.config import PRESETS
from kafka_llm_service_amd.models.furapel import FurapelConfig, FurapelLM
from kafka_llm_service_amd.models.llama import TransformerLM
from kafka_llm_service_amd.models.moe import MoEBlock
from kafka_llm_service_amd.models.rogosun import RogosunConfig, RogosunLM

VOCAB = 32000
LAYERS = {"llama": 4, "mixtral": 2, "budurax": 3, "rogosun": 4, "furapel": 4}
PAGED = ("llama", "mixtral")          # prefix sharing between sequences; the other families compute every token


def _case(family, decode=0, context=0, shared=0, prompts=0, prompt=0, history=0, kv="bf16", width=4096):
    """``decode`` sequences of about ``context`` tokens get one token each; beside them ``prompts`` portions of about
    ``prompt`` tokens, each behind ``history`` tokens of its own; everybody's first ``shared`` tokens are the same."""
    return {"family": family, "width": width, "decode": decode, "context": context, "shared": shared, "prompts": prompts,
            "prompt": prompt, "history": history, "kv": kv}


def listed():
    def named(name, *a, **k):
        return dict(_case(*a, **k), name=name)

    return [
        # one user's chat, token after token: the smallest call, all latency and weight streaming
        named("llama one thread", "llama", decode=1, context=1511),
        # the headline workload's usual step: 64 threads behind one system prompt, each with its own turns
        named("llama 64 threads", "llama", decode=64, context=1344, shared=18000),
        # the same while two users send a new turn
        named("llama new turns", "llama", decode=61, context=1344, shared=18000, prompts=2, prompt=83, history=900),
        # a cold prompt of an odd length: time to the first token
        named("llama prompt", "llama", prompts=1, prompt=4099),
        # long conversations without anything in common on the small cache format
        named("llama fp8 cache", "llama", decode=29, context=7900, kv="fp8"),
        # 128 threads on the mixture of experts
        named("mixtral 128 threads", "mixtral", decode=128, context=1100),
        # a cold prompt on it
        named("mixtral prompt", "mixtral", prompts=1, prompt=1900),
        # a cold prompt on latent attention and the state-space scan
        named("budurax prompt", "budurax", prompts=1, prompt=2048),
        # 64 sequences decoding on it
        named("budurax 64 threads", "budurax", decode=64, context=2048),
        # several users' prompts at once on linear attention, raw-key attention and grouped routing
        named("rogosun prompts", "rogosun", prompts=3, prompt=1100),
        # the largest: a document on softmax, latent and matrix-memory layers with looped layers and 16 experts
        named("furapel document", "furapel", prompts=1, prompt=8192),
        # a small batch decoding on it
        named("furapel 16 threads", "furapel", decode=16, context=2048),
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    family = rng.choice(["llama", "llama", "mixtral", "budurax", "rogosun", "furapel"])
    width = rng.choice([4096, 4096, 2048]) if family != "mixtral" else 4096
    top = 4096 if family in ("llama", "mixtral", "rogosun") else 3000 if family == "budurax" else 7000
    kind = rng.choice(["decode", "prompt", "mixed"])
    kv = rng.choice(["bf16", "bf16", "bf16", "fp8"]) if family == "llama" else "bf16"
    k = {"kv": kv, "width": width}
    if kind != "prompt":
        k["decode"] = _log(rng, 1, 128 if family in PAGED else 64)
        k["context"] = min(_log(rng, 100, 8000), 120000 // k["decode"])
        if family in PAGED and rng.random() < 0.5:
            k["shared"] = _log(rng, 600, 18000)
            k["context"] = min(k["context"], 2000)
    if kind == "prompt":
        k["prompts"] = rng.choice([1, 1, 2, 5])
        k["prompt"] = _log(rng, 17, top // k["prompts"])
    elif kind == "mixed":
        k["prompts"] = rng.choice([1, 2])
        k["prompt"] = _log(rng, 9, 600)
    if kind != "decode" and rng.random() < 0.4:
        k["history"] = _log(rng, 30, 3000)
    return _case(family, **k)


# ---- sizes -------------------------------------------------------------------------------------------------------------
def _lengths(c):
    """Own tokens of the sequences (without the shared ones): ([decoding sequences' contexts], [(history, portion)])."""
    dec = [max(1, c["context"] - (i * 613) % (c["context"] // 3 + 1)) for i in range(c["decode"])]
    pro = [(c["history"], max(1, c["prompt"] - (i * 257) % (c["prompt"] // 4 + 1))) for i in range(c["prompts"])]
    return dec, pro


def _places(n):
    """Offsets of a portion of n tokens whose logits are wanted: the last one, as a server asks."""
    return [n - 1]


def _spec(c):
    """The model's config dict (segment-planned families) or ModelConfig."""
    f, d = c["family"], c["width"]
    H, ff, n = d // 128, 7 * d // 2, LAYERS[c["family"]]
    if f == "llama":
        return dataclasses.replace(PRESETS["llama3-8b"], name="llama-layers", hidden_size=d, intermediate_size=ff, num_layers=n,
                                   num_heads=H, num_kv_heads=H // 4, vocab_size=VOCAB, bos_token_id=1, eos_token_ids=[2])
    if f == "mixtral":
        return dataclasses.replace(PRESETS["mixtral-8x7b"], name="mixtral-layers", num_layers=n)
    out = {"vocab": VOCAB, "width": d, "norm": {"eps": 1e-6}}
    yarn = {"factor": 8.0, "original": 8192, "fast": 32.0, "slow": 1.0}
    if f == "budurax":
        att = {"type": "latent_attention", "mlp": {"kind": "dense", "ff": ff},
               "mixer": {"heads": H, "dim": 128, "rot_dim": 64, "vdim": 128, "kv_rank": 512, "scale": 192 ** -0.5,
                         "rot": {"base": 500000.0, "dims": 64, "scaling": yarn}}}
        ssm = {"type": "mamba2", "mlp": {"kind": "dense", "ff": ff},
               "mixer": {"heads": d // 32, "vdim": 64, "state": 128, "groups": 8, "norm_groups": 8, "conv": 4}}
        return dict(out, architecture="Budurax", layers=[att, ssm, ssm], token_side={"dim": 64})
    if f == "rogosun":
        e = ff // 3 // 256 * 256
        moe = {"kind": "moe", "expert": {"ff": e}, "shared": {"ff": e},
               "router": {"experts": 8, "top": 2, "scale": 2.5, "groups": {"count": 4, "keep": 2}}}
        dense = {"kind": "dense", "ff": ff}
        gla = {"heads": d // 256, "dim": 128, "vdim": 256, "tau": 16.0}
        par = {"left": {"heads": H, "kv_heads": 2, "dim": 128, "vdim": 128, "scale": 128 ** -0.5,
                        "rot": {"base": 100000.0, "dims": 128, "scaling": {"factor": 4.0}}},
               "right": {"heads": H, "kv_heads": H, "dim": 128, "vdim": 128, "conv": 4},
               "left_scale": 0.7, "right_scale": 0.7}
        return dict(out, architecture="Rogosun", layers=[{"type": "gla", "mixer": gla, "mlp": dense},
                                                         {"type": "parallel", "mixer": par, "mlp": moe},
                                                         {"type": "gla", "mixer": gla, "mlp": moe},
                                                         {"type": "parallel", "mixer": par, "mlp": dense}])
    moe = {"kind": "moe", "expert": {"ff": ff * 3 // 8 // 256 * 256}, "router": {"experts": 16, "top": 4}}
    att = {"heads": H, "kv_heads": H // 4, "dim": 128, "vdim": 128, "scale": 128 ** -0.5,
           "rot": {"base": 500000.0, "dims": 64, "scaling": yarn}}
    mem = {"heads": d // 256, "dim": 128, "vdim": 256, "gate_cap": 15.0}
    lat = {"heads": H, "dim": 128, "vdim": 128, "kv_rank": 512, "scale": 128 ** -0.5, "mask": {"size": 1024}}
    return dict(out, architecture="Furapel", embedding={"scale": float(d) ** 0.5}, logit_scale=0.25,
                loop={"start": 1, "stop": 2, "times": 2},
                layers=[{"type": t, "mixer": m, "mlp": moe} for t, m in (("attention", att), ("mlstm", mem), ("attention", att),
                                                                         ("latent_attention", lat))])


def _shapes(c):
    """Tensor names (the checkpoints') -> shapes; a list of three shapes per expert set is written out."""
    f, s = c["family"], _spec(c)
    d, H, out = c["width"], c["width"] // 128, {"embed": (VOCAB, c["width"])}
    if f in PAGED:
        F_, KV = s.intermediate_size, s.kv_size
        for i in range(s.num_layers):
            p = f"l{i}."
            out.update({p + "input_norm": (d,), p + "post_norm": (d,), p + "qkv": (d + 2 * KV, d), p + "o": (d, d)})
            if f == "llama":
                out.update({p + "gate_up": (2 * F_, d), p + "down": (d, F_)})
            else:
                out.update({p + "router": (8, d), p + "w13": (8, 2 * F_, d), p + "w2": (8, d, F_)})
        return dict(out, final_norm=(d,), lm_head=(VOCAB, d))
    if f == "budurax":
        out["side.embed"] = (VOCAB, 64 * len(s["layers"]))
    if f == "furapel":
        out["loop.in"] = (d, 2 * d)

    def norm(name, bias):
        out[name] = (d,)
        if bias:
            out[name + ".b"] = (d,)
        if f == "furapel":
            out[name + ".alpha"] = ()

    for i, L in enumerate(s["layers"]):
        p, m, q = f"l{i}.", L["mixer"], f"l{i}.mix."
        for n in {"budurax": ("norm1", "norm1b", "norm2", "norm2b"), "rogosun": ("norm1", "norm2"),
                  "furapel": ("norm1", "norm2")}[f]:
            norm(p + n, f != "rogosun")
        if f == "budurax":
            if L["type"] == "mamba2":
                inner, C = m["heads"] * 64, m["heads"] * 64 + 2 * 8 * 128
                out.update({q + "in": (inner + C + m["heads"], d), q + "conv": (C, 4), q + "conv.b": (C,),
                            q + "dt_bias": (m["heads"],), q + "A_log": (m["heads"],), q + "D": (m["heads"],),
                            q + "norm": (inner,), q + "o": (d, inner)})
            else:
                out.update({q + "q": (H * 192, d), q + "dkv": (576, d), q + "dkv.norm": (512,), q + "uk": (H * 128, 512),
                            q + "uv": (H * 128, 512), q + "g": (H * 128, d), q + "o": (d, H * 128)})
            out.update({p + "mlp.gate": (L["mlp"]["ff"], d), p + "mlp.up": (L["mlp"]["ff"], d),
                        p + "mlp.down": (d, L["mlp"]["ff"]), p + "shift": (d,), p + "dwa": (i + 2,), p + "side.gate": (64, d),
                        p + "side.proj": (d, 64), p + "side.norm": (d,)})
        elif L["type"] == "gla":
            out.update({q + "q": (d // 2, d), q + "k": (d // 2, d), q + "v": (d, d), q + "g": (d, d), q + "o": (d, d),
                        q + "norm": (256,), q + "a1": (16, d), q + "a2": (d // 2, 16), q + "a2.b": (d // 2,)})
        elif L["type"] == "parallel":
            a, b = q + "left.", q + "right."
            out.update({a + "q": (d, d), a + "k": (256, d), a + "q.norm": (128,), a + "k.norm": (128,), a + "o": (d, d)})
            for n in "qkv":
                out.update({b + n: (d, d), b + n + ".conv": (d, 4)})
            out.update({b + "b": (H, d), b + "A_log": (H,), b + "norm": (128,), b + "a1": (64, d), b + "a2": (d, 64),
                        b + "dt_bias": (d,), b + "g1": (64, d), b + "g2": (d, 64), b + "o": (d, d)})
        elif L["type"] == "mlstm":
            out.update({q + "q": (d // 2, d), q + "k": (d // 2, d), q + "v": (d, d), q + "g": (d, d), q + "o": (d, d),
                        q + "norm": (d,)})
            for n in "if":
                out.update({q + n: (d // 256, d), q + n + ".b": (d // 256,)})
        elif L["type"] == "attention":
            out.update({q + "q": (d, d), q + "k": (d // 4, d), q + "v": (d // 4, d), q + "g": (H, d), q + "o": (d, d)})
        else:
            out.update({q + "q": (d, d), q + "dkv": (512, d), q + "dkv.norm": (512,), q + "uk": (d, 512), q + "uv": (d, 512),
                        q + "o": (d, d)})
        if f == "rogosun" and L["mlp"]["kind"] == "dense":
            out.update({p + "mlp.up": (L["mlp"]["ff"], d), p + "mlp.down": (d, L["mlp"]["ff"])})
        elif f != "budurax":
            e, parts = L["mlp"]["expert"]["ff"], ("gate", "up") if f == "rogosun" else ("up",)
            for x in [f"e{j}" for j in range(L["mlp"]["router"]["experts"])] + (["shared"] if f == "rogosun" else []):
                out.update({f"{p}mlp.{x}.{n}": (e, d) for n in parts})
                out[f"{p}mlp.{x}.down"] = (d, e)
            out[p + "mlp.router"] = (L["mlp"]["router"]["experts"], d)
    norm("final.norm", f != "rogosun")
    return dict(out, head=(VOCAB, d))


#: how far a token's embedding leans towards its experts (first choice first), and the gain of the routers
LEAN = {"mixtral": ([0.30, 0.22], 0.15), "rogosun": ([0.30, 0.22], 0.15), "furapel": ([0.48, 0.40, 0.32, 0.24], 0.08)}


def _weights(c, seed):
    """bf16 tensors on the GPU: norms around one, decays that mostly keep, matrices that keep their input's size."""
    g = torch.Generator(device="cuda").manual_seed(seed)
    d, f, out = c["width"], c["family"], {}
    lean, gain = LEAN.get(f, ([], 0.0))
    E = {"mixtral": 8, "rogosun": 8, "furapel": 16}.get(f, 0)
    signs = torch.randint(0, 2, (E, d), generator=g, device="cuda").float() * 2 - 1

    def rn(*shape, dtype=torch.float32):
        return torch.randn(shape, generator=g, device="cuda", dtype=dtype)

    def ru(*shape):
        return torch.rand(shape, generator=g, device="cuda")

    for name, shape in _shapes(c).items():
        leaf = name.split(".")[-1]
        if name == "embed":
            t = rn(*shape)
            if lean:  # experts of different groups of two, chosen at random
                order = torch.rand(VOCAB, E // 2, generator=g, device="cuda").argsort(1)[:, :len(lean)] * 2 + \
                    torch.randint(0, 2, (VOCAB, len(lean)), generator=g, device="cuda")
                for j, a in enumerate(lean):
                    t += a * signs[order[:, j]]
            if f == "furapel":
                t /= math.sqrt(d)  # (the config scales the rows up again)
        elif leaf == "router":
            t = signs * (gain / math.sqrt(d)) + rn(*shape) * (0.02 / math.sqrt(d))
        elif name == "loop.in":  # mostly keeps the residual and its input
            t = rn(*shape) * (0.2 / math.sqrt(2 * d)) + 0.7 * torch.eye(d, device="cuda").repeat(1, 2)
        elif leaf == "alpha":
            t = 0.7 + 0.1 * rn(*shape)
        elif "norm" in leaf:
            t = (1 + 0.1 * rn(*shape)) * (0.5 if leaf in ("norm1b", "norm2b") or name.endswith("side.norm") else 1)
        elif name.endswith("mix.f.b"):
            t = 2 + 3 * ru(*shape)
        elif name.endswith("a2.b"):
            t = 1 + rn(*shape)
        elif leaf == "b" and len(shape) == 1:
            t = 0.1 * rn(*shape)
        elif leaf == "shift":
            t = ru(*shape)
        elif leaf == "dwa":
            t = ru(*shape) + 0.2
            t /= t.sum()
        elif leaf == "A_log":
            t = torch.log(1 + 7 * ru(*shape)) if f == "budurax" else torch.log(0.5 + 3.5 * ru(*shape))
        elif leaf == "dt_bias":
            t = torch.log(torch.expm1(0.01 + 0.2 * ru(*shape))) if f == "budurax" else -4 + 4 * ru(*shape)
        elif leaf == "D":
            t = 1 + 0.1 * rn(*shape)
        else:
            t = rn(*shape, dtype=torch.bfloat16) * shape[-1] ** -0.5
        out[name] = t.to(torch.bfloat16)
    return out


def _tokens(c, seed):
    """Token ids as lists: (shared, [decoding sequence: context + its next token], [(history, portion)])."""
    g = torch.Generator().manual_seed(seed + 1)
    dec, pro = _lengths(c)

    def ids(n):
        return torch.randint(3, VOCAB, (n,), generator=g).tolist()

    return ids(c["shared"]), [ids(n + 1) for n in dec], [(ids(h), ids(n)) for h, n in pro]


# ---- the engine --------------------------------------------------------------------------------------------------------
def _engine(c, seed):
    W, s = _weights(c, seed), _spec(c)
    dec, pro = _lengths(c)
    own = [n + 1 for n in dec] + [h + n for h, n in pro]
    longest = c["shared"] + max(own)
    blocks = c["shared"] // 16 + sum(n // 16 + 2 for n in own) + 8
    if c["family"] in PAGED:
        mc, model = s, TransformerLM(s, "cuda:0", max_positions=longest + 16)
        for name in ("embed", "lm_head", "final_norm"):
            setattr(model, name, W.pop(name))
        for name in list(W):
            i, kind = name[1:].split(".")
            setattr(model.layers[int(i)], kind, W.pop(name))
        if s.num_experts:
            model.moe = MoEBlock(model)
    else:
        Conf, Model = {"budurax": (BuduraxConfig, BuduraxLM), "rogosun": (RogosunConfig, RogosunLM),
                       "furapel": (FurapelConfig, FurapelLM)}[c["family"]]
        mc = Conf.from_dict(s, name=c["family"])
        model = Model(mc, "cuda:0", max_positions=longest + 16).load_tensors(W)
    return LLMEngine(EngineConfig(model=mc.name, device="cuda:0", num_kv_blocks=blocks, max_num_seqs=len(own) + 1,
                                  max_model_len=longest + 16, kv_dtype=c["kv"]), model_cfg=mc, model=model)


def _plan(eng, portions):
    """The engine's plan of a step over the next tokens of the given sequences, logits at each portion's last token."""
    batch = eng.sched.replay(portions)
    want = {s.seq_id: [] for s, _ in portions}
    for s, a, b in [(s, s.total_len - 1, s.total_len) for s in batch.decode] + batch.prefill:
        want[s.seq_id] = _places(b - a)
    return eng.runner.build_host(batch, want=want)[0], batch


def _advance(eng, portions):
    """A step whose logits nobody wants: the sequences' next tokens go into the caches."""
    host, batch = _plan(eng, portions)
    eng.runner.forward_logits(host)
    for s, b in [(s, s.total_len) for s in batch.decode] + [(s, b) for s, _, b in batch.prefill]:
        s.num_computed = b
        eng.kvm.commit(s.seq_id, b)


def prepare(case, seed):
    eng = _engine(case, seed)
    shared, dec, pro = _tokens(case, seed)
    before = [t[:-1] for t in dec] + [h for h, _ in pro]
    after = [t[-1:] for t in dec] + [n for _, n in pro]
    seqs, fill = [], []
    with torch.inference_mode():
        if shared:
            s = Sequence("shared", list(shared), SamplingParams(max_tokens=1))
            for a in range(0, len(shared), 6000):
                _advance(eng, [(s, min(6000, len(shared) - a))])
        for i, (b, t) in enumerate(zip(before, after)):
            seqs.append(Sequence(f"r{i}", (list(shared) + b) or t, SamplingParams(max_tokens=1)))
            if shared or b:
                fill.append((seqs[-1], seqs[-1].total_len))
            if fill and (i + 1 == len(before) or sum(n - len(shared) for _, n in fill) > 6000):
                _advance(eng, fill)
                fill = []
        for s, t in zip(seqs, after):
            if s.num_computed:
                s.prompt_ids.extend(t)
                eng.kvm.append_tokens(s.seq_id, t)
        host, _ = _plan(eng, [(s, len(t)) for s, t in zip(seqs, after)])
    at = {k: i for i, k in enumerate(host.owners)}
    order = [at[(s.seq_id, _places(len(t))[0])] for s, t in zip(seqs, after)]
    return {"engine": eng, "plan": host, "order": torch.tensor(order, device="cuda:0")}


def run(state):
    return state["engine"].runner.forward_logits(state["plan"]).index_select(0, state["order"])


def work(case):
    """Weights of the step (of the experts that its tokens reach) and the caches and states of its sequences read once, the new
    rows and logits written; the multiply-adds of the projections, the attention and the states."""
    c, f = case, case["family"]
    dec, pro = _lengths(c)
    T = len(dec) + sum(n for _, n in pro)
    n_out = len(dec) + len(pro)
    s, d = _spec(c), c["width"]
    nbytes = flops = 0.0
    reps = [1, 2, 1, 1] if f == "furapel" else [1] * LAYERS[f]
    E, top = {"mixtral": (8, 2), "rogosun": (8, 2), "furapel": (16, 4)}.get(f, (0, 0))
    reached = 1 - (1 - top / E) ** T if E else 0
    for name, shape in _shapes(c).items():
        n = math.prod(shape)
        if name in ("embed", "side.embed"):
            nbytes += T * shape[1] * 2
            continue
        if name in ("lm_head", "head"):
            nbytes, flops = nbytes + 2 * n, flops + 2 * n * n_out
            continue
        times = reps[int(name[1:name.index(".")])] if name[0] == "l" and name[1].isdigit() else 2 if name == "loop.in" else 1
        expert = name.endswith(("w13", "w2")) or ".mlp.e" in name
        nbytes += 2 * n * (reached if expert else 1)
        if len(shape) > 1:
            flops += 2 * n * T * times * (top / E if expert else 1)
    P = c["shared"]
    new = [(P + n, 1) for n in dec] + [(P + h, n) for h, n in pro]
    keys = P + sum(p - P + n for p, n in new)         # distinct positions read
    pairs = sum(n * p + n * (n + 1) / 2 for p, n in new)
    if f in PAGED:
        kvb = 2 * s.kv_size * (1 if c["kv"] == "fp8" else 2)
        nbytes += s.num_layers * kvb * (keys + T)
        flops += s.num_layers * 4.0 * d * pairs
    elif f == "budurax":
        nbytes += 2 * 576 * (keys + T) + 2 * 2 * len(new) * 4 * d * 2 * 128
        flops += 2.0 * (d // 128) * (576 + 512) * pairs + 2 * T * 6.0 * 2 * d * 128
    elif f == "rogosun":
        nbytes += 2 * 2 * 512 * (keys + T) + 4 * 2 * len(new) * 4 * d * 128
        flops += 2 * 4.0 * d * pairs + 4 * T * 6.0 * d * 128
    else:
        near = sum(sum(min(1024, p + 1 + j) for j in range(n)) for p, n in new)
        nbytes += 2 * 2 * 2 * (d // 4) * (keys + T) + 2 * 512 * (sum(min(1024, p) + n for p, n in new) + T)
        nbytes += 2 * 2 * len(new) * 4 * d * 128
        flops += 2 * 4.0 * d * pairs + 2.0 * (d // 128) * 1024 * near + 2 * T * 6.0 * d * 128
    return {"bytes": nbytes + n_out * VOCAB * (2 if f in PAGED else 4), "flops": flops}


def tolerance(case):
    """bf16 products and activations through the layers: the steps are 0.003 (the families with an fp32 residual) to 0.008 (bf16
    residual; 0.005 with experts) from 64 bits, and 0.008 to 0.019 where the residual itself is what the layers read (rogosun)."""
    return {"rel": {"llama": 0.03, "mixtral": 0.02, "budurax": 0.014, "rogosun": 0.03, "furapel": 0.014}[case["family"]]}


# ---- the same in 64 bits, with plain tensor operations ------------------------------------------------------------------
def _rms(x, eps, w=None):
    y = x / torch.sqrt((x * x).mean(-1, keepdim=True) + eps)
    return y if w is None else y * w


def _frequencies(rot):
    """(frequency of every pair, factor on cosine and sine) of a rotation entry of the segment-planned families."""
    dims, base = int(rot["dims"]), float(rot["base"])
    f = torch.tensor([base ** (-2.0 * i / dims) for i in range(dims // 2)], dtype=torch.float64, device="cuda")
    sc = rot.get("scaling")
    if not sc:
        return f, 1.0
    if set(sc) == {"factor"}:
        return f / sc["factor"], 1.0

    def pair(turns):
        return dims * math.log(sc["original"] / (2 * math.pi * turns)) / (2 * math.log(base))

    lo, hi = max(math.floor(pair(sc["fast"])), 0), min(math.ceil(pair(sc["slow"])), dims - 1)
    r = ((torch.arange(dims // 2, dtype=torch.float64, device="cuda") - lo) / max(hi - lo, 0.001)).clamp(0, 1)
    return f / sc["factor"] * r + f * (1 - r), 0.1 * math.log(sc["factor"]) + 1


def _llama_frequencies(s):
    f = s.rope_theta ** (-torch.arange(0, 128, 2, dtype=torch.float64, device="cuda") / 128)
    sc = s.rope_scaling
    if not sc:
        return f
    turns = sc["original_max_position_embeddings"] * f / (2 * math.pi)   # over the original context
    lo, hi = sc["low_freq_factor"], sc["high_freq_factor"]
    r = ((turns - lo) / (hi - lo)).clamp(0, 1)
    return f / sc["factor"] * (1 - r) + f * r


def _turn(x, pos, f, mag=1.0):
    """x [n, heads, D]: dimension i turns with dimension i + len(f)."""
    a = pos.double()[:, None] * f[None]
    co, si, h = (mag * torch.cos(a))[:, None], (mag * torch.sin(a))[:, None], f.numel()
    u, v = x[..., :h], x[..., h:2 * h]
    return torch.cat([u * co - v * si, v * co + u * si, x[..., 2 * h:]], -1)


class _Rows:
    """All rows of the step and of its histories one below the other: per sequence (first row, rows, first position, whether
    it stands on the shared rows, which are the first)."""

    def __init__(self, c, seed):
        shared, dec, pro = _tokens(c, seed)
        runs = ([shared] if shared else []) + dec + [h + n for h, n in pro]
        self.tokens = torch.tensor([t for r in runs for t in r], device="cuda")
        self.runs, at = [], 0
        for i, r in enumerate(runs):
            own = i == 0 and bool(shared)
            self.runs.append((at, len(r), 0 if own else len(shared), bool(shared) and not own))
            at += len(r)
        self.pos = torch.cat([torch.arange(p, p + n, device="cuda") for _, n, p, _ in self.runs])
        self.n_shared = len(shared)
        self.asked = torch.tensor([a + n - 1 for a, n, _, _ in self.runs[1 if shared else 0:]], device="cuda")

    def padded(self, x):
        """[rows, ...] -> [sequences, longest, ...], zeros behind the shorter ones."""
        out = x.new_zeros(len(self.runs), max(n for _, n, _, _ in self.runs), *x.shape[1:])
        for i, (a, n, _, _) in enumerate(self.runs):
            out[i, :n] = x[a:a + n]
        return out

    def flat(self, y):
        return torch.cat([y[i, :n] for i, (_, n, _, _) in enumerate(self.runs)])

    def attend(self, q, k, v, scale, window=None, sink=False):
        """q [rows, H, D], k [rows, G, D], v [rows, G, Dv] -> [rows, H, Dv]; ``sink``: a further score of 0 without a value."""
        H, G = q.shape[1], k.shape[1]
        out = q.new_empty(q.shape[0], H, v.shape[2])
        for a, n, p, on in self.runs:
            kk, vv = (torch.cat([t[:self.n_shared], t[a:a + n]]) if on else t[a:a + n] for t in (k, v))
            first = p - (self.n_shared if on else 0)     # position of the first key
            kk, vv = kk.permute(1, 2, 0).contiguous(), vv.transpose(0, 1).contiguous()
            step = max(16, int(2e9 // (8 * H * kk.shape[2])))
            for b in range(0, n, step):
                e = min(n, b + step)
                lo = 0 if window is None else max(0, p + b - window + 1 - first)
                hi = p + e - first
                qq = q[a + b:a + e].transpose(0, 1).reshape(G, -1, q.shape[2])
                s = (qq @ kk[:, :, lo:hi] * scale).view(H, e - b, hi - lo)
                dist = torch.arange(p + b, p + e, device="cuda")[:, None] - torch.arange(first + lo, first + hi, device="cuda")
                bad = dist < 0 if window is None else (dist < 0) | (dist >= window)
                s.masked_fill_(bad, float("-inf"))
                m = s.amax(-1, keepdim=True)
                m = m.clamp(min=0) if sink else m
                s = torch.exp_(s.sub_(m))
                s /= s.sum(-1, keepdim=True) + (torch.exp(-m) if sink else 0)
                out[a + b:a + e] = (s.view(G, -1, hi - lo) @ vv[:, lo:hi]).view(H, e - b, -1).transpose(0, 1)
        return out


def _by(rows, f, x):
    """f over some rows at a time: what lies between two products of a feed-forward is large."""
    return torch.cat([f(x[a:a + rows]) for a in range(0, x.shape[0], rows)])


def _mm(x, w):
    return x @ w.double().T


def _routed(h, weights, expert):
    y = torch.zeros_like(h)
    for e in range(weights.shape[1]):
        r = weights[:, e].nonzero()[:, 0]
        if r.numel():
            y[r] += weights[r, e:e + 1] * _by(16384, lambda t: expert(e, t), h[r])
    return y


def _chosen(score, by, top):
    """The scores of the ``top`` largest in ``by``, zeros elsewhere."""
    e = by.topk(top, -1).indices
    return torch.zeros_like(score).scatter_(1, e, score.gather(1, e))


def _glu(h, g, u, down, act):
    return _by(16384, lambda t: _mm(act(_mm(t, g)) * _mm(t, u), down), h)


def _exact_paged(c, W, R):
    s, silu = _spec(c), torch.nn.functional.silu
    H, G, eps, F_ = s.num_heads, s.num_kv_heads, s.rms_norm_eps, s.intermediate_size
    x, f = W["embed"][R.tokens].double(), _llama_frequencies(s)
    for i in range(s.num_layers):
        p = f"l{i}."
        qkv = _mm(_rms(x, eps, W[p + "input_norm"].double()), W[p + "qkv"]).view(-1, H + 2 * G, 128)
        q, k = _turn(qkv[:, :H], R.pos, f), _turn(qkv[:, H:H + G], R.pos, f)
        x = x + _mm(R.attend(q, k, qkv[:, H + G:], 128 ** -0.5).flatten(1), W[p + "o"])
        del q, k, qkv
        if i == s.num_layers - 1:
            x = x[R.asked]
        h = _rms(x, eps, W[p + "post_norm"].double())
        if c["family"] == "llama":
            x = x + _glu(h, W[p + "gate_up"][:F_], W[p + "gate_up"][F_:], W[p + "down"], silu)
        else:
            z = torch.softmax(_mm(h, W[p + "router"]), -1)
            w = _chosen(z, z, 2)
            x = x + _routed(h, w / w.sum(-1, keepdim=True), lambda e, t: _glu(t, W[p + "w13"][e, :F_], W[p + "w13"][e, F_:],
                                                                            W[p + "w2"][e], silu))
    return _mm(_rms(x, eps, W["final_norm"].double()), W["lm_head"])


def _before(R, x, w, b):
    """Causal convolution per channel over each sequence (the last column of w is the current row's)."""
    y, taps = R.padded(x), w.shape[1]
    out = torch.zeros_like(y) + b
    for j in range(taps):
        back = taps - 1 - j
        out[:, back:] += y[:, :y.shape[1] - back] * w[:, j].double()
    return R.flat(out)


def _state_space(R, x, B, C, dt, A, D):
    """S_t = exp(A dt) S + dt B x^T, y = S^T C + D x over each sequence, 64 rows at a time; B, C per group of heads."""
    x, B, C, dt = (R.padded(t) for t in (x, B, C, dt))
    n, T, H, P = x.shape
    G = B.shape[2]
    S, out = x.new_zeros(n, G, H // G, B.shape[3], P), []
    low = torch.ones(64, 64, dtype=torch.bool, device="cuda").tril()
    for a in range(0, T, 64):
        xs, Bs, Cs, ds = (t[:, a:a + 64].transpose(1, 2) for t in (x, B, C, dt[..., None]))   # [n, heads, rows, .]
        m = xs.shape[2]
        cum = (A[None, :, None] * ds[..., 0]).cumsum(-1).view(n, G, H // G, m)
        dx = (ds * xs).view(n, G, H // G, m, P)
        L = torch.exp((cum[..., :, None] - cum[..., None, :]).masked_fill(~low[:m, :m], float("-inf")))
        M = (Cs @ Bs.transpose(2, 3))[:, :, None] * L
        y = M @ dx + torch.exp(cum)[..., None] * (Cs[:, :, None] @ S)
        w = torch.exp(cum[..., -1:] - cum)[..., None]
        S = torch.exp(cum[..., -1])[..., None, None] * S + Bs.transpose(2, 3)[:, :, None] @ (w * dx)
        out.append((y.reshape(n, H, m, P) + D[None, :, None, None] * xs).transpose(1, 2))
    return R.flat(torch.cat(out, 1))


def _exact_budurax(c, W, R):
    s, eps, H = _spec(c), 1e-6, c["width"] // 128
    silu, softplus = torch.nn.functional.silu, torch.nn.functional.softplus

    def gelu(t):
        return torch.nn.functional.gelu(t, approximate="tanh")

    def norm(t, name):
        return torch.nn.functional.layer_norm(t, t.shape[-1:], W[name].double(), W[name + ".b"].double(), eps)

    x = W["embed"][R.tokens].double()
    outs = [x]
    for i, L in enumerate(s["layers"]):
        p, m = f"l{i}.mix.", L["mixer"]
        h = norm(x, f"l{i}.norm1")
        mu = W[f"l{i}.shift"][:, None].double()
        h = _before(R, h, torch.cat([mu, 1 - mu], 1), 0.0)
        if L["type"] == "mamba2":
            Hh, inner = m["heads"], m["heads"] * 64
            z = _mm(h, W[p + "in"])
            xbc = silu(_before(R, z[:, inner:2 * inner + 2048], W[p + "conv"], W[p + "conv.b"].double()))
            y = _state_space(R, xbc[:, :inner].view(-1, Hh, 64), xbc[:, inner:inner + 1024].view(-1, 8, 128),
                             xbc[:, inner + 1024:].view(-1, 8, 128),
                             softplus(z[:, -Hh:] + W[p + "dt_bias"].double(), threshold=1e9),
                             -torch.exp(W[p + "A_log"].double()), W[p + "D"].double()).flatten(1) * silu(z[:, :inner])
            y = _mm(_rms(y.view(-1, 8, inner // 8), eps).flatten(1) * W[p + "norm"].double(), W[p + "o"])
        else:
            f, mag = _frequencies(m["rot"])
            dkv = _mm(h, W[p + "dkv"])
            lat = _rms(dkv[:, :512], eps, W[p + "dkv.norm"].double())
            kr = _turn(dkv[:, None, 512:], R.pos, f, mag).expand(-1, H, -1)
            q = _mm(h, W[p + "q"]).view(-1, H, 192)
            q = torch.cat([q[..., :128], _turn(q[..., 128:], R.pos, f, mag)], -1)
            k = torch.cat([_mm(lat, W[p + "uk"]).view(-1, H, 128), kr], -1)
            o = R.attend(q, k, _mm(lat, W[p + "uv"]).view(-1, H, 128), m["scale"]).flatten(1)
            y = _mm(o * torch.sigmoid(_mm(h, W[p + "g"])), W[p + "o"])
        x = x + norm(y, f"l{i}.norm1b")
        p = f"l{i}.mlp."
        x = x + norm(_glu(norm(x, f"l{i}.norm2"), W[p + "gate"], W[p + "up"], W[p + "down"], gelu), f"l{i}.norm2b")
        g = gelu(_mm(x, W[f"l{i}.side.gate"])) * W["side.embed"][R.tokens][:, 64 * i:64 * i + 64].double()
        x = x + _rms(_mm(g, W[f"l{i}.side.proj"]), eps, W[f"l{i}.side.norm"].double())
        outs.append(x)
        x = sum(a * t for a, t in zip(W[f"l{i}.dwa"].double(), outs))
    return _mm(norm(x[R.asked], "final.norm"), W["head"])


def _scan(R, step, *inputs):
    """step(rows of the inputs at one position of all sequences) -> that position's output, in order."""
    cols = [R.padded(t).transpose(0, 1).contiguous() for t in inputs]
    out = [step(*(t[j] for t in cols)) for j in range(cols[0].shape[0])]
    return R.flat(torch.stack(out, 1))


def _matrix_state(S):
    """One position of S <- diag(a) S + k u^T, read S^T q; u = v, or beta (v - S^T k) with a beta."""
    def step(q, k, v, a, beta=None):
        S.mul_(a[..., None])
        u = v if beta is None else beta[..., None] * (v - (k[..., None, :] @ S)[..., 0, :])
        S.add_(k[..., :, None] * u[..., None, :])
        return (q[..., None, :] @ S)[..., 0, :]

    return step


def _exact_rogosun(c, W, R):
    s, eps, d, n = _spec(c), 1e-6, c["width"], len(R.runs)
    H = d // 128
    silu, softplus = torch.nn.functional.silu, torch.nn.functional.softplus
    x = W["embed"][R.tokens].double()

    def w(name):
        return W[name].double()

    for i, L in enumerate(s["layers"]):
        p = f"l{i}.mix."
        if L["type"] == "gla":
            h2 = d // 256
            q, k = (_mm(x, W[p + t]).view(-1, h2, 128) for t in "qk")
            a = torch.sigmoid(_mm(_mm(x, W[p + "a1"]), W[p + "a2"]) + w(p + "a2.b")) ** (1 / 16.0)
            o = _scan(R, _matrix_state(x.new_zeros(n, h2, 128, 256)), q * 128 ** -0.5, k,
                      _mm(x, W[p + "v"]).view(-1, h2, 256), a.view(-1, h2, 128))
            y = _mm(_rms(o, eps, w(p + "norm")).flatten(1) * silu(_mm(x, W[p + "g"])), W[p + "o"])
        else:
            a, b, m = p + "left.", p + "right.", L["mixer"]["left"]
            f, mag = _frequencies(m["rot"])
            v = _mm(x, W[a + "k"]).view(-1, 2, 128)
            q = _turn(_rms(_mm(x, W[a + "q"]).view(-1, H, 128), eps, w(a + "q.norm")), R.pos, f, mag)
            k = _turn(_rms(v, eps, w(a + "k.norm")), R.pos, f, mag)
            y = 0.7 * _mm(R.attend(q, k, v, m["scale"], sink=True).flatten(1), W[a + "o"])
            q, k, v = (silu(_before(R, _mm(x, W[b + t]), W[b + t + ".conv"], 0.0)).view(-1, H, 128) for t in "qkv")
            q, k = (t / torch.sqrt((t * t).sum(-1, keepdim=True) + 1e-6) for t in (q, k))
            dt = softplus(_mm(_mm(x, W[b + "a1"]), W[b + "a2"]) + w(b + "dt_bias"), threshold=1e9).view(-1, H, 128)
            g = torch.exp(-torch.exp(w(b + "A_log"))[:, None] * dt)
            o = _scan(R, _matrix_state(x.new_zeros(n, H, 128, 128)), q * 128 ** -0.5, k, v, g,
                      torch.sigmoid(_mm(x, W[b + "b"])))
            y = y + 0.7 * _mm(_rms(o, eps, w(b + "norm")).flatten(1) * torch.sigmoid(_mm(_mm(x, W[b + "g1"]), W[b + "g2"])),
                              W[b + "o"])
        x = x + _rms(y, eps, w(f"l{i}.norm1"))
        p = f"l{i}.mlp."
        if L["mlp"]["kind"] == "dense":
            y = _by(16384, lambda t: _mm(torch.relu(_mm(t, W[p + "up"])) ** 2, W[p + "down"]), x)
        else:
            z = torch.sigmoid(_mm(x, W[p + "router"]))
            best = z.view(-1, 4, 2).sum(-1).topk(2, -1).indices
            kept = torch.zeros_like(z[:, :4]).scatter_(1, best, 1.0).repeat_interleave(2, 1)
            y = _routed(x, 2.5 * _chosen(z, z * kept, 2), lambda e, t: _glu(t, W[f"{p}e{e}.gate"], W[f"{p}e{e}.up"],
                                                                           W[f"{p}e{e}.down"], silu))
            y = y + _glu(x, W[p + "shared.gate"], W[p + "shared.up"], W[p + "shared.down"], silu)
        x = x + _rms(y, eps, w(f"l{i}.norm2"))
    return _mm(_rms(x[R.asked], eps, w("final.norm")), W["head"])


def _matrix_memory(n, H, D, Dv):
    S = torch.zeros(n, H, D, Dv, dtype=torch.float64, device="cuda")
    nrm, top = S.new_zeros(n, H, D), [S.new_zeros(n, H)]

    def step(q, k, v, ig, fg):
        new = torch.maximum(fg + top[0], ig)
        keep, gain = torch.exp(fg + top[0] - new), torch.exp(ig - new)
        S.mul_(keep[..., None, None]).add_((gain[..., None] * k)[..., :, None] * v[..., None, :])
        nrm.mul_(keep[..., None]).add_(gain[..., None] * k)
        top[0] = new
        den = torch.maximum((nrm * q).sum(-1).abs(), torch.exp(-new)) + 1e-6
        return (q[..., None, :] @ S)[..., 0, :] / den[..., None]

    return step


def _exact_furapel(c, W, R):
    s, eps, d, n = _spec(c), 1e-6, c["width"], len(R.runs)
    H, cap = d // 128, 15.0

    def w(name):
        return W[name].double()

    def norm(t, name):
        return torch.tanh(w(name + ".alpha") * t) * w(name) + w(name + ".b")

    x0 = x = w("embed")[R.tokens] * math.sqrt(d)
    for i, enters in ((0, False), (1, True), (1, True), (2, False), (3, False)):
        L, p, m = s["layers"][i], f"l{i}.mix.", s["layers"][i]["mixer"]
        if enters:
            x = _mm(torch.cat([x, x0], -1), W["loop.in"])
        h = norm(x, f"l{i}.norm1")
        if L["type"] == "attention":
            f, mag = _frequencies(m["rot"])
            q = _turn(_mm(h, W[p + "q"]).view(-1, H, 128), R.pos, f, mag)
            k = _turn(_mm(h, W[p + "k"]).view(-1, H // 4, 128), R.pos, f, mag)
            o = R.attend(q, k, _mm(h, W[p + "v"]).view(-1, H // 4, 128), m["scale"])
            o = o * torch.sigmoid(_mm(h, W[p + "g"]))[:, :, None]
        elif L["type"] == "latent_attention":
            lat = _rms(_mm(h, W[p + "dkv"]), eps, w(p + "dkv.norm"))
            k, v = (_mm(lat, W[p + t]).view(-1, H, 128) for t in ("uk", "uv"))
            o = R.attend(_mm(h, W[p + "q"]).view(-1, H, 128), k, v, m["scale"], window=m["mask"]["size"])
        else:
            H2 = d // 256
            ig, fg = (cap * torch.tanh((_mm(h, W[p + t]) + w(p + t + ".b")) / cap) for t in "if")
            o = _scan(R, _matrix_memory(n, H2, 128, 256), _mm(h, W[p + "q"]).view(-1, H2, 128) * 128 ** -0.5,
                      _mm(h, W[p + "k"]).view(-1, H2, 128), _mm(h, W[p + "v"]).view(-1, H2, 256), ig,
                      torch.nn.functional.logsigmoid(fg))
            o = _rms(o, eps).flatten(1) * w(p + "norm") * torch.sigmoid(_mm(h, W[p + "g"]))
        y = _mm(o.flatten(1), W[p + "o"])
        p, h = f"l{i}.mlp.", norm(x, f"l{i}.norm2")
        z = torch.softmax(_mm(h, W[p + "router"]), -1)
        x = x + y + _routed(h, _chosen(z, z, 4), lambda e, t: _mm(torch.relu(_mm(t, W[f"{p}e{e}.up"])) ** 2,
                                                                 W[f"{p}e{e}.down"]))
    return _mm(norm(x[R.asked], "final.norm"), W["head"]) * 0.25


def exact(case, seed):
    with torch.inference_mode():
        R = _Rows(case, seed)
        f = {"budurax": _exact_budurax, "rogosun": _exact_rogosun, "furapel": _exact_furapel}.get(case["family"], _exact_paged)
        return f(case, _weights(case, seed), R)
