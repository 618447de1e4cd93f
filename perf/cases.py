"""The work that this framework's speed is judged by, through its public entry points.

Each case stands for something a user's program does:
  layer         one call of the packed 1-bit layer (``BitLinearInf``), the drop-in module: a token, a few hundred rows, a prompt batch; float16
                models and, as released checkpoints are stored, float32 ones
  train         one training step's share of a layer (``BitLinear``): forward, then all gradients
  llama_token   one decoded token of a single conversation (``DecodeEngine``)
  llama_batch   one decode step of many conversations (``BatchedDecodeStep``)
  llama_step    one step of continuous batching (``MixedStep``): prompts entering next to decoding requests
  *_prompt      prompts through a hybrid decoder's step engine (Lebepel: sigmoid attention + state space; Serotar: latent attention + experts)
  *_chat        a batch of requests from their prompts through their first tokens, one step per token

Sizes: layer shapes of LLaMA-7B / 13B and of the hybrid configurations of bench.py, with fewer layers (a layer's work repeats), and ragged row
counts.  Decoded tokens are given, not sampled: a near-tie of two logits must not change what the next step computes."""
from __future__ import annotations

import math
import random

import torch

from onebit_amd.bitnet import BitLinearInf
from onebit_amd.engine import BatchedDecodeStep, DecodeEngine, MixedStep
from onebit_amd.lebepel import LebepelConfig, LebepelForCausalLM
from onebit_amd.llama import KVCache, OneBitLlamaConfig, OneBitLlamaForCausalLM
from onebit_amd.serotar import SerotarConfig, SerotarForCausalLM
from onebit_amd.train import BitLinear

DEV = "cuda"
F16, F32, F64, BF16 = torch.float16, torch.float32, torch.float64, torch.bfloat16
VOCAB = 32000

# (in, out) of a 1-bit projection: 7B, 13B, the hybrid widths' feed-forward; the last two are odd ones
SHAPES = [(4096, 4096), (4096, 11008), (11008, 4096), (5120, 13824), (13824, 5120), (2048, 5632), (1024, 2816), (4064, 1000), (1376, 4100)]
# width -> (feed-forward, attention heads, head size, state-space heads, their size, state, groups)
HYBRID = {1024: (2816, 16, 64, 32, 64, 64, 1), 2048: (5632, 16, 128, 64, 64, 128, 1), 4096: (11008, 32, 128, 128, 64, 128, 8)}
# width -> (heads, head size, query rank, latent rank, token input)
LATENT = {1024: (16, 64, 384, 128, 32), 2048: (16, 128, 768, 256, 64), 4096: (32, 128, 1536, 512, 128)}


def listed():
    return [
        # q / o projection of a 7B model for one decoded token: the smallest call, bound by latency
        {"name": "layer_token", "kind": "layer", "dtype": "f16", "rows": 1, "k": 4096, "n": 4096},
        # down projection over a scored continuation or a short prompt, a ragged few hundred rows
        {"name": "layer_rows", "kind": "layer", "dtype": "f16", "rows": 389, "k": 11008, "n": 4096},
        # gate / up projection of a prompt batch, 8 x 2048 tokens
        {"name": "layer_prompt", "kind": "layer", "dtype": "f16", "rows": 16384, "k": 4096, "n": 11008},
        # the same projection of a float32 model (as the released checkpoints are stored) over one prompt
        {"name": "layer_f32", "kind": "layer", "dtype": "f32", "rows": 731, "k": 4096, "n": 11008},
        # distillation training: a layer's forward and backward over 2 x 2048 tokens
        {"name": "train_step", "kind": "train", "dtype": "f16", "rows": 4096, "k": 4096, "n": 11008},
        # one token of one conversation, a few hundred tokens in
        {"name": "llama_token", "kind": "llama_token", "width": 4096, "layers": 8, "context": 397},
        # one token for each of 29 conversations of different lengths
        {"name": "llama_batch", "kind": "llama_batch", "width": 4096, "layers": 8, "rows": 29, "context": 450},
        # four prompts entering next to 20 decoding requests
        {"name": "llama_step", "kind": "llama_step", "width": 4096, "layers": 8, "prompts": 4, "prompt": 500, "rows": 20, "context": 300},
        # long prompts, evaluated as one batch
        {"name": "lebepel_prompt", "kind": "lebepel_prompt", "width": 2048, "layers": 8, "prompts": 4, "prompt": 1900},
        # a batch of requests: prompts, then one step per token
        {"name": "lebepel_chat", "kind": "lebepel_chat", "width": 2048, "layers": 8, "prompts": 12, "prompt": 150, "tokens": 16},
        {"name": "serotar_prompt", "kind": "serotar_prompt", "width": 2048, "layers": 8, "prompts": 4, "prompt": 1900},
        {"name": "serotar_chat", "kind": "serotar_chat", "width": 2048, "layers": 8, "prompts": 12, "prompt": 150, "tokens": 16},
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["layer", "layer", "train", "llama_token", "llama_batch", "llama_step", "lebepel_prompt", "lebepel_chat", "serotar_prompt", "serotar_chat"])
    if kind in ("layer", "train"):
        k, n = rng.choice(SHAPES)
        f32 = rng.random() < 0.3
        most = (16384 * 4096 * 11008 if kind == "layer" else 4096 * 4096 * 11008) // (8 if f32 else 1) // (k * n)
        return {"kind": kind, "dtype": "f32" if f32 else "f16", "rows": _log(rng, 1 if kind == "layer" else 64, min(most, 16384)), "k": k, "n": n}
    if kind.startswith("llama"):
        c = {"kind": kind, "width": rng.choice([2048, 4096]), "layers": rng.choice([2, 4, 8]), "context": _log(rng, 16, 1500)}
        if kind == "llama_batch":
            c["rows"] = rng.randint(2, 48)
        if kind == "llama_step":
            c.update(prompts=rng.randint(1, 8), rows=rng.randint(0, 31))
            c["prompt"] = _log(rng, 20, min(1500, 2000 // c["prompts"]))
            c["context"] = min(c["context"], 500)
        return c
    width = rng.choice([1024, 2048, 2048, 4096])
    c = {"kind": kind, "width": width, "layers": 2 if width == 4096 else rng.choice([4, 8])}
    if kind.endswith("prompt"):
        c["prompts"] = rng.randint(1, 6)
        c["prompt"] = _log(rng, 100, min(2000, 7600 // c["prompts"]))
    else:
        c.update(prompts=rng.randint(1, 20), prompt=_log(rng, 16, 200), tokens=rng.randint(4, 16))
    return c


# ------------------------------------------------------------------------------------------------------------------- inputs --
def _gen(seed):
    return torch.Generator(device=DEV).manual_seed(seed * 7919 + 17)


def _rnd(g, *shape):
    return torch.randn(shape, generator=g, device=DEV)


def _uni(g, lo, hi, *shape):
    return lo + (hi - lo) * torch.rand(shape, generator=g, device=DEV)


def _scale(g, n):
    """A layer's scale vectors: around 0.1, one in ten negative."""
    return _uni(g, 0.05, 0.15, n) * torch.where(torch.rand(n, generator=g, device=DEV) < 0.1, -1.0, 1.0)


def _rows(g, t, k):
    """Activations behind a norm: unit variance, one channel in 512 eight times as large."""
    x = _rnd(g, t, k)
    x[:, ::512] *= 8
    return x


def _packed(g, n, k):
    return torch.randint(0, 256, (n, k // 8), generator=g, device=DEV, dtype=torch.uint8).view(torch.int8)


def _signs(packed):
    """+-1 in 64 bits; 8 signs per byte, lowest bit first, bit 1 = negative."""
    b = packed.view(torch.uint8)
    return 1 - 2 * ((b[:, :, None] >> torch.arange(8, device=b.device, dtype=torch.uint8)) & 1).to(torch.int8).view(b.shape[0], -1).to(F64)


def _layer_inputs(case, seed):
    g, dt = _gen(seed), F16 if case["dtype"] == "f16" else F32
    t, k, n = case["rows"], case["k"], case["n"]
    d = {"x": _rows(g, t, k).to(dt), "g": _scale(g, n).to(dt), "h": _scale(g, k).to(dt)}
    if case["kind"] == "layer":
        d["w"] = _packed(g, n, k)
    else:                                     # latent weights of a pretrained model; the gradient that a scaled loss sends back
        d["w"], d["gy"] = (0.02 * _rnd(g, n, k)).to(dt), (0.01 * _rnd(g, t, n)).to(dt)
    return d


def _llama_config(case):
    w = case["width"]
    return OneBitLlamaConfig(vocab_size=VOCAB, hidden_size=w, intermediate_size=HYBRID[w][0], num_hidden_layers=case["layers"],
                             num_attention_heads=w // 128, max_position_embeddings=2048)


_PROJ = ("self_attn.q_proj", "self_attn.k_proj", "self_attn.v_proj", "self_attn.o_proj", "mlp.gate_proj", "mlp.up_proj", "mlp.down_proj")


def _llama_weights(case, g):
    """A checkpoint in the reference's keys."""
    w, ff = case["width"], HYBRID[case["width"]][0]
    sd = {}
    for i in range(case["layers"]):
        for name in _PROJ:
            k, n = (w, ff) if "gate" in name or "up_" in name else (ff, w) if "down" in name else (w, w)
            p = f"model.layers.{i}.{name}."
            sd[p + "weight"], sd[p + "input_factor"], sd[p + "weight_scale"] = _packed(g, n, k), _scale(g, k).to(F16), _scale(g, n).to(F16)
        for name in ("input_layernorm", "post_attention_layernorm"):
            sd[f"model.layers.{i}.{name}.weight"] = (1 + 0.1 * _rnd(g, w)).to(F16)
    sd["model.embed_tokens.weight"] = _rnd(g, VOCAB, w).to(F16)
    sd["model.norm.weight"] = (1 + 0.1 * _rnd(g, w)).to(F16)
    sd["lm_head.weight"] = (0.02 * _rnd(g, VOCAB, w)).to(F16)
    return sd


def _llama_items(case, seed):
    """[(slot, start, tokens)] of the step, and the cache's length."""
    r, kind = random.Random(seed + 1), case["kind"]
    tok = lambda n: [r.randrange(VOCAB) for _ in range(n)]
    if kind == "llama_token":
        return [(0, case["context"], tok(1))], 512 * (1 + case["context"] // 512)
    length = lambda n: max(1, round(n * r.uniform(0.5, 1)))
    prompts = [length(case["prompt"]) for _ in range(case.get("prompts", 0))]
    items = [(i, 0, tok(n)) for i, n in enumerate(prompts)]
    items += [(len(prompts) + i, length(case["context"]), tok(1)) for i in range(case["rows"])]
    return items, 256 * (1 + max(case["context"], case.get("prompt", 0)) // 256)


def _llama_inputs(case, seed):
    g = _gen(seed)
    sd = _llama_weights(case, g)
    items, max_len = _llama_items(case, seed)
    cfg = _llama_config(case)
    shape = (1 + max(i[0] for i in items), cfg.num_attention_heads, max_len, cfg.head_dim)
    # keys and values of the tokens before: what a layer norm leaves, unit variance
    caches = [tuple(_rnd(g, *shape).to(F16) for _ in range(2)) for _ in range(case["layers"])]
    return sd, items, max_len, cfg, caches


def _hybrid_config(case):
    w = case["width"]
    ff, ah, ad, sh, sd, n, gr = HYBRID[w]
    dense = {"kind": "dense", "ff": ff}
    if case["kind"].startswith("lebepel"):
        ssm = {"type": "mamba2", "mixer": {"heads": sh, "groups": gr, "state": n, "vdim": sd, "conv": 4, "norm_groups": gr}, "mlp": dense}
        att = {"type": "attention", "mixer": {"heads": ah, "kv_heads": ah, "dim": ad, "vdim": ad, "scale": ad ** -0.5}, "mlp": dense}
        return LebepelConfig(vocab_size=VOCAB, width=w, layers=[ssm, att] * (case["layers"] // 2), norm_eps=1e-5, residual_mult=0.5, logit_softcap=30.0,
                             max_positions=4096)
    h, d, qr, kr, side = LATENT[w]
    mix = {"heads": h, "dim": d, "vdim": d, "q_rank": qr, "kv_rank": kr, "scale": d ** -0.5}
    moe = {"kind": "moe", "expert": {"ff": ff // 8}, "shared": {"ff": ff // 4}, "router": {"experts": 32, "identity": 8, "top": 6, "groups": {"count": 8, "keep": 4}}}
    return SerotarConfig(vocab_size=VOCAB, width=w, norm_eps=1e-5, embed_scale=1.0, bigram={"buckets": 4 * VOCAB - 1, "mul_prev": 53, "mul_cur": 11}, side_dim=side,
                         layers=[{"type": "latent_attention", "mixer": mix, "mlp": moe if i else dense} for i in range(case["layers"])])


def _hybrid_weights(case, g):
    """bfloat16 tensors of every name of the checkpoint: products N(0, 1 / fan-in), the others in the ranges that training leaves them in."""
    out = {}
    for name, shape in _hybrid_config(case).tensor_shapes().items():
        leaf = name.rsplit(".", 1)[-1]
        if name in ("embed", "bigram", "side.embed"):
            t = _rnd(g, *shape)
        elif name == "pos":
            t = 0.3 * _rnd(g, *shape)
        elif leaf == "dwa":
            t = 0.2 * _rnd(g, *shape)
            t[-1] += 1
        elif case["kind"].startswith("lebepel") and leaf in ("norm1", "norm") and "mix" not in name:
            t = 0.1 * _rnd(g, *shape)
        elif leaf in ("norm", "norm1", "norm2", "ls1", "ls2"):
            t = 1 + 0.1 * _rnd(g, *shape)
        elif leaf in ("r1", "r2", "pb", "A_log", "dt_bias"):
            lo, hi = {"r1": (0.3, 1.0), "r2": (0.05, 0.5), "pb": (-4.0, -2.0), "A_log": (0.0, 1.5), "dt_bias": (-4.0, -1.0)}[leaf]
            t = _uni(g, lo, hi, *shape)
        elif leaf == "D":
            t = 1 + 0.2 * _rnd(g, *shape)
        elif leaf == "act":
            t = 0.5 * _rnd(g, *shape)
        elif leaf == "correction":
            t = 0.1 * _rnd(g, *shape) / shape[0] ** 0.5
        elif len(shape) == 2:
            t = _rnd(g, *shape) / shape[1] ** 0.5
        else:
            t = 0.1 * _rnd(g, *shape)
        out[name] = t.to(BF16)
    return out


def _hybrid_tokens(case, seed):
    """Token lists of the prompts, and the given tokens of every request."""
    r = random.Random(seed + 1)
    lens = [max(2, round(case["prompt"] * r.uniform(0.6, 1))) for _ in range(case["prompts"])]
    tok = lambda n: [r.randrange(VOCAB) for _ in range(n)]
    return [tok(n) for n in lens], [tok(case.get("tokens", 0)) for _ in lens]


def _scored(n):
    """Rows of a prompt whose logits are asked for: the continuation that is scored, or the last one."""
    return min(n, 64)


def prepare(case, seed):
    kind = case["kind"]
    if kind == "layer":
        d = _layer_inputs(case, seed)
        m = BitLinearInf(case["k"], case["n"], device=DEV, dtype=d["x"].dtype)
        m.weight.data, m.input_factor.data, m.weight_scale.data = d["w"], d["h"], d["g"]
        return {"run": _run_layer, "module": m, "x": d["x"]}
    if kind == "train":
        d = _layer_inputs(case, seed)
        m = BitLinear(case["k"], case["n"], device=DEV, dtype=d["x"].dtype)
        m.weight.data, m.input_factor.data, m.weight_scale.data = d["w"], d["h"], d["g"]
        return {"run": _run_train, "module": m, "x": d["x"].requires_grad_(True), "gy": d["gy"]}
    if kind.startswith("llama"):
        sd, items, max_len, cfg, caches = _llama_inputs(case, seed)
        with torch.device("meta"):
            model = OneBitLlamaForCausalLM(cfg, F16)
        model = model.to_empty(device=DEV)
        model.load_state_dict(sd, assign=True)
        for p in model.parameters():
            p.requires_grad_(False)
        if kind == "llama_token":
            eng = DecodeEngine(model, max_len=max_len)
            for mine, given in zip(eng.cache.layers, caches):
                for a, b in zip(mine, given):
                    a.copy_(b)
            return {"run": _run_llama_token, "engine": eng, "item": items[0], "caches": eng.cache.layers}
        if kind == "llama_batch":
            splits = -(-max_len // 256) if max_len > 256 else 0
            eng = BatchedDecodeStep(model, caches, len(items), max_len, keep_logits=True, attn_splits=splits, attn_chunk=256)
            eng.tokens.copy_(torch.tensor([i[2][0] for i in items], dtype=torch.int32))
            eng.pos.copy_(torch.tensor([i[1] for i in items], dtype=torch.int32))
            return {"run": _run_llama_batch, "engine": eng, "caches": caches}
        eng = MixedStep(model, caches, len(caches[0][0]), max_len, max_rows=sum(len(i[2]) for i in items), keep_logits=True)
        return {"run": _run_llama_step, "engine": eng, "items": items, "caches": caches}
    cfg, w = _hybrid_config(case), _hybrid_weights(case, _gen(seed))
    model = (LebepelForCausalLM if kind.startswith("lebepel") else SerotarForCausalLM)(cfg, w, BF16, DEV)
    prompts, more = _hybrid_tokens(case, seed)
    eng = model.step_engine(len(prompts), max(map(len, prompts)) + len(more[0]), max_rows=sum(map(len, prompts)))
    if kind.endswith("prompt"):
        return {"run": _run_prompt, "engine": eng, "items": [(i, 0, p, _scored(len(p))) for i, p in enumerate(prompts)]}
    steps = [[(i, len(p) + t, more[i][t:t + 1]) for i, p in enumerate(prompts)] for t in range(len(more[0]))]
    state = {"run": _run_chat, "engine": eng, "items": [(i, 0, p) for i, p in enumerate(prompts)], "steps": steps}
    _run_chat(state)                          # a server's engine has served before
    return state


# --------------------------------------------------------------------------------------------------------------------- runs --
def run(state):
    return state["run"](state)


def _run_layer(s):
    with torch.no_grad():
        return s["module"](s["x"])


def _run_train(s):
    m, x = s["module"], s["x"]
    y = m(x)
    gx, gw, gg, gh = torch.autograd.grad(y, [x, m.weight, m.weight_scale, m.input_factor], s["gy"])
    return {"y": y.detach(), "x": gx, "weight": gw, "weight_scale": gg, "input_factor": gh}


def _out(s, logits):
    return {"logits": logits, "caches": [list(c) for c in s["caches"]]}


def _run_llama_token(s):
    eng, (_, start, tokens) = s["engine"], s["item"]
    eng.set_state(tokens[0], start)
    eng.step()
    return _out(s, eng.logits())


def _run_llama_batch(s):
    s["engine"].launch()
    return _out(s, s["engine"].logits)


def _run_llama_step(s):
    n = len(s["items"])
    s["engine"].launch(s["items"])
    return _out(s, s["engine"].logits[:n])


def _run_prompt(s):
    n = sum(i[3] for i in s["items"])
    s["engine"].launch(s["items"])
    return s["engine"].logits[:n]


def _run_chat(s):
    eng, n = s["engine"], len(s["items"])
    eng.launch(s["items"])
    out = [eng.logits[:n].clone()]
    for step in s["steps"]:
        eng.launch(step)
        out.append(eng.logits[:n].clone())
    return torch.stack(out)


# --------------------------------------------------------------------------------------------------------------------- work --
def work(case):
    kind = case["kind"]
    if kind in ("layer", "train"):
        t, k, n = case["rows"], case["k"], case["n"]
        e = 2 if case["dtype"] == "f16" else 4
        if kind == "layer":
            return {"bytes": n * k // 8 + e * (t * k + t * n + k + n), "flops": 2 * t * k * n}
        return {"bytes": e * (2 * t * k + 2 * t * n + 2 * n * k + 2 * (k + n)), "flops": 6 * t * k * n}
    w, layers, ff = case["width"], case["layers"], HYBRID[case["width"]][0]
    if kind.startswith("llama"):
        items = _llama_items(case, 0)[0]
        rows, outs, par = sum(len(i[2]) for i in items), len(items), layers * (4 * w * w + 3 * w * ff)
        pairs = sum(sum(range(i[1] + 1, i[1] + len(i[2]) + 1)) for i in items)                     # (query, key) pairs of a head
        kv = sum(i[1] + 2 * len(i[2]) for i in items) * 2 * w * 2 * layers
        return {"bytes": par // 8 + 2 * VOCAB * w + kv + 2 * w * rows + 2 * VOCAB * outs, "flops": 2 * rows * par + 4 * pairs * w * layers + 2 * outs * w * VOCAB}
    prompts, more = _hybrid_tokens(case, 0)
    cfg, leb, total = _hybrid_config(case), kind.startswith("lebepel"), {"bytes": 0, "flops": 0}
    r = None if leb else cfg.layers[-1]["mlp"]["router"]
    shapes = [(k, s) for k, s in cfg.tensor_shapes().items() if k[0] == "l" and k[1].isdigit() and len(s) == 2 and "conv" not in k]

    def step(rows, pairs, cached, outs):
        flops, read = 2 * outs * w * VOCAB, 2 * VOCAB * w + 4 * VOCAB * outs + 2 * w * rows
        for k, s in shapes:
            routed = ".mlp.e" in k
            flops += 2 * rows * s[0] * s[1] * (r["top"] / (r["experts"] + r["identity"]) if routed else 1)
            read += 2 * s[0] * s[1] * ((1 - (1 - r["top"] / (r["experts"] + r["identity"])) ** rows) if routed else 1)
        for lay in cfg.layers:
            m = lay["mixer"]
            if lay["type"] == "mamba2":
                flops += 6 * rows * m["heads"] * m["state"] * m["vdim"]
                read += 8 * len(prompts) * m["heads"] * m["state"] * m["vdim"]
            else:
                flops += 2 * pairs * m["heads"] * (m["dim"] + m["vdim"])
                read += 2 * cached * (m["heads"] * (m["dim"] + m["vdim"]) if leb else m["kv_rank"])
        total["bytes"] += read
        total["flops"] += flops
    lens = [len(p) for p in prompts]
    step(sum(lens), sum(n * (n + 1) // 2 for n in lens), sum(lens), sum(_scored(n) if kind.endswith("prompt") else 1 for n in lens))
    for t in range(len(more[0])):
        ctx = sum(lens) + (t + 1) * len(lens)
        step(len(lens), ctx, ctx, len(lens))
    return {k: int(v) for k, v in total.items()}


def tolerance(case):
    """About four times what the outputs are off from the same sums in 64 bits: float16 layers 4e-4, float32 ones 2e-7 (gradients sum over more
    rows), the 1-bit LLaMA up to 3e-3 at its logits, Lebepel 5e-3, Serotar 5e-3 to 1.2e-2 (a near-tie between two experts may fall either way)."""
    kind = case["kind"]
    if kind in ("layer", "train"):
        return {"rel": 1e-5, "max": 1e-3} if case["dtype"] == "f32" else {"rel": 2e-3, "max": 0.05}
    if kind.startswith("llama"):
        return {"rel": 1e-2, "max": 0.2}
    return {"rel": 2e-2, "max": 0.2} if kind.startswith("lebepel") else {"rel": 3e-2, "max": 0.99}


# ----------------------------------------------------------------------------------------------------- the same in 64 bits --
def exact(case, seed):
    kind = case["kind"]
    with torch.no_grad():
        if kind == "layer":
            d = _layer_inputs(case, seed)
            return _layer_norm(_one_bit(d["x"].to(F64), d["w"], d["h"], d["g"]))
        if kind == "train":
            return _exact_train(_layer_inputs(case, seed))
        if kind.startswith("llama"):
            return _exact_llama(case, seed)
        logits, lens = _exact_hybrid(case, seed)
        if kind.endswith("prompt"):
            return torch.cat([logits[i, n - _scored(n):n] for i, n in enumerate(lens)])
        return torch.stack([torch.stack([logits[i, n - 1 + t] for i, n in enumerate(lens)]) for t in range(case["tokens"] + 1)])


def _one_bit(x, w, h, g):
    return ((x * h.to(F64)) @ _signs(w).T) * g.to(F64)


def _layer_norm(u, eps=1e-5):
    u = u - u.mean(-1, keepdim=True)
    return u / torch.sqrt((u * u).mean(-1, keepdim=True) + eps)


def _rms(x, eps):
    return x / torch.sqrt((x * x).mean(-1, keepdim=True) + eps)


def _silu(z):
    return z * torch.sigmoid(z)


def _exact_train(d):
    x, w, h, g, gy = (d[k].to(F64) for k in ("x", "w", "h", "g", "gy"))
    s = torch.sign(w)
    a = x * h
    z = a @ s.T
    u = z * g
    c = u - u.mean(-1, keepdim=True)
    r = 1 / torch.sqrt((c * c).mean(-1, keepdim=True) + 1e-5)
    y = c * r
    gu = r * (gy - gy.mean(-1, keepdim=True) - y * (gy * y).mean(-1, keepdim=True))
    gz = gu * g
    ga = gz @ s
    return {"y": y, "x": ga * h, "weight": (gz.T @ a) * (1.001 - torch.tanh(w) ** 2), "weight_scale": (gu * z).sum(0), "input_factor": (ga * x).sum(0)}


def _exact_llama(case, seed):
    sd, items, _, cfg, caches = _llama_inputs(case, seed)
    H, D = cfg.num_attention_heads, cfg.head_dim
    pos = torch.cat([torch.arange(i[1], i[1] + len(i[2])) for i in items]).to(DEV)
    freq = 10000.0 ** (-torch.arange(0, D, 2, device=DEV, dtype=F64) / D)
    angle = (pos.to(F64)[:, None] * freq).repeat(1, 2)
    cos, sin = angle.cos()[:, None], angle.sin()[:, None]
    turn = lambda t: t * cos + torch.cat([-t[..., D // 2:], t[..., :D // 2]], -1) * sin
    x = sd["model.embed_tokens.weight"][torch.tensor([t for i in items for t in i[2]], device=DEV)].to(F64)
    rows = x.shape[0]
    after = []
    for i in range(case["layers"]):
        pre = f"model.layers.{i}."
        proj = lambda v, name: _layer_norm(_one_bit(v, *(sd[f"{pre}{name}.{q}"] for q in ("weight", "input_factor", "weight_scale"))))
        norm = lambda v, name: _rms(v, cfg.rms_norm_eps) * sd[pre + name + ".weight"].to(F64)
        v = norm(x, "input_layernorm")
        q, k, val = (proj(v, f"self_attn.{n}_proj").view(rows, H, D) for n in "qkv")
        q, k = turn(q), turn(k)
        kc, vc = (c.to(F64) for c in caches[i])
        out, row = torch.empty_like(q), 0
        for slot, start, tokens in items:
            n = len(tokens)
            end, mine = start + n, slice(row, row + n)
            kc[slot, :, start:end], vc[slot, :, start:end] = k[mine].transpose(0, 1), val[mine].transpose(0, 1)
            s = q[mine].transpose(0, 1) @ kc[slot, :, :end].transpose(1, 2) / D ** 0.5
            s = s.masked_fill(torch.ones(n, end, dtype=torch.bool, device=DEV).triu(start + 1), -math.inf)
            out[mine] = (s.softmax(-1) @ vc[slot, :, :end]).transpose(0, 1)
            row += n
        x = x + proj(out.reshape(rows, -1), "self_attn.o_proj")
        v = norm(x, "post_attention_layernorm")
        x = x + proj(_silu(proj(v, "mlp.gate_proj")) * proj(v, "mlp.up_proj"), "mlp.down_proj")
        after.append([kc, vc])
    last = torch.tensor([len(i[2]) for i in items], device=DEV).cumsum(0) - 1
    x = _rms(x[last], cfg.rms_norm_eps) * sd["model.norm.weight"].to(F64)
    logits = x @ sd["lm_head.weight"].to(F64).T
    return {"logits": logits[0] if case["kind"] == "llama_token" else logits, "caches": after}


def _exact_hybrid(case, seed):
    """Logits [requests, positions, vocabulary] of whole sequences, shorter ones padded behind their end (every position looks back only)."""
    cfg, w = _hybrid_config(case), _hybrid_weights(case, _gen(seed))
    w = {k: v.to(F64) if v.numel() < 1 << 24 else v for k, v in w.items()}
    prompts, more = _hybrid_tokens(case, seed)
    S = max(len(p) + len(m) for p, m in zip(prompts, more))
    tokens = torch.tensor([(p + m + [0] * S)[:S] for p, m in zip(prompts, more)], device=DEV)
    x = (_exact_lebepel if case["kind"].startswith("lebepel") else _exact_serotar)(cfg, w, tokens)
    # (only rows that are compared go through the head)
    first = min(len(p) - _scored(len(p)) for p in prompts) if case["kind"].endswith("prompt") else min(len(p) - 1 for p in prompts)
    logits = x.new_zeros(x.shape[0], S, VOCAB)
    logits[:, first:] = x[:, first:] @ w["head"].to(F64).T
    if case["kind"].startswith("lebepel"):
        logits = cfg.logit_softcap * torch.tanh(logits / cfg.logit_softcap)
    return logits, [len(p) for p in prompts]


def _exact_lebepel(cfg, w, tokens):
    B, S = tokens.shape
    eps = cfg.norm_eps
    x = w["embed"][tokens].to(F64) + w["pos"][:S].to(F64)
    t = torch.arange(S, device=DEV)
    dist, later = (t[:, None] - t[None]).clamp(min=0).to(F64), t[None] > t[:, None]
    for i, lay in enumerate(cfg.layers):
        p, m = f"l{i}.", lay["mixer"]
        W = lambda n: w[p + n].to(F64)
        h, H = _rms(x, eps) * (1 + W("norm1")), m["heads"]
        if lay["type"] == "attention":
            q, k, v = (h @ W(f"mix.{n}").T + W(f"mix.{n}.b") for n in "qkv")
            q, k = _rms(q.view(B, S, H, -1), eps), _rms(k.view(B, S, H, -1), eps)
            v = v.view(B, S, H, -1)
            o = torch.empty_like(v)
            for j in range(H):
                s = q[:, :, j] @ k[:, :, j].transpose(1, 2) * m["scale"] - W("mix.r1")[j] * torch.log1p(W("mix.r2")[j] * dist) + W("mix.pb")[j]
                o[:, :, j] = torch.sigmoid(s).masked_fill(later, 0.0) @ v[:, :, j]
            s = o.reshape(B, S, -1) @ W("mix.o").T + W("mix.o.b")
        else:
            P, N, G = m["vdim"], m["state"], m["groups"]
            z, u, dt = (h @ W("mix.in").T).split([H * P, H * P + 2 * G * N, H], dim=-1)
            taps, c = W("mix.conv"), W("mix.conv.b").expand_as(u).clone()
            for b in range(m["conv"]):
                c[:, b:] += taps[:, m["conv"] - 1 - b] * u[:, :S - b]
            xs, Bm, Cm = _silu(c).split([H * P, G * N, G * N], dim=-1)
            xs, Bm, Cm = xs.view(B, S, H, P), Bm.view(B, S, G, N).repeat_interleave(H // G, 2), Cm.view(B, S, G, N).repeat_interleave(H // G, 2)
            dt = torch.nn.functional.softplus(dt + W("mix.dt_bias"))
            decay = torch.exp(-torch.exp(W("mix.A_log")) * dt)
            y, state = torch.empty_like(xs), x.new_zeros(B, H, N, P)
            for n in range(S):
                state = decay[:, n, :, None, None] * state + (dt[:, n, :, None] * Bm[:, n])[..., None] * xs[:, n, :, None]
                y[:, n] = (Cm[:, n, :, None] @ state)[:, :, 0] + W("mix.D")[:, None] * xs[:, n]
            v = y.reshape(B, S, -1) * _silu(z)
            s = (_rms(v.view(B, S, m["norm_groups"], -1), eps).reshape(B, S, -1) * W("mix.norm")) @ W("mix.o").T
        x = x + cfg.residual_mult * (s + (_silu(h @ W("mlp.gate").T) * (h @ W("mlp.up").T)) @ W("mlp.down").T)
    return _rms(x, eps) * (1 + w["final.norm"].to(F64))


def _exact_serotar(cfg, w, tokens):
    B, S = tokens.shape
    eps, bg = cfg.norm_eps, cfg.bigram
    row = torch.full_like(tokens, bg["buckets"])
    row[:, 1:] = (tokens[:, :-1] * bg["mul_prev"] + tokens[:, 1:] * bg["mul_cur"]) % bg["buckets"]
    x = (w["embed"][tokens].to(F64) * cfg.embed_scale + w["bigram"][row].to(F64)).view(B * S, -1)
    later = torch.ones(S, S, dtype=torch.bool, device=DEV).triu(1)
    seen = [x]
    for i, lay in enumerate(cfg.layers):
        p, m, mlp = f"l{i}.", lay["mixer"], lay["mlp"]
        W = lambda n: w[p + n].to(F64)
        q = (_rms(x @ W("mix.dq").T, eps) * W("mix.dq.norm")) @ W("mix.uq").T
        c = _rms(x @ W("mix.dkv").T, eps) * W("mix.dkv.norm")
        q, k, v = (t.view(B, S, m["heads"], -1) for t in (q, c @ W("mix.uk").T, c @ W("mix.uv").T))
        o = torch.empty_like(v)
        for j in range(m["heads"]):
            o[:, :, j] = (q[:, :, j] @ k[:, :, j].transpose(1, 2) * m["scale"]).masked_fill(later, -math.inf).softmax(-1) @ v[:, :, j]
        x = x + _rms(o.reshape(B * S, -1) @ W("mix.o").T, eps) * (W("norm1") * W("ls1"))
        if mlp["kind"] == "dense":
            z, (a, b) = x @ W("mlp.up").T, torch.nn.functional.softplus(W("mlp.act"))
            f = torch.where(z > 0, a * z * z, (0.5 + b) * (torch.expm1(z.clamp(max=0)) - z)) + 0.5 * z
            f = f @ W("mlp.down").T
        else:
            r = mlp["router"]
            gated = lambda v, e: (_silu(v @ W(e + "gate").T) * (v @ W(e + "up").T)) @ W(e + "down").T
            s = (x @ W("mlp.router").T).softmax(-1)
            choice = s + W("mlp.correction")
            groups = choice.view(B * S, r["groups"]["count"], -1)
            best = groups.amax(-1).topk(r["groups"]["keep"], dim=1).indices
            hidden = torch.ones(groups.shape[:2], dtype=torch.bool, device=DEV).scatter_(1, best, False)
            top = groups.masked_fill(hidden[..., None], -math.inf).view(B * S, -1).topk(r["top"], dim=1).indices
            weight = torch.zeros_like(s).scatter_(1, top, s.gather(1, top))
            f = gated(x, "mlp.shared.") + weight[:, r["experts"]:].sum(1, keepdim=True) * x
            for e in range(r["experts"]):
                at = weight[:, e].nonzero()[:, 0]
                f[at] += weight[at, e, None] * gated(x[at], f"mlp.e{e}.")
        x = x + _rms(f, eps) * (W("norm2") * W("ls2"))
        e = w["side.embed"][tokens.view(-1), i * cfg.side_dim:(i + 1) * cfg.side_dim].to(F64)
        z = torch.nn.functional.gelu(x @ W("side.gate").T, approximate="tanh")
        x = x + _rms((z * e) @ W("side.proj").T, eps) * W("side.norm")
        seen.append(x)
        x = sum(a * v for a, v in zip(W("dwa"), seen))
    return (_rms(x, eps) * w["final.norm"].to(F64)).view(B, S, -1)
