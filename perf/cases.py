"""Steps of the serving engine, timed as the engine runs them: packed prompts (``LLMEngine.feed``) and
decode steps of running sequences (``DecodeRunner.launch`` with one step in flight).

Models are layer stacks at the two widths of ``bench.py --design`` (2048 with 16 heads on 4, 4096 with
32 on 8; four layers; vocabulary 32,000), bf16, random weights:

  llama     grouped-query attention and a gated feed-forward
  mixtral   the same attention, 16 experts a quarter as wide, 4 per token
  ralesun   latent attention with window, sink and feed-forward, bare gated delta-rule layers
  garesun   matrix memory, latent attention, retention, attention over the same latents, each beside
            20 squared-relu experts (4 per token) and a shared one, with token inputs

A case: family, width, phase ("prefill" or "decode"), sequences n, tokens: the mean length of the
prompts, or of the contexts that are decoded.  Lengths are ragged, from three quarters to five
quarters of the mean.  Outputs are the logits of each sequence's last token, as the model gives them.
"""
from __future__ import annotations

import dataclasses
import math

import numpy as np
import torch

from drtc_amd.engine import LLMEngine, Request
from drtc_amd.models import build_model
from drtc_amd.models.config import (ChannelDelta, Experts, HybridConfig, LatentAttention, Layer, MatrixMemory,
                                    ModelConfig, Retention, retention_decays)

FAMILIES = ("llama", "mixtral", "ralesun", "garesun")
SIZES = {2048: (16, 4, 7168), 4096: (32, 8, 14336)}  # width -> heads, kv heads, feed-forward
VOCAB, DIM, EPS, BLOCK = 32000, 128, 1e-5, 32
ROUTER = 4.0  # trained routers decide more clearly than random ones: their logits this much wider
EMBED = 200.0  # and tokens stand out of the residual stream: embeddings four times a unit row, in all designs
MOST_PROMPT = 16384  # tokens of a packed step


def listed():
    def case(name, family, width, phase, n, tokens):
        return {"name": name, "family": family, "width": width, "phase": phase, "n": n, "tokens": tokens}

    return [
        # one chat request alone on the service: its prompt, then its tokens one after the other
        case("llama prompt of one", "llama", 4096, "prefill", 1, 148),
        case("llama decode of one", "llama", 2048, "decode", 1, 160),
        # a few users with a long channel history behind them
        case("llama decode 16 x 1000", "llama", 4096, "decode", 16, 1000),
        # the smart replies of a full batch: the workload of bench.py
        case("llama decode 1024 x 150", "llama", 4096, "decode", 1024, 150),
        # long documents to summarise
        case("llama prompts 4 x 4000", "llama", 2048, "prefill", 4, 4000),
        # suggestions from a mixture of experts: few users, many users, a chunk of their prompts
        case("mixtral decode 13 x 700", "mixtral", 4096, "decode", 13, 700),
        case("mixtral decode 224 x 300", "mixtral", 2048, "decode", 224, 300),
        case("mixtral prompts 64 x 190", "mixtral", 4096, "prefill", 64, 190),
        # the designs with recurrent layers: long prompts, long generations, many users
        case("ralesun prompts 4 x 3500", "ralesun", 2048, "prefill", 4, 3500),
        case("ralesun decode 64 x 1500", "ralesun", 4096, "decode", 64, 1500),
        case("garesun prompts 15 x 1000", "garesun", 4096, "prefill", 15, 1000),
        case("garesun decode 200 x 500", "garesun", 2048, "decode", 200, 500),
    ]


def draw(rng):
    def size(lo, hi):  # spread over the logarithm
        return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))

    family, width, phase = rng.choice(FAMILIES), rng.choice(sorted(SIZES)), rng.choice(("prefill", "decode"))
    if phase == "prefill":
        tokens = size(24, 4000)
        n = size(1, max(1, min(64, 15000 // tokens)))
    else:
        tokens = size(24, 4000)
        n = size(1, max(1, min(1024 if family in ("llama", "mixtral") else 256, 150_000 // tokens)))
    return {"family": family, "width": width, "phase": phase, "n": n, "tokens": tokens}


def _lengths(case):
    """Longest first, as the engine orders large batches."""
    golden = (math.sqrt(5) - 1) / 2
    return sorted((max(1, int(case["tokens"] * (0.75 + 0.5 * ((i + 1) * golden % 1)))) for i in range(case["n"])),
                  reverse=True)


def _config(case):
    family, W = case["family"], case["width"]
    H, G, ff = SIZES[W]
    name = f"{family}-{W}"
    if family == "llama":
        return ModelConfig(name, VOCAB, W, ff, 4, H, G, DIM)
    if family == "mixtral":
        return ModelConfig(name, VOCAB, W, ff // 4, 4, H, G, DIM, num_experts=16, experts_per_token=4)
    if family == "ralesun":
        att = LatentAttention(H, DIM, 64, DIM, 512, 192 ** -0.5, 1024, 500000.0, 64)
        return HybridConfig(name, VOCAB, W, (Layer(att, ff), Layer(ChannelDelta(H, H, DIM, DIM, 4, 128, 128))) * 2,
                            norm_eps=EPS)
    att = LatentAttention(H, DIM, 64, DIM, 512, 192 ** -0.5, None, 500000.0, 64, False, True)
    mixers = (MatrixMemory(H, DIM, DIM, 15.0), att, Retention(H, DIM, DIM, retention_decays(H), 500000.0, DIM),
              dataclasses.replace(att, kv_from=1))
    return HybridConfig(name, VOCAB, W,
                        tuple(Layer(m, ff // 4, experts=Experts(20, 4), shared=ff // 2) for m in mixers),
                        norm_eps=EPS, act="relu2", block="joint", norm="layer", embed_scale=4.0, side_dim=W // 16)


class _Tensors:
    """Checkpoint tensors by name, made in the order in which they are asked for."""

    def __init__(self, seed):
        self.gen = torch.Generator(device="cuda").manual_seed(seed)
        self.made = {}

    def add(self, name, *shape, std=0.02, mean=0.0):
        t = torch.empty(*shape, dtype=torch.bfloat16, device="cuda")
        self.made[name] = t.normal_(mean, std, generator=self.gen)

    def uniform(self, name, *shape, lo, hi):
        t = torch.empty(*shape, dtype=torch.bfloat16, device="cuda")
        self.made[name] = t.uniform_(lo, hi, generator=self.gen)


def _checkpoint(cfg, seed):
    """A ralesun or garesun checkpoint."""
    W, T = cfg.hidden_size, _Tensors(seed)
    add, joint = T.add, cfg.block == "joint"
    add("embed", cfg.vocab_size, W, std=1.0 if joint else 0.02 * EMBED)
    if joint:
        add("side.embed", cfg.vocab_size, cfg.num_layers * cfg.side_dim, std=1.0)

    def norm(name):
        add(name, W, std=0.1, mean=1.0)
        if not joint:
            add(name + ".b", W, std=0.05)
            T.made[name + ".alpha"] = torch.tensor(0.8)

    for i, l in enumerate(cfg.layers):
        m, p, q = l.mixer, f"l{i}.mix.", f"l{i}.mlp."
        norm(f"l{i}.norm1")
        H, vd = m.heads, m.heads * m.vdim
        if isinstance(m, LatentAttention):
            add(p + "q", H * (m.dim + m.rot_dim), W)
            if m.kv_from is None:
                add(p + "dkv", m.kv_rank + m.rot_dim, W)
                add(p + "dkv.norm", m.kv_rank, std=0.1, mean=1.0)
            add(p + "uk", H * m.dim, m.kv_rank, std=m.kv_rank ** -0.5)
            add(p + "uv", vd, m.kv_rank, std=m.kv_rank ** -0.5)
            if m.sink:
                add(p + "sink", H, std=1.0)
            if m.gate:
                add(p + "g", H, W)
        elif isinstance(m, ChannelDelta):
            kd = m.kv_heads * m.dim
            for x, n in (("q", kd), ("k", kd), ("v", vd)):
                add(p + x, n, W)
                add(f"{p}{x}.conv", n, m.conv, std=m.conv ** -0.5)
            add(p + "b", H, W)
            add(p + "a1", m.decay_rank, W)
            add(p + "a2", H * m.dim, m.decay_rank, std=m.decay_rank ** -0.5)
            add(p + "g1", m.gate_rank, W)
            add(p + "g2", vd, m.gate_rank, std=m.gate_rank ** -0.5)
            T.uniform(p + "A_log", H, lo=-1.0, hi=1.0)
            T.uniform(p + "dt_bias", H * m.dim, lo=-5.0, hi=1.0)
            add(p + "norm", m.vdim, std=0.1, mean=1.0)
        else:
            for x, n in (("q", H * m.dim), ("k", H * m.dim), ("v", vd), ("g", vd)):
                add(p + x, n, W)
            if isinstance(m, MatrixMemory):
                for x, mean in (("i", 0.0), ("f", 5.0)):
                    add(p + x, H, W)
                    add(f"{p}{x}.b", H, std=1.0, mean=mean)
                add(p + "norm", vd, std=0.1, mean=1.0)
        add(p + "o", W, vd)
        if joint:
            add(q + "router", l.experts.count, W, std=0.02 * ROUTER)
            for e in range(l.experts.count):
                add(f"{q}e{e}.up", l.ff, W)
                add(f"{q}e{e}.down", W, l.ff)
            add(q + "shared.up", l.shared, W)
            add(q + "shared.down", W, l.shared)
            add(f"l{i}.side.gate", cfg.side_dim, W)
            add(f"l{i}.side.proj", W, cfg.side_dim)
            add(f"l{i}.side.norm", W, std=0.1, mean=1.0)
        elif l.ff:
            norm(f"l{i}.norm2")
            add(q + "gate", l.ff, W)
            add(q + "up", l.ff, W)
            add(q + "down", W, l.ff)
    norm("final.norm")
    add("head", cfg.vocab_size, W)
    return T.made


def _model(case, seed):
    cfg = _config(case)
    if isinstance(cfg, HybridConfig):
        return build_model(cfg, "cuda", tensors=_checkpoint(cfg, seed))
    model = build_model(cfg, "cuda", seed=seed, full_then_shard=False)
    model.embed.mul_(EMBED)
    for L in model.layers if cfg.is_moe else ():
        L["router"].mul_(ROUTER)
    return model


def _tokens(case, seed):
    """Prompts, and the token that each sequence decodes behind its context."""
    rng = np.random.default_rng([7, seed])
    return [rng.integers(3, VOCAB, n).tolist() for n in _lengths(case)], rng.integers(3, VOCAB, case["n"]).astype(np.int32)


def prepare(case, seed):
    model, (prompts, tokens), n = _model(case, seed), _tokens(case, seed), case["n"]
    slots = 1024 if n > 256 else 256 if n > 64 else 64
    blocks = sum(len(p) // BLOCK + 2 for p in prompts)
    eng = LLMEngine(model, max_batch=slots, max_model_len=max(512, len(prompts[0]) + 64), num_blocks=blocks + 2)
    if case["phase"] == "prefill":
        return {"engine": eng, "prompts": prompts}
    reqs, at = [Request([]) for _ in range(n)], 0
    while at < n:  # the contexts, in packed steps
        end, total = at, 0
        while end < n and (end == at or total + len(prompts[end]) <= MOST_PROMPT):
            total += len(prompts[end])
            end += 1
        eng.feed([(r, p, []) for r, p in zip(reqs[at:end], prompts[at:end])])
        at = end
    eng.runner.read_logits(n)
    pos = eng.ctx[:n].copy()
    for r in reqs:  # room for the decoded token
        if eng.ctx[r.slot] // BLOCK >= len(r.blocks):
            r.blocks += eng.alloc.allocate(1)
            eng.bt[r.slot, :len(r.blocks)] = r.blocks
    slots = eng.bt[np.arange(n), pos // BLOCK].astype(np.int64) * BLOCK + pos % BLOCK
    step = (n, tokens, pos, pos + 1, slots, eng.bt[:n].copy(), np.full(n, 1.0, np.float32), np.full(n, 64, np.int32),
            np.full(n, 0.95, np.float32), eng.sstate[:n].copy())
    return {"engine": eng, "requests": reqs, "step": step, "flying": None}


def run(state):
    eng = state["engine"]
    if "prompts" in state:
        reqs = [Request([]) for _ in state["prompts"]]
        rows = eng.feed([(r, p, [len(p) - 1]) for r, p in zip(reqs, state["prompts"])])
        for r in reqs:
            eng.release(r)
        return torch.cat(rows)
    # one step in flight: a step is read when the next one has been enqueued
    handle = eng.runner.launch(*state["step"])
    if state["flying"] is not None:
        eng.runner.wait(state["flying"])
    state["flying"] = handle
    n = state["step"][0]
    return eng.runner.logits[eng.runner.bucket(n)][:n]


def work(case):
    """Weights that the tokens meet, cached rows and states read, rows and states written, logits."""
    W, n, prefill = case["width"], case["n"], case["phase"] == "prefill"
    H, _, ff = SIZES[W]
    lens = _lengths(case)
    rows = sum(lens) if prefill else n
    pairs = sum(l * (l + 1) / 2 for l in lens) if prefill else sum(l + 1.0 for l in lens)
    layers, cfg = 4, _config(case)
    weights = 2.0 * W * VOCAB  # the head, bytes
    flops, moved = 2.0 * W * VOCAB * n, rows * W * 2.0 + n * VOCAB * 2.0

    def experts(count, top, params):  # (bytes of the experts that are met, flops)
        met = count * (1 - (1 - top / count) ** rows)
        return 2.0 * met * params, 2.0 * rows * top * params

    for i in range(layers):
        # the last layer of a prompt step ends with one row of each sequence
        tail = n if prefill and i == layers - 1 else rows
        if case["family"] in ("llama", "mixtral"):
            G = cfg.num_kv_heads
            qkv, out = W * (H + 2 * G) * DIM, W * H * DIM
            weights += 2.0 * (qkv + out)
            flops += 2.0 * (rows * qkv + tail * out) + 4.0 * pairs * H * DIM
            moved += 4.0 * G * DIM * ((0 if prefill else sum(lens)) + rows)
            if case["family"] == "llama":
                weights += 2.0 * 3 * W * ff
                flops += 2.0 * tail * 3 * W * ff
            else:
                b, f = experts(16, 4, 3 * W * ff // 4)
                weights, flops = weights + b, flops + f * tail / rows
            continue
        m, l = cfg.layers[i].mixer, cfg.layers[i]
        if isinstance(m, LatentAttention):
            near = [min(x, m.window or x) for x in lens]
            seen = sum(min(x, y) * (x + 1) - min(x, y) ** 2 / 2 for x, y in zip(lens, near)) if prefill else sum(near)
            proj = W * H * (m.dim + m.rot_dim) + (W * (m.kv_rank + m.rot_dim) if m.kv_from is None else 0)
            up = 2 * H * DIM * m.kv_rank
            weights += 2.0 * (proj + up + W * H * DIM)
            per = 2.0 * (m.dim + m.rot_dim + m.vdim) if prefill else 2.0 * (2 * m.kv_rank + m.rot_dim)
            flops += 2.0 * (rows * (proj + up) + tail * W * H * DIM) + H * per * seen
            moved += 2.0 * (m.kv_rank + m.rot_dim) * ((0 if prefill else sum(near)) + rows)
        else:
            proj = W * (3 * H * DIM + (2 * 128 + H if isinstance(m, ChannelDelta) else H * DIM))
            if isinstance(m, ChannelDelta):
                proj += 128 * 2 * H * DIM
            weights += 2.0 * (proj + W * H * DIM)
            flops += 2.0 * (rows * proj + tail * W * H * DIM) + rows * H * DIM * DIM * (8.0 if isinstance(m, ChannelDelta) else 6.0)
            moved += 4.0 * H * DIM * DIM * n * (1 if prefill else 2)
        if l.experts:
            b, f = experts(20, 4, 2 * W * ff // 4)
            weights += b + 2.0 * (2 * W * l.shared + 2 * W * cfg.side_dim)
            flops += (f / rows + 2.0 * (2 * W * l.shared + 2 * W * cfg.side_dim)) * tail
            moved += 2.0 * tail * cfg.side_dim
        elif l.ff:
            weights += 2.0 * 3 * W * l.ff
            flops += 2.0 * tail * 3 * W * l.ff
    return {"bytes": weights + moved, "flops": flops}


def tolerance(case):
    """bf16 rows and products leave 0.004 to 0.012 between these logits and those in 64 bits; where two
    experts are nearly equal, rounding may choose the other one, which is more for single rows."""
    return {"rel": 0.03 if case["family"] in ("mixtral", "garesun") else 0.02}


# ------------------------------------------------------------------ the same in 64 bits
def exact(case, seed):
    cfg = _config(case)
    family = case["family"]
    if family in ("llama", "mixtral"):
        m = _model(case, seed)
        weights = {"embed": m.embed, "head": m.lm_head, "final.norm": m.final_norm}
        for i, L in enumerate(m.layers):
            weights.update({f"l{i}.{k}": t for k, t in L.items()})
        del m
    else:
        weights = _checkpoint(cfg, seed)
    get = _Weights(weights)
    prompts, tokens = _tokens(case, seed)
    if case["phase"] == "decode":
        prompts = [p + [int(t)] for p, t in zip(prompts, tokens)]
    layers = {"llama": _attention_layer, "mixtral": _attention_layer, "ralesun": _serial_layer, "garesun": _joint_layer}
    out, at = [], 0
    while at < len(prompts):  # groups of sequences, padded behind to the longest (the first)
        longest = len(prompts[at])
        group = prompts[at:at + max(1, 20000 // longest)]
        at += len(group)
        lens = torch.tensor([len(p) for p in group], device="cuda")
        ids = torch.zeros(len(group), longest, dtype=torch.long)
        for i, p in enumerate(group):
            ids[i, :len(p)] = torch.tensor(p)
        ids = ids.cuda()
        x, carry = get("embed", rows=ids), {}
        if family == "garesun":
            x = x * cfg.embed_scale
        for i in range(4):
            last = lens - 1 if i == 3 else None
            x = layers[family](get, cfg, i, x, ids, last, carry)
        if family == "ralesun":
            x = _dyt(x, get, "final.norm")
        elif family == "garesun":
            x = _layer_norm(x) * get("final.norm")
        else:
            x = _rms(x) * get("final.norm")
        out.append(x @ get("head").T)
        del x, carry
    return torch.cat(out)


class _Weights:
    def __init__(self, tensors):
        self.tensors = tensors

    def __call__(self, name, rows=None, part=None):
        t = self.tensors[name]
        if part is not None:
            t = t[part]
        return (t if rows is None else t[rows]).double()


def _rms(x):
    return x * torch.rsqrt((x * x).mean(-1, keepdim=True) + EPS)


def _layer_norm(x):
    d = x - x.mean(-1, keepdim=True)
    return d * torch.rsqrt((d * d).mean(-1, keepdim=True) + EPS)


def _dyt(x, get, name):
    return torch.tanh(float(get.tensors[name + ".alpha"]) * x) * get(name) + get(name + ".b")


def _silu(x):
    return x * torch.sigmoid(x)


def _gelu(x):
    return torch.nn.functional.gelu(x, approximate="tanh")


def _pick(x, last):
    """Each sequence's last row."""
    return x if last is None else x[torch.arange(x.shape[0], device=x.device), last]


def _angles(length, dims, base):
    speed = base ** (-torch.arange(0, dims, 2, dtype=torch.float64, device="cuda") / dims)
    a = torch.arange(length, dtype=torch.float64, device="cuda")[:, None, None] * speed
    return torch.cos(a), torch.sin(a)


def _turn_halves(x, base):
    """[g, L, heads, D], components half of D apart."""
    c, s = _angles(x.shape[1], x.shape[-1], base)
    u, v = x.chunk(2, -1)
    return torch.cat([u * c - v * s, v * c + u * s], -1)


def _turn_pairs(x, base):
    """[g, L, heads, D], neighbours."""
    c, s = _angles(x.shape[1], x.shape[-1], base)
    u, v = x[..., 0::2], x[..., 1::2]
    return torch.stack([u * c - v * s, v * c + u * s], -1).flatten(-2)


def _causal(q, k, v, scale, window=None, sink=None):
    """q [g, L, H, d], k [g, L, H, d], v [g, L, H, dv] -> [g, L, H dv]; heads a few at a time."""
    g, L, H, _ = q.shape
    at = torch.arange(L, device="cuda")
    hidden = at[:, None] < at[None, :]
    if window is not None:
        hidden = hidden | (at[:, None] - at[None, :] >= window)
    out = torch.empty(g, L, H, v.shape[-1], dtype=torch.float64, device="cuda")
    few = max(1, int(1e9 / (L * L * g)))
    for h in range(0, H, few):
        e = min(H, h + few)
        s = torch.matmul(q[:, :, h:e].transpose(1, 2), k[:, :, h:e].permute(0, 2, 3, 1)) * scale
        s = s.masked_fill_(hidden, -math.inf)
        if sink is not None:
            s = torch.cat([s, sink[h:e].view(1, -1, 1, 1).expand(g, e - h, L, 1)], -1)
        p = torch.softmax(s, -1)[..., :L]
        out[:, :, h:e] = torch.matmul(p, v[:, :, h:e].transpose(1, 2)).transpose(1, 2)
    return out.flatten(2)


def _routed(z, x, top, one):
    """Weighted sum of the chosen experts' outputs; ``one(e, rows)``: an expert."""
    flat, z = x.reshape(-1, x.shape[-1]), z.reshape(-1, z.shape[-1])
    best = z.topk(top, -1)
    w, y = torch.softmax(best.values, -1), torch.zeros_like(flat)
    for e in range(z.shape[1]):
        rows, k = torch.nonzero(best.indices == e, as_tuple=True)
        if rows.numel():
            y.index_add_(0, rows, one(e, flat[rows]) * w[rows, k, None])
    return y.reshape(x.shape)


def _attention_layer(get, cfg, i, x, ids, last, carry):
    p, H, G = f"l{i}.", cfg.num_heads, cfg.num_kv_heads
    h = _rms(x) * get(p + "ln_in")
    q, k, v = (h @ get(p + "qkv").T).unflatten(-1, (-1, DIM)).split([H, G, G], 2)
    q, k = _turn_halves(q, cfg.rope_theta), _turn_halves(k, cfg.rope_theta)
    k, v = k.repeat_interleave(H // G, 2), v.repeat_interleave(H // G, 2)
    x = _pick(x, last) + _pick(_causal(q, k, v, DIM ** -0.5), last) @ get(p + "o").T
    h, ff = _rms(x) * get(p + "ln_post"), cfg.intermediate_size

    def mlp(r, up, down):
        g, u = (r @ up.T).split(ff, -1)
        return (_silu(g) * u) @ down.T

    if not cfg.is_moe:
        return x + mlp(h, get(p + "gate_up"), get(p + "down"))
    return x + _routed(h @ get(p + "router").T, h, cfg.experts_per_token,
                       lambda e, r: mlp(r, get(p + "gate_up", part=e), get(p + "down", part=e)))


def _latent(get, p, m, h, held):
    """-> (heads' outputs, latent rows)."""
    g, L, _ = h.shape
    H, d, r = m.heads, m.dim, m.rot_dim
    if held is None:
        kv = h @ get(p + "dkv").T
        held = _rms(kv[..., :m.kv_rank]) * get(p + "dkv.norm"), _turn_pairs(kv[..., None, m.kv_rank:], m.rot_base)
    c, kr = held
    q = (h @ get(p + "q").T).view(g, L, H, d + r)
    q = torch.cat([q[..., :d], _turn_pairs(q[..., d:], m.rot_base)], -1)
    k = torch.cat([(c @ get(p + "uk").T).view(g, L, H, d), kr.expand(g, L, H, r)], -1)
    v = (c @ get(p + "uv").T).view(g, L, H, m.vdim)
    return _causal(q, k, v, m.scale, m.window, get(p + "sink") if m.sink else None), held


def _conv(x, w):
    taps = w.shape[1]
    padded = torch.nn.functional.pad(x, (0, 0, taps - 1, 0))
    return sum(padded[:, j:j + x.shape[1]] * w[:, j] for j in range(taps))


def _unit(x):
    return x * torch.rsqrt((x * x).sum(-1, keepdim=True) + 1e-6)


def _delta(get, p, m, h):
    g, L, _ = h.shape
    H, d, dv = m.heads, m.dim, m.vdim
    q, k, v = (_silu(_conv(h @ get(p + x).T, get(f"{p}{x}.conv"))).view(g, L, H, -1) for x in "qkv")
    q, k = _unit(q) * d ** -0.5, _unit(k)
    beta = torch.sigmoid(h @ get(p + "b").T)
    raw = (h @ get(p + "a1").T) @ get(p + "a2").T + get(p + "dt_bias")
    step = torch.nn.functional.softplus(raw, threshold=700).view(g, L, H, d)
    decay = torch.exp(-torch.exp(get(p + "A_log"))[:, None] * step)
    S, o = h.new_zeros(g, H, d, dv), torch.empty_like(v)
    for t in range(L):
        S *= decay[:, t, :, :, None]
        u = beta[:, t, :, None] * (v[:, t] - (k[:, t, :, None] @ S)[:, :, 0])
        S += k[:, t, :, :, None] * u[:, :, None]
        o[:, t] = (q[:, t, :, None] @ S)[:, :, 0]
    gate = torch.sigmoid((h @ get(p + "g1").T) @ get(p + "g2").T).view(g, L, H, dv)
    return (_rms(o) * get(p + "norm") * gate).flatten(2)


def _memory(get, p, m, h):
    """Matrix memory, or retention: the same recurrence with a fixed decay and no normaliser."""
    g, L, _ = h.shape
    H, d = m.heads, m.dim
    q, k, v = ((h @ get(p + x).T).view(g, L, H, -1) for x in "qkv")
    z = h @ get(p + "g").T
    S, o = h.new_zeros(g, H, d, m.vdim), torch.empty_like(v)
    if isinstance(m, Retention):
        q, k = _turn_halves(q, m.rot_base), _turn_halves(k, m.rot_base) * d ** -0.5
        keep = torch.tensor(m.decay, dtype=torch.float64, device="cuda")[:, None, None]
        for t in range(L):
            S = S * keep + k[:, t, :, :, None] * v[:, t, :, None]
            o[:, t] = (q[:, t, :, None] @ S)[:, :, 0]
        return _rms(o).flatten(2) * _silu(z)
    q = q * d ** -0.5
    i, f = (m.gate_cap * torch.tanh((h @ get(p + x).T + get(f"{p}{x}.b")) / m.gate_cap) for x in "if")
    f = torch.nn.functional.logsigmoid(f)
    N, top = h.new_zeros(g, H, d), h.new_zeros(g, H)
    for t in range(L):
        new = torch.maximum(f[:, t] + top, i[:, t])
        keep, put = torch.exp(f[:, t] + top - new)[..., None], torch.exp(i[:, t] - new)[..., None]
        S = S * keep[..., None] + (put * k[:, t])[..., None] * v[:, t, :, None]
        N, top = N * keep + put * k[:, t], new
        den = torch.maximum((N * q[:, t]).sum(-1).abs(), torch.exp(-top)) + 1e-6
        o[:, t] = (q[:, t, :, None] @ S)[:, :, 0] / den[..., None]
    return _rms(o).flatten(2) * get(p + "norm") * torch.sigmoid(z)


def _serial_layer(get, cfg, i, x, ids, last, carry):
    m, p, q = cfg.layers[i].mixer, f"l{i}.mix.", f"l{i}.mlp."
    h = _dyt(x, get, f"l{i}.norm1")
    a = _delta(get, p, m, h) if isinstance(m, ChannelDelta) else _latent(get, p, m, h, None)[0]
    x = _pick(x, last) + _pick(a, last) @ get(p + "o").T
    if cfg.layers[i].ff:
        h = _dyt(x, get, f"l{i}.norm2")
        x = x + (_gelu(h @ get(q + "gate").T) * (h @ get(q + "up").T)) @ get(q + "down").T
    return x


def _joint_layer(get, cfg, i, x, ids, last, carry):
    l, p, q, side = cfg.layers[i], f"l{i}.mix.", f"l{i}.mlp.", cfg.side_dim
    h = _layer_norm(x) * get(f"l{i}.norm1")
    if isinstance(l.mixer, LatentAttention):
        a, carry[i] = _latent(get, p, l.mixer, h, carry.get(l.mixer.kv_from))
        a = a * torch.sigmoid(h @ get(p + "g").T).repeat_interleave(l.mixer.vdim, -1)
    else:
        a = _memory(get, p, l.mixer, h)
    x, h, ids = _pick(x, last), _pick(h, last), _pick(ids, last)

    def mlp(r, name):
        return torch.relu(r @ get(name + "up").T).square() @ get(name + "down").T

    x = x + _pick(a, last) @ get(p + "o").T + mlp(h, q + "shared.") + _routed(
        h @ get(q + "router").T, h, l.experts.top, lambda e, r: mlp(r, f"{q}e{e}."))
    own = get("side.embed", rows=ids)[..., i * side:(i + 1) * side]
    return x + _rms((_gelu(x @ get(f"l{i}.side.gate").T) * own) @ get(f"l{i}.side.proj").T) * get(f"l{i}.side.norm")
