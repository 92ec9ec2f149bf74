"""The workloads whose speed is watched: steps of whole models through `Engine.step`.

A case names a model (`design`, `size`, `layers`, `dtype`, for the dense decoder perhaps a sliding `window`) and
what a serving program asks of it:

  decode    `batch` sequences with about `context` cached tokens each take `steps` one-token steps, the tokens given on
            the device as a generation loop gives them; then the sequences are cut back to where they were
  prompt    `batch` new sequences of `tokens` tokens in all, packed in one step; the last token's logits are wanted
  turn      one sequence goes on by `tokens` tokens behind `context` cached ones while `batch` - 1 others take one
            token each, all in one step
  request   `batch` new sequences of `tokens` tokens in all; the logits of the last `places` of each are wanted (a
            scored completion); then `steps` one-token steps: the designs with a state per sequence, which cannot be
            cut back, go through both directions in one pass

Lengths are ragged: a case's total is dealt out unevenly over its sequences by the seed. Weights are random (the
engine's own generator, from the seed), token ids uniform. Outputs are fp32 logits.
"""
import math

import numpy as np
import torch

import hector_engine_amd as he
from hector_engine_amd.parts.base import BuildEnv
from hector_engine_amd.registry import build_model, config_from_dict
from hector_engine_amd.weights.random_init import random_tensor

F64 = torch.float64

# layer sizes: the benchmark's 7B and 32B shapes, the sizes of a 0.5B model of the same family, and the sizes the
# benchmark compares the other designs at
DENSE = {
    "0.5b": dict(hidden_size=896, num_attention_heads=14, num_key_value_heads=2, head_dim=64, intermediate_size=4864,
                 vocab_size=151936, tie_word_embeddings=True),
    "7b": dict(hidden_size=3584, num_attention_heads=28, num_key_value_heads=4, head_dim=128, intermediate_size=18944,
               vocab_size=152064, tie_word_embeddings=False),
    "32b": dict(hidden_size=5120, num_attention_heads=40, num_key_value_heads=8, head_dim=128, intermediate_size=27648,
                vocab_size=152064, tie_word_embeddings=False),
}
SIZES = {
    "w2048": dict(width=2048, heads=16, kv_heads=4, dim=128, vdim=128, ff=8192),
    "w3584": dict(width=3584, heads=28, kv_heads=4, dim=128, vdim=128, ff=18944),
    "w4096": dict(width=4096, heads=32, kv_heads=8, dim=64, vdim=128, ff=14336),
}
VOCAB = 32000


def listed():
    return [
        # the smallest steps: a 0.5B model answering one user, where launches and latency count
        dict(name="decode_small_b1", kind="decode", design="qwen2", size="0.5b", layers=24, dtype="bfloat16", window=0, batch=1, context=512, steps=8),
        # one user, and a handful of users, of a 7B model (the benchmark's headline and its point at batch 1)
        dict(name="decode_7b_b1", kind="decode", design="qwen2", size="7b", layers=28, dtype="bfloat16", window=0, batch=1, context=2048, steps=8),
        dict(name="decode_7b_b8", kind="decode", design="qwen2", size="7b", layers=28, dtype="bfloat16", window=0, batch=8, context=2048, steps=8),
        # a full server: many users with long contexts, where keys and values weigh as much as weights
        dict(name="decode_7b_b64_long", kind="decode", design="qwen2", size="7b", layers=8, dtype="bfloat16", window=0, batch=64, context=4100, steps=8),
        # one prompt, and a packed batch of ragged prompts
        dict(name="prompt_7b_2048", kind="prompt", design="qwen2", size="7b", layers=28, dtype="bfloat16", window=0, batch=1, tokens=2048),
        dict(name="prompt_7b_packed", kind="prompt", design="qwen2", size="7b", layers=28, dtype="bfloat16", window=0, batch=8, tokens=12001),
        # a conversation's next turn joins seven users that decode
        dict(name="turn_7b_b8", kind="turn", design="qwen2", size="7b", layers=28, dtype="bfloat16", window=0, batch=8, context=2500, tokens=203),
        # the 32-bit path, both directions
        dict(name="prompt_7b_fp32", kind="prompt", design="qwen2", size="7b", layers=8, dtype="float32", window=0, batch=1, tokens=1003),
        dict(name="decode_7b_b4_fp32", kind="decode", design="qwen2", size="7b", layers=8, dtype="float32", window=0, batch=4, context=700, steps=8),
        # the designs with a state per sequence and routed feed-forwards, both directions in a pass
        dict(name="penasun_request", kind="request", design="penasun", size="w2048", layers=4, dtype="bfloat16", batch=2, tokens=2048, places=32, steps=8),
        dict(name="butolorn_request", kind="request", design="butolorn", size="w3584", layers=4, dtype="bfloat16", batch=1, tokens=2048, places=32, steps=8),
        dict(name="domorax_request", kind="request", design="domorax", size="w2048", layers=4, dtype="bfloat16", batch=4, tokens=3001, places=16, steps=8),
    ]


def _log(rng, lo, hi):
    return max(lo, min(hi, int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))))


def draw(rng):
    kind = rng.choice(["decode", "decode", "prompt", "prompt", "turn", "fp32", "request", "request", "request"])
    if kind == "request":
        design = rng.choice(["penasun", "butolorn", "domorax"])
        batch = rng.choice([1, 1, 2, 3, 4, 8])
        return dict(kind=kind, design=design, size=rng.choice(sorted(SIZES)), layers=rng.choice([2, 4]) if design != "domorax" else 4,
                    dtype="float32" if rng.random() < (0.4 if design == "domorax" else 0.15) else "bfloat16", batch=batch,
                    tokens=max(24 * batch, _log(rng, 24, 3001)), places=rng.choice([1, 8, 16]), steps=rng.choice([4, 8]))
    dense = dict(design="qwen2", size=rng.choice(["0.5b", "7b", "7b", "32b"]), layers=rng.choice([4, 8]), dtype="bfloat16", window=0)
    if kind == "fp32":
        kind = rng.choice(["decode", "prompt"])
        dense.update(dtype="float32", size=rng.choice(["0.5b", "7b"]), layers=4)
        if kind == "decode":
            return dict(dense, kind=kind, batch=_log(rng, 1, 16), context=_log(rng, 16, 1003), steps=8)
        return dict(dense, kind=kind, batch=rng.choice([1, 1, 3]), tokens=_log(rng, 16, 1003))
    small = dense["size"] == "0.5b"       # (of the small model no steps of 17 to 64 rows: they were refused when this file was written)
    if kind == "decode":
        return dict(dense, kind=kind, batch=_log(rng, 1, 16 if small else 64), context=_log(rng, 64, 4100), steps=8)
    if kind == "prompt":
        batch = rng.choice([1, 1, 2, 5, 8])
        return dict(dense, kind=kind, window=rng.choice([0, 0, 1024]), batch=batch, tokens=max(65 if small else 8 * batch, _log(rng, 16, 12001)))
    return dict(dense, kind=kind, batch=_log(rng, 2, 16), context=_log(rng, 64, 2500), tokens=_log(rng, 65 if small else 8, 700))


# ---- models ---------------------------------------------------------------------------

def model_dict(case):
    design, L = case["design"], case["layers"]
    if design == "qwen2":
        d = dict(DENSE[case["size"]], architectures=["Qwen2ForCausalLM"], num_hidden_layers=L, rope_theta=1000000.0,
                 rms_norm_eps=1e-6, max_position_embeddings=32768)
        if case["window"]:
            d.update(use_sliding_window=True, sliding_window=case["window"], max_window_layers=L // 2)
        return d
    z = SIZES[case["size"]]
    base = dict(vocab=VOCAB, width=z["width"], norm=dict(eps=1e-6))
    if design == "penasun":
        scan = dict(type="mamba2", mixer=dict(heads=2 * z["width"] // 64, vdim=64, state=128, groups=8, conv=4, norm_groups=8))
        attention = dict(type="attention", mixer=dict(heads=z["heads"], kv_heads=z["kv_heads"], dim=z["dim"] // 2, vdim=z["vdim"],
                                                      scale=(z["dim"] // 2) ** -0.5, diff=0.6, q_temp=dict(coef=0.1, every=512)))
        mlp = dict(kind="moe", expert=dict(ff=z["ff"] // 4, limit=7.0),
                   router=dict(experts=16, identity=2, top=4, scale=1.0, groups=dict(count=3, keep=2)))
        return dict(base, architecture="Penasun", layers=[dict(l, mlp=mlp) for l in (scan, attention)] * (L // 2))
    if design == "butolorn":
        attention = dict(heads=z["heads"], kv_heads=z["kv_heads"], dim=z["dim"], vdim=z["vdim"], scale=z["dim"] ** -0.5,
                         rot=dict(base=1000000.0, dims=z["dim"] // 2))
        pair = dict(left=attention, left_scale=1.0, right_scale=1.0,
                    right=dict(heads=z["width"] // 256, dim=128, vdim=256, gate_cap=15.0))
        mlp = dict(kind="dense", ff=z["ff"])
        return dict(base, architecture="Butolorn", embedding=dict(scale=1.0), token_side=dict(dim=64),
                    loop=dict(start=0, stop=0, times=1),
                    layers=[dict(type="parallel", mixer=pair, mlp=mlp), dict(type="attention", mixer=attention, mlp=mlp)] * (L // 2))
    delta = dict(type="delta", mixer=dict(heads=z["heads"], kv_heads=z["kv_heads"], dim=z["dim"], vdim=z["vdim"], conv=4))
    latent = dict(type="latent_attention", mixer=dict(
        heads=z["heads"], dim=z["dim"], rot_dim=64, vdim=z["vdim"], kv_rank=192, q_rank=z["width"] // 2,
        scale=(z["dim"] + 64) ** -0.5, mask=dict(size=1024),
        rot=dict(base=10000.0, dims=64, scaling=dict(factor=4.0, original=1024, fast=32.0, slow=1.0))))
    wide = max(z["dim"], z["vdim"])
    attention = dict(type="attention", mixer=dict(heads=z["heads"], kv_heads=z["kv_heads"], dim=wide, vdim=wide, conv=4, scale=wide ** -0.5))
    moe = dict(kind="moe", expert=dict(ff=z["ff"] // 4), router=dict(experts=16, top=4), shared=dict(ff=z["ff"] // 4))
    return dict(base, architecture="Domorax", residual_mult=0.5, norm=dict(eps=1e-6, groups=4),
                layers=[dict(delta, mlp=moe), dict(latent, mlp=moe), dict(delta, mlp=dict(kind="dense", ff=z["ff"])), dict(attention, mlp=moe)])


def vocabulary(case):
    return DENSE[case["size"]]["vocab_size"] if case["design"] == "qwen2" else VOCAB


def deal(rng, total, parts):
    """`total` tokens dealt out over `parts` sequences: shares between about half and half as much again of the mean."""
    share = rng.uniform(0.5, 1.5, parts)
    n = np.maximum(1, np.floor(total * share / share.sum()).astype(int))
    n[int(np.argmax(n))] += total - int(n.sum())
    return [int(v) for v in n]


def plan(case, seed):
    """The tokens of every sequence: (cached before the pass, fed by the pass's first step, fed one by one after it)."""
    rng = np.random.default_rng([seed, 77])
    V, B, kind = vocabulary(case), case["batch"], case["kind"]

    def ids(n):
        return rng.integers(0, V, n).tolist()
    if kind == "decode":
        return [(ids(n), [], ids(case["steps"])) for n in deal(rng, case["context"] * B, B)]
    if kind == "turn":
        lengths = deal(rng, case["context"] * B, B)
        return [(ids(n), ids(case["tokens"] if i == B - 1 else 1), []) for i, n in enumerate(lengths)]
    return [([], ids(n), ids(case.get("steps", 0))) for n in deal(rng, case["tokens"], B)]


# ---- one pass ---------------------------------------------------------------------------

def prepare(case, seed):
    seqs = plan(case, seed)
    longest = max(len(a) + len(b) + len(c) for a, b, c in seqs)
    pages = sum(-(-(len(a) + len(b) + len(c)) // 64) for a, b, c in seqs)
    engine = he.Engine(config=config_from_dict(model_dict(case)), seed=seed, dtype=case["dtype"], max_tokens=64 * (pages + 1),
                       max_slots=case["batch"], max_seq_len=longest)
    state = dict(case=case, engine=engine, seqs=seqs, slots=[],
                 after=torch.tensor([c for _, _, c in seqs], dtype=torch.int32).t().contiguous().to(engine.device))
    if case["kind"] in ("decode", "turn"):
        state["slots"] = [engine.acquire() for _ in seqs]
        for i in range(0, len(seqs), 4):        # the contexts, a few sequences a step
            engine.step([he.StepEntry(s, a, []) for s, (a, _, _) in zip(state["slots"][i:i + 4], seqs[i:i + 4])])
    if seqs[0][2]:                              # room for every one-token step's logits
        state["logits"] = torch.empty((len(seqs[0][2]), len(seqs), vocabulary(case)), dtype=torch.float32, device=engine.device)
    engine.synchronize()
    return state


def wanted(case, n):
    return list(range(max(0, n - case.get("places", 1)), n))


def run(state):
    case, engine, seqs, out = state["case"], state["engine"], state["seqs"], {}
    keep = case["kind"] in ("decode", "turn")
    slots = state["slots"] if keep else [engine.acquire() for _ in seqs]
    if seqs[0][1]:
        first = engine.step([he.StepEntry(s, b, wanted(case, len(b))) for s, (_, b, _) in zip(slots, seqs)])
        out["first"] = first if not seqs[0][2] else first.clone()      # (a step's logits are valid until the next step)
    for j in range(len(seqs[0][2])):
        logits = engine.step([he.StepEntry(s, [c[j]], [0]) for s, (_, _, c) in zip(slots, seqs)], device_tokens=state["after"][j])
        out["after"] = state["logits"]
        out["after"][j].copy_(logits)
    for s, (a, _, _) in zip(slots, seqs):
        if keep:
            engine.truncate(s, len(a))
        else:
            engine.release(s)
    return out


# ---- what a pass cannot do without ---------------------------------------------------------

def work(case):
    """Every weight read once a step (of the experts those that some token uses), keys and values of every earlier
    token read once and of every new one written, states read and written, logits written; two operations a weight
    and token and the attention's products."""
    es = 2 if case["dtype"] == "bfloat16" else 4
    specs = build_model(config_from_dict(model_dict(case)), BuildEnv(torch.device("cpu"), getattr(torch, case["dtype"]))).tensor_specs()
    V, B, seqs = vocabulary(case), case["batch"], plan(case, 0)
    dense = expert = tables = 0
    for name, spec in specs.items():
        n = math.prod(spec.shape)
        if name.startswith("model.embed") or name in ("embed", "side.embed"):
            tables += n if name == "embed" and "head" not in specs or case["size"] == "0.5b" else 0       # tied: read as the head
        elif ".mlp.e" in name:
            expert += n
        elif name in ("head", "lm_head.weight"):
            tables += n
        else:
            dense += n
    d = model_dict(case)
    if case["design"] == "qwen2":
        H, G, hd, e = d["num_attention_heads"], d["num_key_value_heads"], d["head_dim"], d["head_dim"]
        attending = [(H, G, hd, e, case["window"] if l >= case["layers"] // 2 else 0) for l in range(case["layers"])]
    else:
        attending = []
        for l in d["layers"]:
            m = l["mixer"].get("left", l["mixer"])
            if l["type"] in ("attention", "parallel"):
                maps = 2 if case["design"] == "penasun" else 1
                attending.append((maps * m["heads"], maps * m["kv_heads"], m["dim"], m["vdim"], 0))
            elif l["type"] == "latent_attention":
                attending.append((m["heads"], 1, m["kv_rank"] + m["rot_dim"], 0, m["mask"]["size"]))
    top, experts = (4, 16) if expert else (0, 1)

    def step(news, befores, wants):
        rows = sum(news)
        used = 1 - (1 - top / experts) ** rows if expert else 0
        nbytes = es * (dense + used * expert + tables) + 4 * wants * V
        flops = 2.0 * rows * (dense + expert * top / experts) + 2.0 * wants * tables
        for H, G, dim, e, window in attending:
            for n, before in zip(news, befores):
                first = min(before, window) if window else before
                pairs = sum(min(before + i + 1, window) if window else before + i + 1 for i in (range(n) if window else ()))
                pairs = pairs or n * before + n * (n + 1) // 2
                nbytes += es * G * (dim + e) * (first + n)
                flops += 2.0 * H * (dim + (e or dim)) * pairs
        return nbytes, flops

    total = [0.0, 0.0]
    before = [len(a) for a, _, _ in seqs]
    todo = []
    if seqs[0][1]:
        news = [len(b) for _, b, _ in seqs]
        todo.append((news, list(before), sum(len(wanted(case, n)) for n in news)))
        before = [x + n for x, n in zip(before, news)]
    for _ in seqs[0][2]:
        todo.append(([1] * B, list(before), B))
        before = [x + 1 for x in before]
    for t in todo:
        nb, fl = step(*t)
        total[0] += nb
        total[1] += fl
    return {"bytes": total[0], "flops": total[1]}


def tolerance(case):
    """About four times what the path differs from its 64-bit form where that is a few roundings (32-bit: 2e-6), and what
    two correct implementations differ by where bf16 activations pass through all layers (from the 64-bit form: 1 % at
    4 layers, 3 % at 8, 6.5 % at 28)."""
    if case["dtype"] == "float32":
        return {"rel": 1e-5}
    if case["design"] == "domorax":      # unnormed rows into a router: near ties fall either way (from the 64-bit form: up to 20 %)
        return {"rel": 0.3}
    if case["design"] == "penasun":      # a router behind a norm: 1 to 5 %
        return {"rel": 0.15}
    return {"rel": round(0.025 * math.sqrt(case["layers"]), 3)}


# ---- the same in 64 bits -----------------------------------------------------------------

def rms(x, eps=1e-6):
    return x / torch.sqrt((x * x).mean(-1, keepdim=True) + eps)


def silu(z):
    return z * torch.sigmoid(z)


def gelu_tanh(z):
    return 0.5 * z * (1.0 + torch.tanh(math.sqrt(2.0 / math.pi) * (z + 0.044715 * z ** 3)))


def softplus(z):
    return torch.logaddexp(z, torch.zeros_like(z))


def rotate(x, dims, freqs, mult=1.0, interleaved=False):
    """x [T, heads, d] at the positions 0..: pairs of the first `dims` dims turn by position * frequency (the angle is
    a product of the frequencies' type: the dense decoder's is a float32 one by its definition)."""
    a = (torch.arange(x.shape[0], dtype=freqs.dtype, device=x.device)[:, None] * freqs.to(x.device)).to(F64)
    c, s = (torch.cos(a) * mult)[:, None], (torch.sin(a) * mult)[:, None]
    out = x.clone()
    i, j = (slice(0, dims, 2), slice(1, dims, 2)) if interleaved else (slice(0, dims // 2), slice(dims // 2, dims))
    out[..., i] = x[..., i] * c - x[..., j] * s
    out[..., j] = x[..., j] * c + x[..., i] * s
    return out


def plain_freqs(dims, base):
    return torch.tensor([base ** (-2.0 * i / dims) for i in range(dims // 2)], dtype=F64)


def yarn_freqs(r, base, sc):
    f = plain_freqs(r, base)

    def dim_of(turns):
        return r * math.log(sc["original"] / (2 * math.pi * turns)) / (2 * math.log(base))
    lo, hi = max(math.floor(dim_of(sc["fast"])), 0), min(math.ceil(dim_of(sc["slow"])), r - 1)
    ramp = ((torch.arange(r // 2, dtype=F64) - lo) / max(hi - lo, 0.001)).clamp(0, 1)
    return f / sc["factor"] * ramp + f * (1 - ramp), 0.1 * math.log(sc["factor"]) + 1.0


def attend(q, k, v, scale, window=0, sink=None, slopes=None):
    """Causal attention, q [T, H, d], k [T, G, d], v [T, G, e]; sink [H]: one more term in the denominator."""
    T, H, G = q.shape[0], q.shape[1], k.shape[1]
    at = torch.arange(T, device=q.device)
    gap = at[:, None] - at[None, :]
    hidden = (gap < 0) | (gap >= window) if window else gap < 0
    out = []
    for h in range(H):
        g = h // (H // G)
        s = (q[:, h] @ k[:, g].t().contiguous()) * scale
        if slopes is not None:
            s = s - slopes[h] * gap
        s = s.masked_fill(hidden, -math.inf)
        if sink is not None:
            s = torch.cat([s, sink[h].expand(T, 1)], 1)
        p = torch.softmax(s, -1)
        out.append(p[:, :T] @ v[:, g])
    return torch.stack(out, 1)


def conv(u, taps):
    K = taps.shape[1]
    padded = torch.cat([u.new_zeros(K - 1, u.shape[1]), u])
    return sum(taps[:, j] * padded[j:j + u.shape[0]] for j in range(K))


class Plain:
    """One model in 64 bits, sequences one after another through a layer at a time; its weights are the engine's, made
    from the same seed."""

    def __init__(self, case, seed):
        self.d, self.case, self.seed = model_dict(case), case, seed
        self.dtype = getattr(torch, case["dtype"])
        self.specs = build_model(config_from_dict(self.d), BuildEnv(torch.device("cpu"), self.dtype)).tensor_specs()

    def w(self, name):
        return random_tensor(name, self.specs[name], self.seed, self.dtype, "cuda").to(F64)

    def logits(self, seqs, places):
        d, qwen2 = self.d, self.case["design"] == "qwen2"
        table = self.w("model.embed_tokens.weight" if qwen2 else "embed")
        xs = [table[torch.tensor(s, device="cuda")] for s in seqs]
        tied = d["tie_word_embeddings"] if qwen2 else "head" not in self.specs
        kept = [[x] for x in xs]
        del table
        for l in range(self.case["layers"]):
            xs = getattr(self, self.case["design"])(l, xs, seqs, kept)
        out = torch.cat([x[p] for x, p in zip(xs, places)])
        if qwen2:
            normed, head = rms(out) * self.w("model.norm.weight"), "model.embed_tokens.weight" if tied else "lm_head.weight"
        else:
            groups = d["norm"].get("groups", 1)
            normed = rms(out.reshape(len(out), groups, -1)).reshape(out.shape) * self.w("final.norm")
            head = "embed" if tied else "head"
        return normed @ self.w(head).t()

    # each: layer l over all sequences' streams; returns the new ones

    def qwen2(self, l, xs, seqs, kept):
        d, p = self.d, f"model.layers.{l}."
        H, G, hd = d["num_attention_heads"], d["num_key_value_heads"], d["head_dim"]
        window = self.case["window"] if l >= self.case["layers"] // 2 else 0
        f = plain_freqs(hd, d["rope_theta"]).float()
        w = {n: (self.w(f"{p}self_attn.{n}_proj.weight"), self.w(f"{p}self_attn.{n}_proj.bias")) for n in "qkv"}
        n1, o = self.w(p + "input_layernorm.weight"), self.w(p + "self_attn.o_proj.weight")
        new = []
        for x in xs:
            h = rms(x) * n1
            q, k, v = ((h @ w[n][0].t() + w[n][1]).reshape(len(x), -1, hd) for n in "qkv")
            y = attend(rotate(q, hd, f), rotate(k, hd, f), v, hd ** -0.5, window)
            new.append(x + y.reshape(len(x), H * hd) @ o.t())
        del w, o
        n2, gate, up, down = (self.w(p + n + ".weight") for n in ("post_attention_layernorm", "mlp.gate_proj", "mlp.up_proj", "mlp.down_proj"))
        return [x + (silu(h @ gate.t()) * (h @ up.t())) @ down.t() for x in new for h in [rms(x) * n2]]

    def penasun(self, l, xs, seqs, kept):
        layer, pre = self.d["layers"][l], f"l{l}."
        m, mix = layer["mixer"], pre + "mix."
        n1, n2 = self.w(pre + "norm1"), self.w(pre + "norm2")
        mixer = self.ssm if layer["type"] == "mamba2" else self.diff_attention
        xs = [x + mixer(rms(x) * n1, mix, m) for x in xs]
        r, mlp = layer["mlp"]["router"], pre + "mlp."
        experts = [[self.w(f"{mlp}e{e}.{n}") for n in ("gate", "up", "down")] for e in range(r["experts"])]
        router, correction, limit = self.w(mlp + "router"), self.w(mlp + "correction"), layer["mlp"]["expert"]["limit"]
        new = []
        for x in xs:
            h = rms(x) * n2
            s = torch.softmax(h @ router.t(), -1)
            c = (s + correction).reshape(len(x), r["groups"]["count"], -1)
            keep = torch.topk(c.max(-1).values, r["groups"]["keep"], -1).indices
            masked = torch.full_like(c, -math.inf).scatter(1, keep[..., None].expand(-1, -1, c.shape[2]),
                                                           c.gather(1, keep[..., None].expand(-1, -1, c.shape[2])))
            chosen = torch.topk(masked.reshape(len(x), -1), r["top"], -1).indices
            share = torch.zeros_like(s).scatter(1, chosen, s.gather(1, chosen)) * r["scale"]
            y = h * share[:, r["experts"]:].sum(-1, keepdim=True)
            for e, (gate, up, down) in enumerate(experts):
                rows = (share[:, e] != 0).nonzero()[:, 0]
                g, u = (h[rows] @ gate.t()).clamp(max=limit), (h[rows] @ up.t()).clamp(-limit, limit)
                y[rows] += share[rows, e:e + 1] * ((g * torch.sigmoid(1.702 * g) * (u + 1)) @ down.t())
            new.append(x + y)
        return new

    def ssm(self, h, p, m):
        R, P, N, Q, T = m["heads"], m["vdim"], m["state"], m["groups"], len(h)
        inner = R * P
        proj = h @ self.w(p + "in").t()
        z, dt = proj[:, :inner], softplus(proj[:, 2 * inner + 2 * Q * N:] + self.w(p + "dt_bias"))
        xbc = silu(conv(proj[:, inner:2 * inner + 2 * Q * N], self.w(p + "conv")) + self.w(p + "conv.b"))
        x = xbc[:, :inner].reshape(T, R, P)
        Bs, Cs = (t.reshape(T, Q, N).repeat_interleave(R // Q, 1) for t in (xbc[:, inner:inner + Q * N], xbc[:, inner + Q * N:]))
        decay, Bd = torch.exp(-torch.exp(self.w(p + "A_log")) * dt), Bs * dt[..., None]
        S, y = h.new_zeros(R, N, P), torch.empty_like(x)
        for t in range(T):
            S = torch.baddbmm(S * decay[t, :, None, None], Bd[t][:, :, None], x[t][:, None, :])
            y[t] = torch.bmm(Cs[t][:, None, :], S)[:, 0]
        y = (y + self.w(p + "D")[:, None] * x).reshape(T, inner) * silu(z)
        return (rms(y.reshape(T, m["norm_groups"], -1)).reshape(T, inner) * self.w(p + "norm")) @ self.w(p + "o").t()

    def diff_attention(self, h, p, m):
        H, G, dim, e, T = m["heads"], m["kv_heads"], m["dim"], m["vdim"], len(h)
        q, k, v = (h @ self.w(p + n).t() + self.w(p + n + ".b") for n in "qkv")
        q, k, v = q.reshape(T, H, 2, dim), k.reshape(T, G, 2, dim), v.reshape(T, G, e)
        at = torch.arange(T, dtype=F64, device=h.device)
        q = q * (1 + m["q_temp"]["coef"] * torch.log((at + 1).div(m["q_temp"]["every"], rounding_mode="floor") + 1))[:, None, None, None]
        one, two = (math.exp(float((self.w(p + f"lq{i}") * self.w(p + f"lk{i}")).sum())) for i in (1, 2))
        a, b = (attend(q[:, :, i], k[:, :, i], v, m["scale"]) for i in (0, 1))
        y = rms(a - (one - two + m["diff"]) * b) * (1 - m["diff"])
        return y.reshape(T, H * e) @ self.w(p + "o").t() + self.w(p + "o.b")

    def butolorn(self, l, xs, seqs, kept):
        layer, p, side = self.d["layers"][l], f"l{l}.", self.d["token_side"]["dim"]
        w = {n: self.w(p + n) for n in ("norm1", "norm1b", "norm2", "norm2b", "mlp.up", "mlp.down", "side.gate", "side.proj", "side.norm")}
        rows = self.w("side.embed")[:, l * side:(l + 1) * side]
        new = []
        for x, ids in zip(xs, seqs):
            h = rms(x) * w["norm1"]
            if layer["type"] == "attention":
                y = self.rotated_attention(h, p + "mix.", layer["mixer"], False)
            else:
                y = layer["mixer"]["left_scale"] * self.rotated_attention(h, p + "mix.left.", layer["mixer"]["left"], True) \
                    + layer["mixer"]["right_scale"] * self.memory(h, p + "mix.right.", layer["mixer"]["right"])
            x = x + rms(y) * w["norm1b"]
            x = x + rms((((rms(x) * w["norm2"]) @ w["mlp.up"].t()).clamp(min=0) ** 2) @ w["mlp.down"].t()) * w["norm2b"]
            y = (gelu_tanh(x @ w["side.gate"].t()) * rows[torch.tensor(ids, device="cuda")]) @ w["side.proj"].t()
            new.append(x + rms(y) * w["side.norm"])
        return new

    def rotated_attention(self, h, p, m, beside):
        T = len(h)
        q, k, v = (h @ self.w(p + n).t() for n in "qkv")
        if beside:
            q, k = rms(q) * self.w(p + "q.norm"), rms(k) * self.w(p + "k.norm")
        else:
            q, k, v = q + self.w(p + "q.b"), k + self.w(p + "k.b"), v + self.w(p + "v.b")
        dims = m["rot"]["dims"]
        f = plain_freqs(dims, m["rot"]["base"])
        q, k = (rotate(t.reshape(T, -1, m["dim"]), dims, f, interleaved=beside) for t in (q, k))
        y = attend(q, k, v.reshape(T, -1, m["vdim"]), m["scale"], sink=h.new_zeros(m["heads"]) if beside else None).reshape(T, -1)
        if beside:
            y = y * torch.sigmoid(h @ self.w(p + "g").t())
        return y @ self.w(p + "o").t()

    def memory(self, h, p, m):
        H, dim, e, cap, T = m["heads"], m["dim"], m["vdim"], m["gate_cap"], len(h)
        q, k, v = ((h @ self.w(p + n).t()).reshape(T, H, -1) for n in "qkv")
        q = q * dim ** -0.5
        gate_in, keep = (cap * torch.tanh((h @ self.w(p + n).t() + self.w(p + n + ".b")) / cap) for n in "if")
        keep = -softplus(-keep)
        S, n, top, y = h.new_zeros(H, dim, e), h.new_zeros(H, dim), h.new_zeros(H), torch.empty_like(v)
        for t in range(T):
            new = torch.maximum(keep[t] + top, gate_in[t])
            old, take = torch.exp(keep[t] + top - new), torch.exp(gate_in[t] - new)
            kt = k[t] * take[:, None]
            S = torch.baddbmm(S * old[:, None, None], kt[:, :, None], v[t][:, None, :])
            n, top = n * old[:, None] + kt, new
            y[t] = torch.bmm(q[t][:, None, :], S)[:, 0] / (torch.maximum((n * q[t]).sum(-1).abs(), torch.exp(-top)) + 1e-6)[:, None]
        return (rms(y).reshape(T, H * e) * self.w(p + "norm") * torch.sigmoid(h @ self.w(p + "g").t())) @ self.w(p + "o").t()

    def domorax(self, l, xs, seqs, kept):
        layer, p, d = self.d["layers"][l], f"l{l}.", self.d
        m, mix, mlp = layer["mixer"], p + "mix.", layer["mlp"]
        groups, mult = d["norm"]["groups"], d["residual_mult"]

        def normed(y, name):
            return rms(y.reshape(len(y), groups, -1)).reshape(y.shape) * self.w(p + name)
        mixer = {"delta": self.delta, "latent_attention": self.latent, "attention": self.conv_attention}[layer["type"]]
        xs = [x + mult * normed(mixer(x, mix, m), "norm1") for x in xs]
        ff = self.poly_ff if mlp["kind"] == "dense" else self.routed_ff
        xs = [x + mult * normed(ff(x, p + "mlp.", mlp), "norm2") for x in xs]
        weights, new = self.w(p + "dwa"), []
        for x, k in zip(xs, kept):
            k.append(x)
            new.append(sum(weights[j] * k[j] for j in range(l + 2)))
        return new

    def delta(self, h, p, m):
        H, G, dim, e, T = m["heads"], m["kv_heads"], m["dim"], m["vdim"], len(h)
        q, k, v = (silu(conv(h @ self.w(p + n).t(), self.w(p + n + ".conv"))) for n in "qkv")

        def unit(x):
            return x / torch.sqrt((x * x).sum(-1, keepdim=True) + 1e-6)
        q, k = (unit(t.reshape(T, G, dim)).repeat_interleave(H // G, 1) for t in (q, k))
        q, v = q * dim ** -0.5, v.reshape(T, H, e)
        beta = torch.sigmoid(h @ self.w(p + "b").t())
        g = torch.exp(-torch.exp(self.w(p + "A_log")) * softplus(h @ self.w(p + "a").t() + self.w(p + "dt_bias")))
        S, o = h.new_zeros(H, dim, e), torch.empty_like(v)
        for t in range(T):
            S = S * g[t, :, None, None]
            u = beta[t][:, None] * (v[t] - torch.bmm(k[t][:, None, :], S)[:, 0])
            S = torch.baddbmm(S, k[t][:, :, None], u[:, None, :])
            o[t] = torch.bmm(q[t][:, None, :], S)[:, 0]
        y = rms(o) * self.w(p + "norm") * silu(h @ self.w(p + "g").t()).reshape(T, H, e)
        return y.reshape(T, H * e) @ self.w(p + "o").t()

    def latent(self, h, p, m):
        H, dim, r, e, rank, T = m["heads"], m["dim"], m["rot_dim"], m["vdim"], m["kv_rank"], len(h)
        q = ((rms(h @ self.w(p + "dq").t()) * self.w(p + "dq.norm")) @ self.w(p + "uq").t()).reshape(T, H, dim + r)
        down = h @ self.w(p + "dkv").t()
        c = rms(down[:, :rank]) * self.w(p + "dkv.norm")
        k, v = (c @ self.w(p + "uk").t()).reshape(T, H, dim), (c @ self.w(p + "uv").t()).reshape(T, H, e)
        f, mult = yarn_freqs(r, m["rot"]["base"], m["rot"]["scaling"])
        q = torch.cat([q[..., :dim], rotate(q[..., dim:], r, f, mult)], -1)
        k = torch.cat([k, rotate(down[:, rank:].reshape(T, 1, r), r, f, mult).expand(T, H, r)], -1)
        y = attend(q, k, v, m["scale"], m["mask"]["size"], self.w(p + "sink"))
        return y.reshape(T, H * e) @ self.w(p + "o").t()

    def conv_attention(self, h, p, m):
        H, dim, T = m["heads"], m["dim"], len(h)
        q, k = (conv(h @ self.w(p + n).t(), self.w(p + n + ".conv")).reshape(T, -1, dim) for n in "qk")
        slopes = [2.0 ** (-8.0 * (i + 1) / H) for i in range(H)]
        y = attend(rms(q) * self.w(p + "q.norm"), rms(k) * self.w(p + "k.norm"), k, m["scale"], slopes=slopes)
        return y.reshape(T, H * dim) @ self.w(p + "o").t()

    def poly_ff(self, h, p, mlp):
        z = h @ self.w(p + "up").t()
        a, b, c, e = self.w(p + "act").tolist()
        return (a * rms(z) + b * rms(z * z) + c * rms(z * z * z) + e) @ self.w(p + "down").t()

    def routed_ff(self, h, p, mlp):
        def expert(x, name):
            return (silu(x @ self.w(p + name + ".gate").t()) * (x @ self.w(p + name + ".up").t())) @ self.w(p + name + ".down").t()
        z = h @ self.w(p + "router").t()
        best = torch.topk(z, mlp["router"]["top"], -1)
        share = torch.zeros_like(z).scatter(1, best.indices, torch.softmax(best.values, -1))
        y = torch.sigmoid(h @ self.w(p + "shared.sg").t()) * expert(h, "shared")
        for e in range(mlp["router"]["experts"]):
            rows = (share[:, e] != 0).nonzero()[:, 0]
            y[rows] += share[rows, e:e + 1] * expert(h[rows], f"e{e}")
        return y


def exact(case, seed):
    seqs = plan(case, seed)
    tokens = sum(len(a) + len(b) + len(c) for a, b, c in seqs)
    d = model_dict(case)
    if case["design"] == "domorax" and case["dtype"] == "bfloat16":
        return None           # (bf16 turns its router's near ties over; its 32-bit cases hold the same arithmetic to 1e-5)
    if case["design"] == "qwen2" and 2.0 * tokens * case["layers"] * d["hidden_size"] * (3 * d["intermediate_size"] + 2 * d["hidden_size"]) > 3e14:
        return None           # (the full server's contexts: minutes in 64 bits)
    model = Plain(case, seed)
    first = [[len(a) + w for w in wanted(case, len(b))] if b else [] for a, b, _ in seqs]
    after = [list(range(len(a) + len(b), len(a) + len(b) + len(c))) for a, b, c in seqs]
    rows = model.logits([a + b + c for a, b, c in seqs], [torch.tensor(f + a, dtype=torch.long, device="cuda") for f, a in zip(first, after)])
    parts = rows.split([len(f) + len(a) for f, a in zip(first, after)])
    out = {}
    if first[0]:
        out["first"] = torch.cat([x[:len(f)] for x, f in zip(parts, first)])
    if after[0]:
        out["after"] = torch.stack([x[len(f):] for x, f in zip(parts, first)], 1)
    return out
