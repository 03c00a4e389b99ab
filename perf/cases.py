"""What is measured of this library's speed: passes through its public entry points as a program that serves or
scores text makes them.

A pass of a language-model case takes its sequences' slots, runs their prompts in one step (`Model.step`, ragged and
packed), lets a late prompt come in by portions while the others go on by a token (`Model.step` again: the mixed steps
of continuous batching), then continues every sequence by one token a step through the captured decode graphs
(`Engine.graphed`), and gives the slots back.  The continuations' tokens are given beforehand, as when a known text is
scored or a draft is checked, so that the logits of two implementations can be compared; every step's logits are
returned.  A `sample` case is the choice of the next tokens from given logits.

Weights are random, drawn on the GPU from the seed (N(0, 0.02), norm weights N(0, 0.1)); prompts are uniform random ids.
Only architectures without routed experts are here: two correct implementations in bfloat16 choose different experts
wherever two scores nearly tie, and their logits then cannot be held to a tolerance.
"""
import hashlib
import math
import random

import torch

DEVICE = "cuda:0"
CONTEXT = 8192

# ---- the models: sizes of the benchmark (`python -m trapetum_amd bench`, also with --compare) ---------------------------
# The two recurrent designs have fewer layers than there (the benchmark's --layers): in bfloat16 their random weights
# carry a rounding error on from layer to layer (26 layers of Besulix are 3 to 5 per cent off what 64 bits give), and two
# correct implementations have to be within 3 per cent of each other.
_GEMMA = dict(num_hidden_layers=26, hidden_size=2304, num_attention_heads=8, num_key_value_heads=4, head_dim=256,
              intermediate_size=9216, vocab_size=256000, rms_norm_eps=1e-6, rope_theta=10000.0, sliding_window=4096,
              query_pre_attn_scalar=256, attn_logit_softcapping=50.0, final_logit_softcapping=30.0,
              max_position_embeddings=CONTEXT)
_GEMMA_9B = dict(_GEMMA, num_hidden_layers=42, hidden_size=3584, num_attention_heads=16, num_key_value_heads=8,
                 intermediate_size=14336)


def _besulix():
    D, I = 2304, 9216
    left = {"heads": 16, "kv_heads": 4, "dim": 128, "vdim": 128, "scale": 128 ** -0.5, "rot": {"base": 250000.0, "dims": 64},
            "mask": {"size": 1024}}
    par = {"type": "parallel", "mixer": {"left": left, "left_scale": 0.8, "right": {"heads": D // 64, "dim": 64}, "right_scale": 0.9},
           "mlp": {"kind": "dense", "ff": I, "limit": 7.0}}
    mem = {"type": "mlstm", "mixer": {"heads": D // 256, "dim": 128, "vdim": 256, "gate_cap": 15.0}, "mlp": None}
    return {"architecture": "Besulix", "vocab": 256000, "width": D, "norm": {"eps": 1e-6}, "logit_softcap": 30.0,
            "layers": [par if i % 2 == 0 else mem for i in range(6)]}


def _kaderax():
    D, I, heads = 2304, 9216, 18
    lat = {"heads": 16, "dim": 128, "rot_dim": 64, "vdim": 128, "kv_rank": 192, "q_rank": 768, "scale": 192 ** -0.5,
           "rot": {"base": 10000.0, "dims": 64}}
    par = {"left": {"heads": 8, "kv_heads": 4, "dim": 256, "vdim": 256, "scale": 256 ** -0.5, "softcap": 50.0, "bias_max": 128,
                    "q_temp": {"coef": 0.1, "every": 256}}, "left_scale": 0.7,
           "right": {"heads": heads, "dim": 128, "vdim": 128, "decay": [1.0 - 2.0 ** (-1.0 - 8.0 * i / heads) for i in range(heads)]},
           "right_scale": 0.6}
    layers = [{"type": "parallel" if i % 3 == 2 else "latent_attention", "mixer": par if i % 3 == 2 else lat,
               "mlp": {"kind": "dense", "ff": I}} for i in range(9)]
    return {"architecture": "Kaderax", "vocab": 256000, "width": D, "norm": {"eps": 1e-6}, "residual_mult": 0.5, "layers": layers,
            "loop": {"start": 3, "stop": 6, "times": 2}}


_SIZES = {"gemma2-2b": _GEMMA, "gemma2-9b": _GEMMA_9B, "besulix-2b": _besulix(), "kaderax-2b": _kaderax()}


# ---- the cases ------------------------------------------------------------------------------------------------------------
def _lm(model, prompts, new=0, late=0, portion=0, dtype="bfloat16", want="last"):
    """prompts: their lengths; late: the length of a prompt that comes in by `portion` tokens a step while the others go
    on; new: steps of one token for every sequence; want: "last", or "all" for the logits of every prompt row."""
    return {"kind": "lm", "model": model, "dtype": dtype, "prompts": ",".join(str(n) for n in prompts), "late": late,
            "portion": portion, "new": new, "want": want}


def listed():
    cases = {
        # the smallest call: the next tokens of eight running requests, chosen with the default sampling options
        "sample_8": {"kind": "sample", "rows": 8, "vocab": 256000, "temperature": 0.8, "top_k": 256, "top_p": 0.95},
        # one user's short question and its answer: a batch of one, latency and launches
        "chat_1": _lm("gemma2-2b", [23], new=32),
        # the benchmark's batch: eight requests of unequal prompts, then decoding together
        "chat_8": _lm("gemma2-2b", [64, 511, 9, 130, 257, 700, 35, 96], new=32),
        # a server at the batch where its throughput is best: many short requests
        "batch_64": _lm("gemma2-2b", [3 + (i * 29) % 61 for i in range(64)], new=16),
        # a long document arrives while three requests run: portions beside single tokens, past the window of 4,096
        "document": _lm("gemma2-2b", [150, 611, 48], new=16, late=7001, portion=2048),
        # the benchmark's prefill: one prompt of 2,048 tokens, its last row's logits
        "prefill_2048": _lm("gemma2-2b", [2048]),
        # texts of odd lengths are scored: the logits of all rows
        "score_ragged": _lm("gemma2-2b", [333, 97, 1021, 5, 260], want="all"),
        # the largest: four prompts at the 9B sizes, 8,191 tokens in one step
        "prefill_9b": _lm("gemma2-9b", [2048, 1999, 2500, 1644]),
        # eight requests at the 9B sizes: a decode step that is mostly its weights
        "chat_8_9b": _lm("gemma2-9b", [20, 33, 7, 64, 51, 18, 40, 29], new=12),
        # the engine in 32-bit arithmetic, as a check of another run is made: prompts and a few tokens
        "chat_f32": _lm("gemma2-2b", [201, 31, 77], new=8, dtype="float32"),
        # recurrent layers (matrix memory, time mixing) beside chunked attention: the prompts' scans and the states' steps
        "recurrent": _lm("besulix-2b", [700, 333, 64, 1025], new=16),
        # attention through a latent, linear attention beside biased attention, layers run twice
        "latent": _lm("kaderax-2b", [512, 77, 1300, 260], new=16),
    }
    return [dict(c, name=n) for n, c in cases.items()]


def _logint(rng, lo, hi):
    return min(hi, max(lo, int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))))


def draw(rng):
    kind = rng.choice(["sample", "chat", "chat", "batch", "document", "prefill", "score", "chat_9b", "prefill_9b", "f32", "recurrent", "latent"])
    if kind == "sample":
        k = rng.choice([0, 1, _logint(rng, 2, 1024), _logint(rng, 2, 1024)])
        return {"kind": "sample", "rows": _logint(rng, 1, 64), "vocab": _logint(rng, 32000, 256000), "temperature": round(rng.uniform(0.3, 1.5), 2),
                "top_k": k, "top_p": 1.0 if k == 0 else round(rng.uniform(0.5, 1.0), 3)}
    if kind == "chat":
        return _lm("gemma2-2b", [_logint(rng, 4, 700) for _ in range(rng.randint(1, 12))], new=rng.randint(8, 32))
    if kind == "batch":
        return _lm("gemma2-2b", [_logint(rng, 2, 100) for _ in range(rng.randint(13, 64))], new=rng.randint(6, 16))
    if kind == "document":
        return _lm("gemma2-2b", [_logint(rng, 8, 700) for _ in range(rng.randint(0, 6))], new=rng.randint(1, 16),
                   late=rng.randint(1500, 7400), portion=rng.choice([512, 1000, 2048]))
    if kind in ("prefill", "score"):
        most, lengths = (8192 if kind == "prefill" else 2000), []
        for _ in range(rng.randint(1, 8)):
            n = _logint(rng, 5, 4000)
            if sum(lengths) + n <= most:
                lengths.append(n)
        return _lm("gemma2-2b", lengths or [most], want="all" if kind == "score" else "last")
    if kind == "chat_9b":
        return _lm("gemma2-9b", [_logint(rng, 4, 200) for _ in range(rng.randint(1, 16))], new=rng.randint(4, 12))
    if kind == "prefill_9b":
        return _lm("gemma2-9b", [_logint(rng, 300, 2040) for _ in range(rng.randint(1, 4))])
    if kind == "f32":
        return _lm("gemma2-2b", [_logint(rng, 4, 250) for _ in range(rng.randint(1, 4))], new=rng.randint(1, 8), dtype="float32")
    return _lm("besulix-2b" if kind == "recurrent" else "kaderax-2b", [_logint(rng, 8, 1300) for _ in range(rng.randint(1, 4))],
               new=rng.randint(2, 16))


# ---- inputs -----------------------------------------------------------------------------------------------------------------
def _key(seed, name):
    return int.from_bytes(hashlib.sha256(f"{seed}:{name}".encode()).digest()[:7], "little")


def _drawn(seed, name, shape, kind, dtype):
    """A weight as a model folder would hold it: `kind` as the model declares it."""
    g = torch.Generator(device=DEVICE).manual_seed(_key(seed, name))
    t = torch.empty(shape, dtype=torch.float32, device=DEVICE).normal_(0.0, 0.1 if kind in ("norm", "gain") else 0.02, generator=g)
    if kind == "gain":
        t += 1.0
    return t if dtype == "float32" else t.to(torch.bfloat16)


class _Weights:
    """A weight source for `load_into`."""

    def __init__(self, layout, seed, dtype):
        self.layout, self.seed, self.stored = layout, seed, dtype

    def names(self):
        return list(self.layout)

    def shape(self, name):
        return tuple(self.layout[name].shape)

    def dtype(self, name):
        return torch.float32 if self.stored == "float32" else torch.bfloat16

    def tensor(self, name):
        return _drawn(self.seed, name, self.shape(name), self.layout[name].init, self.stored)


def _config(model):
    from trapetum_amd.config import BesulixConfig, Gemma2Config, KaderaxConfig
    sizes = _SIZES[model]
    if model.startswith("gemma2"):
        return Gemma2Config.from_kwargs(**sizes)
    return (BesulixConfig if model.startswith("besulix") else KaderaxConfig).from_dict(sizes)


def _vocab(model):
    s = _SIZES[model]
    return s["vocab_size"] if "vocab_size" in s else s["vocab"]


def _lengths(case):
    return [int(n) for n in case["prompts"].split(",") if n]


def _steps(case):
    """The pass as steps: [(sequence, first position, tokens)] of each; the late prompt is the last sequence."""
    lengths = _lengths(case)
    at = list(lengths)
    steps = [[(i, 0, n) for i, n in enumerate(lengths)]] if lengths else []
    if case["late"]:
        late, o = len(lengths), 0
        while o < case["late"]:
            c = min(case["portion"], case["late"] - o)
            steps.append([(i, at[i], 1) for i in range(late)] + [(late, o, c)])
            at = [p + 1 for p in at]
            o += c
        at.append(o)
    for _ in range(case["new"]):
        steps.append([(i, p, 1) for i, p in enumerate(at)])
        at = [p + 1 for p in at]
    return steps, at                                        # at: each sequence's tokens in the end


def _tokens(case, seed):
    rng = random.Random(_key(seed, "tokens"))
    n = _vocab(case["model"])
    return [[rng.randrange(n) for _ in range(k)] for k in _steps(case)[1]]


def prepare(case, seed):
    if case["kind"] == "sample":
        from trapetum_amd.engine.runtime import Runtime
        from trapetum_amd.sampling.sampler import RequestSampling, Sampler, SamplingParams
        g = torch.Generator(device=DEVICE).manual_seed(_key(seed, "logits"))
        logits = torch.randn((case["rows"], case["vocab"]), generator=g, device=DEVICE) * 2.0
        logits = 30.0 * torch.tanh(logits / 30.0)           # as a capped head leaves them
        params = SamplingParams(temperature=case["temperature"], top_k=case["top_k"], top_p=case["top_p"])
        return {"case": case, "logits": logits, "sampler": Sampler(Runtime(device=DEVICE), params),
                "requests": [RequestSampling(seed, i, [1]) for i in range(case["rows"])]}
    from trapetum_amd.engine import Engine
    from trapetum_amd.engine.model import Model
    from trapetum_amd.engine.runtime import Runtime
    from trapetum_amd.registry import architecture
    from trapetum_amd.weights import load_into
    config = _config(case["model"])
    model = Model(architecture(config.architecture).build_spec(config), Runtime(dtype=case["dtype"], device=DEVICE))
    load_into(model, _Weights(model.tensor_layout(), seed, case["dtype"]))
    steps, totals = _steps(case)
    tokens = _tokens(case, seed)
    engine = Engine(model, config, max_tokens_in_cache=sum(-(-n // 64) * 64 for n in totals), max_context=CONTEXT,
                    max_batch=len(totals))
    plan = [([i for i, _, _ in s], [c for _, _, c in s], [t for i, p, c in s for t in tokens[i][p:p + c]]) for s in steps]
    return {"case": case, "engine": engine, "plan": plan, "sequences": len(totals)}


# ---- one pass ------------------------------------------------------------------------------------------------------------------
def run(state):
    case = state["case"]
    if case["kind"] == "sample":
        return state["sampler"].choose_on_device(state["logits"], state["requests"])
    engine = state["engine"]
    model, cache = engine.model, engine.cache
    slots = [cache.acquire() for _ in range(state["sequences"])]
    out = []
    try:
        first_decode = len(state["plan"]) - case["new"]
        for i, (who, counts, tokens) in enumerate(state["plan"]):
            mine = [slots[s] for s in who]
            if i >= first_decode:                           # its logits lie in the graph's memory until its next step
                out.append(engine.graphed.step(mine, tokens).clone())
            else:
                want = list(range(len(tokens))) if case["want"] == "all" else None
                out.append(model.step(cache, mine, tokens, counts=counts, want=want))
    finally:
        for s in slots:
            cache.release(s)
    return out


# ---- what a pass cannot do without -------------------------------------------------------------------------------------------
def _per_token(model):
    """(elements of the matrices that a token passes through, of the head, [(query width, key/value elements per cached
    token, window) of each attention], multiply-adds of recurrences) of one forward."""
    s = _SIZES[model]
    if model.startswith("gemma2"):
        D, hd, H, G, I, n = (s[k] for k in ("hidden_size", "head_dim", "num_attention_heads", "num_key_value_heads", "intermediate_size", "num_hidden_layers"))
        layer = D * (H + 2 * G) * hd + H * hd * D + 3 * D * I
        return n * layer, s["vocab_size"] * D, [(H * hd * 2, 2 * G * hd, s["sliding_window"] if i % 2 == 0 else None) for i in range(n)], 0
    D, total, attn, rec = s["width"], 0, [], 0
    order, loop = list(range(len(s["layers"]))), s.get("loop")
    if loop:
        order = order[:loop["stop"]] + order[loop["start"]:loop["stop"]] * (loop["times"] - 1) + order[loop["stop"]:]
        total += loop["times"] * 2 * D * D
    for i in order:
        l = s["layers"][i]
        m = l["mixer"]
        if l["mlp"] is not None:
            total += 3 * D * l["mlp"]["ff"]
        if l["type"] == "mlstm":
            H, dk, dv = m["heads"], m["dim"], m["vdim"]
            total += D * (2 * H * dk + 3 * H * dv + 2 * H)
            rec += 3 * H * dk * dv
        elif l["type"] == "latent_attention":
            H, dn, dr, dv, R, Q = m["heads"], m["dim"], m["rot_dim"], m["vdim"], m["kv_rank"], m["q_rank"]
            total += D * (Q + R + dr) + Q * H * (dn + dr) + R * H * (dn + dv) + 2 * D * H * dv
            attn.append((H * (dn + dr + dv), R + dr, None))
        else:
            a, r = m["left"], m["right"]
            H, G, d, dv = a["heads"], a["kv_heads"], a["dim"], a["vdim"]
            total += D * (H * d + G * (d + dv) + H * dv)
            attn.append((H * (d + dv), G * (d + dv), a["mask"]["size"] if "mask" in a else None))
            rd, rv = r["dim"], r.get("vdim", r["dim"])
            total += 3 * D * r["heads"] * rv + 2 * D * r["heads"] * rd
            rec += 3 * r["heads"] * rd * rv
    return total, s["vocab"] * D, attn, rec


def work(case):
    if case["kind"] == "sample":
        n = case["rows"] * case["vocab"]
        return {"bytes": 4 * n, "flops": 2 * n}
    matrices, head, attn, rec = _per_token(case["model"])
    size = 4 if case["dtype"] == "float32" else 2
    vocab = _vocab(case["model"])
    b = f = 0
    for step in _steps(case)[0]:
        rows = sum(c for _, _, c in step)
        wanted = rows if case["want"] == "all" else len(step)
        b += (matrices + head) * size + wanted * vocab * 4
        f += 2 * (rows * (matrices + rec) + wanted * head)
        for width, kept, window in attn:
            for _, start, c in step:
                seen = lambda p: p + 1 if window is None else min(p + 1, window)  # noqa: E731
                b += (min(start, window or start) + c) * kept * size
                f += 2 * width * (c * (seen(start) + seen(start + c - 1)) // 2)
    return {"bytes": b, "flops": f}


# What the widths give: the engine's logits are 0.7 to 1.7 per cent (relative 2-norm) off float64 in bfloat16 after all
# layers, and two implementations that round elsewhere differ by 1.4 times that; in float32 they are 4e-6 to 5e-6 off.  Chosen
# tokens are whole numbers and the same.
def tolerance(case):
    if case["kind"] == "sample":
        return "exact"
    return {"rel": 2e-5, "max": 1e-3} if case["dtype"] == "float32" else {"rel": 0.03, "max": 0.5}


# ---- the same in 64 bits -----------------------------------------------------------------------------------------------------
F64 = torch.float64


def _rms(x, eps):
    return x / torch.sqrt((x * x).mean(-1, keepdim=True) + eps)


def _turn(x, base, dims, neighbours=False, sign=1.0):
    """x [T, heads, n] at positions 0 ..: the first `dims` elements turn in pairs (i, i + dims / 2), or neighbours."""
    half = dims // 2
    a = sign * torch.arange(x.shape[0], dtype=F64, device=x.device)[:, None] * base ** (-2.0 * torch.arange(half, dtype=F64, device=x.device) / dims)
    c, s = torch.cos(a)[:, None], torch.sin(a)[:, None]
    u, v = (x[..., 0:dims:2], x[..., 1:dims:2]) if neighbours else (x[..., :half], x[..., half:dims])
    pair = [u * c - v * s, v * c + u * s]
    turned = torch.stack(pair, -1).flatten(-2) if neighbours else torch.cat(pair, -1)
    return torch.cat([turned, x[..., dims:]], -1)


def _attend(q, k, v, scale, cap=None, visible=None, bias=None, sink=None):
    """q [T, H, d], k [T, G, d], v [T, G, dv]: causal softmax attention, head after head."""
    T, H = q.shape[:2]
    ok = torch.ones(T, T, dtype=torch.bool, device=q.device).tril()
    if visible is not None:
        ok &= visible
    out = torch.empty((T, H, v.shape[2]), dtype=F64, device=q.device)
    for h in range(H):
        g = h // (H // k.shape[1])
        s = (q[:, h] @ k[:, g].t().contiguous()) * scale
        if cap:
            s = cap * torch.tanh(s / cap)
        if bias is not None:
            s = s + bias(h)
        s.masked_fill_(~ok, -math.inf)
        top = s.max(-1, keepdim=True).values
        if sink is not None:
            top = torch.clamp(top, min=float(sink[h]))
        e = torch.exp(s - top)
        z = e.sum(-1, keepdim=True)
        if sink is not None:
            z = z + torch.exp(sink[h] - top)
        out[:, h] = (e / z) @ v[:, g].contiguous()
    return out.flatten(1)


def _gelu(z):
    return 0.5 * z * (1.0 + torch.tanh(math.sqrt(2.0 / math.pi) * (z + 0.044715 * z ** 3)))


def _silu(z):
    return z * torch.sigmoid(z)


def _split(x, parts):
    """Rows of several sequences, packed -> each sequence's."""
    return torch.split(x, parts)


def _gemma_rows(s, w, rows, parts):
    D, H, G, hd, I, eps = (s[k] for k in ("hidden_size", "num_attention_heads", "num_key_value_heads", "head_dim", "intermediate_size", "rms_norm_eps"))
    table = w("model.embed_tokens.weight", (s["vocab_size"], D))
    x = table[rows] * math.sqrt(D)
    norm = lambda v, name: _rms(v, eps) * (1.0 + w(name + ".weight", (D,), "norm"))  # noqa: E731
    for i in range(s["num_hidden_layers"]):
        p = f"model.layers.{i}."
        n = norm(x, p + "input_layernorm")
        q, k, v = (n @ w(p + f"self_attn.{c}_proj.weight", (m * hd, D)).T for c, m in (("q", H), ("k", G), ("v", G)))
        a = []
        for qs, ks, vs in zip(_split(q, parts), _split(k, parts), _split(v, parts)):
            T = qs.shape[0]
            at = torch.arange(T, device=qs.device)
            near = at[:, None] - at[None, :] < s["sliding_window"] if i % 2 == 0 else None
            a.append(_attend(_turn(qs.view(T, H, hd), s["rope_theta"], hd), _turn(ks.view(T, G, hd), s["rope_theta"], hd), vs.view(T, G, hd),
                             s["query_pre_attn_scalar"] ** -0.5, s["attn_logit_softcapping"], near))
        x = x + norm(torch.cat(a) @ w(p + "self_attn.o_proj.weight", (D, H * hd)).T, p + "post_attention_layernorm")
        n = norm(x, p + "pre_feedforward_layernorm")
        m = _gelu(n @ w(p + "mlp.gate_proj.weight", (I, D)).T) * (n @ w(p + "mlp.up_proj.weight", (I, D)).T)
        x = x + norm(m @ w(p + "mlp.down_proj.weight", (D, I)).T, p + "post_feedforward_layernorm")
    x = norm(x, "model.norm")
    return x, table, s["final_logit_softcapping"]


def _besulix_rows(s, w, rows, parts):
    D, eps = s["width"], s["norm"]["eps"]
    x = _rms(w("embed", (s["vocab"], D))[rows], eps) * w("embed.norm", (D,), "gain")

    def chunked(h, p, m):
        H, G, d, dv, C = m["heads"], m["kv_heads"], m["dim"], m["vdim"], m["mask"]["size"]
        base, dims = m["rot"]["base"], m["rot"]["dims"]
        q, k, v = (h @ w(p + c, (n, D)).T + w(p + c + ".b", (n,), "norm") for c, n in (("q", H * d), ("k", G * d), ("v", G * dv)))
        temp, sink = w(p + "temp", (H,), "gain"), w(p + "sink", (H,), "norm")
        out = []
        for qs, ks, vs in zip(_split(q, parts), _split(k, parts), _split(v, parts)):
            T = qs.shape[0]
            c = torch.arange(T, device=h.device) // C
            qs = _turn(qs.view(T, H, d), base, dims) * temp[:, None]
            a = _attend(qs, _turn(ks.view(T, G, d), base, dims), _turn(vs.view(T, G, dv), base, dv), m["scale"],
                        visible=c[:, None] == c[None, :], sink=sink)
            out.append(_turn(a.view(T, H, dv), base, dv, sign=-1.0).flatten(1))
        return torch.cat(out) @ w(p + "o", (D, H * dv)).T

    def time_mix(h, p, m):
        H, d = m["heads"], m["dim"]
        before = torch.cat([torch.cat([torch.zeros_like(t[:1]), t[:-1]]) for t in _split(h, parts)])
        mixed = {c: h + (before - h) * w(p + "mu." + c, (D,), "norm") for c in "rkvgw"}
        r, k, v = ((mixed[c] @ w(p + c, (H * d, D)).T).view(-1, H, d) for c in "rkv")
        gate = _silu(mixed["g"] @ w(p + "g", (H * d, D)).T)
        rank = D // 16
        low = torch.tanh(mixed["w"] @ w(p + "w1", (rank, D)).T) @ w(p + "w2", (H * d, rank)).T
        decay = torch.exp(-torch.exp(low + w(p + "w0", (H * d,), "norm"))).view(-1, H, d)
        u, o, at = w(p + "u", (H, d), "norm"), [], 0
        for n in parts:
            S = torch.zeros((H, d, d), dtype=F64, device=h.device)
            for t in range(at, at + n):
                kv = k[t][:, :, None] * v[t][:, None, :]
                o.append(((S + u[:, :, None] * kv) * r[t][:, :, None]).sum(1))
                S = decay[t][:, :, None] * S + kv
            at += n
        y = _rms(torch.stack(o), eps).flatten(1) * w(p + "norm", (H * d,), "gain") * gate
        return y @ w(p + "o", (D, H * d)).T

    def memory(h, p, m):
        H, dk, dv, cap = m["heads"], m["dim"], m["vdim"], m["gate_cap"]
        q = (h @ w(p + "q", (H * dk, D)).T).view(-1, H, dk) * dk ** -0.5
        k = (h @ w(p + "k", (H * dk, D)).T).view(-1, H, dk)
        v = (h @ w(p + "v", (H * dv, D)).T).view(-1, H, dv)
        gi, gf = (cap * torch.tanh((h @ w(p + c, (H, D)).T + w(p + c + ".b", (H,), "norm")) / cap) for c in "if")
        gf = torch.nn.functional.logsigmoid(gf)
        o, at = [], 0
        for n in parts:
            S = torch.zeros((H, dk, dv), dtype=F64, device=h.device)
            N, top = torch.zeros((H, dk), dtype=F64, device=h.device), torch.zeros(H, dtype=F64, device=h.device)
            for t in range(at, at + n):
                new = torch.maximum(gf[t] + top, gi[t])
                keep, take = torch.exp(gf[t] + top - new), torch.exp(gi[t] - new)
                tk = take[:, None] * k[t]
                S, N, top = keep[:, None, None] * S + tk[:, :, None] * v[t][:, None, :], keep[:, None] * N + tk, new
                den = torch.maximum((N * q[t]).sum(-1).abs(), torch.exp(-top)) + 1e-6
                o.append((S * q[t][:, :, None]).sum(1) / den[:, None])
            at += n
        y = _rms(torch.stack(o), eps).flatten(1) * w(p + "norm", (H * dv,), "gain") * torch.sigmoid(h @ w(p + "g", (H * dv, D)).T)
        return y @ w(p + "o", (D, H * dv)).T

    for i, layer in enumerate(s["layers"]):
        p, m = f"l{i}.", layer["mixer"]
        h = _rms(x, eps) * w(p + "norm1", (D,), "gain")
        if layer["type"] == "mlstm":
            x = x + memory(h, p + "mix.", m)
        else:
            x = x + m["left_scale"] * chunked(h, p + "mix.left.", m["left"]) + m["right_scale"] * time_mix(h, p + "mix.right.", m["right"])
        if layer["mlp"] is not None:
            L, I = layer["mlp"]["limit"], layer["mlp"]["ff"]
            h = _rms(x, eps) * w(p + "norm2", (D,), "gain")
            g = torch.clamp(h @ w(p + "mlp.gate", (I, D)).T, max=L)
            u = torch.clamp(h @ w(p + "mlp.up", (I, D)).T, min=-L, max=L)
            x = x + (g * torch.sigmoid(1.702 * g) * (u + 1.0)) @ w(p + "mlp.down", (D, I)).T
    x = _rms(x, eps) * w("final.norm", (D,), "gain")
    return x, w("head", (s["vocab"], D)), s["logit_softcap"]


def _kaderax_rows(s, w, rows, parts):
    D, eps = s["width"], s["norm"]["eps"]
    start = w("embed", (s["vocab"], D))[rows]

    def latent(h, p, m):
        H, dn, dr, dv, R, Q = m["heads"], m["dim"], m["rot_dim"], m["vdim"], m["kv_rank"], m["q_rank"]
        cq = _rms(h @ w(p + "dq", (Q, D)).T, eps) * w(p + "dq.norm", (Q,), "gain")
        q = cq @ w(p + "uq", (H * (dn + dr), Q)).T
        down = h @ w(p + "dkv", (R + dr, D)).T
        c = _rms(down[:, :R], eps) * w(p + "dkv.norm", (R,), "gain")
        k, v = c @ w(p + "uk", (H * dn, R)).T, c @ w(p + "uv", (H * dv, R)).T
        sink, out = w(p + "sink", (H,), "norm"), []
        for qs, ks, vs, rot in zip(*(_split(t, parts) for t in (q, k, v, down[:, R:]))):
            T = qs.shape[0]
            qs = qs.view(T, H, dn + dr)
            turned = _turn(torch.cat([qs[:, :, dn:], rot.view(T, 1, dr)], 1), m["rot"]["base"], m["rot"]["dims"], neighbours=True)
            out.append(_attend(torch.cat([qs[:, :, :dn], turned[:, :H]], -1),
                               torch.cat([ks.view(T, H, dn), turned[:, H:].expand(T, H, dr)], -1), vs.view(T, H, dv), m["scale"], sink=sink))
        return (torch.cat(out) * torch.sigmoid(h @ w(p + "g", (H * dv, D)).T)) @ w(p + "o", (D, H * dv)).T

    def biased(h, p, m):
        H, G, d, dv = m["heads"], m["kv_heads"], m["dim"], m["vdim"]
        q, k, v = (h @ w(p + c, (n, D)).T for c, n in (("q", H * d), ("k", G * d), ("v", G * dv)))
        table, gate = w(p + "rel", (32, H), "norm"), torch.sigmoid(h @ w(p + "g", (H, D)).T)
        B, out = table.shape[0], []
        for qs, ks, vs in zip(_split(q, parts), _split(k, parts), _split(v, parts)):
            T = qs.shape[0]
            row = [n if n < B // 2 else min(B - 1, B // 2 + int(math.floor(math.log(n / (B // 2)) / math.log(m["bias_max"] / (B // 2)) * (B - B // 2))))
                   for n in range(T)]
            at = torch.arange(T, device=h.device)
            which = torch.tensor(row, device=h.device)[torch.clamp(at[:, None] - at[None, :], min=0)]
            warm = torch.tensor([1.0 + m["q_temp"]["coef"] * math.log((i + 1) // m["q_temp"]["every"] + 1) for i in range(T)], dtype=F64, device=h.device)
            out.append(_attend(qs.view(T, H, d) * warm[:, None, None], ks.view(T, G, d), vs.view(T, G, dv), m["scale"], m["softcap"],
                               bias=lambda hh: table[:, hh][which]))
        y = torch.cat(out).view(-1, H, dv) * gate[:, :, None]
        return y.flatten(1) @ w(p + "o", (D, H * dv)).T

    def linear(h, p, m):
        H, d, dv = m["heads"], m["dim"], m["vdim"]
        q, k, v = (_silu(h @ w(p + c, (H * n, D)).T).view(-1, H, n) for c, n in (("q", d), ("k", d), ("v", dv)))
        out = []
        for qs, ks, vs in zip(_split(q, parts), _split(k, parts), _split(v, parts)):
            at = torch.arange(qs.shape[0], dtype=F64, device=h.device)
            gap = at[:, None] - at[None, :]
            one = [(qs[:, i] @ ks[:, i].t().contiguous() * torch.where(gap >= 0, m["decay"][i] ** gap.clamp(min=0), 0.0)) @ vs[:, i].contiguous() for i in range(H)]
            out.append(torch.cat(one, 1))
        y = _rms(torch.cat(out), eps) * w(p + "norm", (H * dv,), "gain") * torch.sigmoid(h @ w(p + "g", (H * dv, D)).T)
        return y @ w(p + "o", (D, H * dv)).T

    loop, order = s["loop"], [(i, False) for i in range(s["loop"]["start"])]
    for _ in range(loop["times"]):
        order += [(i, i == loop["start"]) for i in range(loop["start"], loop["stop"])]
    order += [(i, False) for i in range(loop["stop"], len(s["layers"]))]
    x, mult = start, s["residual_mult"]
    for i, enters in order:
        p, layer = f"l{i}.", s["layers"][i]
        m = layer["mixer"]
        if enters:
            x = torch.cat([x, start], 1) @ w("loop.in", (D, 2 * D)).T
        h = _rms(x, eps) * w(p + "norm1", (D,), "gain")
        if layer["type"] == "parallel":
            y = m["left_scale"] * biased(h, p + "mix.left.", m["left"]) + m["right_scale"] * linear(h, p + "mix.right.", m["right"])
        else:
            y = latent(h, p + "mix.", m)
        x = x + mult * y
        h = _rms(x, eps) * w(p + "norm2", (D,), "gain")
        I = layer["mlp"]["ff"]
        x = x + mult * ((_gelu(h @ w(p + "mlp.gate", (I, D)).T) * (h @ w(p + "mlp.up", (I, D)).T)) @ w(p + "mlp.down", (D, I)).T)
    return _rms(x, eps) * w("final.norm", (D,), "gain"), w("head", (s["vocab"], D)), None


def exact(case, seed):
    if case["kind"] == "sample":
        return None
    steps, totals = _steps(case)
    s, tokens = _SIZES[case["model"]], _tokens(case, seed)

    def w(name, shape, kind="matrix"):
        return _drawn(seed, name, shape, kind, case["dtype"]).to(F64)

    rows = torch.tensor([t for seq in tokens for t in seq], device=DEVICE)
    forward = {"gemma2": _gemma_rows, "besulix": _besulix_rows, "kaderax": _kaderax_rows}[case["model"].split("-")[0]]
    x, head, cap = forward(s, w, rows, totals)
    first = [sum(totals[:i]) for i in range(len(totals))]
    out = []
    for i, step in enumerate(steps):
        if case["want"] == "all" and i < len(steps) - case["new"]:
            at = [first[q] + p + j for q, p, c in step for j in range(c)]
        else:
            at = [first[q] + p + c - 1 for q, p, c in step]
        z = x[torch.tensor(at, device=DEVICE)] @ head.T
        out.append(z if cap is None else cap * torch.tanh(z / cap))
    return out
