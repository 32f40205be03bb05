"""What this engine's users have it do, as cases that can be timed and checked: steps of `ModelRunner.step`, the call
that every token of a served or replayed request passes through.

A case is one step over a model with random weights.  `decode` requests hold a context in the paged cache and bring one
token each; `prompts` requests bring a whole prompt, or its next portion behind the `prompt_held` tokens that earlier steps
ran; every request gets the logits of its last token.  A pass is that step, and it is the same step every time: the tokens
of requests that hold a context are taken back after it (reserved, run, not committed), the others are released.  The model is loaded once for all states that use it, as a server keeps
one.  The routed designs (experts chosen per token) are left out: in bfloat16 a rounding may choose another expert, so
that no tolerance can be stated for their outputs.
"""
import dataclasses
import gc
import itertools
import math

import numpy as np
import torch

from ginfer_amd import ModelRunner, StepEntry, config_from_dict
from ginfer_amd.parts.model import build_model
from ginfer_amd.weights.random_init import bind_random_weights

DTYPES = {"bfloat16": torch.bfloat16, "float32": torch.float32}
PAGE = 16
WEIGHT_SEED = 0


# ------------------------------------------------------------------------------------------------ the models
def _qwen2(hidden, heads, kv_heads, ff, vocab, theta):
    return dict(architectures=["Qwen2ForCausalLM"], model_type="qwen2", num_hidden_layers=28, hidden_size=hidden,
                num_attention_heads=heads, num_key_value_heads=kv_heads, head_dim=128, intermediate_size=ff, vocab_size=vocab,
                rope_theta=theta, rms_norm_eps=1e-6, tie_word_embeddings=False, max_position_embeddings=32768,
                use_sliding_window=False, sliding_window=4096, max_window_layers=28)


def _titozen():
    """Two recurrent layers (HGRN2) to one of attention over a cached latent, at the 1.5B shape's layer sizes."""
    mlp = dict(kind="dense", ff=8960, limit=7.0)
    recurrent = dict(type="hgrn2", mixer=dict(heads=12, dim=64, vdim=128), mlp=mlp)
    latent = dict(type="latent_attention", mlp=mlp, mixer=dict(heads=12, dim=128, vdim=128, q_rank=768, kv_rank=256,
                                                               scale=128 ** -0.5, mask=dict(size=1024)))
    return dict(architecture="Titozen", vocab=32768, width=1536, norm=dict(eps=1e-5), canon=dict(taps=4),
                layers=[latent if i % 3 == 2 else recurrent for i in range(6)])


def _puguzen():
    """Gated linear attention, retention, and attention over a window and pooled blocks, in turn, at the same sizes."""
    mlp = dict(kind="dense", ff=8960)
    gla = dict(type="gla", mixer=dict(heads=12, dim=64, vdim=128, tau=16.0, rank=64), mlp=mlp)
    retention = dict(type="retention", mlp=mlp, mixer=dict(heads=12, dim=64, vdim=128, rot=dict(base=1e6, dims=64),
                                                           decay=[1.0 - 2.0 ** (-5 - 4.0 * h / 12) for h in range(12)]))
    attention = dict(type="attention", mlp=mlp, mixer=dict(heads=12, kv_heads=2, dim=128, vdim=128, scale=0.1,
                                                           mask=dict(size=1024, pool=64), rot=dict(base=5e5, dims=64)))
    return dict(architecture="Puguzen", vocab=32768, width=1536, norm=dict(eps=1e-5),
                layers=[(gla, retention, attention)[i % 3] for i in range(6)])


# tokens: what the cache holds, room for four states of the largest case or draw of this model
MODELS = {
    "qwen2-1.5b": dict(config=_qwen2(1536, 12, 2, 8960, 151936, 10000.0), tokens=1 << 20),
    "qwen2-7b": dict(config=_qwen2(3584, 28, 4, 18944, 152064, 1e6), tokens=1 << 19),
    "titozen-1.5b": dict(config=_titozen(), tokens=1 << 19),
    "puguzen-1.5b": dict(config=_puguzen(), tokens=1 << 19),
}
MAX_REQUESTS = 320
MAX_LENGTH = 32768

_loaded = {}         # the one model that this process serves: (model, dtype) -> ModelRunner


def _runner(model, dtype):
    key = (model, dtype)
    if key not in _loaded:
        _loaded.clear()
        gc.collect()
        torch.cuda.empty_cache()
        entry = MODELS[model]
        _loaded[key] = ModelRunner(None, dtype=dtype, config=config_from_dict(entry["config"]), random_seed=WEIGHT_SEED,
                                   page_size=PAGE, num_pages=entry["tokens"] // PAGE, max_requests=MAX_REQUESTS,
                                   max_model_len=MAX_LENGTH)
        _Weights(model, dtype, _loaded[key].model).bind()
    return _loaded[key]


class _Weights:
    """The weights of a model, drawn by the engine's generator: the engine's model is bound to them, and by name they are
    64-bit tensors, made when they are asked for.  The Qwen2 shapes get an embedding of unit size and sublayers whose
    outputs are small beside the stream, as trained models have them; with all matrices drawn alike the stream would be
    the sum of its sublayers, and roundings would grow from layer to layer to several percent of the logits."""

    def __init__(self, model, dtype, bound=None):
        self.specs = dict(_unbound(model, dtype).weight_specs())
        self.dtype, self.bound = DTYPES[dtype], bound
        if model.startswith("qwen2"):
            for name, spec in self.specs.items():
                if name.endswith(("o_proj.weight", "down_proj.weight")):
                    self.specs[name] = dataclasses.replace(spec, std=0.02 / math.sqrt(56))
                elif name == "model.embed_tokens.weight":
                    self.specs[name] = dataclasses.replace(spec, std=1.0)

    def bind(self):
        bind_random_weights(self, WEIGHT_SEED, torch.device("cuda"))
        return self

    def weight_specs(self):
        return self.specs

    def bind_weights(self, tensors):
        self.tensors = tensors
        if self.bound is not None:
            self.bound.bind_weights(tensors)

    def __getitem__(self, name):
        return self.tensors[name].to(torch.float64)


def _unbound(model, dtype):
    return build_model(config_from_dict(MODELS[model]["config"]).model_spec(), DTYPES[dtype], device=None)


# ------------------------------------------------------------------------------------------------ the cases
def _case(model, name=None, dtype="bfloat16", decode=0, context_from=0, context_to=0, prompts=0, prompt_from=0, prompt_to=0,
          prompt_held=0):
    c = dict(model=model, dtype=dtype, decode=decode, context_from=context_from, context_to=context_to, prompts=prompts,
             prompt_from=prompt_from, prompt_to=prompt_to, prompt_held=prompt_held)
    return c if name is None else dict(c, name=name)


def listed():
    return [
        # one user in a chat: the time per token that they see
        _case("qwen2-1.5b", "decode_one", decode=1, context_from=2048, context_to=2048),
        # a few users with long chats: the decode step that the benchmark reports
        _case("qwen2-1.5b", "decode_eight", decode=8, context_from=4000, context_to=4090),
        # a busy server: as many requests as the engine runs by default, at all stages of their answers
        _case("qwen2-1.5b", "decode_busy", decode=64, context_from=2048, context_to=3072),
        # questions about long documents
        _case("qwen2-1.5b", "decode_long", decode=4, context_from=13001, context_to=16384),
        # the prompt whose throughput the benchmark reports
        _case("qwen2-1.5b", "prompt_2048", prompts=1, prompt_from=2048, prompt_to=2048),
        # ten chat prompts that arrive together: the time to their first tokens
        _case("qwen2-1.5b", "prompts_chat", prompts=10, prompt_from=13, prompt_to=19),
        # requests that arrive while others are answered
        _case("qwen2-1.5b", "mixed_arrivals", decode=32, context_from=130, context_to=900, prompts=2, prompt_from=101, prompt_to=157),
        # the larger model on a busy server: decode alone, and beside the portion of a longer prompt that fills the step's budget
        _case("qwen2-7b", "decode_7b", decode=64, context_from=300, context_to=1500),
        _case("qwen2-7b", "mixed_7b", decode=48, context_from=300, context_to=1500, prompts=1, prompt_from=2000, prompt_to=2000,
              prompt_held=2048),
        # the true 32-bit path, by which a model's logits are checked: a replayed step of prompts and single tokens
        _case("qwen2-1.5b", "mixed_32bit", dtype="float32", decode=6, context_from=200, context_to=700, prompts=2, prompt_from=61, prompt_to=180),
        # the other designs of mixers: recurrences with a state per request beside attention over a latent, decoded; gated
        # linear attention, retention and pooled attention over a prompt
        _case("titozen-1.5b", "decode_titozen", decode=16, context_from=1000, context_to=2000),
        _case("puguzen-1.5b", "prompt_puguzen", prompts=1, prompt_from=2048, prompt_to=2048),
    ]


def draw(rng):
    def spread(lo, hi):                       # over the logarithm, odd numbers as often as even ones
        return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))
    model, dtype = rng.choice([("qwen2-1.5b", "bfloat16")] * 6 + [("qwen2-7b", "bfloat16")] * 2 +
                              [("qwen2-1.5b", "float32"), ("titozen-1.5b", "bfloat16"), ("puguzen-1.5b", "bfloat16")])
    small = dtype == "float32"
    kind = rng.choice(["decode", "decode", "prompts", "mixed"])
    c = dict(model=model, dtype=dtype)
    if kind != "prompts":
        longest = dict([("qwen2-1.5b", 16384)]).get(model, 2000) if not small else 900
        most_tokens = 64 * 2600 if model == "qwen2-1.5b" and not small else 64 * 900
        c["decode"] = spread(1, 16 if small else 64)
        c["context_to"] = min(spread(100, longest), most_tokens // c["decode"])
        c["context_from"] = max(1, int(c["context_to"] * rng.uniform(0.3, 1.0)))
    if kind != "decode":
        c["prompts"] = spread(1, 4 if small else 10)
        total = spread(8 * c["prompts"], 400 if small else 2000)
        each = total // c["prompts"]
        c["prompt_from"] = max(1, int(each * rng.uniform(0.6, 1.0)))
        c["prompt_to"] = max(c["prompt_from"], 2 * each - c["prompt_from"] if c["prompts"] > 1 else each)
        if rng.random() < 0.3:
            c["prompt_held"] = spread(16, 2048 if not small else 400)
    return _case(**c)


def _lengths(n, lo, hi):
    """n lengths from hi down to lo: ragged ones, as requests have them."""
    return [hi - (hi - lo) * i // max(n - 1, 1) for i in range(n)]


def contexts(case):
    return _lengths(case["decode"], case["context_from"], case["context_to"])


def prompt_lengths(case):
    return _lengths(case["prompts"], case["prompt_from"], case["prompt_to"])


# ------------------------------------------------------------------------------------------------ inputs and passes
_ids = itertools.count()


class State:
    """A model, the requests whose contexts are in its cache and the entries of the step; gives the requests back at its
    end."""

    def __init__(self, runner):
        self.runner, self.held, self.fresh, self.entries = runner, [], [], []

    def __del__(self):
        for rid, _ in self.held:
            self.runner.release(rid)


def _requests(case, seed):
    """[(tokens, how many of them the cache holds)] of the step's requests, the decoding ones first."""
    g = np.random.default_rng(seed)
    vocab = config_from_dict(MODELS[case["model"]]["config"]).model_spec().vocab_size
    sizes = [(n + 1, n) for n in contexts(case)] + [(case["prompt_held"] + n, case["prompt_held"]) for n in prompt_lengths(case)]
    return [(g.integers(0, vocab, n), held) for n, held in sizes]


def prepare(case, seed):
    runner = _runner(case["model"], case["dtype"])
    s = State(runner)
    batch, room = [], 8192                     # contexts are filled in steps of this many tokens
    for ids, held in _requests(case, seed):
        rid, at = next(_ids), 0
        while at < held:
            n = min(room, held - at)
            batch.append(StepEntry(rid, ids[at:at + n]))
            at, room = at + n, room - n
            if room == 0:
                runner.step(batch)
                batch, room = [], 8192
        (s.held.append((rid, len(ids) - held)) if held else s.fresh.append(rid))
        s.entries.append(StepEntry(rid, ids[held:], [len(ids) - held - 1]))
    if batch:
        runner.step(batch)
    return s


def run(state):
    runner, cache = state.runner, state.runner.cache
    for rid, n in state.held:
        cache.append(rid, n)
    logits = runner.step(state.entries, borrow=True)
    for rid, _ in state.held:
        cache.cancel(rid)
    for rid in state.fresh:
        runner.release(rid)
    out = {"first": logits[:1]}                # the rows that `exact` computes by themselves
    if logits.shape[0] > 1:
        out["last"] = logits[-1:]
    if logits.shape[0] > 2:
        out["others"] = logits[1:-1]
    return out


# ------------------------------------------------------------------------------------------------ what a pass needs
def work(case):
    """Weights, the visible part of the cache and the logits once; two operations a weight and token, four a coordinate
    of a visible key's head, and the recurrences' own."""
    d, size = MODELS[case["model"]]["config"], 2 if case["dtype"] == "bfloat16" else 4
    specs = _unbound(case["model"], case["dtype"]).weight_specs()
    embedding = {n: s for n, s in specs.items() if n in ("embed", "model.embed_tokens.weight")}
    (vocab, width), tied = next(iter(embedding.values())).shape, case["model"].startswith("puguzen")
    layers = sum(math.prod(s.shape) for n, s in specs.items() if n not in embedding) - (0 if tied else vocab * width)
    new = [1] * case["decode"] + prompt_lengths(case)
    held = contexts(case) + [case["prompt_held"]] * case["prompts"]
    T, R = sum(new), len(new)
    bytes_ = size * (layers + vocab * width + T * width) + 4 * R * vocab
    flops = 2.0 * T * layers + 2.0 * R * vocab * width

    def pairs(window):                          # visible (token, key) pairs, and keys of the cache that are read
        n = sum(sum(min(h + i + 1, window) for i in range(t)) for t, h in zip(new, held))
        return n, sum(min(h, window) for h in held)
    if case["model"].startswith("qwen2"):
        n, read = pairs(1 << 30)
        per_token = 2 * d["num_key_value_heads"] * 128 * size
        bytes_ += 28 * per_token * (read + T)
        flops += 28 * 4.0 * d["num_attention_heads"] * 128 * n
        return {"bytes": bytes_, "flops": flops}
    n, read = pairs(1024)
    for l in d["layers"]:
        m = l["mixer"]
        if "mask" not in m:                     # a recurrence: its state is read and written, in 32-bit
            state = m["heads"] * m["dim"] * m["vdim"]
            bytes_ += 4 * state * (R + sum(1 for h in held if h))
            flops += 6.0 * state * T
        elif "kv_rank" in m:
            bytes_ += size * m["kv_rank"] * (read + T)
            flops += 4.0 * m["heads"] * 128 * n
        else:
            pooled = sum(sum(max(0, h + i + 1 - 1024) // 64 for i in range(t)) for t, h in zip(new, held))
            bytes_ += 2 * size * m["kv_heads"] * 128 * (read + T + sum(max(0, h - 1024) // 64 for h in held))
            flops += 4.0 * m["heads"] * 128 * (n + pooled)
    return {"bytes": bytes_, "flops": flops}


def tolerance(case):
    """About four times what the engine shows against the same step in 64 bits: activations and cache rounded to
    bfloat16 through all layers, or 32-bit sums throughout."""
    if case["dtype"] == "float32":
        return {"rel": 5e-6}
    return {"rel": {"qwen2-1.5b": 0.01, "qwen2-7b": 0.028, "titozen-1.5b": 0.02, "puguzen-1.5b": 0.025}[case["model"]]}


# ------------------------------------------------------------------------------------------------ the same in 64 bits
F64 = torch.float64


def _unit_rms(x, eps):
    return x / torch.sqrt((x * x).mean(dim=-1, keepdim=True) + eps)


def _angles(frequencies, T):
    """Angles as every implementation of the design makes them: 32-bit positions times 32-bit frequencies."""
    return (torch.arange(T, dtype=torch.float32)[:, None] * frequencies[None, :]).to(device="cuda", dtype=F64)


def _turn_halves(x, angles):
    c, s, half = torch.cos(angles)[:, None], torch.sin(angles)[:, None], angles.shape[1]
    lo, hi = x[..., :half], x[..., half:2 * half]
    return torch.cat([lo * c - hi * s, hi * c + lo * s, x[..., 2 * half:]], dim=-1)


def _turn_neighbours(x, angles):
    c, s, dims = torch.cos(angles)[:, None], torch.sin(angles)[:, None], 2 * angles.shape[1]
    out = x.clone()
    out[..., 0:dims:2] = x[..., 0:dims:2] * c - x[..., 1:dims:2] * s
    out[..., 1:dims:2] = x[..., 1:dims:2] * c + x[..., 0:dims:2] * s
    return out


def _attend(q, k, v, scale, weigh):
    """q [T, H, D] over k, v [T, G, ...], a few hundred tokens and one head at a time; weigh(scores [n, T], rows, head)
    makes the weights of tokens `rows` over all keys."""
    T, H = q.shape[:2]
    out = torch.empty((T, H, v.shape[2]), dtype=F64, device=q.device)
    for h in range(H):
        g = h * k.shape[1] // H
        for a in range(0, T, 2048):
            rows = torch.arange(a, min(a + 2048, T), device=q.device)
            out[rows, h] = weigh((q[rows, h] @ k[:, g].t()) * scale, rows[:, None], h) @ v[:, g]
    return out


def _exact_qwen2(w, d, ids):
    T, eps, hd = len(ids), d["rms_norm_eps"], 128
    j = torch.arange(hd // 2, dtype=torch.float32) / float(hd // 2)
    angles = _angles(1.0 / torch.pow(torch.tensor(d["rope_theta"], dtype=torch.float32), j), T)
    keys = torch.arange(T, device="cuda")[None, :]

    def weigh(s, rows, h):
        return torch.softmax(s.masked_fill_(keys > rows, -math.inf), dim=-1)
    x = w["model.embed_tokens.weight"][ids]
    for i in range(d["num_hidden_layers"]):
        p = "model.layers.%d." % i
        n = _unit_rms(x, eps) * w[p + "input_layernorm.weight"]
        q, k, v = ((n @ w[p + "self_attn.%s_proj.weight" % c].t() + w[p + "self_attn.%s_proj.bias" % c]).view(T, -1, hd) for c in "qkv")
        a = _attend(_turn_halves(q, angles), _turn_halves(k, angles), v, hd ** -0.5, weigh)
        x = x + a.view(T, -1) @ w[p + "self_attn.o_proj.weight"].t()
        n = _unit_rms(x, eps) * w[p + "post_attention_layernorm.weight"]
        g = n @ w[p + "mlp.gate_proj.weight"].t()
        x = x + (g * torch.sigmoid(g) * (n @ w[p + "mlp.up_proj.weight"].t())) @ w[p + "mlp.down_proj.weight"].t()
    return (_unit_rms(x[-1:], eps) * w["model.norm.weight"]) @ w["lm_head.weight"].t()


def _recurrence(q, k, v, decay):
    """S_t = diag(decay_t) S_(t-1) + k_t v_t^T, o_t = S_t^T q_t per head, token by token."""
    S = torch.zeros((q.shape[1], q.shape[2], v.shape[2]), dtype=F64, device=q.device)
    out = torch.empty_like(v)
    for t in range(q.shape[0]):
        S = torch.baddbmm(S * decay[t][:, :, None], k[t][:, :, None], v[t][:, None, :])
        out[t] = (S * q[t][:, :, None]).sum(dim=1)
    return out


def _exact_titozen(w, d, ids):
    T, W, eps = len(ids), d["width"], d["norm"]["eps"]
    keys = torch.arange(T, device="cuda")[None, :]
    even = torch.arange(W // 2, dtype=F64)
    a = _angles(torch.pow(torch.tensor(10000.0, dtype=F64), -2.0 * even / W).to(torch.float32), T)
    x = _unit_rms(w["embed"][ids] + torch.stack([torch.sin(a), torch.cos(a)], dim=-1).view(T, W), eps) * w["embed.norm"]
    for i, l in enumerate(d["layers"]):
        p, m = "l%d." % i, l["mixer"]
        H, D, V = m["heads"], m["dim"], m["vdim"]
        taps = w[p + "canon1"]
        h = x + sum(taps[:, j] * torch.cat([x.new_zeros((taps.shape[1] - 1 - j, W)), x])[:T] for j in range(taps.shape[1]))
        mix = lambda name, u=None: (h if u is None else u) @ w[p + "mix." + name].t()      # noqa: E731
        if l["type"] == "hgrn2":
            low = w[p + "mix.lower"]
            f = (low + (1 - low) * torch.sigmoid(mix("f") + w[p + "mix.f.b"])).view(T, H, D)
            o = _recurrence(torch.nn.functional.silu(mix("q")).view(T, H, D), 1 - f, mix("v").view(T, H, V), f)
            o = _unit_rms(o, eps) * w[p + "mix.norm"]
        else:
            cq = _unit_rms(mix("dq"), eps) * w[p + "mix.dq.norm"]
            c = _unit_rms(mix("dkv"), eps) * w[p + "mix.dkv.norm"]
            sink = w[p + "mix.sink"]

            def weigh(s, rows, head):
                s = s.masked_fill_((keys > rows) | (keys <= rows - m["mask"]["size"]), -math.inf)
                return torch.softmax(torch.cat([s, sink[head].expand(s.shape[0], 1)], dim=1), dim=-1)[:, :T]
            o = _attend(mix("uq", cq).view(T, H, D), mix("uk", c).view(T, H, D), mix("uv", c).view(T, H, V), m["scale"], weigh)
            o = o * torch.sigmoid(mix("g"))[:, :, None]
        x = x + _unit_rms(mix("o", o.reshape(T, H * V)), eps) * w[p + "norm1"]
        L = l["mlp"]["limit"]
        g, u = torch.clamp(x @ w[p + "mlp.gate"].t(), max=L), torch.clamp(x @ w[p + "mlp.up"].t(), -L, L)
        x = x + _unit_rms((g * torch.sigmoid(1.702 * g) * (u + 1)) @ w[p + "mlp.down"].t(), eps) * w[p + "norm2"]
    return (_unit_rms(x[-1:], eps) * w["final.norm"]) @ w["head"].t()


def _exact_puguzen(w, d, ids):
    T, eps = len(ids), d["norm"]["eps"]

    def angles(rot):
        return _angles(torch.tensor([rot["base"] ** (-2.0 * i / rot["dims"]) for i in range(rot["dims"] // 2)]).to(torch.float32), T)
    x = w["embed"][ids]
    for i, l in enumerate(d["layers"]):
        p, m = "l%d." % i, l["mixer"]
        H, D, V = m["heads"], m["dim"], m["vdim"]
        n = _unit_rms(x, eps) * (1 + w[p + "norm1"])
        mix = lambda name: n @ w[p + "mix." + name].t()                                    # noqa: E731
        q, k, v = mix("q").view(T, H, D), mix("k").view(T, -1, D), mix("v").view(T, -1, V)
        if l["type"] == "gla":
            z = mix("a1") @ w[p + "mix.a2"].t() + w[p + "mix.a2.b"]
            decay = torch.sigmoid(z).pow(1.0 / m["tau"]).view(T, H, D)
            o = _unit_rms(_recurrence(q / math.sqrt(D), k, v, decay), eps) * w[p + "mix.norm"]
        elif l["type"] == "retention":
            a = angles(m["rot"])
            decay = torch.tensor(m["decay"], dtype=F64, device="cuda")[None, :, None].expand(T, H, D)
            o = _unit_rms(_recurrence(_turn_halves(q, a), _turn_halves(k, a) / math.sqrt(D), v, decay), eps)
        else:
            a, size, pool, bias = angles(m["rot"]), m["mask"]["size"], m["mask"]["pool"], w[p + "mix.pb"]
            q, k = _unit_rms(_turn_neighbours(q, a), eps), _unit_rms(_turn_neighbours(k, a), eps)
            blocks = T // pool
            k, v = (torch.cat([u, u[:blocks * pool].view(blocks, pool, u.shape[1], u.shape[2]).mean(dim=1)]) for u in (k, v))
            token, last = torch.arange(T, device="cuda")[None, :], torch.arange(1, blocks + 1, device="cuda")[None, :] * pool - 1

            def weigh(s, rows, head):
                seen = torch.cat([(token <= rows) & (token > rows - size), last <= rows - size], dim=1)
                return torch.sigmoid(s + bias[head]) * seen
            o = _attend(q, k, v, m["scale"], weigh)
        g = mix("g")
        o = o.reshape(T, H * V) * (torch.sigmoid(g) if l["type"] == "attention" else g * torch.sigmoid(g))
        mixed = o @ w[p + "mix.o"].t()
        ff = (torch.relu(n @ w[p + "mlp.gate"].t()) * (n @ w[p + "mlp.up"].t())) @ w[p + "mlp.down"].t()
        x = x + torch.sigmoid(n @ w[p + "rg1"].t() + w[p + "rg1.b"]) * mixed + torch.sigmoid(n @ w[p + "rg2"].t() + w[p + "rg2.b"]) * ff
    return (_unit_rms(x[-1:], eps) * (1 + w["final.norm"])) @ w["embed"].t()


def exact(case, seed):
    """The first and the last request's logits, each request recomputed as a whole sequence; the other rows have none."""
    every = [ids for ids, _ in _requests(case, seed)]
    forward = {"qwen2": _exact_qwen2, "titozen": _exact_titozen, "puguzen": _exact_puguzen}[case["model"].split("-")[0]]
    w, d = _Weights(case["model"], case["dtype"]).bind(), MODELS[case["model"]]["config"]
    rows = [forward(w, d, torch.from_numpy(ids).to("cuda")) for ids in ([every[0], every[-1]] if len(every) > 1 else every)]
    out = dict(zip(("first", "last"), rows))
    if len(every) > 2:
        out["others"] = None
    return out
