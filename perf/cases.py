"""What this framework is used for, as cases that can be timed and compared: prompts, generation, serving and sampling through
the public entry points (``Llama`` and its relatives, sessions, ``ContinuousBatcher``, ``sample_next_token``).

A case is a dict of plain values; ``prepare`` makes what a program holds before the call, ``run`` is the call, ``exact`` the
same outputs from plain torch in 64 bits.  Models are the repository's benchmark sizes with random weights.  A trained model's
next token is mostly decided, one with independent random weights is not: its best two logits lie within one bf16 step every
few dozen tokens.  So token embeddings are large against the layers' contributions and the vocabulary projection holds
them in another order: every token has one likely successor, about 20 % to 90 % of the probability.
"""

import math
import random

import torch
import torch.nn.functional as F

from ohara_amd.batching import ContinuousBatcher
from ohara_amd.bitnet import BitLlama
from ohara_amd.llama import Config, Llama
from ohara_amd.phi import Phi, PhiConfig
from ohara_amd.sampling import SamplingConfig, sample_next_token

DEV = "cuda"
BF16 = torch.bfloat16

# The sizes of this repository's benchmark: the d12 Llama that its headline is quoted on, a wider Llama with grouped heads,
# the ternary Llama, the mixture of experts and Phi-2.
MODELS = {
    "d12": dict(vocab_size=65536, hidden_size=768, intermediate_size=3072, num_attention_heads=6, num_hidden_layers=12,
                max_sequence_length=4096),
    "gqa": dict(vocab_size=32000, hidden_size=2048, intermediate_size=5632, num_attention_heads=16, num_key_value_heads=4,
                num_hidden_layers=8, max_sequence_length=4608),
    "bitnet": dict(vocab_size=32000, hidden_size=2048, intermediate_size=5632, num_attention_heads=16, num_hidden_layers=24,
                   max_sequence_length=2048),
    "moe": dict(vocab_size=32000, hidden_size=1024, intermediate_size=512, num_attention_heads=16, num_hidden_layers=16,
                max_sequence_length=2048, moe_num_experts=64, moe_experts_per_tok=8, moe_grouped=True,
                moe_num_shared_experts=1),
    "phi2": dict(vocab_size=51200, hidden_size=2560, num_attention_heads=32, num_hidden_layers=32, max_sequence_length=2048),
}
BIT_LINEARS = ("attn.key", "attn.query", "attn.value", "attn.proj", "ff.gate", "ff.up", "ff.down")


def listed():
    return [
        # the choice of one token with the chat defaults (temperature 0.8, top-p 0.95): once per token of every reply
        dict(name="sample_chat", task="sample", batch=1, vocab=65536, temperature=0.8, top_k=0, top_p=0.95),
        # the time to the first token of a short question
        dict(name="prompt_short", task="prompt", model="d12", batch=1, prompt=128),
        # eight prompts at once: the throughput of reading
        dict(name="prompt_batch", task="prompt", model="d12", batch=8, prompt=1024),
        # a document of odd length, most of the context window
        dict(name="prompt_long", task="prompt", model="gqa", batch=1, prompt=4001),
        # the next turn of four conversations, every position's logits (scoring, or drafts to be checked)
        dict(name="next_turn", task="extend", model="gqa", batch=4, prompt=1900, new=48),
        # one user's reply: the headline workload's prompt and context window
        dict(name="reply_one", task="generate", model="d12", batch=1, prompt=1024, new=64),
        # a batch of replies
        dict(name="reply_batch", task="generate", model="d12", batch=32, prompt=512, new=32),
        # the same over the int8 cache, for the memory it saves
        dict(name="reply_int8", task="generate", model="gqa", batch=16, prompt=700, new=32, int8=True),
        # replies of the ternary model, the mixture of experts and Phi-2, the last two driven token by token
        dict(name="reply_bitnet", task="generate", model="bitnet", batch=1, prompt=300, new=24),
        dict(name="reply_moe", task="generate", model="moe", batch=24, prompt=160, new=12),
        dict(name="reply_phi", task="generate", model="phi2", batch=1, prompt=700, new=8),
        # a server's slots: sixteen prompts of different lengths join, and are decoded together
        dict(name="serve", task="serve", model="d12", batch=16, prompt=800, new=16),
    ]


def _spread(rng, low, high):
    """A whole number between the two, even over its logarithm."""
    return min(high, max(low, round(math.exp(rng.uniform(math.log(low), math.log(high + 0.5))))))


def _one(rng):
    task = rng.choice(["sample", "prompt", "prompt", "extend", "generate", "generate", "int8", "serve"])
    if task == "sample":
        k = rng.choice([0, 0, 50])
        return dict(task="sample", batch=_spread(rng, 1, 64), vocab=rng.choice([32000, 51200, 65536]),
                    temperature=rng.choice([0.8, 1.0]), top_k=k, top_p=rng.choice([0.9, 0.95]))
    if task == "prompt":
        model = rng.choice(["d12", "d12", "gqa", "gqa", "moe", "phi2"])
        window = MODELS[model]["max_sequence_length"]
        batch = _spread(rng, 1, 8)
        return dict(task=task, model=model, batch=batch, prompt=_spread(rng, 16, min(window - 8, 8192 // batch)))
    if task == "extend":
        model = rng.choice(["d12", "gqa"])
        return dict(task=task, model=model, batch=_spread(rng, 1, 8), prompt=_spread(rng, 200, 3500), new=_spread(rng, 2, 200))
    if task == "int8":
        return dict(task="generate", model=rng.choice(["d12", "gqa"]), batch=_spread(rng, 1, 16), prompt=_spread(rng, 16, 1024),
                    new=_spread(rng, 4, 32), int8=True)
    if task == "serve":
        return dict(task=task, model=rng.choice(["d12", "gqa"]), batch=_spread(rng, 2, 24), prompt=_spread(rng, 64, 1024),
                    new=_spread(rng, 4, 16))
    model, most = rng.choice([("d12", 32), ("d12", 32), ("gqa", 16), ("bitnet", 8), ("moe", 24), ("phi2", 2)])
    slow = model in ("bitnet", "moe", "phi2")
    return dict(task=task, model=model, batch=_spread(rng, 1, most), prompt=_spread(rng, 16, 400 if slow else 1024),
                new=_spread(rng, 2, 12 if slow else 64))


def _cost(case):
    w = work(case)
    return w["bytes"] / 5e12 + w["flops"] / 5e14


def draw(rng):
    most = max(_cost(c) for c in listed())
    while True:
        case = _one(rng)
        if _cost(case) <= most:
            return case


# -- models ---------------------------------------------------------------------------------------------------------------


def _numbers(name):
    """width, feed-forward width, heads, key / value heads, head width, layers, vocabulary"""
    c = MODELS[name]
    d, H = c["hidden_size"], c["num_attention_heads"]
    return (d, c.get("intermediate_size", 4 * d), H, c.get("num_key_value_heads") or H, d // H, c["num_hidden_layers"],
            c["vocab_size"])


def _weights(name):
    """A state dict under the names that the constructors take."""
    d, ff, H, G, D, layers, vocab = _numbers(name)
    g = torch.Generator(device=DEV).manual_seed(11)

    def n(*shape, std=0.02):
        return torch.randn(*shape, generator=g, device=DEV, dtype=torch.float32).mul_(std).to(BF16)

    back = 0.02 / math.sqrt(2 * layers)  # the projections that add to the stream, as models of this kind are initialised
    one = lambda k: (1 + 0.1 * torch.randn(k, generator=g, device=DEV)).to(BF16)  # noqa: E731
    emb = n(vocab, d, std=1.0)
    successor = torch.randperm(vocab, generator=g, device=DEV)
    head = torch.empty_like(emb)
    head[successor] = (emb.float() * (14.0 / d)).to(BF16)
    if name == "phi2":
        w = {"wte.weight": emb, "lm_head.weight": head, "lm_head.bias": n(vocab), "ln.weight": one(d), "ln.bias": n(d)}
        for i in range(layers):
            p = f"layers.{i}."
            w[p + "ln.weight"], w[p + "ln.bias"] = one(d), n(d)
            for m, (rows, cols) in {"mixer.q_proj": (d, d), "mixer.k_proj": (d, d), "mixer.v_proj": (d, d), "mixer.dense": (d, d),
                                    "mlp.fc1": (ff, d), "mlp.fc2": (d, ff)}.items():
                w[p + m + ".weight"] = n(rows, cols, std=back if m in ("mixer.dense", "mlp.fc2") else 0.02)
                w[p + m + ".bias"] = n(rows)
        return w
    w = {"token_emb.weight": emb, "vocab_proj.weight": head, "norm.weight": one(d)}
    # the rotary tables, rounded to bf16 as a model moved to bf16 rounds its buffers
    span = torch.arange(2 * MODELS[name]["max_sequence_length"]).float()
    angle = torch.outer(span, 1.0 / (100000.0 ** (torch.arange(0, D, 2).float() / D)))
    w["freq_cos"], w["freq_sin"] = torch.cos(angle).to(DEV, BF16), torch.sin(angle).to(DEV, BF16)
    shapes = {"attn.key": (G * D, d), "attn.query": (H * D, d), "attn.value": (G * D, d), "attn.proj": (d, H * D),
              "ff.gate": (ff, d), "ff.up": (ff, d), "ff.down": (d, ff)}
    for i in range(layers):
        p = f"layers.{i}."
        w[p + "norm1.weight"], w[p + "norm2.weight"] = one(d), one(d)
        for m, (rows, cols) in shapes.items():
            if name == "bitnet":
                w[p + m + ".ternary"] = torch.randint(-1, 2, (rows, cols), device=DEV, generator=g, dtype=torch.int8)
                w[p + m + ".gamma"] = torch.tensor(0.004)
                w[p + m + ".rms_norm.weight"] = one(cols)
            elif name != "moe" or m.startswith("attn"):
                w[p + m + ".weight"] = n(rows, cols, std=back if m in ("attn.proj", "ff.down") else 0.02)
        if name == "moe":
            E = MODELS[name]["moe_num_experts"]
            w[p + "ff.w_gate"], w[p + "ff.w_up"], w[p + "ff.w_down"] = n(E, d, ff), n(E, d, ff), n(E, ff, d, std=back)
            w[p + "ff.router.weight"] = n(E, d, std=1.0 / math.sqrt(d))
            w[p + "ff.router_bias"] = torch.zeros(E, device=DEV, dtype=BF16)
            w[p + "ff.shared_gate.weight"], w[p + "ff.shared_up.weight"] = n(ff, d), n(ff, d)
            w[p + "ff.shared_down.weight"] = n(d, ff, std=back)
    return w


_loaded = {}


def _model(name):
    """A program loads its model once and answers every request with it."""
    if name not in _loaded:
        w = _weights(name)
        if name == "phi2":
            _loaded[name] = Phi(PhiConfig(**MODELS[name]), w, device=DEV)
        else:
            _loaded[name] = (BitLlama if name == "bitnet" else Llama)(Config(**MODELS[name]), w, device=DEV)
    return _loaded[name]


# -- the cases ------------------------------------------------------------------------------------------------------------

GREEDY = SamplingConfig(temperature=0)


def _ids(case, seed):
    """Token ids of the prompt, and of what follows it."""
    g = torch.Generator(device=DEV).manual_seed(seed)
    vocab = MODELS[case["model"]]["vocab_size"]
    return torch.randint(0, vocab, (case["batch"], case["prompt"] + case.get("new", 0)), generator=g, device=DEV)


def _lengths(case):
    """A server's prompts: anything from an eighth of the longest to the longest."""
    rng = random.Random(case["prompt"])
    return [rng.randint(max(1, case["prompt"] // 8), case["prompt"]) for _ in range(case["batch"])]


def _logits_to_sample(case, seed):
    """A language model's logits: a wide bell and a few dozen tokens far above it."""
    g = torch.Generator(device=DEV).manual_seed(seed)
    B, V = case["batch"], case["vocab"]
    x = torch.randn(B, V, generator=g, device=DEV) * 2.0
    likely = torch.randint(0, V, (B, 40), generator=g, device=DEV)
    x.scatter_add_(1, likely, 14.0 - 3.0 * torch.arange(1, 41, device=DEV).float().log().expand(B, 40))
    return x.to(BF16).view(B, 1, V), torch.rand(B, generator=g, device=DEV)


def prepare(case, seed):
    task = case["task"]
    if task == "sample":
        logits, u = _logits_to_sample(case, seed)
        rule = SamplingConfig(temperature=case["temperature"], top_k=case["top_k"], top_p=case["top_p"])
        return dict(case=case, logits=logits, u=u, rule=rule)
    model, ids = _model(case["model"]), _ids(case, seed)
    B, P, new = case["batch"], case["prompt"], case.get("new", 0)
    s = dict(case=case, model=model, prompt=ids[:, :P].contiguous(), more=ids[:, P:].contiguous())
    if task == "serve":
        s["prompts"] = [row[:n].cpu() for row, n in zip(s["prompt"], _lengths(case))]
        s["batcher"] = ContinuousBatcher(model, B)
        return s
    s["cache"] = model.build_kv_cache(B, int8=case.get("int8", False))
    if task == "extend":
        model(s["prompt"], s["cache"], 0, last_only=True)
    elif task == "generate" and hasattr(model, "session"):
        # an engine keeps its session, with the captured graphs in it, from one request to the next
        s["session"] = model.session(B, new, kv_cache=s["cache"])
        s["session"].prefill(s["prompt"])
        if new > 1:
            s["session"].run(1)
    return s


def _rewind(cache, length):
    """Back to the first ``length`` tokens: a new request, or an edited turn."""
    for c in cache:
        c.length, c.lengths = length, None
        if length == 0:
            c.batch_size = None


def _answer(case, cache, length, **out):
    """The outputs, and the state a call leaves: the last layer's keys and values, which rest on every earlier layer's.  (Rows
    in int8 codes are left out: a code moves by one with the last bit of what it stands for.)"""
    if not case.get("int8"):
        out["keys"], out["values"] = cache[-1].key[:, :length], cache[-1].value[:, :length]
    return out


def run(s):
    case = s["case"]
    task = case["task"]
    if task == "sample":
        return sample_next_token(s["logits"], s["rule"], u=s["u"])
    P, new, model = case["prompt"], case.get("new", 0), s["model"]
    if task == "prompt":
        _rewind(s["cache"], 0)
        return _answer(case, s["cache"], P, logits=model(s["prompt"], s["cache"], 0, last_only=True))
    if task == "extend":
        _rewind(s["cache"], P)
        return _answer(case, s["cache"], P + new, logits=model(s["more"], s["cache"], P))
    if task == "serve":
        b = s["batcher"]
        for slot in range(case["batch"]):
            if b.active[slot]:
                b.remove(slot)
        first = b.add_many(s["prompts"])
        rest = b.steps(new - 1) if new > 1 else {}
        tokens = torch.tensor([[tok, *rest.get(slot, [])] for slot, tok in first])
        return dict(tokens=tokens, keys=[b.cache[-1].key[slot, :n] for slot, n in enumerate(b.lengths)],
                    values=[b.cache[-1].value[slot, :n] for slot, n in enumerate(b.lengths)])
    if "session" in s:
        sess = s["session"]
        sess.restart()
        sess.prefill(s["prompt"])
        sess.run(new - 1)
        return _answer(case, s["cache"], P + new - 1, tokens=sess.tokens(), logits=sess.logits)
    # a model without a session: one call per token
    cache, feed, at, tokens = s["cache"], s["prompt"], 0, []
    _rewind(cache, 0)
    for _ in range(new):
        logits = model(feed, cache, at, last_only=True)
        at += feed.shape[1]
        feed = sample_next_token(logits, GREEDY)
        tokens.append(feed)
    return _answer(case, cache, at, tokens=torch.cat(tokens, 1), logits=logits)


# -- what a pass cannot do without ----------------------------------------------------------------------------------------


def work(case):
    if case["task"] == "sample":
        return {"bytes": 2 * case["batch"] * case["vocab"], "flops": 0}
    name, B, P, new = case["model"], case["batch"], case["prompt"], case.get("new", 0)
    d, ff, H, G, D, layers, vocab = _numbers(name)
    attn = d * D * (2 * H + 2 * G)
    ffn = 2 * d * ff if name == "phi2" else 3 * d * ff
    active, E = attn + ffn, 0
    if name == "moe":
        k, E = MODELS[name]["moe_experts_per_tok"], MODELS[name]["moe_num_experts"]
        active = attn + (k + 1) * ffn + E * d

    def weights(tokens):  # bytes of one call over so many tokens
        if name == "bitnet":
            return layers * (attn + ffn) / 4 + 2 * vocab * d
        if name == "moe":
            touched = E * (1 - (1 - k / E) ** tokens)
            return 2 * (layers * (attn + (touched + 1) * ffn + E * d) + vocab * d)
        return 2 * (layers * active + vocab * d)

    row = layers * 2 * G * (D + 8 if case.get("int8") else 2 * D)  # a position's keys and values

    def call(sequences, start, tokens, rows_out):  # bytes and flops of one call of the model
        pairs = sequences * (tokens * start + tokens * (tokens + 1) / 2)
        by = weights(sequences * tokens) + row * sequences * (start + tokens) + 2 * sequences * (tokens * d + rows_out * vocab)
        return by, 2 * sequences * (tokens * layers * active + rows_out * vocab * d) + 4 * layers * H * D * pairs

    if case["task"] == "extend":
        calls = [call(B, P, new, new)]
    elif case["task"] == "prompt":
        calls = [call(B, 0, P, 1)]
    elif case["task"] == "serve":  # lengths run from an eighth of the longest to the longest
        mean = (P / 8 + P) / 2
        calls = [call(1, 0, mean, 1)] * B + [call(B, mean + i, 1, 1) for i in range(new - 1)]
    else:
        calls = [call(B, 0, P, 1)] + [call(B, P + i, 1, 1) for i in range(new - 1)]
    return {"bytes": sum(c[0] for c in calls), "flops": sum(c[1] for c in calls)}


def tolerance(case):
    if case["task"] == "sample":
        return "exact"
    # Measured at these sizes: bf16 activations leave the logits 0.005 to 0.01 off 64 bits, and the same tokens in two calls
    # instead of one (sums in another order) 0.004 off each other, a few values 0.1.  An int8 code that rounds the other way
    # moves its whole row in the ternary model, an expert that wins by a hair the token's in the mixture of experts.
    return {"rel": 0.03, "max": 0.5, "differ": 0.01} if case["model"] in ("bitnet", "moe") else {"rel": 0.02, "max": 0.3, "differ": 0.01}


# -- the same in 64 bits --------------------------------------------------------------------------------------------------


def _rms(x, w):
    return x * torch.rsqrt(x.square().mean(-1, keepdim=True) + 1e-5) * w.double()


class _Plain:
    """A model's forward pass in 64 bits, over caches that are lists of [keys, values] of shape (B, heads, length, D)."""

    def __init__(self, case):
        self.name, self.int8 = case["model"], case.get("int8", False)
        self.w = _weights(self.name)
        self.d, self.ff, self.H, self.G, self.D, self.layers, self.vocab = _numbers(self.name)

    def cache(self):
        return [[None, None] for _ in range(self.layers)]

    def linear(self, name, x):
        if name + ".ternary" in self.w:
            x = _rms(x, self.w[name + ".rms_norm.weight"])
            s = 127.0 / x.abs().amax(-1, keepdim=True).clamp(min=1e-5)
            x = (x * s).round().clamp(-128, 127) / s
            return x @ self.w[name + ".ternary"].double().t() * float(self.w[name + ".gamma"])
        y = x @ self.w[name + ".weight"].double().t()
        return y + self.w[name + ".bias"].double() if name + ".bias" in self.w else y

    def heads(self, x, n):
        B, S, _ = x.shape
        return x.view(B, S, n, self.D).transpose(1, 2)

    def rotate(self, x, start):
        c, s = (self.w[t][start:start + x.shape[2]].double() for t in ("freq_cos", "freq_sin"))
        e, o = x[..., 0::2], x[..., 1::2]
        return torch.stack([e * c - o * s, e * s + o * c], -1).flatten(-2)

    def rotate_phi(self, x):  # the first 40 % of a head's features, the two halves of them paired
        n = int(0.4 * self.D)
        half = n // 2
        rate = torch.exp(-torch.arange(0.0, half, device=x.device) * (math.log(10000.0) / half))
        angle = (torch.arange(x.shape[2], device=x.device).float().view(-1, 1) * rate).float()
        c, s = angle.cos().double(), angle.sin().double()
        a, b = x[..., :half], x[..., half:n]
        return torch.cat([a * c - b * s, a * s + b * c, x[..., n:]], -1)

    def stored(self, x):
        if not self.int8:
            return x
        low, high = x.amin(-1, keepdim=True), x.amax(-1, keepdim=True)
        step = ((high - low) / 255).clamp(min=1e-8)
        return ((x - low) / step - 128).round().clamp(-128, 127).add(128) * step + low

    def attend(self, p, x, kv, start):
        phi = self.name == "phi2"
        names = ("mixer.q_proj", "mixer.k_proj", "mixer.v_proj", "mixer.dense") if phi else ("attn.query", "attn.key",
                                                                                            "attn.value", "attn.proj")
        q, k, v = (self.heads(self.linear(p + m, x), n) for m, n in zip(names, (self.H, self.G, self.G)))
        if not phi:
            q, k = self.rotate(q, start), self.rotate(k, start)
        k, v = self.stored(k), self.stored(v)
        kv[0], kv[1] = (new if old is None else torch.cat([old, new], 2) for old, new in zip(kv, (k, v)))
        k, v = kv
        if phi:
            q = self.rotate_phi(F.pad(q, (0, 0, start, 0)))[:, :, start:]
            k = self.rotate_phi(k)
        B, S, L = x.shape[0], x.shape[1], k.shape[2]
        hidden = torch.arange(L, device=DEV) > start + torch.arange(S, device=DEV).view(-1, 1)
        out = torch.empty(B, S, self.H * self.D, dtype=torch.float64, device=DEV)
        for b in range(B):
            for g in range(self.G):
                qs = slice(g * (self.H // self.G), (g + 1) * (self.H // self.G))
                score = (q[b, qs] @ k[b, g].t() / math.sqrt(self.D)).masked_fill(hidden, -math.inf)
                out[b, :, qs.start * self.D:qs.stop * self.D] = (score.softmax(-1) @ v[b, g]).transpose(0, 1).flatten(1)
        return self.linear(p + names[3], out)

    def experts(self, p, x):
        rows = x.reshape(-1, self.d)
        best = (rows @ self.w[p + "ff.router.weight"].double().t()).topk(MODELS[self.name]["moe_experts_per_tok"])
        share, y = best.values.softmax(-1), torch.zeros_like(rows)
        for e in range(MODELS[self.name]["moe_num_experts"]):
            at, nth = (best.indices == e).nonzero(as_tuple=True)
            gate, up, down = (self.w[p + m][e].double() for m in ("ff.w_gate", "ff.w_up", "ff.w_down"))
            r = rows[at]
            y.index_add_(0, at, (F.silu(r @ gate) * (r @ up)) @ down * share[at, nth, None])
        z = F.silu(self.linear(p + "ff.shared_gate", rows)) * self.linear(p + "ff.shared_up", rows)
        return (y + self.linear(p + "ff.shared_down", z)).view_as(x)

    def __call__(self, ids, cache, start):
        w = self.w
        if self.name == "phi2":
            x = w["wte.weight"][ids].double()
            norm = lambda t, p: F.layer_norm(t, (self.d,), w[p + "weight"].double(), w[p + "bias"].double(), 1e-5)  # noqa: E731
            for i in range(self.layers):
                p = f"layers.{i}."
                h = norm(x, p + "ln.")
                x = x + self.attend(p, h, cache[i], start) + self.linear(
                    p + "mlp.fc2", F.gelu(self.linear(p + "mlp.fc1", h), approximate="tanh"))
            return lambda rows: self.linear("lm_head", norm(x[:, rows], "ln."))
        x = w["token_emb.weight"][ids].double()
        for i in range(self.layers):
            p = f"layers.{i}."
            x = x + self.attend(p, _rms(x, w[p + "norm1.weight"]), cache[i], start)
            h = _rms(x, w[p + "norm2.weight"])
            x = x + (self.experts(p, h) if self.name == "moe" else self.linear(
                p + "ff.down", F.silu(self.linear(p + "ff.gate", h)) * self.linear(p + "ff.up", h)))
        return lambda rows: self.linear("vocab_proj", _rms(x[:, rows], w["norm.weight"]))

    def generate(self, prompt, new):
        """(tokens, the last step's logits, the cache)"""
        cache, feed, at, tokens = self.cache(), prompt, 0, []
        for _ in range(new):
            logits = self(feed, cache, at)(slice(-1, None))
            at += feed.shape[1]
            feed = logits.argmax(-1)
            tokens.append(feed)
        return torch.cat(tokens, 1), logits, cache


def _rows(cache):
    """The last layer's keys and values in the order of a cache's tensors."""
    return (t.transpose(1, 2) for t in cache[-1])


@torch.no_grad()
def exact(case, seed):
    task = case["task"]
    if task == "sample":
        return None  # whole numbers
    plain, ids, P, new = _Plain(case), _ids(case, seed), case["prompt"], case.get("new", 0)
    if task == "serve":
        out = [plain.generate(ids[b:b + 1, :n], new) for b, n in enumerate(_lengths(case))]
        keys, values = zip(*((t[0] for t in _rows(cache)) for _, _, cache in out))
        return dict(tokens=torch.cat([t for t, _, _ in out]).cpu(), keys=list(keys), values=list(values))
    if task == "generate":
        tokens, logits, cache = plain.generate(ids[:, :P], new)
        out = dict(tokens=tokens, logits=logits[:, 0] if case["model"] in ("d12", "gqa", "bitnet") else logits)
    else:
        cache = plain.cache()
        logits = plain(ids[:, :P], cache, 0)
        out = dict(logits=plain(ids[:, P:], cache, P)(slice(None)) if task == "extend" else logits(slice(-1, None)))
    if not case.get("int8"):
        out["keys"], out["values"] = _rows(cache)
    return out
