"""What this library's speed is measured on: requests to a Llama engine through ``Engine.step`` and ``Engine.sample``.

A serving process loads a model once and then answers requests, so a state holds one request (or a batch of
requests that start together) beside the process's engine, and a pass answers it from its first prompt token to its
last logits: slots are taken, the prompts run (in one packed step, or in portions), every further token is a
decode step that returns its logits, and the slots are given back. The tokens that are fed are the request's own
(as a caller does who replays, scores or samples by rules of its own); the float32 cases pick them with the engine's
sampler instead. The sizes are those of ``bench.py``: the layers of Llama-3.2-1B, Llama-3.2-3B and Llama-3.1-8B, all
of them, with random weights.
"""
import functools
import math
import zlib

import numpy as np
import torch

import gpullama3_java_amd as g


def _config(hidden, intermediate, layers, heads, head_dim, factor, tied):
    return {"architectures": ["LlamaForCausalLM"], "vocab_size": 128256, "hidden_size": hidden, "intermediate_size": intermediate,
            "num_hidden_layers": layers, "num_attention_heads": heads, "num_key_value_heads": 8, "head_dim": head_dim,
            "max_position_embeddings": 131072, "rms_norm_eps": 1e-5, "rope_theta": 500000.0, "hidden_act": "silu",
            "tie_word_embeddings": tied,
            "rope_scaling": {"rope_type": "llama3", "factor": factor, "low_freq_factor": 1.0, "high_freq_factor": 4.0,
                             "original_max_position_embeddings": 8192}}


SHAPES = {"1b": _config(2048, 8192, 16, 32, 64, 32.0, True),
          "3b": _config(3072, 8192, 28, 24, 128, 32.0, True),
          "8b": _config(4096, 14336, 32, 32, 128, 8.0, False)}
CACHE_TOKENS = {"1b": 65536, "3b": 32768, "8b": 32768}
SLOTS = 64


# ------------------------------------------------------------------------------------------------ the cases
def _request(name, shape, lengths, new=0, chunk=0, want="last", dtype="bfloat16", greedy=False):
    """``lengths``: the prompts' lengths; ``new``: decode steps; ``chunk``: a prompt comes in portions of that many tokens;
    ``want``: logits of the last token of a prompt or of all; ``greedy``: the sampler picks the tokens that are fed."""
    return {"name": name, "kind": "request", "shape": shape, "dtype": dtype, "lengths": ",".join(str(n) for n in lengths), "new": new,
            "chunk": chunk, "want": want, "greedy": greedy}


def _spread(n, lo, hi):
    """n lengths from lo to hi, evenly spread over their logarithm, in an order that mixes short and long ones."""
    got = [int(round(lo * (hi / lo) ** (i / max(1, n - 1)))) for i in range(n)]
    return [got[(i * 37) % n] for i in range(n)] if math.gcd(37, n) == 1 else got


def listed():
    return [
        # one token for each of eight requests, picked by temperature and top-p from their logits
        {"name": "sample_8", "kind": "sample", "shape": "1b", "dtype": "bfloat16", "rows": 8, "temperature": 0.8, "top_p": 0.95},
        # a short question to a small model, one user: prompt latency, then 32 tokens one by one
        _request("turn_1b", "1b", [37], new=32),
        # the benchmark's batch: eight users with 512-token prompts
        _request("batch8_1b", "1b", [512] * 8, new=32),
        # a busy server: 64 users with short prompts of unequal lengths
        _request("batch64_1b", "1b", _spread(64, 24, 200), new=24),
        # a prompt of the usual size, first token wanted
        _request("prompt_1b", "1b", [2048]),
        # texts whose every token is scored
        _request("score_1b", "1b", [317, 1203, 701], want="all"),
        # a long document and a few tokens about it
        _request("long_1b", "1b", [16384], new=16),
        # eight requests of very unequal lengths in one packed step, then decode
        _request("unequal8_3b", "3b", [1752, 96, 1390, 211, 803, 1101, 377, 156], new=16),
        # a document that comes in portions (the cache holds what came before), then a question about it
        _request("portions_3b", "3b", [4543], chunk=512, new=4),
        # the largest model: one user's turn, and its longest prompt
        _request("turn_8b", "8b", [150], new=16),
        _request("prompt_8b", "8b", [8192]),
        # the true 32-bit path: two prompts, the next tokens picked by the engine
        _request("float32_1b", "1b", [333, 180], new=16, dtype="float32", greedy=True),
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["sample", "turn", "batch", "batch", "prompt", "prompt", "score", "portions", "float32"])
    shape = rng.choice(["1b", "1b", "1b", "3b", "3b", "8b"])
    most = {"1b": 16384, "3b": 8192, "8b": 6144}[shape]         # prompt tokens of a request
    if kind == "sample":
        case = {"kind": "sample", "shape": "1b", "dtype": "bfloat16", "rows": _log(rng, 1, 64), "temperature": round(rng.uniform(0.5, 1.2), 2),
                "top_p": rng.choice([0.9, 0.95, 0.98])}
        return case
    if kind == "turn":
        case = _request("", shape, [_log(rng, 5, 700)], new=rng.randint(8, 32))
    elif kind == "batch":
        n = _log(rng, 2, 64)
        longest = max(40, most // (2 * n))
        case = _request("", shape, [_log(rng, 16, longest) for _ in range(n)], new=rng.randint(8, 24))
    elif kind == "prompt":
        case = _request("", shape, [_log(rng, 16, most)], new=rng.choice([0, 0, 4]))
    elif kind == "score":
        case = _request("", shape, [_log(rng, 32, 1200) for _ in range(rng.randint(1, 4))], want="all")
    elif kind == "portions":
        case = _request("", shape, [_log(rng, 1000, most // 2)], chunk=rng.randint(200, 1100), new=rng.randint(0, 8))
    else:
        case = _request("", "1b", [_log(rng, 8, 256) for _ in range(rng.randint(1, 4))], new=rng.randint(2, 12), dtype="float32", greedy=True)
    del case["name"]
    return case


# ------------------------------------------------------------------------------------------------ what a program has in hand
def _std(c, name):
    """How widely a matrix is drawn: 0.02, the embedding and the head 0.05 (logits of 2 to 3, as trained models have), and
    the matrices whose products go into the residual rows so narrowly that all layers together change a row about
    as much as the row was to begin with. (Drawn with 0.02 as well, every layer would drown what came before it, and
    rounding to 16 bits would grow from layer to layer to several per cent, which says nothing about a kernel.)"""
    if "embed" in name or "lm_head" in name:
        return 0.05
    if "o_proj" in name or "down_proj" in name:
        total = 0.5 * 0.02 * math.sqrt(c["hidden_size"] * c["intermediate_size"] * c["num_hidden_layers"])
        return 0.05 / total * (4.0 if "o_proj" in name else 1.0)
    return 0.02


def _tensor(shape, dtype, name, size):
    """A weight: N(0, _std) for a matrix, 1 + N(0, 0.1) for a norm's vector, from the model and the name alone."""
    gen = torch.Generator(device="cuda").manual_seed(zlib.crc32((shape + ":" + name).encode()))
    t = torch.empty(size, dtype=torch.bfloat16, device="cuda")
    if len(size) == 1:
        t = (1.0 + 0.1 * torch.randn(size, generator=gen, device="cuda")).to(torch.bfloat16)
    else:
        t.normal_(0.0, _std(SHAPES[shape], name), generator=gen)
    return t.to(getattr(torch, dtype))


def _layer_sizes(c):
    d, F, q, kv = c["hidden_size"], c["intermediate_size"], c["num_attention_heads"] * c["head_dim"], c["num_key_value_heads"] * c["head_dim"]
    return {"input_layernorm": (d,), "self_attn.q_proj": (q, d), "self_attn.k_proj": (kv, d), "self_attn.v_proj": (kv, d),
            "self_attn.o_proj": (d, q), "post_attention_layernorm": (d,), "mlp.gate_proj": (F, d), "mlp.up_proj": (F, d),
            "mlp.down_proj": (d, F)}


def _outer_sizes(c):
    out = {"model.embed_tokens.weight": (c["vocab_size"], c["hidden_size"]), "model.norm.weight": (c["hidden_size"],)}
    if not c["tie_word_embeddings"]:
        out["lm_head.weight"] = (c["vocab_size"], c["hidden_size"])
    return out


@functools.lru_cache(maxsize=None)
def _engine(shape, dtype):
    """The process's engine for a model: loaded once, used for every request."""
    c = SHAPES[shape]
    sizes = dict(_outer_sizes(c))
    for i in range(c["num_hidden_layers"]):
        sizes.update({f"model.layers.{i}.{k}.weight": v for k, v in _layer_sizes(c).items()})
    weights = {name: _tensor(shape, dtype, name, size) for name, size in sizes.items()}
    return g.Engine(g.config_from_dict(c), weights, dtype=dtype, device="cuda:0", max_tokens=CACHE_TOKENS[shape], n_slots=SLOTS)


def _tokens(case, seed):
    """The request's tokens: one list a sequence, its prompt and what is fed after it."""
    rng = np.random.default_rng([int(seed), 77])
    vocab = SHAPES[case["shape"]]["vocab_size"]
    return [rng.integers(0, vocab, int(n) + case["new"]).tolist() for n in case["lengths"].split(",")]


def _logits(case, seed):
    """Logits as a trained model's are: a long tail and some tokens well above it."""
    gen = torch.Generator(device="cuda").manual_seed(int(seed))
    rows, vocab = case["rows"], SHAPES[case["shape"]]["vocab_size"]
    x = 2.0 * torch.randn(rows, vocab, generator=gen, device="cuda")
    at = torch.randint(0, vocab, (rows, 40), generator=gen, device="cuda")
    return x.scatter(1, at, 10.0 + 3.0 * torch.randn(rows, 40, generator=gen, device="cuda"))


def prepare(case, seed):
    engine = _engine(case["shape"], case["dtype"])
    if case["kind"] == "sample":
        rng = np.random.default_rng([int(seed), 78])
        n = case["rows"]
        return {"case": case, "engine": engine, "logits": _logits(case, seed), "temperatures": [case["temperature"]] * n,
                "top_ps": [case["top_p"]] * n, "uniforms": rng.random(n).astype(np.float32).tolist()}
    tokens = _tokens(case, seed)
    prompts = [t[:int(n)] for t, n in zip(tokens, case["lengths"].split(","))]
    fed = [t[len(p):] for t, p in zip(tokens, prompts)]
    return {"case": case, "engine": engine, "prompts": prompts, "fed": fed}


# ------------------------------------------------------------------------------------------------ a pass
def run(state):
    case, engine = state["case"], state["engine"]
    if case["kind"] == "sample":
        return engine.sample(state["logits"], state["temperatures"], state["top_ps"], state["uniforms"])
    prompts, fed = state["prompts"], state["fed"]
    slots = [engine.take_slot() for _ in prompts]
    logits, picked = [], []
    try:
        if case["chunk"]:
            (prompt,) = prompts
            cuts = list(range(0, len(prompt), case["chunk"]))
            for lo in cuts[:-1]:
                engine.step([(slots[0], prompt[lo:lo + case["chunk"]])], want="none")
            logits.append(engine.step([(slots[0], prompt[cuts[-1]:])]))
        else:
            logits.append(engine.step(list(zip(slots, prompts)), want=case["want"]))
        for k in range(case["new"]):
            if case["greedy"]:
                nxt = engine.sample(logits[-1], [0.0] * len(slots), [1.0] * len(slots), [0.0] * len(slots))
                picked.append(nxt)
            else:
                nxt = [f[k] for f in fed]
            logits.append(engine.step([(s, [t]) for s, t in zip(slots, nxt)]))
    finally:
        for s in slots:
            engine.give_back_slot(s)
    return {"logits": logits, "picked": picked} if case["greedy"] else logits


# ------------------------------------------------------------------------------------------------ what a pass cannot do without
def work(case):
    c = SHAPES[case["shape"]]
    if case["kind"] == "sample":
        return {"bytes": 4.0 * case["rows"] * (c["vocab_size"] + 1), "flops": 0.0}
    es = 2 if case["dtype"] == "bfloat16" else 4
    L, V, d = c["num_hidden_layers"], c["vocab_size"], c["hidden_size"]
    layers = L * sum(int(np.prod(s)) for s in _layer_sizes(c).values())
    head = V * d
    kv = 2 * L * c["num_key_value_heads"] * c["head_dim"]                   # elements a cached token holds
    attn = 4 * L * c["num_attention_heads"] * c["head_dim"]                 # flops a pair of query and key takes
    nbytes = flops = 0.0

    def step(counts, before, rows):
        nonlocal nbytes, flops
        T = sum(counts)
        pairs = sum(n * b + n * (n + 1) // 2 for n, b in zip(counts, before))
        nbytes += es * (layers + (head if rows else 0) + T * d + kv * (sum(before) + T)) + 4.0 * rows * V
        flops += 2.0 * layers * T + 2.0 * head * rows + float(attn) * pairs

    lengths = [int(n) for n in case["lengths"].split(",")]
    if case["chunk"]:
        (n,) = lengths
        for lo in range(0, n, case["chunk"]):
            k = min(case["chunk"], n - lo)
            step([k], [lo], 1 if lo + k == n else 0)
    else:
        step(lengths, [0] * len(lengths), sum(lengths) if case["want"] == "all" else len(lengths))
    for k in range(case["new"]):
        step([1] * len(lengths), [n + k for n in lengths], len(lengths))
    return {"bytes": nbytes, "flops": flops}


# ------------------------------------------------------------------------------------------------ how far results may be off
def tolerance(case):
    if case["kind"] == "sample":
        return "exact"                              # the same definition, the same uniform number: the same token
    if case["dtype"] == "float32":
        return {"rel": 1e-5, "max": 1e-4, "differ": 0.0}         # (2e-6 from the 64-bit logits over 16 layers)
    # bfloat16 rows through all layers: 0.0037 to 0.0062 from the 64-bit logits, four times that where two roundings meet
    return {"rel": 0.02, "max": 0.15}


def _rotation(c, n):
    """cos and sin [n, head_dim / 2] by the model's definition: frequency and angle in float32, then in 64 bits."""
    f32, r = np.float32, c["rope_scaling"]
    freq = np.zeros(c["head_dim"] // 2, dtype=f32)
    for j in range(c["head_dim"] // 2):
        f = f32(1.0 / math.pow(c["rope_theta"], 2 * j / c["head_dim"]))
        old, lo, hi = (f32(r[k]) for k in ("original_max_position_embeddings", "low_freq_factor", "high_freq_factor"))
        length = f32(2.0 * math.pi / float(f))
        if length > f32(old / lo):
            f = f32(f / f32(r["factor"]))
        elif length >= f32(old / hi):
            smooth = f32(f32(f32(old / length) - lo) / f32(hi - lo))
            f = f32(f32(f32(f32(1.0) - smooth) * f / f32(r["factor"])) + f32(smooth * f))
        freq[j] = f
    angle = torch.from_numpy((np.arange(n, dtype=f32)[:, None] * freq[None, :]).astype(np.float64)).cuda()
    return angle.cos(), angle.sin()


def _plain(case, seqs, rows):
    """The decoder in 64 bits over whole sequences: logits at ``rows[b]`` of sequence b, one tensor a sequence."""
    c, shape, dtype = SHAPES[case["shape"]], case["shape"], case["dtype"]
    hs, H, G = c["head_dim"], c["num_attention_heads"], c["num_key_value_heads"]
    cuts = np.cumsum([0] + [len(s) for s in seqs])
    cos, sin = _rotation(c, max(len(s) for s in seqs))
    at = torch.cat([torch.arange(len(s)) for s in seqs]).cuda()
    cos, sin = cos[at][:, None, :], sin[at][:, None, :]

    def weight(name, size):
        return _tensor(shape, dtype, name, size).double()

    def norm(x, w):
        return x * torch.rsqrt(x.square().mean(-1, keepdim=True) + c["rms_norm_eps"]) * w

    def rotate(x):
        a, b = x[..., :hs // 2], x[..., hs // 2:]
        return torch.cat([a * cos - b * sin, b * cos + a * sin], -1)

    sizes = _layer_sizes(c)
    table = _tensor(shape, dtype, "model.embed_tokens.weight", _outer_sizes(c)["model.embed_tokens.weight"])
    x = table[torch.tensor([t for s in seqs for t in s], device="cuda")].double()
    for i in range(c["num_hidden_layers"]):
        w = {k: weight(f"model.layers.{i}.{k}.weight", v) for k, v in sizes.items()}
        h = norm(x, w["input_layernorm"])
        q = rotate((h @ w["self_attn.q_proj"].T).view(-1, H, hs))
        k = rotate((h @ w["self_attn.k_proj"].T).view(-1, G, hs))
        v = (h @ w["self_attn.v_proj"].T).view(-1, G, hs)
        o = torch.empty_like(q)
        for lo, hi in zip(cuts[:-1], cuts[1:]):
            for first in range(lo, hi, 2048):
                last = min(hi, first + 2048)
                hidden = torch.arange(lo, last, device="cuda")[None, :] > torch.arange(first, last, device="cuda")[:, None]
                for head in range(H):
                    kv = head // (H // G)
                    s = (q[first:last, head] @ k[lo:last, kv].T) / math.sqrt(hs)
                    o[first:last, head] = torch.softmax(s.masked_fill_(hidden, -math.inf), -1) @ v[lo:last, kv]
        x = x + o.reshape(-1, H * hs) @ w["self_attn.o_proj"].T
        h = norm(x, w["post_attention_layernorm"])
        x = x + (torch.nn.functional.silu(h @ w["mlp.gate_proj"].T) * (h @ w["mlp.up_proj"].T)) @ w["mlp.down_proj"].T
    x = norm(x, weight("model.norm.weight", (c["hidden_size"],)))
    head = (table if c["tie_word_embeddings"] else _tensor(shape, dtype, "lm_head.weight", _outer_sizes(c)["lm_head.weight"])).double()
    return [x[lo + torch.tensor(r, device="cuda")] @ head.T for lo, r in zip(cuts[:-1], rows)]


def exact(case, seed):
    """What ``run`` returns, in 64 bits, by plain torch. The float32 cases feed the tokens that these logits pick."""
    if case["kind"] == "sample":
        return None
    tokens, lengths = _tokens(case, seed), [int(n) for n in case["lengths"].split(",")]
    if not case["greedy"]:
        whole = case["want"] == "all"
        rows = [list(range(n)) if whole else list(range(n - 1, n + case["new"])) for n in lengths]
        got = _plain(case, tokens, rows)
        return [torch.cat(got)] if whole else [torch.stack([x[k] for x in got]) for k in range(1 + case["new"])]
    seqs = [t[:n] for t, n in zip(tokens, lengths)]
    logits = []
    for _ in range(1 + case["new"]):
        logits.append(torch.cat(_plain(case, seqs, [[len(s) - 1] for s in seqs])))
        seqs = [s + [int(t)] for s, t in zip(seqs, logits[-1].argmax(-1).tolist())]
    return {"logits": logits, "picked": [x.argmax(-1).tolist() for x in logits[:-1]]}
