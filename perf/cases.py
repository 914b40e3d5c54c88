"""The work that programs have this engine do, as cases that can be timed: decode steps, prompts and mixed steps.

Every case is one step of a serving loop through the engine's public pieces: a batch of ``StepEntry`` goes through the
step function (``Engine.runner``, or ``Engine.graphs`` for a step of single tokens, as ``Engine.step`` chooses), the
sampler turns the logits into tokens on the device, and nobody waits.  A pass leaves the books as it found them (a
prompt's pages go back, a decoded token's position is taken again), so that it can be repeated.

Models have the layer sizes of the presets (``llama-3.2-1b``, ``llama-3.2-3b``, ``llama-3.1-8b``) with a part of the
layers, and ``mogisun-linear``: the Mogisun design with gated linear attention at the 3B shape's widths and dense
feed-forwards.  Fewer layers than the models have keep what rounding to bfloat16 does to the logits small enough to
tell it from a mistake (the error grows with depth); the work of a layer is what it is at full depth.  For the same
reason weights are drawn as models are initialised for training, so that a layer adds to the stream and does not
replace it: N(0, 0.02), the products that end a sublayer narrower by the root of twice the layers, embeddings N(0, 0.1),
gains 1 + N(0, 0.1); token ids are uniform.  Routed experts are left out of the cases: with random weights
a rounding difference changes which expert a token takes now and then, and with it the logits by more than any tolerance.
The sampled tokens are not among the outputs for the same reason: the two best of 128,256 random logits nearly tie in
every twentieth row.

A case: ``model``, ``layers``, ``dtype``; ``rows`` requests that bring one token each, over contexts around ``context``
tokens (``ragged``: from half to one and a half times as many, else all equal); ``prompt`` tokens of one further request
over ``past`` earlier ones; ``want``: logits of the ``last`` place of each request or of ``all``; ``sampling``:
``greedy`` or ``filtered`` (temperature, top-k, top-p).
"""

import math

import torch

VOCAB = 128256
PAGE = 16

_SHAPES = {
    # hidden, query heads, key/value heads, head size, feed-forward, rope factor, tied head
    "llama-3.2-1b": (2048, 32, 8, 64, 8192, 32.0, True),
    "llama-3.2-3b": (3072, 24, 8, 128, 8192, 32.0, True),
    "llama-3.1-8b": (4096, 32, 8, 128, 14336, 8.0, False),
    "mogisun-linear": (3072, 24, 24, 128, 8192, None, False),
}
_RANK, _TAU, _CAP = 64, 16.0, 30.0       # of the linear attention's decays; the cap of its model's logits
_EPS = 1e-5


def _case(model, layers, rows=0, context=0, ragged=False, prompt=0, past=0, dtype="bfloat16", want="last", sampling="greedy"):
    return {"model": model, "layers": layers, "dtype": dtype, "rows": rows, "context": context, "ragged": ragged,
            "prompt": prompt, "past": past, "want": want, "sampling": sampling}


def listed():
    named = [
        # one user at the start of a chat with the smallest model: the shortest step there is, latency and launches
        ("decode 1 row of 40", _case("llama-3.2-1b", 8, rows=1, context=40)),
        # the headline: eight users with 2,048-token contexts
        ("decode 8 rows of 2048", _case("llama-3.2-3b", 8, rows=8, context=2048)),
        # a full server: 64 users whose contexts differ, sampled as chat programs sample
        ("decode 64 ragged rows", _case("llama-3.2-3b", 4, rows=64, context=2048, ragged=True, sampling="filtered")),
        # a server in the middle of its day: an odd number of users, between the few-row products and the full batch
        ("decode 27 ragged rows", _case("llama-3.2-1b", 8, rows=27, context=700, ragged=True, sampling="filtered")),
        # a few users with long documents: the cache is most of what a step reads
        ("decode 3 rows of 12000", _case("llama-3.1-8b", 4, rows=3, context=12000, ragged=True)),
        # the headline's prompt: 2,048 tokens in one step
        ("prompt 2048", _case("llama-3.2-3b", 8, prompt=2048)),
        # a long document run as one step, of a size that divides nothing
        ("prompt 7001", _case("llama-3.1-8b", 4, prompt=7001)),
        # a chat turn: a short prompt of odd size
        ("prompt 45", _case("llama-3.2-3b", 8, prompt=45, sampling="filtered")),
        # continuous batching: a portion of 449 tokens over 1,024 beside 63 decoding users (512 tokens a step)
        ("63 rows beside 449 of a prompt", _case("llama-3.2-1b", 8, rows=63, context=700, ragged=True, prompt=449, past=1024)),
        # trace replay in the 32-bit path: logits at every place, decoded tokens beside a portion
        ("float32 3 rows beside 300", _case("llama-3.2-1b", 4, rows=3, context=200, ragged=True, prompt=300, dtype="float32", want="all")),
        # linear attention with a state: a prompt, and eight users decoding
        ("linear prompt 2048", _case("mogisun-linear", 4, prompt=2048)),
        ("linear decode 8 rows", _case("mogisun-linear", 4, rows=8, context=500, ragged=True)),
    ]
    return [dict(c, name=name) for name, c in named]


def draw(rng):
    """A step of one of the kinds above: sizes spread over their logarithm, odd ones as likely as even ones."""
    size = lambda lo, hi: int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))
    model, layers = rng.choice([("llama-3.2-1b", 8), ("llama-3.2-3b", 8), ("llama-3.1-8b", 4), ("llama-3.2-3b", 8),
                                ("mogisun-linear", 4)])
    sampling = rng.choice(["greedy", "filtered"])
    kind = rng.choice(["decode", "decode", "prompt", "prompt", "mixed", "float32"])
    if model == "mogisun-linear":      # its states cannot go back to before a portion: decode or whole prompts
        kind = "decode" if kind == "decode" else "prompt"
    if kind == "prompt":
        past = 0 if model == "mogisun-linear" or rng.random() < 0.7 else size(16, 8192)
        top = 7001 if past == 0 else 2048
        return _case(model, layers, prompt=size(2, 4096 if model == "mogisun-linear" else top), past=past, sampling=sampling)
    if kind == "float32":
        return _case("llama-3.2-1b", 4, rows=rng.randint(1, 8), context=size(16, 600), ragged=True,
                     prompt=rng.choice([0, size(2, 600)]), dtype="float32", want="all", sampling=sampling)
    if kind == "mixed":
        rows = size(1, 63)
        return _case(model, layers, rows=rows, context=size(64, 1500), ragged=True, prompt=size(16, 2048), past=rng.choice([0, size(16, 2048)]),
                     sampling=sampling)
    rows = size(1, 64)
    most = 1500 if model == "mogisun-linear" else min(16000, 120000 // rows)
    return _case(model, layers, rows=rows, context=size(16, most), ragged=rng.random() < 0.7, sampling=sampling)


# ---------------------------------------------------------------------------------------------------------
# the model's configuration and weights
# ---------------------------------------------------------------------------------------------------------

def _config(case):
    from simple_inference_amd import preset

    if case["model"] != "mogisun-linear":
        return dict(preset(case["model"]), num_hidden_layers=case["layers"])
    width, heads, _, dim, ff, _, _ = _SHAPES["mogisun-linear"]
    layer = {"type": "gla", "mixer": {"dim": dim, "vdim": dim, "heads": heads, "tau": _TAU, "rank": _RANK},
             "mlp": {"kind": "dense", "ff": ff}}
    return {"architecture": "Mogisun", "vocab": VOCAB, "width": width, "norm": {"eps": _EPS}, "logit_scale": 1.0,
            "logit_softcap": _CAP, "loop": {"start": 0, "stop": case["layers"], "times": 1},
            "layers": [layer] * case["layers"]}


def _weight_shapes(case):
    """Checkpoint name -> shape; one number for a gain or a bias, two for a matrix."""
    hidden, heads, kv, dim, ff, _, tied = _SHAPES[case["model"]]
    if case["model"] == "mogisun-linear":
        out = {"embed": (VOCAB, hidden), "loop.in": (hidden, 2 * hidden), "final.norm": (hidden,), "head": (VOCAB, hidden)}
        for i in range(case["layers"]):
            p = f"l{i}."
            for name in ("q", "k", "v", "g"):
                out[p + "mix." + name] = (heads * dim, hidden)
            out.update({p + "mix.o": (hidden, heads * dim), p + "mix.norm": (dim,), p + "mix.a1": (_RANK, hidden),
                        p + "mix.a2": (heads * dim, _RANK), p + "mix.a2.b": (heads * dim,),
                        p + "norm1": (hidden,), p + "norm2": (hidden,),
                        p + "mlp.gate": (ff, hidden), p + "mlp.up": (ff, hidden), p + "mlp.down": (hidden, ff)})
            for name in ("rg1", "rg2"):
                out.update({p + name: (hidden, hidden), p + name + ".b": (hidden,)})
        return out
    out = {"model.embed_tokens.weight": (VOCAB, hidden), "model.norm.weight": (hidden,)}
    if not tied:
        out["lm_head.weight"] = (VOCAB, hidden)
    for i in range(case["layers"]):
        p = f"model.layers.{i}."
        out.update({
            p + "input_layernorm.weight": (hidden,), p + "post_attention_layernorm.weight": (hidden,),
            p + "self_attn.q_proj.weight": (heads * dim, hidden), p + "self_attn.k_proj.weight": (kv * dim, hidden),
            p + "self_attn.v_proj.weight": (kv * dim, hidden), p + "self_attn.o_proj.weight": (hidden, heads * dim),
            p + "mlp.gate_proj.weight": (ff, hidden), p + "mlp.up_proj.weight": (ff, hidden), p + "mlp.down_proj.weight": (hidden, ff)})
    return out


def _weights(case, seed):
    """bfloat16 weights (as checkpoints hold them) in one fixed order from one generator on the GPU."""
    gen = torch.Generator(device="cuda")
    gen.manual_seed(1000003 * seed + 17)
    out = {}
    for name, shape in _weight_shapes(case).items():
        t = torch.empty(shape, dtype=torch.bfloat16, device="cuda").normal_(0.0, 1.0, generator=gen)
        if len(shape) == 2:
            ends = name.endswith((".o", ".down", "o_proj.weight", "down_proj.weight"))
            t.mul_(0.1 if "embed" in name else 0.02 / math.sqrt(2 * case["layers"]) if ends else 0.02)
        elif name.endswith(".b"):
            t.mul_(0.1)
        else:
            t.mul_(0.1).add_(1.0)
        out[name] = t
    return out


def _tokens(case, seed):
    """([tokens of each decoding request: its context and the token that the pass brings], the prompt's past, the prompt)."""
    gen = torch.Generator()
    gen.manual_seed(7919 * seed + 5)
    lengths = [case["context"]] * case["rows"]
    if case["ragged"]:
        half = max(1, case["context"] // 2)
        lengths = [half + int(torch.randint(0, case["context"] + 1, (1,), generator=gen)) for _ in lengths]
    ids = lambda n: torch.randint(0, VOCAB, (n,), generator=gen).tolist()
    return [ids(n + 1) for n in lengths], ids(case["past"]), ids(case["prompt"])


# ---------------------------------------------------------------------------------------------------------
# a state and a pass
# ---------------------------------------------------------------------------------------------------------

class _State:
    pass


def prepare(case, seed):
    """An engine with its weights, the contexts of its requests in the cache, its graph captured: what a server
    holds when the step comes."""
    from simple_inference_amd import Engine, EngineConfig, SamplingParams
    from simple_inference_amd.engine import StepEntry
    from simple_inference_amd.engine.build import build_model, default_kernels

    decoding, past, prompt = _tokens(case, seed)
    longest = max([len(t) for t in decoding] + [len(past) + len(prompt)])
    pages = sum(-(-len(t) // PAGE) for t in decoding) + -(-(len(past) + len(prompt)) // PAGE)
    rows = len(decoding) + (1 if prompt else 0)
    cfg = EngineConfig(max_running=rows, max_seq_len=max(4096, -(-(longest + 1) // 1024) * 1024), dtype=case["dtype"],
                       chunk_tokens=max(512, len(prompt) + len(decoding)), eos_id=-1, block_size=PAGE,
                       num_kv_blocks=pages + 8, device="cuda:0")
    kernels = default_kernels()
    model, model_cfg = build_model(_config(case), cfg, kernels)
    weights = _weights(case, seed)
    wanted = model.expected_tensors()
    assert {n: tuple(s.shape) for n, s in wanted.items()} == {n: tuple(t.shape) for n, t in weights.items()}
    for name, spec in wanted.items():
        if spec.role == "vector" or case["dtype"] == "float32":
            weights[name] = weights[name].float()
    model.bind(weights)
    s = _State()
    s.engine = engine = Engine(model, model_cfg, cfg, kernels)
    s.decoding, s.prompt, s.past = [], [], 0
    s.repeats = case["model"] != "mogisun-linear"      # a prompt's positions can be taken again; a state's cannot
    contexts = []
    for i, t in enumerate(decoding):
        engine.cache.admit(i + 1, len(t), cfg.chunk_tokens)
        contexts.append((i + 1, t[:-1]))
        s.decoding.append(StepEntry(i + 1, [t[-1]], [0]))
    s.prompt_id, s.prompt_len = len(decoding) + 1, len(past) + len(prompt)
    if prompt:
        s.prompt = prompt
        s.want = list(range(len(prompt))) if case["want"] == "all" else [len(prompt) - 1]
        if past:
            engine.cache.admit(s.prompt_id, s.prompt_len, cfg.chunk_tokens)
            contexts.append((s.prompt_id, past))
            s.past = len(past)
    batch, room = [], 16384
    for rid, tokens in contexts:      # the contexts, up to 16,384 tokens a step
        if batch and len(tokens) > room:
            engine.runner.run(batch)
            batch, room = [], 16384
        batch.append(StepEntry(rid, tokens))
        room -= len(tokens)
    if batch:
        engine.runner.run(batch)
    emitted = len(decoding) + (len(s.want) if prompt else 0)
    params = {"greedy": lambda i: SamplingParams(max_new_tokens=64),
              "filtered": lambda i: SamplingParams(temperature=0.8, top_k=50, top_p=0.9, seed=seed + i, max_new_tokens=64)}
    s.params = [params[case["sampling"]](i) for i in range(emitted)]
    s.draws = [3] * emitted
    s.graph = not prompt and engine.graphs is not None and engine.graphs.can_run(s.decoding)
    if s.graph:
        bucket = engine.graphs.bucket_of(len(s.decoding)), engine.graphs.kv_bucket_of(longest)
        engine.graphs.capture(*bucket)
    s.StepEntry = StepEntry
    torch.cuda.synchronize()
    return s


def run(s):
    """One step: the logits at the places asked for, one row each, in the order decoding requests, prompt."""
    engine, entries = s.engine, s.decoding
    if s.prompt:
        if not s.past:
            engine.cache.admit(s.prompt_id, s.prompt_len, engine.cfg.chunk_tokens)
        entries = entries + [s.StepEntry(s.prompt_id, s.prompt, s.want)]
    logits = engine.graphs.run(entries) if s.graph else engine.runner.run(entries)
    engine.sampler.sample_on_device(logits, s.params, s.draws)
    for e in s.decoding:
        engine.cache.retract(e.req, 1)
    if s.prompt:
        if s.past:
            engine.cache.retract(s.prompt_id, len(s.prompt))
        else:
            engine.cache.release(s.prompt_id)
    return logits


# ---------------------------------------------------------------------------------------------------------
# what a pass cannot do without, and how exactly it is known
# ---------------------------------------------------------------------------------------------------------

def work(case):
    hidden, heads, kv, dim, ff, _, tied = _SHAPES[case["model"]]
    el = 2 if case["dtype"] == "bfloat16" else 4
    n, rows, prompt, past = case["layers"], case["rows"], case["prompt"], case["past"]
    context = case["context"] + (0.5 if case["ragged"] else 0)
    tokens = rows + prompt
    emitted = rows + ((prompt if case["want"] == "all" else 1) if prompt else 0)
    layer = sum(math.prod(s) for name, s in _weight_shapes(dict(case, layers=1)).items() if len(s) == 2 and
                (name.startswith("l0.") or ".layers." in name))
    head = VOCAB * hidden
    once = 2 * hidden * hidden if case["model"] == "mogisun-linear" else 0       # the re-mix with the embedding
    flops = 2 * tokens * (n * layer + once) + 2 * emitted * head
    moved = el * (n * layer + once + head + tokens * hidden) + 4 * emitted * VOCAB
    if case["model"] == "mogisun-linear":
        flops += n * tokens * heads * dim * dim * 6
        moved += n * 4 * heads * dim * dim * (2 * rows + (1 if prompt else 0))   # a decoded token's state in and out
    else:
        seen = rows * (context + 1) + prompt * past + prompt * (prompt + 1) / 2
        flops += n * 4 * heads * dim * seen
        moved += n * 2 * kv * dim * el * (rows * (context + 1) + past + prompt)
    return {"bytes": moved, "flops": flops}


def tolerance(case):
    """Two correct implementations differ by up to the sum of their errors.  Measured against ``exact``: float32 4e-6 to
    5e-6 (sums in another order); bfloat16 0.8e-2 to 1.6e-2 over 4 or 8 layers, the largest single difference 0.08 of the logits' size."""
    if case["dtype"] == "float32":
        return {"rel": 2e-5, "max": 2e-4}
    return {"rel": 3e-2, "max": 0.25}


def _inv_freq(dim, factor):
    f = 1.0 / (500000.0 ** (torch.arange(0, dim, 2, dtype=torch.float32) / dim))
    out = []
    for x in f.tolist():
        wave = 2 * math.pi / x
        if wave < 8192 / 4.0:
            out.append(x)
        elif wave > 8192 / 1.0:
            out.append(x / factor)
        else:
            smooth = (8192 / wave - 1.0) / (4.0 - 1.0)
            out.append((1 - smooth) * x / factor + smooth * x)
    return torch.tensor(out, dtype=torch.float32)


def _rms(x, gain=None):
    y = x * torch.rsqrt((x * x).mean(-1, keepdim=True) + _EPS)
    return y if gain is None else y * gain


def _causal(q, k, v):
    """Softmax attention of one sequence in 64 bits, q [T, H, D], k and v [T, G, D], some heads and rows at a time."""
    T, H, D = q.shape
    G = k.shape[1]
    out = torch.empty_like(q)
    place = torch.arange(T, device=q.device)
    block = max(64, min(T, (1 << 27) // T))
    for g in range(G):
        kt, vg = k[:, g].t().contiguous(), v[:, g].contiguous()
        for a in range(g * (H // G), (g + 1) * (H // G)):
            for lo in range(0, T, block):
                hi = min(T, lo + block)
                scores = (q[lo:hi, a].contiguous() @ kt[:, :hi]) * D ** -0.5
                scores.masked_fill_(place[None, :hi] > place[lo:hi, None], float("-inf"))
                out[lo:hi, a] = torch.softmax(scores, -1) @ vg[:hi]
    return out


def _linear(q, k, v, alpha):
    """The gated linear recurrence of several sequences at once: [B, T, H, D] each, token by token."""
    B, T, H, D = q.shape
    state = q.new_zeros(B, H, D, v.shape[-1])
    out = torch.empty_like(v)
    for t in range(T):
        state = alpha[:, t, :, :, None] * state + k[:, t, :, :, None] * v[:, t, :, None, :]
        out[:, t] = (state * q[:, t, :, :, None]).sum(2)
    return out


@torch.no_grad()
def exact(case, seed):
    """The same logits from whole sequences in 64 bits, without a cache.  Rotation tables are those of the model's
    definition (positions times frequencies as 32-bit products)."""
    hidden, heads, kv, dim, ff, factor, tied = _SHAPES[case["model"]]
    decoding, past, prompt = _tokens(case, seed)
    sequences = decoding + ([past + prompt] if prompt else [])
    total = sum(len(t) for t in sequences)
    if total > 140000:
        return None      # longer than about 20 seconds
    w = _weights(case, seed)
    linear = case["model"] == "mogisun-linear"
    embed = w["embed" if linear else "model.embed_tokens.weight"]
    lengths = [len(t) for t in sequences]
    starts = [sum(lengths[:i]) for i in range(len(lengths))]
    flat = torch.tensor([t for s in sequences for t in s], device="cuda")
    x = embed[flat].double()
    wide = lambda name: w[name].double()

    def by_rows(f, rows, step=16384):
        return torch.cat([f(rows[i:i + step]) for i in range(0, rows.shape[0], step)])

    if linear:
        x = by_rows(lambda r: torch.cat([r, r], -1) @ wide("loop.in").t(), x)
    else:
        angles = torch.arange(max(lengths), device="cuda", dtype=torch.float32)[:, None] * _inv_freq(dim, factor).cuda()[None, :]
        cos, sin = angles.cos().double(), angles.sin().double()

    def rotate(y, n):
        a, b = y[..., :dim // 2], y[..., dim // 2:]
        c, d = cos[:n, None], sin[:n, None]
        return torch.cat([a * c - b * d, b * c + a * d], -1)

    def swiglu(h, gate, up, down):
        return by_rows(lambda r: (torch.nn.functional.silu(r @ gate.t()) * (r @ up.t())) @ down.t(), h)

    for i in range(case["layers"]):
        if linear:
            p = f"l{i}."
            h = _rms(x, wide(p + "norm1"))
            q, k, v, g = (by_rows(lambda r: r @ wide(p + "mix." + n).t(), h).view(total, heads, dim) for n in "qkvg")
            z = (h @ wide(p + "mix.a1").t()) @ wide(p + "mix.a2").t() + wide(p + "mix.a2.b")
            alpha = torch.exp(torch.nn.functional.logsigmoid(z) / _TAU).view(total, heads, dim)
            longest = max(lengths)

            def padded(y, fill):       # every sequence from its first token on, shorter ones padded behind their last
                out = y.new_full((len(lengths), longest, heads, dim), fill)
                for s, n in enumerate(lengths):
                    out[s, :n] = y[starts[s]:starts[s] + n]
                return out
            o = _linear(padded(q * dim ** -0.5, 0.0), padded(k, 0.0), padded(v, 0.0), padded(alpha, 1.0))
            o = torch.cat([o[s, :n] for s, n in enumerate(lengths)])
            o = (_rms(o, wide(p + "mix.norm")) * torch.nn.functional.silu(g)).reshape(total, heads * dim)
            mixed = o @ wide(p + "mix.o").t()
            x = x + torch.sigmoid(h @ wide(p + "rg1").t() + wide(p + "rg1.b")) * mixed
            h = _rms(x, wide(p + "norm2"))
            x = x + torch.sigmoid(h @ wide(p + "rg2").t() + wide(p + "rg2.b")) * swiglu(
                h, wide(p + "mlp.gate"), wide(p + "mlp.up"), wide(p + "mlp.down"))
            continue
        p = f"model.layers.{i}."
        h = _rms(x, wide(p + "input_layernorm.weight"))
        q = by_rows(lambda r: r @ wide(p + "self_attn.q_proj.weight").t(), h).view(total, heads, dim)
        k = by_rows(lambda r: r @ wide(p + "self_attn.k_proj.weight").t(), h).view(total, kv, dim)
        v = by_rows(lambda r: r @ wide(p + "self_attn.v_proj.weight").t(), h).view(total, kv, dim)
        o = torch.cat([_causal(rotate(q[b:b + n], n), rotate(k[b:b + n], n), v[b:b + n]) for b, n in zip(starts, lengths)])
        del q, k, v, h
        x += by_rows(lambda r: r @ wide(p + "self_attn.o_proj.weight").t(), o.view(total, heads * dim))
        del o
        x += swiglu(_rms(x, wide(p + "post_attention_layernorm.weight")), wide(p + "mlp.gate_proj.weight"),
                    wide(p + "mlp.up_proj.weight"), wide(p + "mlp.down_proj.weight"))
    places = [b + n - 1 for b, n in zip(starts[:len(decoding)], lengths)]
    if prompt:
        end = starts[-1] + lengths[-1]
        places += list(range(end - len(prompt), end)) if case["want"] == "all" else [end - 1]
    gain, head = ("final.norm", "head") if linear else ("model.norm.weight", "model.embed_tokens.weight" if tied else "lm_head.weight")
    z = _rms(x[torch.tensor(places, device="cuda")], wide(gain))
    z = torch.cat([z @ w[head][j:j + 16384].double().t() for j in range(0, VOCAB, 16384)], -1)
    return _CAP * torch.tanh(z / _CAP) if linear else z
