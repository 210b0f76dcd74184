"""What this engine is timed on: whole pieces of work through its public entry points.

Three kinds of case:

* "trace": requests with given tokens run through `ModelRunner.step`, the step function that generation, the scheduler's
  engine and trace replay all call, in the steps that continuous batching makes of them (decoded tokens first, then the
  prompts under way and waiting in portions of at most `chunk`, at most `budget` rows a step).  Outputs: every step's logits.
* "generate": `Engine.generate` with its scheduler and samplers, half of the requests greedy and half with sampling options.
  Outputs: the tokens.  In 32-bit, where a token does not hang on a rounding.
* Both on GPT-2 shapes (Medium, Large, XL) and, for the trace, on a model of linear recurrences beside attention (Pafivik) with
  dense feed-forwards: a choice of experts in bfloat16 has near ties that go either way, and two right answers then differ.

A program keeps its model, its cache and its captured graphs, so `prepare` makes them and runs the work twice, as a server
warms up before it takes requests.  Weights and tokens come from the seed.
"""
import random

import torch

# The GPT-2 shapes of the repository's benchmark: (layers, width); heads of 64, inner size four times the width.
SHAPES = {"medium": (24, 1024), "large": (36, 1280), "xl": (48, 1600)}
GPT2_VOCAB, PAF_VOCAB = 50257, 32000


def _gpt2(name, shape, **more):
    layers, width = SHAPES[shape]
    return dict(dict(name=name, kind="trace", model="gpt2", layers=layers, width=width, head=64, positions=1024, dtype="bfloat16",
                     page=16, requests=1, low=1, high=1, new=0, chunk=1024, budget=8192, want_all=False), **more)


def _pafivik(name, **more):
    return dict(dict(name=name, kind="trace", model="pafivik", layers=4, width=1024, positions=2048, dtype="bfloat16", page=16,
                     requests=1, low=1, high=1, new=0, chunk=1024, budget=8192, want_all=False), **more)


def listed():
    return [
        # a single user's short exchange with the smallest shape: nothing but the latency of one row's chain of kernels
        _gpt2("medium b1", "medium", low=40, high=40, new=32),
        # the same with the largest shape and a long prompt
        _gpt2("xl b1", "xl", low=512, high=512, new=24),
        # a handful of users: the repository's headline batch, contexts of different lengths
        _gpt2("xl b8", "xl", requests=8, low=384, high=560, new=32),
        # a loaded server: the cache is as many bytes as the weights
        _gpt2("xl b64", "xl", requests=64, low=64, high=400, new=16),
        # a throughput job: an odd number of many short requests, products of some hundreds of rows
        _gpt2("large b203", "large", requests=203, low=8, high=64, new=12),
        # the prompt phase alone: two full prompts in one step
        _gpt2("xl prefill 2x1024", "xl", requests=2, low=1024, high=1024),
        # scoring of a set of texts of all lengths, as many rows in a step as fit
        _gpt2("large prefill ragged", "large", requests=23, low=17, high=1000),
        # continuous batching: decoded rows beside portions of the prompts that arrive
        _gpt2("large mixed", "large", requests=24, low=16, high=768, new=16, chunk=192, budget=320),
        # the 32-bit engine as a checker: whole texts, every place's logits
        _gpt2("medium f32 replay", "medium", dtype="float32", requests=2, low=1024, high=1024, want_all=True),
        # the 32-bit engine generating, scheduler and samplers included
        _gpt2("medium f32 generate", "medium", kind="generate", dtype="float32", requests=8, low=16, high=160, new=40, chunk=512,
              budget=2048),
        # a model of linear recurrences beside an attention layer: its prompt phase and its decoding
        _pafivik("pafivik prefill", requests=3, low=400, high=1024),
        _pafivik("pafivik b8", requests=8, low=32, high=256, new=40),
    ]


def _log_int(rng, low, high):
    return int(round(low * (high / low) ** rng.random()))


def draw(rng):
    """One more case of the same ranges: other widths, depths, head sizes, numbers of requests and lengths, pages."""
    what = rng.choice(["decode", "decode", "decode", "prefill", "prefill", "mixed", "float32", "generate", "pafivik", "pafivik"])
    heads, head = rng.randint(8, 25), rng.choice([64, 64, 64, 48, 80, 128])
    width = heads * head if head <= 64 else max(1, heads * 64 // head) * head
    c = dict(kind="trace", model="gpt2", layers=_log_int(rng, 6, 48), width=width, head=head, positions=1024, dtype="bfloat16",
             page=rng.choice([16, 16, 32, 64]), requests=1, low=1, high=1, new=0, chunk=1024, budget=8192, want_all=False)

    def lengths(most):
        a, b = _log_int(rng, 8, most), _log_int(rng, 8, most)
        c.update(low=min(a, b), high=max(a, b))
    if what == "decode":
        c.update(requests=_log_int(rng, 1, 220), new=rng.randint(10, 24))
        lengths(max(16, min(700, 16000 // c["requests"])))
    elif what == "prefill":
        c.update(requests=_log_int(rng, 1, 20))
        lengths(1000)
    elif what == "mixed":
        c.update(requests=rng.randint(6, 24), new=rng.randint(8, 16), chunk=rng.choice([64, 100, 192, 256]), budget=rng.choice([256, 320, 500]))
        lengths(500)
    elif what == "float32":
        c.update(dtype="float32", layers=_log_int(rng, 4, 24), requests=_log_int(rng, 1, 6), new=rng.randint(0, 12))
        lengths(600)
    elif what == "generate":
        c.update(kind="generate", dtype="float32", layers=_log_int(rng, 4, 16), requests=_log_int(rng, 1, 12), new=rng.randint(12, 32),
                 chunk=512, budget=2048)
        lengths(300)
    else:
        c = dict(_pafivik(""), width=rng.choice([512, 1024, 1024, 1536, 2048]), layers=rng.randint(3, 8), page=c["page"],
                 requests=_log_int(rng, 1, 48), new=rng.choice([0, rng.randint(8, 32)]))
        del c["name"]
        lengths(max(16, min(1000, 6000 // c["requests"])))
    biggest = [work(k) for k in listed()]
    most = {k: max(w[k] for w in biggest) for k in ("bytes", "flops")}
    if c["dtype"] == "float32":       # (32-bit rows cost as many times more)
        most["flops"] = max(w["flops"] for w, k in zip(biggest, listed()) if k["dtype"] == "float32")
    while c["layers"] > 2 and any(work(c)[k] > most[k] for k in most):
        c["layers"] = c["layers"] * 3 // 4
    while c["requests"] > 1 and any(work(c)[k] > most[k] for k in most):
        c["requests"] = c["requests"] * 3 // 4
    return c


# -- requests and the steps they make -------------------------------------------------------------------------------------

def _requests(case, seed):
    """-> [(tokens fed, length of the prompt)]: every request's prompt and the tokens that follow it.  The lengths are spread
    over low .. high and do not change with the seed, so that every seed's pass is the same amount of work."""
    rng = random.Random(seed)
    n, low, high = case["requests"], case["low"], case["high"]
    vocab = GPT2_VOCAB if case["model"] == "gpt2" else PAF_VOCAB
    spread = [low + (high - low) * k // max(1, n - 1) for k in range(n)]
    random.Random(1).shuffle(spread)
    more = 0 if case["kind"] == "generate" else case["new"]
    return [([rng.randrange(vocab) for _ in range(p + more)], p) for p in spread]


def _steps(case, requests):
    """-> a list of steps, each a list of (request, first place, places, wanted places among them)."""
    fed, waiting, running, steps = [0] * len(requests), list(range(len(requests))), [], []
    while waiting or running:
        left, step = case["budget"], []
        for r in running:
            prompt = requests[r][1]
            if fed[r] >= prompt and left > 0:
                step.append((r, fed[r], 1, [0]))
                left -= 1
        for r in running + waiting:
            prompt = requests[r][1]
            if fed[r] < prompt and left > 0:
                n = min(case["chunk"], left, prompt - fed[r])
                step.append((r, fed[r], n, list(range(n)) if case["want_all"] else [n - 1] if fed[r] + n == prompt else []))
                left -= n
        for r, _, n, _ in step:
            if r in waiting:
                waiting.remove(r)
                running.append(r)
            fed[r] += n
        running = [r for r in running if fed[r] < len(requests[r][0])]
        steps.append(step)
    return steps


# -- models -----------------------------------------------------------------------------------------------------------------

def _config(case):
    if case["model"] == "gpt2":
        return dict(architectures=["GPT2LMHeadModel"], n_layer=case["layers"], n_embd=case["width"], n_head=case["width"] // case["head"],
                    n_inner=4 * case["width"], vocab_size=GPT2_VOCAB, n_positions=case["positions"], layer_norm_epsilon=1e-5,
                    activation_function="gelu_new")
    width = case["width"]
    H = width // 128
    ff = dict(kind="dense", ff=4 * width)
    delta = dict(type="channel_delta", mlp=ff, mixer=dict(heads=H, kv_heads=max(1, H // 2), dim=64, vdim=128, conv=4, decay_rank=64,
                                                           gate_rank=64))
    kinds = [dict(type="lightning", mlp=ff, mixer=dict(heads=H, dim=64, vdim=128, decay=[1.0 - 2.0 ** -(5 + 3 * h / H) for h in range(H)])),
             delta,
             dict(type="attention", mlp=ff, mixer=dict(heads=width // 64, kv_heads=max(1, width // 256), dim=64, vdim=64, scale=0.125,
                                                        rot=dict(base=10000.0, dims=64))),
             delta]
    return dict(architecture="Pafivik", vocab=PAF_VOCAB, width=width, norm=dict(eps=1e-5), embedding=dict(scale=1.0), residual_mult=0.5,
                layers=[kinds[i % 4] for i in range(case["layers"])], max_positions=case["positions"])


def _tensors(case):
    """{name in a checkpoint: (shape, mean, standard deviation, whether it is a matrix)}, matrices as a checkpoint stores them."""
    W, t = case["width"], {}

    def vector(name, n, mean, std):
        t[name] = ((n,) if isinstance(n, int) else n, mean, std, False)

    def matrix(name, a, b, std=0.02):
        t[name] = ((a, b), 0.0, std, True)
    if case["model"] == "gpt2":
        matrix("wte.weight", GPT2_VOCAB, W)
        matrix("wpe.weight", case["positions"], W)
        for i in range(case["layers"]):
            p = f"h.{i}."
            for n in ("ln_1", "ln_2"):
                vector(p + n + ".weight", W, 1.0, 0.02), vector(p + n + ".bias", W, 0.0, 0.01)
            for n, a, b in (("attn.c_attn", W, 3 * W), ("attn.c_proj", W, W), ("mlp.c_fc", W, 4 * W), ("mlp.c_proj", 4 * W, W)):
                matrix(p + n + ".weight", a, b), vector(p + n + ".bias", b, 0.0, 0.01)
        vector("ln_f.weight", W, 1.0, 0.02), vector("ln_f.bias", W, 0.0, 0.01)
        return t
    matrix("embed", PAF_VOCAB, W)
    for i, layer in enumerate(_config(case)["layers"]):
        m, p, wide = layer["mixer"], f"l{i}.", W ** -0.5
        for n in ("norm1", "norm1b", "norm2", "norm2b"):
            vector(p + n, W, 1.0, 0.1)
        vector(p + "ls1", W, 1.0, 0.2), vector(p + "ls2", W, 1.0, 0.2)
        H, dk, dv = m["heads"], m["dim"], m["vdim"]
        if layer["type"] == "lightning":
            for n, rows in (("q", H * dk), ("k", H * dk), ("v", H * dv), ("g", H * dv)):
                matrix(p + "mix." + n, rows, W, wide)
            vector(p + "mix.norm", H * dv, 1.0, 0.1)
        elif layer["type"] == "channel_delta":
            G = m["kv_heads"]
            for n, rows in (("q", G * dk), ("k", G * dk), ("v", H * dv)):
                matrix(p + "mix." + n, rows, W, wide), vector(p + "mix." + n + ".conv", (rows, m["conv"]), 0.0, 0.4)
            matrix(p + "mix.b", H, W, wide)
            matrix(p + "mix.a1", m["decay_rank"], W, wide), matrix(p + "mix.a2", H * dk, m["decay_rank"], m["decay_rank"] ** -0.5)
            matrix(p + "mix.g1", m["gate_rank"], W, wide), matrix(p + "mix.g2", H * dv, m["gate_rank"], m["gate_rank"] ** -0.5)
            vector(p + "mix.A_log", H, -0.75, 0.7), vector(p + "mix.dt_bias", H * dk, -1.0, 1.0), vector(p + "mix.norm", dv, 1.0, 0.1)
        else:
            G = m["kv_heads"]
            for n, rows in (("q", H * dk), ("k", G * dk), ("v", G * dv)):
                matrix(p + "mix." + n, rows, W), vector(p + "mix." + n + ".b", rows, 0.0, 0.01)
        matrix(p + "mix.o", W, H * dv)
        ff = layer["mlp"]["ff"]
        matrix(p + "mlp.up", ff, W, wide), vector(p + "mlp.up.b", ff, 0.0, 0.01), vector(p + "mlp.act", 2, 0.5, 0.3)
        matrix(p + "mlp.down", W, ff), vector(p + "mlp.down.b", W, 0.0, 0.01)
        vector(p + "dwa", i + 2, 1.0 / (i + 2), 0.1)
    vector("final.norm", W, 1.0, 0.1)
    return t


def _weights(case, seed):
    """{name: tensor} on the GPU as a checkpoint holds them: matrices in the case's type, vectors in 32-bit."""
    g = torch.Generator(device="cuda").manual_seed(seed * 1000003 + 17)
    kind, out = getattr(torch, case["dtype"]), {}
    for name, (shape, mean, std, is_matrix) in _tensors(case).items():
        x = torch.randn(shape, generator=g, device="cuda").mul_(std)
        out[name] = x.to(kind) if is_matrix else x.add_(mean)
    return out


# -- the program ------------------------------------------------------------------------------------------------------------

class State:
    pass


def prepare(case, seed):
    from denno_beta_amd.config import EngineOptions, resolve_architecture
    from denno_beta_amd.engine import Engine, ModelRunner, SamplingParams, StepEntry
    s = State()
    config = _config(case)
    arch = resolve_architecture(config)
    cfg = arch.config_cls.from_dict(config)
    spec = arch.build(cfg)
    files, held = _weights(case, seed), {}
    for p in spec.param_specs():
        x = torch.cat([files[name] for name, _ in p.pieces()], dim=p.concat_dim) if p.sources is not None else files[p.name]
        held[p.name] = (x.t() if p.transpose else x).contiguous()
    del files
    requests = _requests(case, seed)
    n, longest = len(requests), max(len(t) for t, _ in requests) + (case["new"] if case["kind"] == "generate" else 0)
    pages = -(-(longest + 1) // case["page"])
    options = EngineOptions(dtype=case["dtype"], page_size=case["page"], cache_tokens=n * pages * case["page"], max_live=n,
                            max_batch_tokens=case["budget"], prefill_chunk=case["chunk"], seed=0)
    s.runner = ModelRunner(spec, held, options, cfg)
    del held
    if case["kind"] == "generate":
        s.engine = Engine(s.runner, options)
        s.prompts = [t for t, _ in requests]
        s.params = [SamplingParams(max_tokens=case["new"], temperature=0.0, ignore_eos=True) if r % 2 == 0 else
                    SamplingParams(max_tokens=case["new"], temperature=0.8, top_p=0.9, repetition_penalty=1.1, seed=r, ignore_eos=True)
                    for r in range(n)]
    else:
        s.engine = None
        s.steps = [[StepEntry(r, requests[r][0][at:at + count], want) for r, at, count, want in step] for step in _steps(case, requests)]
        s.requests = range(n)
    for _ in range(2):       # the graphs of its steps' shapes are captured (one that holds portions at its second step)
        run(s)
    return s


def run(state):
    if state.engine is not None:
        out = state.engine.generate(state.prompts, state.params)
        return [torch.tensor(tokens) for tokens in out]
    runner, logits, started = state.runner, [], set()
    for step in state.steps:
        for e in step:
            if e.rid not in started:
                runner.start_request(e.rid)
                started.add(e.rid)
        out = runner.step(step)
        if out.shape[0]:
            logits.append(out)
    for r in state.requests:
        runner.end_request(r)
    return logits


# -- what it cannot do without ------------------------------------------------------------------------------------------------

def work(case):
    """Every step reads the weights that its rows need and the live requests' cache once and writes its own keys and values and
    its logits; two operations a weight and row, four a pair of query and key element."""
    size = 2 if case["dtype"] == "bfloat16" else 4
    names = _tensors(case)
    vocab = GPT2_VOCAB if case["model"] == "gpt2" else PAF_VOCAB
    table = "wte.weight" if case["model"] == "gpt2" else "embed"
    W = case["width"]
    head = vocab * W
    layer_weights = sum(a[0][0] * a[0][1] for n, a in names.items() if a[3] and n not in (table, "wpe.weight"))
    if case["model"] == "gpt2":
        kv, qwidth = case["layers"] * 2 * W, W
        attentions, state = case["layers"], 0
    else:
        kinds = [layer["type"] for layer in _config(case)["layers"]]
        attentions = kinds.count("attention")
        kv, qwidth = attentions * 2 * max(1, W // 256) * 64, W
        state = (len(kinds) - attentions) * (W // 128) * 64 * 128       # a matrix per head, in 32-bit, read and written
    requests = _requests(case, 0)
    if case["kind"] == "generate":
        requests = [(t + [0] * (case["new"] - 1), p) for t, p in requests]
    nbytes = flops = 0.0
    for step in _steps(case, requests):
        rows, wanted = sum(n for _, _, n, _ in step), sum(len(w) for _, _, _, w in step)
        nbytes += (layer_weights + (head if wanted else 0)) * size + wanted * vocab * 4 + rows * W * size
        nbytes += kv * size * sum(at + n for _, at, n, _ in step) + kv * size * rows + 8.0 * state * len(step)
        flops += 2.0 * rows * layer_weights + 2.0 * wanted * head + 4.0 * rows * state
        flops += 4.0 * attentions * qwidth * sum(n * at + n * (n + 1) / 2 for _, at, n, _ in step)
    return {"bytes": nbytes, "flops": flops}


def tolerance(case):
    # Measured against `exact`, and about four times that: bfloat16 logits of 4 to 48 layers are 0.4 to 0.75 % off in the 2-norm
    # (five times as much of a row's scale at the worst place), the 32-bit engine's 6e-7; a 32-bit token may differ where two
    # logits are closer than that.
    if case["dtype"] == "float32":
        return {"rel": 3e-6, "max": 5e-5, "differ": 0.01}
    return {"rel": 0.03 if case["model"] == "pafivik" else 0.025, "max": 0.25}


# -- the same in 64 bits, plainly ---------------------------------------------------------------------------------------------

def _layer_norm(x, w, b):
    x = x - x.mean(-1, keepdim=True)
    return x / torch.sqrt((x * x).mean(-1, keepdim=True) + 1e-5) * w + b


def _attend(q, k, v, scale, first):
    """q [n, H, d] at positions first .. first + n - 1 over k, v [t, G, d], causal."""
    n, H, d = q.shape
    t, G = k.shape[0], k.shape[1]
    k, v = (x.repeat_interleave(H // G, dim=1).permute(1, 0, 2).contiguous() for x in (k, v))
    scores = torch.matmul(q.permute(1, 0, 2).contiguous(), k.transpose(1, 2).contiguous()) * scale
    later = torch.arange(t, device=q.device)[None, :] > first + torch.arange(n, device=q.device)[:, None]
    return torch.matmul(torch.softmax(scores.masked_fill(later, float("-inf")), -1), v).permute(1, 0, 2).reshape(n, -1)


def _gpt2_exact(case, w, sequences, firsts, caches):
    """The rows of the final norm for the sequences' tokens, which stand at positions firsts[r] ...; caches: per layer and
    sequence the keys and values so far, which grow (None: none are kept)."""
    W, H, dev = case["width"], case["width"] // case["head"], "cuda"
    tokens = torch.tensor([t for s in sequences for t in s], device=dev)
    at = torch.cat([torch.arange(f, f + len(s), device=dev) for s, f in zip(sequences, firsts)])
    x = w["wte.weight"][tokens] + w["wpe.weight"][at]
    for i in range(case["layers"]):
        p = f"h.{i}."
        h = _layer_norm(x, w[p + "ln_1.weight"], w[p + "ln_1.bias"])
        qkv = (h @ w[p + "attn.c_attn.weight"] + w[p + "attn.c_attn.bias"]).view(-1, 3, H, case["head"])
        out, o = [], 0
        for r, s in enumerate(sequences):
            q, k, v = (qkv[o:o + len(s), j] for j in range(3))
            o += len(s)
            if caches is not None:
                if caches[i][r] is not None:
                    k, v = torch.cat([caches[i][r][0], k]), torch.cat([caches[i][r][1], v])
                caches[i][r] = (k, v)
            out.append(_attend(q, k, v, case["head"] ** -0.5, firsts[r]))
        x = x + torch.cat(out) @ w[p + "attn.c_proj.weight"] + w[p + "attn.c_proj.bias"]
        h = _layer_norm(x, w[p + "ln_2.weight"], w[p + "ln_2.bias"])
        u = h @ w[p + "mlp.c_fc.weight"] + w[p + "mlp.c_fc.bias"]
        u = 0.5 * u * (1 + torch.tanh((2 / torch.pi) ** 0.5 * (u + 0.044715 * u ** 3)))
        x = x + u @ w[p + "mlp.c_proj.weight"] + w[p + "mlp.c_proj.bias"]
    return _layer_norm(x, w["ln_f.weight"], w["ln_f.bias"])


def _rms(x, weight, eps=1e-5):
    return x / torch.sqrt((x * x).mean(-1, keepdim=True) + eps) * weight


def _silu(x):
    return x * torch.sigmoid(x)


def _pafivik_exact(case, w, sequences):
    """The rows of the final norm, sequence behind sequence; every sequence begins at position 0."""
    cfg, dev = _config(case), "cuda"
    lens = [len(s) for s in sequences]
    x = w["embed"][torch.tensor([t for s in sequences for t in s], device=dev)]
    T, S = max(lens), len(lens)
    row = torch.cat([torch.arange(n, device=dev) * S + r for r, n in enumerate(lens)])       # a row's place in [time, sequence]
    place = torch.cat([torch.arange(n, device=dev) for n in lens])

    def by_time(y):
        out = torch.zeros((T * S,) + y.shape[1:], dtype=y.dtype, device=dev)
        out[row] = y
        return out.view((T, S) + y.shape[1:])
    history = [x]
    for i, layer in enumerate(cfg["layers"]):
        p, m = (lambda name, i=i: w[f"l{i}.{name}"]), layer["mixer"]
        H, dk, dv = m["heads"], m["dim"], m["vdim"]
        h = _rms(x, p("norm1"))
        if layer["type"] == "attention":
            G, out, o = m["kv_heads"], [], 0
            q, k, v = ((h @ p("mix." + n).T + p("mix." + n + ".b")).view(-1, g, 64) for n, g in (("q", H), ("k", G), ("v", G)))
            angle = place[:, None].double() * 10000.0 ** (-torch.arange(0, 64, 2, device=dev).double() / 64)[None, :]
            cos, sin = torch.cos(angle)[:, None], torch.sin(angle)[:, None]
            q, k = (torch.stack([z[..., 0::2] * cos - z[..., 1::2] * sin, z[..., 1::2] * cos + z[..., 0::2] * sin], -1).flatten(-2) for z in (q, k))
            for n in lens:
                out.append(_attend(q[o:o + n], k[o:o + n], v[o:o + n], m["scale"], 0))
                o += n
            y = torch.cat(out)
        elif layer["type"] == "lightning":
            q, k, v = (by_time(_silu(h @ p("mix." + n).T).view(-1, H, d)) for n, d in (("q", dk), ("k", dk), ("v", dv)))
            decay = torch.tensor(m["decay"], dtype=torch.float64, device=dev).view(1, H, 1, 1)
            state, o = torch.zeros(S, H, dk, dv, dtype=torch.float64, device=dev), torch.empty(T, S, H, dv, dtype=torch.float64, device=dev)
            for t in range(T):
                state = decay * state + k[t].unsqueeze(-1) * v[t].unsqueeze(-2)
                o[t] = (state * q[t].unsqueeze(-1)).sum(-2)
            y = _rms(o.view(T * S, H * dv)[row], p("mix.norm")) * torch.sigmoid(h @ p("mix.g").T)
        else:
            G, taps = m["kv_heads"], m["conv"]

            def convolved(n):
                z = by_time(h @ p("mix." + n).T)
                z = torch.cat([z.new_zeros((taps - 1,) + z.shape[1:]), z])
                return _silu(sum(p("mix." + n + ".conv")[:, j] * z[j:j + T] for j in range(taps)))
            q, k, v = convolved("q").view(T, S, G, dk), convolved("k").view(T, S, G, dk), convolved("v").view(T, S, H, dv)
            q, k = ((z / torch.sqrt((z * z).sum(-1, keepdim=True) + 1e-6)).repeat_interleave(H // G, dim=2) for z in (q, k))
            q = q * dk ** -0.5
            beta = by_time(torch.sigmoid(h @ p("mix.b").T))
            step = torch.nn.functional.softplus((h @ p("mix.a1").T) @ p("mix.a2").T + p("mix.dt_bias"), threshold=1e9).view(-1, H, dk)
            fade = by_time(torch.exp(-torch.exp(p("mix.A_log"))[None, :, None] * step))
            state, o = torch.zeros(S, H, dk, dv, dtype=torch.float64, device=dev), torch.empty(T, S, H, dv, dtype=torch.float64, device=dev)
            for t in range(T):
                state = fade[t].unsqueeze(-1) * state
                u = beta[t].unsqueeze(-1) * (v[t] - (state * k[t].unsqueeze(-1)).sum(-2))
                state = state + k[t].unsqueeze(-1) * u.unsqueeze(-2)
                o[t] = (state * q[t].unsqueeze(-1)).sum(-2)
            gate = torch.sigmoid((h @ p("mix.g1").T) @ p("mix.g2").T).view(-1, H, dv)
            y = (_rms(o.view(T * S, H, dv)[row], p("mix.norm")) * gate).view(-1, H * dv)
        x = x + cfg["residual_mult"] * (_rms(y @ p("mix.o").T, p("norm1b")) * p("ls1"))
        h = _rms(x, p("norm2"))

        z, (a, b) = h @ p("mlp.up").T + p("mlp.up.b"), torch.nn.functional.softplus(p("mlp.act"), threshold=1e9)
        low = z.clamp(max=0)
        y = torch.where(z > 0, a * z * z + 0.5 * z, (0.5 + b) * (torch.expm1(low) - low) + 0.5 * z) @ p("mlp.down").T + p("mlp.down.b")
        x = x + cfg["residual_mult"] * (_rms(y, p("norm2b")) * p("ls2"))
        history.append(x)
        x = sum(p("dwa")[j] * history[j] for j in range(i + 2))
    return _rms(x, w["final.norm"])


def exact(case, seed):
    w = {name: x.double() for name, x in _weights(case, seed).items()}
    requests = _requests(case, seed)
    if case["kind"] == "generate":
        out = []
        for r, (prompt, _) in enumerate(requests):
            if r % 2:
                out.append(None)          # (a sampled request has no such value: its draws are the engine's own)
                continue
            caches, tokens, feed = [[None] for _ in range(case["layers"])], [], prompt
            while len(tokens) < case["new"]:
                rows = _gpt2_exact(case, w, [feed], [len(prompt) + len(tokens) - len(feed) if tokens else 0], caches)
                tokens.append(int((w["wte.weight"] @ rows[-1]).argmax()))
                feed = tokens[-1:]
            out.append(torch.tensor(tokens))
        return out
    sequences = [t for t, _ in requests]
    if case["model"] == "gpt2":
        rows, table = [], w["wte.weight"]
        for at in range(0, len(sequences), 16):
            part = sequences[at:at + 16]
            rows.append(_gpt2_exact(case, w, part, [0] * len(part), None))
        rows = torch.cat(rows)
    else:
        rows, table = _pafivik_exact(case, w, sequences), w["embed"]
    first = [0]
    for s in sequences:
        first.append(first[-1] + len(s))
    steps = [[first[r] + at + j for r, at, _, want in step for j in want] for step in _steps(case, requests)]
    return [rows[torch.tensor(places, device="cuda")] @ table.T for places in steps if places]
