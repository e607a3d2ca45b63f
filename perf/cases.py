"""Sessions of the engine that are timed: prompts go in, in portions under a token budget and beside the requests that already
decode, then every request decodes one token a step, until all have their tokens. A pass is one whole session through
``CacheManager.open``, ``ModelRunner.step`` and ``CacheManager.close``, on a model that is loaded and an engine that is up. The
tokens are given (as ``bin/trace_run`` is given them), so a session's outputs are the logits of its steps.

The models: GPT-2 at the sizes of the repository's benchmark, in bfloat16 and in float32, and at the benchmark's middle size one
model with softmax attention, latent attention and experts (Kelasun) and one with recurrent states beside attention (Lelatar).
"""
import math
import random

import torch

GPT2_SIZES = {  # width, heads, layers
    "small": (768, 12, 12),
    "medium": (1024, 16, 24),
    "xl": (1600, 25, 48),
    "7b": (4096, 32, 32),
}
GPT2_VOCAB, OTHER_VOCAB = 50257, 32000
PAGE = 16


# ---- the cases ----------------------------------------------------------------------------------------------------------
def _case(name, arch, size, dtype, requests, shortest, longest, new, budget=2048, score=False):
    """``requests`` prompts of ``shortest`` .. ``longest`` tokens, ``new`` decoded tokens each; at most ``budget`` prompt tokens a step;
    ``score``: the logits of every prompt token are wanted, not the last one's alone."""
    return {"name": name, "arch": arch, "size": size, "dtype": dtype, "requests": requests, "shortest": shortest, "longest": longest,
            "new": new, "budget": budget, "score": score}


def listed():
    return [
        # one user's short question to the smallest model: a few tokens a step, latency and launches count
        _case("small_one_user", "gpt2", "small", "bfloat16", 1, 24, 24, 24),
        # a handful of users of a middle-sized model, prompts of a sentence or two
        _case("xl_few_users", "gpt2", "xl", "bfloat16", 6, 17, 90, 32),
        # a busy server: portions of 256 prompt tokens beside the requests that decode already, in every step
        _case("xl_busy_server", "gpt2", "xl", "bfloat16", 24, 33, 301, 24, budget=256),
        # a long document into the benchmark's model: prefill alone
        _case("7b_long_prompt", "gpt2", "7b", "bfloat16", 1, 2048, 2048, 0),
        # the benchmark's decode batch of 8, ragged prompts
        _case("7b_batch_8", "gpt2", "7b", "bfloat16", 8, 70, 200, 32),
        # a large decode batch: weights and caches both count
        _case("7b_batch_64", "gpt2", "7b", "bfloat16", 64, 48, 131, 20),
        # 32-bit: a small batch generates, as in checks of a model against another implementation
        _case("small_float32", "gpt2", "small", "float32", 4, 100, 203, 16),
        # 32-bit: the logits of every token of a document, as in an evaluation
        _case("medium_float32_score", "gpt2", "medium", "float32", 1, 777, 777, 0, score=True),
        # prompts into a model of latent attention, attention and experts
        _case("kelasun_prompts", "kelasun", "2k", "bfloat16", 2, 990, 1040, 0),
        # the same model decodes a batch: some of the experts a step
        _case("kelasun_batch_8", "kelasun", "2k", "bfloat16", 8, 100, 230, 32),
        # prompts into a model of recurrences beside attention
        _case("lelatar_prompts", "lelatar", "2k", "bfloat16", 3, 301, 999, 0),
        # the same model decodes a larger batch
        _case("lelatar_batch_32", "lelatar", "2k", "bfloat16", 32, 40, 150, 32),
    ]


def draw(rng: random.Random):
    """One more case: a model, then its sizes, spread over the logarithm of what the listed cases span."""

    def spread(lo, hi):
        return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))

    arch, size, dtype = rng.choice([("gpt2", "small", "bfloat16"), ("gpt2", "xl", "bfloat16"), ("gpt2", "7b", "bfloat16"), ("gpt2", "7b", "bfloat16"),
                                    ("gpt2", "small", "float32"), ("gpt2", "medium", "float32"),
                                    ("kelasun", "2k", "bfloat16"), ("lelatar", "2k", "bfloat16")])
    if rng.random() < 0.4:  # prompts alone
        longest = spread(64, 777 if dtype == "float32" else 1000 if size in ("small", "xl") else 2000)  # within the model's positions
        requests = rng.randint(1, max(1, min(4, (2048 if dtype == "bfloat16" else 777) // longest)))
        c = _case("", arch, size, dtype, requests, max(1, longest - rng.randint(0, longest // 2)), longest, 0, score=dtype == "float32" and rng.random() < 0.5)
    else:
        requests = spread(1, {"small": 32 if dtype == "bfloat16" else 4, "medium": 4, "xl": 24, "7b": 32, "2k": 32}[size])
        longest = spread(12, 200)
        c = _case("", arch, size, dtype, requests, max(1, longest - rng.randint(0, longest // 2)), longest, rng.randint(6, {"7b": 14, "medium": 8}.get(size, 24 if dtype == "bfloat16" else 16)),
                  budget=rng.choice([256, 2048]))
        while len(plan(c)) > 60:  # outputs come one a step
            c["requests"] = max(1, c["requests"] // 2)
    del c["name"]
    return c


def prompt_lengths(c):
    span = c["longest"] - c["shortest"] + 1
    return [c["longest"] - (i * 37) % span for i in range(c["requests"])]


def plan(c):
    """The session's steps: lists of (request, first position, tokens, places whose logits are wanted). Decoding requests come
    first, then prompt portions under the budget, oldest request first."""
    lens = prompt_lengths(c)
    fed, steps = [0] * len(lens), []
    while any(f < n + c["new"] for f, n in zip(fed, lens)):
        step, left = [], c["budget"]
        step += [(r, fed[r], 1, (0,)) for r, n in enumerate(lens) if n <= fed[r] < n + c["new"]]
        for r, n in enumerate(lens):
            if fed[r] < n and left > 0:
                k = min(left, n - fed[r])
                step.append((r, fed[r], k, tuple(range(k)) if c["score"] else (k - 1,) if fed[r] + k == n else ()))
                left -= k
        for r, _, k, _ in step:
            fed[r] += k
        steps.append(step)
    return steps


# ---- configurations -----------------------------------------------------------------------------------------------------
def config(c):
    if c["arch"] == "gpt2":
        width, heads, layers = GPT2_SIZES[c["size"]]
        return {"model_type": "gpt2", "n_layer": layers, "n_embd": width, "n_head": heads, "n_inner": 4 * width, "vocab_size": GPT2_VOCAB,
                "n_positions": 1024 if width < 2048 else 2048, "layer_norm_epsilon": 1e-5, "activation_function": "gelu_new"}
    width, heads, kv_heads, dim, vdim, ff, runs = 2048, 16, 4, 128, 64, 8192, 8
    base = {"vocab": OTHER_VOCAB, "width": width, "norm": {"eps": 1e-6}}
    if c["arch"] == "kelasun":
        attention = {"heads": heads, "kv_heads": kv_heads, "dim": dim, "vdim": vdim, "scale": dim ** -0.5, "q_temp": {"coef": 0.1, "every": 2048}}
        latent = {"heads": heads, "dim": dim, "rot_dim": 32, "vdim": vdim, "kv_rank": 224, "q_rank": width // 2, "scale": (dim + 32) ** -0.5,
                  "rot": {"dims": 32, "base": 500000.0, "scaling": {"factor": 8.0, "original": 4096, "fast": 32.0, "slow": 1.0}}}
        mlp = {"kind": "moe", "expert": {"ff": ff // 4}, "router": {"experts": 32, "top": 4}, "shared": {"ff": ff // 4}}
        layers = [{"type": ("attention", "latent_attention")[i % 2], "mixer": dict((attention, latent)[i % 2]), "mlp": dict(mlp)} for i in range(runs)]
        return {"architecture": "Kelasun", **base, "postln_alpha": 2.0, "logit_scale": 0.5, "layers": layers}
    left = {"heads": heads, "kv_heads": kv_heads, "dim": dim, "vdim": vdim, "scale": dim ** -0.5, "rot": {"dims": dim // 2, "base": 500000.0}}
    right = {"heads": heads, "kv_heads": heads // 2, "dim": dim, "vdim": vdim, "conv": 4}
    mamba = {"heads": width // 32, "vdim": 64, "state": 128, "groups": 4, "norm_groups": 4, "conv": 4}
    layers = [{"type": "parallel", "mixer": {"left": dict(left), "right": dict(right)}, "mlp": {"kind": "dense", "ff": 5376}} if i % 2 == 0 else
              {"type": "mamba2", "mixer": dict(mamba), "mlp": None} for i in range(runs - 2)]
    return {"architecture": "Lelatar", **base, "layers": layers, "loop": {"start": 2, "stop": 4, "times": 2}, "token_side": {"dim": width // 16}}


def layer_order(cfg):
    """Lelatar's layers in the order they run, each with the number of the loop's pass that begins before it (None: none does)."""
    n, loop = len(cfg["layers"]), cfg["loop"]
    a, b = loop["start"], loop["stop"]
    return [(i, None) for i in range(a)] + [(i, t if i == a else None) for t in range(loop["times"]) for i in range(a, b)] + [(i, None) for i in range(b, n)]


def shapes(cfg):
    """Checkpoint tensor -> (shape, mean, standard deviation). Matrices keep the size of what they multiply, norm weights lie around
    one; routers are decided, as trained ones are (the last chosen expert's weight is small beside the first's), and a sublayer's result is
    small beside the stream, so that a router's near ties, which rounding alone decides, do not take the logits over."""
    s = {}
    if cfg.get("model_type") == "gpt2":
        d, f, std = cfg["n_embd"], cfg["n_inner"], 0.02
        s["wte.weight"], s["wpe.weight"] = ((cfg["vocab_size"], d), 0, std), ((cfg["n_positions"], d), 0, std)
        norms = ["ln_f"]
        for i in range(cfg["n_layer"]):
            norms += [f"h.{i}.ln_1", f"h.{i}.ln_2"]
            for name, a, b in (("attn.c_attn", d, 3 * d), ("attn.c_proj", d, d), ("mlp.c_fc", d, f), ("mlp.c_proj", f, d)):
                s[f"h.{i}.{name}.weight"], s[f"h.{i}.{name}.bias"] = ((a, b), 0, std), ((b,), 0, std)
        for n in norms:
            s[n + ".weight"], s[n + ".bias"] = ((d,), 1, 0.02), ((d,), 0, 0.02)
        return s
    D, V = cfg["width"], cfg["vocab"]

    def mat(name, rows, cols, gain=1.0):
        s[name] = ((rows, cols), 0, gain / math.sqrt(cols))

    def vec(name, n, mean, std=0.2):
        s[name] = ((n,), mean, std)

    s["embed"] = ((V, D), 0, 1.0)
    mat("head", V, D, 2.0)
    stored_one = 0 if cfg["architecture"] == "Lelatar" else 1  # Lelatar stores its stream norms' weights as the distance from one
    vec("final.norm", D, stored_one)
    for i, L in enumerate(cfg["layers"]):
        m, p, q, mlp = L["mixer"], f"l{i}.", f"l{i}.mix.", L["mlp"]
        vec(p + "norm1", D, stored_one)
        if mlp is not None:
            vec(p + "norm2", D, stored_one)
        if L["type"] == "mamba2":
            H, P, N, G = m["heads"], m["vdim"], m["state"], m["groups"]
            inner, conv = H * P, H * P + 2 * G * N
            mat(q + "in", inner + conv + H, D)
            s[q + "conv"] = ((conv, m["conv"]), 0, 0.7)
            vec(q + "conv.b", conv, 0), vec(q + "dt_bias", H, -2, 1.0), vec(q + "A_log", H, 0, 1.0), vec(q + "D", H, 0.5, 0.5), vec(q + "norm", inner, 1)
            mat(q + "o", D, inner)
        if L["type"] == "latent_attention":
            H, dk, dr, dv, R, Q = (m[k] for k in ("heads", "dim", "rot_dim", "vdim", "kv_rank", "q_rank"))
            mat(q + "dq", Q, D), mat(q + "uq", H * (dk + dr), Q), mat(q + "dkv", R + dr, D), mat(q + "uk", H * dk, R), mat(q + "uv", H * dv, R)
            vec(q + "dq.norm", Q, 1.5, 0.3), vec(q + "dkv.norm", R, 1.2, 0.3)
            mat(q + "g", H * dv, D, 1.5), mat(q + "o", D, H * dv)
        if L["type"] in ("attention", "parallel"):
            a, q1 = (m, q) if L["type"] == "attention" else (m["left"], q + "left.")
            H, G, dk, dv = a["heads"], a["kv_heads"], a["dim"], a["vdim"]
            mat(q1 + "q", H * dk, D), mat(q1 + "k", G * dk, D), mat(q1 + "v", G * dv, D)
            vec(q1 + "q.norm", H * dk, 1.5, 0.3), vec(q1 + "k.norm", G * dk, 1.5, 0.3), vec(q1 + "sink", H, 1, 1.0)
            if L["type"] == "attention":
                mat(q1 + "g", H, D, 1.5)
            mat(q1 + "o", D, H * dv)
        if L["type"] == "parallel":
            r, q2 = m["right"], q + "right."
            H, G, dk, dv = r["heads"], r["kv_heads"], r["dim"], r["vdim"]
            for n, ch in (("q", G * dk), ("k", G * dk), ("v", H * dv)):
                mat(q2 + n, ch, D)
                s[q2 + n + ".conv"] = ((ch, r["conv"]), 0, 0.7)
            mat(q2 + "a", H, D), mat(q2 + "b", H, D), mat(q2 + "g", H * dv, D, 1.5), mat(q2 + "o", D, H * dv)
            vec(q2 + "dt_bias", H, -2, 1.0), vec(q2 + "A_log", H, 0, 1.0), vec(q2 + "norm", dv, 1)
            vec(q + "left.out", D, 1), vec(q + "right.out", D, 1)
        if mlp is not None and mlp["kind"] == "moe":
            mat(p + "mlp.router", mlp["router"]["experts"], D, 8.0)
            for n, F in [(f"e{e}", mlp["expert"]["ff"]) for e in range(mlp["router"]["experts"])] + [("shared", mlp["shared"]["ff"])]:
                mat(f"{p}mlp.{n}.up", F, D), mat(f"{p}mlp.{n}.down", D, F, 0.3)
        elif mlp is not None:
            mat(p + "mlp.gate", mlp["ff"], D), mat(p + "mlp.up", mlp["ff"], D), mat(p + "mlp.down", D, mlp["ff"])
        if cfg.get("token_side"):
            d = cfg["token_side"]["dim"]
            mat(p + "side.gate", d, D), mat(p + "side.proj", D, d), vec(p + "side.norm", D, 0.5)
    if cfg.get("token_side"):
        s["side.embed"] = ((V, len(cfg["layers"]) * cfg["token_side"]["dim"]), 0, 1.0)
    if cfg.get("loop"):
        mat("loop.in", D, 2 * D)
        s["loop.step"] = ((cfg["loop"]["times"], D), 0, 0.3)
    return s


# ---- a session on the engine --------------------------------------------------------------------------------------------
def weights(c, seed):
    g = torch.Generator(device="cuda").manual_seed(seed)
    dtype = getattr(torch, c["dtype"])
    return {n: torch.empty(shape, dtype=dtype, device="cuda").normal_(mean, std, generator=g) for n, (shape, mean, std) in shapes(config(c)).items()}


def token_ids(c, seed):
    g = torch.Generator().manual_seed(seed)
    vocab = GPT2_VOCAB if c["arch"] == "gpt2" else OTHER_VOCAB
    return [torch.randint(0, vocab, (n + c["new"],), generator=g).tolist() for n in prompt_lengths(c)]


def prepare(c, seed):
    from levanter_amd.config import InferenceEngineConfig, LmConfig
    from levanter_amd.engine import InferenceEngine
    from levanter_amd.engine.loading import make_env
    from levanter_amd.parts import DecoderLm

    pages = max(-(-(n + c["new"]) // PAGE) for n in prompt_lengths(c))
    engine_config = InferenceEngineConfig(max_seqs=c["requests"], page_size=PAGE, max_pages_per_seq=pages, max_pages=c["requests"] * pages,
                                          compute_dtype=c["dtype"], max_prefill_size=c["budget"], max_seqs_in_prefill=c["requests"])
    model = DecoderLm(LmConfig.from_dict(config(c)).model_spec(), weights(c, seed), make_env(c["dtype"]))
    engine = InferenceEngine.from_model_with_config(model, config=engine_config)
    state = {"engine": engine, "plan": plan(c), "tokens": token_ids(c, seed + 1)}
    run(state)  # the engine has served a session before: kernels are loaded, step shapes have been seen
    state["tokens"] = token_ids(c, seed)
    return state


def run(state):
    from levanter_amd.engine import StepEntry

    engine, tokens = state["engine"], state["tokens"]
    handles = [engine.cache.open(r) for r in range(len(tokens))]
    logits = [engine.runner.step([StepEntry(handles[r], tokens[r][p:p + n], want) for r, p, n, want in step]) for step in state["plan"]]
    for h in handles:
        engine.cache.close(h)
    return logits


# ---- what a session cannot do without -----------------------------------------------------------------------------------
def _kv_and_state(cfg):
    """(cached numbers a token, multiply-adds per query and key it sees, state numbers a request) of all layers together."""
    if cfg.get("model_type") == "gpt2":
        return 2 * cfg["n_embd"] * cfg["n_layer"], 2 * cfg["n_embd"] * cfg["n_layer"], 0
    cached = pairs = state = 0
    for i, _ in layer_order(cfg) if cfg.get("loop") else [(i, None) for i in range(len(cfg["layers"]))]:
        L = cfg["layers"][i]
        m = L["mixer"]
        if L["type"] == "latent_attention":
            cached += m["kv_rank"] + m["rot_dim"]
            pairs += m["heads"] * (2 * m["kv_rank"] + m["rot_dim"])
        elif L["type"] == "mamba2":
            state += m["heads"] * m["vdim"] * m["state"]
        else:
            a = m.get("left", m)
            cached += a["kv_heads"] * (a["dim"] + a["vdim"])
            pairs += a["heads"] * (a["dim"] + a["vdim"])
            if "right" in m:
                state += m["right"]["heads"] * m["right"]["dim"] * m["right"]["vdim"]
    return cached, pairs, state


def work(c):
    """Every step reads the matrices its tokens need once (of the experts those that its tokens choose) and the cache its tokens see, and
    writes the new cache entries and the wanted logits; states are read and written once a request and step."""
    cfg = config(c)
    size = 2 if c["dtype"] == "bfloat16" else 4
    runs = {}  # how often a layer runs in a step: one in a loop is read once and multiplied with every time
    for i, _ in layer_order(cfg) if cfg.get("loop") else []:
        runs[f"l{i}"] = runs.get(f"l{i}", 0) + 1
    matrices = products = experts = head = 0  # numbers read, numbers multiplied with per token, of the experts, of the head
    for name, (shape, _, _) in shapes(cfg).items():
        n = math.prod(shape)
        if name in ("wte.weight", "head"):
            head = n
        elif name in ("wpe.weight", "embed", "side.embed"):
            pass  # a row a token
        elif ".mlp.e" in name:
            experts += n
        else:
            matrices += n
            products += n * runs.get(name.split(".")[0], 1)
    vocab = GPT2_VOCAB if c["arch"] == "gpt2" else OTHER_VOCAB
    cached, pairs, state = _kv_and_state(cfg)
    n_experts, top = (32, 4) if c["arch"] == "kelasun" else (1, 1)
    byte = flop = 0.0
    for step in plan(c):
        T, rows = sum(n for _, _, n, _ in step), sum(len(w) for *_, w in step)
        touched = 1.0 - (1.0 - top / n_experts) ** T
        seen = sum(n * p + n * (n + 1) // 2 for _, p, n, _ in step)
        byte += size * (matrices + experts * touched + (head if rows else 0) + cached * sum(p + n for _, p, n, _ in step)) + 4.0 * rows * vocab + 8.0 * state * len(step)
        flop += 2.0 * T * (products + experts * top / n_experts) + 2.0 * rows * head + 2.0 * pairs * seen + 4.0 * state * T
    return {"bytes": byte, "flops": flop}


def tolerance(c):
    """Measured against ``exact``: 1.6e-6 .. 2.3e-6 in 32 bits; in bfloat16 0.004 .. 0.007 (GPT-2), 0.012 (Lelatar), 0.005 .. 0.013 (Kelasun, where
    a token now and then chooses another last expert)."""
    if c["dtype"] == "float32":
        return {"rel": 1e-5}
    return {"rel": 0.025 if c["arch"] == "gpt2" else 0.03}


# ---- the same sessions in 64 bits, plainly ------------------------------------------------------------------------------
class _Plain:
    """A model's logits for whole sequences in float64: all sequences' tokens one behind the other, ``self.spans`` says where each lies."""

    def __init__(self, c, seed):
        self.c, self.cfg, self.w = c, config(c), weights(c, seed)
        self.tokens = token_ids(c, seed)
        self.spans, at = [], 0
        for t in self.tokens:
            self.spans.append((at, at + len(t)))
            at += len(t)
        self.ids = torch.tensor([x for t in self.tokens for x in t], device="cuda")
        self.pos = torch.cat([torch.arange(len(t), device="cuda") for t in self.tokens])

    def W(self, name):
        return self.w[name].double()

    def lin(self, x, name):
        return x @ self.W(name).T

    def rms(self, x, w, eps):
        y = x / torch.sqrt((x * x).mean(-1, keepdim=True) + eps)
        return y if w is None else y * w

    def layer_norm(self, x, w, b, eps):
        d = x - x.mean(-1, keepdim=True)
        return d / torch.sqrt((d * d).mean(-1, keepdim=True) + eps) * w + b

    def attention(self, q, k, v, scale, slopes=None, sinks=None):
        """q ``[N, H, d]``, k ``[N, G, d]``, v ``[N, G, dv]`` -> ``[N, H * dv]``: causal softmax attention inside each sequence; a term
        -slope times the distance on the scores and exp(sink) in the denominator where given."""
        H, G = q.shape[1], k.shape[1]
        out = []
        for a, b in self.spans:
            far = (self.pos[a:b, None] - self.pos[None, a:b]).double()
            Q, K, Vv = (t[a:b].transpose(0, 1) for t in (q, k, v))
            K, Vv = K.repeat_interleave(H // G, 0).contiguous(), Vv.repeat_interleave(H // G, 0).contiguous()
            s = torch.matmul(Q.contiguous(), K.transpose(1, 2).contiguous()) * scale
            if slopes is not None:
                s = s - slopes[:, None, None] * far
            s = s.masked_fill(far < 0, -math.inf)
            if sinks is not None:
                s = torch.cat([s, sinks[:, None, None].expand(H, b - a, 1)], 2)
            p = torch.softmax(s, -1)[:, :, :b - a].contiguous()
            out.append(torch.matmul(p, Vv).transpose(0, 1).reshape(b - a, -1))
        return torch.cat(out)

    def turn(self, x, freqs, neighbours, magnitude=1.0):
        """x ``[N, heads, d]``: pairs of dimensions, neighbours or half the turned part apart, turn by position * frequency."""
        n = freqs.numel()
        a = self.pos.double()[:, None] * freqs[None]
        cos, sin = magnitude * torch.cos(a)[:, None], magnitude * torch.sin(a)[:, None]
        one, two = (slice(0, 2 * n, 2), slice(1, 2 * n, 2)) if neighbours else (slice(0, n), slice(n, 2 * n))
        out = x.clone()
        out[..., one], out[..., two] = x[..., one] * cos - x[..., two] * sin, x[..., two] * cos + x[..., one] * sin
        return out

    # -- GPT-2
    def gpt2(self):
        cfg, N = self.cfg, self.ids.numel()
        eps, H, d = cfg["layer_norm_epsilon"], cfg["n_head"], cfg["n_embd"]
        norm = lambda x, n: self.layer_norm(x, self.W(n + ".weight"), self.W(n + ".bias"), eps)
        lin = lambda x, n: x @ self.W(n + ".weight") + self.W(n + ".bias")
        x = self.w["wte.weight"][self.ids].double() + self.w["wpe.weight"][self.pos].double()
        for i in range(cfg["n_layer"]):
            q, k, v = (t.reshape(N, H, d // H) for t in lin(norm(x, f"h.{i}.ln_1"), f"h.{i}.attn.c_attn").split(d, 1))
            x = x + lin(self.attention(q, k, v, (d // H) ** -0.5), f"h.{i}.attn.c_proj")
            z = lin(norm(x, f"h.{i}.ln_2"), f"h.{i}.mlp.c_fc")
            x = x + lin(0.5 * z * (1 + torch.tanh(math.sqrt(2 / math.pi) * (z + 0.044715 * z ** 3))), f"h.{i}.mlp.c_proj")
        return norm(x, "ln_f"), lambda h: self.lin(h, "wte.weight")

    # -- Kelasun
    def kelasun_latent(self, h, p, m):
        N, H, dk, dv, R, eps = h.shape[0], m["heads"], m["dim"], m["vdim"], m["kv_rank"], self.cfg["norm"]["eps"]
        q = self.lin(self.rms(self.lin(h, p + "dq"), self.W(p + "dq.norm"), eps), p + "uq").view(N, H, -1)
        down = self.lin(h, p + "dkv")
        latent = self.rms(down[:, :R], self.W(p + "dkv.norm"), eps)
        rot = m["rot"]
        dims, base, sc = rot["dims"], rot["base"], rot["scaling"]
        plain = torch.tensor([base ** (-2.0 * i / dims) for i in range(dims // 2)], dtype=torch.float64, device="cuda")
        where = [dims * math.log(sc["original"] / (2 * math.pi * sc[k])) / (2 * math.log(base)) for k in ("fast", "slow")]
        lo, hi = max(math.floor(where[0]), 0), min(math.ceil(where[1]), dims - 1)
        ramp = ((torch.arange(dims // 2, device="cuda").double() - lo) / max(hi - lo, 0.001)).clamp(0, 1)
        turn = lambda x: self.turn(x, ramp * plain / sc["factor"] + (1 - ramp) * plain, True, 0.1 * math.log(sc["factor"]) + 1)
        k = torch.cat([self.lin(latent, p + "uk").view(N, H, dk), turn(down[:, None, R:]).expand(N, H, -1)], 2)
        o = self.attention(torch.cat([q[..., :dk], turn(q[..., dk:])], 2), k, self.lin(latent, p + "uv").view(N, H, dv), m["scale"])
        return self.lin(o * torch.sigmoid(self.lin(h, p + "g")), p + "o")

    def kelasun_attention(self, h, p, m):
        N, H, G, dk, dv, eps = h.shape[0], m["heads"], m["kv_heads"], m["dim"], m["vdim"], self.cfg["norm"]["eps"]
        warm = 1 + m["q_temp"]["coef"] * torch.log(torch.floor((self.pos.double() + 1) / m["q_temp"]["every"]) + 1)
        q = self.rms(self.lin(h, p + "q"), self.W(p + "q.norm"), eps) * warm[:, None]
        k = self.rms(self.lin(h, p + "k"), self.W(p + "k.norm"), eps)
        slopes = torch.tensor([2.0 ** (-8.0 * (i + 1) / H) for i in range(H)], dtype=torch.float64, device="cuda")
        o = self.attention(q.view(N, H, dk), k.view(N, G, dk), self.lin(h, p + "v").view(N, G, dv), m["scale"], slopes, self.W(p + "sink"))
        return self.lin((o.view(N, H, dv) * torch.sigmoid(self.lin(h, p + "g"))[:, :, None]).reshape(N, -1), p + "o")

    def kelasun_experts(self, h, p, mlp):
        expert = lambda t, n: self.lin(self.lin(t, f"{p}{n}.up").clamp(min=0) ** 2, f"{p}{n}.down")
        best = self.lin(h, p + "router").topk(mlp["router"]["top"], -1)
        share = torch.softmax(best.values, -1)
        y = expert(h, "shared")
        for e in range(mlp["router"]["experts"]):
            rows, choice = (best.indices == e).nonzero(as_tuple=True)
            y[rows] += share[rows, choice][:, None] * expert(h[rows], f"e{e}")
        return y

    def kelasun(self):
        cfg = self.cfg
        x = self.w["embed"][self.ids].double()
        after = lambda x, y, n: self.layer_norm(cfg["postln_alpha"] * x + y, self.W(n), 0, cfg["norm"]["eps"])
        for i, L in enumerate(cfg["layers"]):
            mixer = self.kelasun_attention if L["type"] == "attention" else self.kelasun_latent
            x = after(x, mixer(x, f"l{i}.mix.", L["mixer"]), f"l{i}.norm1")
            x = after(x, self.kelasun_experts(x, f"l{i}.mlp.", L["mlp"]), f"l{i}.norm2")
        return self.layer_norm(x, self.W("final.norm"), 0, cfg["norm"]["eps"]), lambda h: self.lin(h, "head") * cfg["logit_scale"]

    # -- Lelatar
    def conv(self, x, taps, bias=None):
        """Causal convolution of every channel inside each sequence, then x * sigmoid(x)."""
        out = torch.zeros_like(x)
        K = taps.shape[1]
        for a, b in self.spans:
            for k in range(min(K, b - a)):
                out[a + k:b] += x[a:b - k] * taps[:, K - 1 - k]
        out = out if bias is None else out + bias
        return out * torch.sigmoid(out)

    def padded(self, x):
        return torch.nn.utils.rnn.pad_sequence([x[a:b] for a, b in self.spans], batch_first=True)

    def unpadded(self, y):
        return torch.cat([y[i, :b - a] for i, (a, b) in enumerate(self.spans)])

    def lelatar_mamba(self, h, p, m):
        H, P, S, G, eps = m["heads"], m["vdim"], m["state"], m["groups"], self.cfg["norm"]["eps"]
        inner, N = H * P, h.shape[0]
        z, xbc, dt = self.lin(h, p + "in").split([inner, inner + 2 * G * S, H], 1)
        x, B, C = self.conv(xbc, self.W(p + "conv"), self.W(p + "conv.b")).split([inner, G * S, G * S], 1)
        dt = torch.nn.functional.softplus(dt + self.W(p + "dt_bias"), threshold=1000)
        wide = lambda t: self.padded(t.reshape(N, G, S).repeat_interleave(H // G, 1))
        X, B, C = self.padded(x.reshape(N, H, P)), wide(B), wide(C)
        keep, step = self.padded(torch.exp(-torch.exp(self.W(p + "A_log")) * dt)), self.padded(dt)
        B = B * step[..., None]
        state = torch.zeros(X.shape[0], H, S, P, dtype=torch.float64, device="cuda")
        y = torch.empty_like(X)
        for t in range(X.shape[1]):
            state = keep[:, t, :, None, None] * state + B[:, t, :, :, None] * X[:, t, :, None, :]
            y[:, t] = (state * C[:, t, :, :, None]).sum(2)
        y = self.unpadded(y + self.W(p + "D")[:, None] * X).reshape(N, inner) * (z * torch.sigmoid(z))
        return self.lin(self.rms(y.view(N, m["norm_groups"], -1), None, eps).reshape(N, inner) * self.W(p + "norm"), p + "o")

    def lelatar_attention(self, h, p, m):
        N, H, G, dk, dv, eps = h.shape[0], m["heads"], m["kv_heads"], m["dim"], m["vdim"], self.cfg["norm"]["eps"]
        n, base = m["rot"]["dims"], m["rot"]["base"]
        freqs = torch.tensor([base ** (-2.0 * i / n) for i in range(n // 2)], dtype=torch.float64, device="cuda")
        q = self.turn(self.rms(self.lin(h, p + "q"), self.W(p + "q.norm"), eps).view(N, H, dk), freqs, False)
        k = self.turn(self.rms(self.lin(h, p + "k"), self.W(p + "k.norm"), eps).view(N, G, dk), freqs, False)
        return self.lin(self.attention(q, k, self.lin(h, p + "v").view(N, G, dv), m["scale"], sinks=self.W(p + "sink")), p + "o")

    def lelatar_delta(self, h, p, m):
        N, H, G, d, dv, eps = h.shape[0], m["heads"], m["kv_heads"], m["dim"], m["vdim"], self.cfg["norm"]["eps"]
        q, k, v = (self.conv(self.lin(h, p + n), self.W(p + n + ".conv")) for n in ("q", "k", "v"))
        unit = lambda x: x / torch.sqrt((x * x).sum(-1, keepdim=True) + 1e-6)
        wide = lambda t: self.padded(unit(t.view(N, G, d)).repeat_interleave(H // G, 1))
        Q, K, Vv = wide(q) * d ** -0.5, wide(k), self.padded(v.reshape(N, H, dv))
        beta = self.padded(torch.sigmoid(self.lin(h, p + "b")))
        keep = self.padded(torch.exp(-torch.exp(self.W(p + "A_log")) * torch.nn.functional.softplus(self.lin(h, p + "a") + self.W(p + "dt_bias"), threshold=1000)))
        state = torch.zeros(Q.shape[0], H, d, dv, dtype=torch.float64, device="cuda")
        o = torch.empty_like(Vv)
        for t in range(Q.shape[1]):
            state = keep[:, t, :, None, None] * state
            new = beta[:, t, :, None] * (Vv[:, t] - (state * K[:, t, :, :, None]).sum(2))
            state = state + K[:, t, :, :, None] * new[:, :, None, :]
            o[:, t] = (state * Q[:, t, :, :, None]).sum(2)
        g = self.lin(h, p + "g")
        return self.lin(self.rms(self.unpadded(o), self.W(p + "norm"), eps).reshape(N, -1) * (g * torch.sigmoid(g)), p + "o")

    def lelatar(self):
        cfg, eps, side = self.cfg, self.cfg["norm"]["eps"], self.cfg["token_side"]["dim"]
        norm = lambda x, n: self.rms(x, 1 + self.W(n), eps)
        silu = lambda z: z * torch.sigmoid(z)
        x = x0 = self.w["embed"][self.ids].double()
        for i, run in layer_order(cfg):
            L, p = cfg["layers"][i], f"l{i}."
            if run is not None:
                x = self.lin(torch.cat([x, x0], 1), "loop.in") + self.W("loop.step")[run]
            h = norm(x, p + "norm1")
            if L["type"] == "mamba2":
                x = x + self.lelatar_mamba(h, p + "mix.", L["mixer"])
            else:
                left = self.rms(self.lelatar_attention(h, p + "mix.left.", L["mixer"]["left"]), self.W(p + "mix.left.out"), eps)
                right = self.rms(self.lelatar_delta(h, p + "mix.right.", L["mixer"]["right"]), self.W(p + "mix.right.out"), eps)
                x = x + 0.5 * (left + right)
            if L["mlp"] is not None:
                h = norm(x, p + "norm2")
                x = x + self.lin(silu(self.lin(h, p + "mlp.gate")) * self.lin(h, p + "mlp.up"), p + "mlp.down")
            row = self.w["side.embed"][self.ids][:, i * side:(i + 1) * side].double()
            z = self.lin(x, p + "side.gate")
            z = 0.5 * z * (1 + torch.tanh(math.sqrt(2 / math.pi) * (z + 0.044715 * z ** 3)))
            x = x + self.rms(self.lin(z * row, p + "side.proj"), self.W(p + "side.norm"), eps)
        return norm(x, "final.norm"), lambda h: self.lin(h, "head")


@torch.no_grad()
def exact(c, seed):
    m = _Plain(c, seed)
    h, head = getattr(m, c["arch"])()
    return [head(h[[m.spans[r][0] + p + w for r, p, _, want in step for w in want]]) for step in plan(c)]
