"""What a user of the engine has it do, as cases that can be timed and compared.

A case is one call after another of the step function (`ModelRunner.step`, which generation and trace
replay both go through) on a model of random weights: a number of live requests that decode on by a
token each, beside new requests whose prompts enter whole or in portions and that are taken out
again when their last portion has given its logits. What a case returns are the logits. Live
requests keep what they have decoded, so a pass over a state finds their contexts a token longer
than the pass before, as in generation.

    model      "0.6b", "8b" (Qwen3ForCausalLM at the sizes bench.py gives those names) or "surasun"
               (Mamba-2, Griffin's recurrent unit, softmax attention beside retention, a residual in
               four streams; bench.py's "base")
    dtype      "bfloat16" or "float32"
    live       requests that decode, one token each a step
    context    tokens the longest of them holds; `shortest` the shortest, the others in between
    prompts    new requests, `tokens` prompt tokens in all, of uneven lengths
    portion    prompt tokens a step takes in at most (0: all of them in one step)
"""

import hashlib
import math

import torch

PAGE = 16                  # tokens of a cache page, the engine's default
ROOM = 2048                # tokens a live request may grow by
FILL = 8192                # prompt tokens a step takes in while live requests are filled

QWEN3 = {
    "0.6b": dict(vocab_size=151936, hidden_size=1024, num_hidden_layers=28, num_attention_heads=16,
                 num_key_value_heads=8, head_dim=128, intermediate_size=4096, rms_norm_eps=1e-5, rope_theta=100000.0),
    "8b": dict(vocab_size=151936, hidden_size=4096, num_hidden_layers=36, num_attention_heads=32,
               num_key_value_heads=8, head_dim=128, intermediate_size=12288, rms_norm_eps=1e-6, rope_theta=1000000.0),
}
SURASUN = dict(vocab=32768, width=2048, streams=4, ff=6144, eps=1e-5,
               mamba2=dict(heads=64, vdim=64, state=128, groups=1, conv=4, norm_groups=1),
               rglru=dict(width=2048, blocks=8, conv=4),
               left=dict(heads=16, kv_heads=4, dim=128, vdim=128, scale=128 ** -0.5, softcap=50.0,
                         rot=dict(dims=64, base=10000.0)),
               right=dict(heads=8, dim=128, vdim=256, rot=dict(dims=128, base=10000.0),
                          decay=[1.0 - 2.0 ** (-5 - i) for i in range(8)]),
               scales=(0.5, 0.5), layers=(("mamba2", False), ("rglru", True), ("parallel", True), ("mamba2", False)))


def _width(case):
    return SURASUN["width"] if case["model"] == "surasun" else QWEN3[case["model"]]["hidden_size"]


def _vocab(case):
    return SURASUN["vocab"] if case["model"] == "surasun" else QWEN3[case["model"]]["vocab_size"]


def _std(case):
    """The deviation of the random weights: 0.02 at a width of 1,024 and as much less as keeps a product's
    results there at any width, where depth does not make rounding grow past what it is in a trained model."""
    return 0.64 * _width(case) ** -0.5


def _case(name, model, dtype="bfloat16", live=0, context=0, shortest=None, prompts=0, tokens=0, portion=0):
    case = {"model": model, "dtype": dtype, "live": live, "context": context,
            "shortest": context if shortest is None else shortest, "prompts": prompts, "tokens": tokens, "portion": portion}
    return dict(case, name=name) if name else case


def listed():
    return [
        # one user of the small model, in the middle of an answer: launches and latency are everything
        _case("decode_0.6b_1", "0.6b", live=1, context=1100),
        # the reference's own load: 20 requests in flight, 512 tokens in and up to 512 out
        _case("decode_0.6b_20", "0.6b", live=20, context=1030, shortest=512),
        # three short questions that arrive together
        _case("prompts_0.6b_3x67", "0.6b", prompts=3, tokens=201),
        # the float32 path as trace replay uses it: two prompts beside three requests that decode
        _case("float32_0.6b_mixed", "0.6b", "float32", live=3, context=150, shortest=40, prompts=2, tokens=333),
        # the headline's three batch sizes, behind prompts of 2,048 tokens
        _case("decode_8b_1", "8b", live=1, context=2060),
        _case("decode_8b_8", "8b", live=8, context=2060, shortest=2048),
        _case("decode_8b_64", "8b", live=64, context=2060, shortest=2048),
        # the headline's prompt, whole in one step
        _case("prompt_8b_2048", "8b", prompts=1, tokens=2048),
        # a document: as many tokens as the headline's context holds
        _case("prompt_8b_8192", "8b", prompts=1, tokens=8192),
        # continuous batching: a prompt enters in portions of 512 beside 23 requests that decode
        _case("portions_8b_1300", "8b", live=23, context=3000, shortest=150, prompts=1, tokens=1300, portion=512),
        # the design with recurrent mixers and streams, decoding and taking a prompt in
        _case("decode_surasun_8", "surasun", live=8, context=1100, shortest=900),
        _case("prompt_surasun_2048", "surasun", prompts=1, tokens=2048),
    ]


def _between(rng, low, high):
    """A whole number between the two, spread over their logarithm."""
    return max(low, min(high, round(math.exp(rng.uniform(math.log(low), math.log(high + 0.499))))))


def draw(rng):
    model = rng.choice(["0.6b", "0.6b", "8b", "8b", "8b", "surasun"])
    dtype = "float32" if model == "0.6b" and rng.random() < 0.25 else "bfloat16"
    most = 600 if dtype == "float32" else 8192 if model == "8b" else 4096
    kind = rng.choice(["decode", "decode", "prompts", "portions"])
    live = context = shortest = prompts = tokens = portion = 0
    if kind != "prompts":
        live = _between(rng, 1, 8 if dtype == "float32" else 64 if kind == "decode" else 40)
        context = _between(rng, 100, 400 if dtype == "float32" else min(4096, 120000 // live))
        shortest = rng.randint(max(1, context // 4), context)
    if kind != "decode":
        prompts = rng.randint(1, 3)
        tokens = _between(rng, 16, most if kind == "prompts" else min(most, 1500))
        portion = 512 if kind == "portions" else 0
    return _case(None, model, dtype, live, context, shortest, prompts, tokens, portion)


# ---- what a user's program has in hand ----

def _config(case):
    if case["model"] == "surasun":
        from qwen3_from_scratch_amd.config.surasun_config import SurasunConfig

        c = SURASUN
        mixers = {"mamba2": c["mamba2"], "rglru": c["rglru"],
                  "parallel": {"left": c["left"], "right": c["right"], "left_scale": c["scales"][0], "right_scale": c["scales"][1]}}
        return SurasunConfig.from_dict({
            "architecture": "Surasun", "vocab": c["vocab"], "width": c["width"], "norm": {"eps": c["eps"]},
            "residual_mult": 1.0, "streams": c["streams"],
            "layers": [{"type": kind, "mixer": mixers[kind], "mlp": {"kind": "dense", "ff": c["ff"]} if fed else None}
                       for kind, fed in c["layers"]]})
    from qwen3_from_scratch_amd.config import ModelConfig

    return ModelConfig.from_dict(dict(QWEN3[case["model"]], architectures=["Qwen3ForCausalLM"], hidden_act="silu",
                                      max_position_embeddings=40960, tie_word_embeddings=False))


def _contexts(case):
    n, longest, shortest = case["live"], case["context"], case["shortest"]
    return [longest - (longest - shortest) * i // max(1, n - 1) for i in range(n)]


def _prompt_lengths(case):
    n, total = case["prompts"], case["tokens"]
    lengths = [max(1, total * 2 * (i + 1) // (n * (n + 1))) for i in range(n - 1)]
    return lengths + [max(1, total - sum(lengths))] if n else []


def _plan(case):
    """Per step of a pass: the prompts' slices as (prompt, first token, end)."""
    portion = case["portion"] or case["tokens"]
    steps, slices, room = [], [], portion
    for p, length in enumerate(_prompt_lengths(case)):
        at = 0
        while at < length:
            n = min(room, length - at)
            slices.append((p, at, at + n))
            at, room = at + n, room - n
            if room == 0:
                steps.append(slices)
                slices, room = [], portion
    if slices:
        steps.append(slices)
    return steps or [[]]


def _tokens(case, seed):
    """(tokens of every live request: what it holds, then as many as it may decode; tokens of every prompt)"""
    gen = torch.Generator().manual_seed(int(seed))

    def some(n):
        return torch.randint(0, _vocab(case), (n,), generator=gen).tolist()

    return [some(n + ROOM) for n in _contexts(case)], [some(n) for n in _prompt_lengths(case)]


def prepare(case, seed):
    from qwen3_from_scratch_amd.engine import ModelRunner, StepEntry, random_model

    live, prompts = _tokens(case, seed)
    held = _contexts(case)
    model = random_model(_config(case), dtype=case["dtype"], device="cuda:0", seed=int(seed), std=_std(case))
    pages = sum(-(-(n + ROOM) // PAGE) for n in held) + sum(-(-len(p) // PAGE) for p in prompts) + 1
    runner = ModelRunner(model, PAGE, pages, max_requests=max(1, len(live) + len(prompts)))
    # as SyncEngine.warmup() does it: what is built at first use is built
    runner.step([StepEntry("warm", [1, 2, 3], [2])])
    runner.finish("warm")
    # the live requests' contexts but their last token, then that one as a decode step
    entries, room = [], FILL
    for i, tokens in enumerate(live):
        at = 0
        while at < held[i] - 1:
            n = min(room, held[i] - 1 - at)
            entries.append(StepEntry("live %d" % i, tokens[at:at + n], []))
            at, room = at + n, room - n
            if room == 0:
                runner.step(entries)
                entries, room = [], FILL
    if entries:
        runner.step(entries)
    if live:
        runner.step([StepEntry("live %d" % i, [tokens[n - 1]], [0]) for i, (tokens, n) in enumerate(zip(live, held))])
    return {"runner": runner, "live": live, "at": held, "prompts": prompts, "plan": _plan(case)}


def run(state):
    from qwen3_from_scratch_amd.engine import StepEntry

    runner, outputs = state["runner"], []
    for slices in state["plan"]:
        entries = [StepEntry("live %d" % i, [tokens[at]], [0]) for i, (tokens, at) in enumerate(zip(state["live"], state["at"]))]
        state["at"] = [at + 1 for at in state["at"]]
        ended = []
        for p, first, end in slices:
            tokens = state["prompts"][p]
            last = end == len(tokens)
            entries.append(StepEntry("prompt %d" % p, tokens[first:end], [end - first - 1] if last else []))
            if last:
                ended.append("prompt %d" % p)
        logits = runner.step(entries)
        for request in ended:
            runner.finish(request)
        if len(state["plan"]) > 1:
            logits = logits.clone()            # the next step may write over them
        outputs.append(logits)
    return outputs


# ---- what a pass cannot do without ----

def _sequences(case):
    """Per sequence of a pass: (tokens it holds before, new tokens, rows of logits)"""
    steps = len(_plan(case))
    return [(n, steps, steps) for n in _contexts(case)] + [(0, n, 1) for n in _prompt_lengths(case)]


def work(case):
    size = 4 if case["dtype"] == "float32" else 2
    steps = len(_plan(case))
    sequences = _sequences(case)
    new, rows = sum(n for _, n, _ in sequences), sum(r for _, _, r in sequences)
    if case["model"] == "surasun":
        c = SURASUN
        W, vocab, m, r, left, right = c["width"], c["vocab"], c["mamba2"], c["rglru"], c["left"], c["right"]
        inner = m["heads"] * m["vdim"]
        mamba = W * (2 * inner + 2 * m["groups"] * m["state"] + m["heads"]) + W * inner
        unit = 3 * W * r["width"] + 2 * r["width"] ** 2 // r["blocks"]
        both = (W * (2 * left["heads"] + 2 * left["kv_heads"]) * left["dim"] + left["heads"] * W
                + right["heads"] * W * (2 * right["dim"] + 3 * right["vdim"]))
        weights = 2 * mamba + unit + both + 2 * 3 * W * c["ff"]
        # beside the products: a recurrence's update and read, three multiply-adds a number of state
        states = 2 * m["heads"] * m["state"] * m["vdim"] + right["heads"] * right["dim"] * right["vdim"]
        each = weights + 3 * states
        held_each = states + 2 * (m["conv"] - 1) * (inner + 2 * m["groups"] * m["state"]) + r["conv"] * r["width"]
        cached, pair = left["kv_heads"] * (left["dim"] + left["vdim"]), left["heads"] * (left["dim"] + left["vdim"])
    else:
        c = QWEN3[case["model"]]
        W, D, layers, vocab, held_each = c["hidden_size"], c["head_dim"], c["num_hidden_layers"], c["vocab_size"], 0
        H, G = c["num_attention_heads"], c["num_key_value_heads"]
        weights = each = layers * ((H + 2 * G) * D * W + H * D * W + 3 * W * c["intermediate_size"])
        cached, pair = layers * 2 * G * D, layers * H * 2 * D
    seen = sum(held + i + 1 for held, n, _ in sequences for i in range(n))
    read = sum(held for held, _, _ in sequences) * steps
    kept = 4 * held_each * sum(2 * steps if held else 1 for held, _, _ in sequences)
    return {"bytes": size * (steps * (weights + vocab * W) + cached * (read + new) + new * W) + 4 * rows * vocab + kept,
            "flops": 2 * (new * each + rows * vocab * W + seen * pair)}


def tolerance(case):
    """The same tokens cut into steps in other ways (other kernels, other orders of the sums) give logits that
    differ by 0.007 to 0.009 ("0.6b"), about 0.01 ("8b") and 0.015 to 0.018 ("surasun") in bfloat16, and by up to
    3e-6 in float32; a pass is off `exact` by 0.008 to 0.013, 0.03 ("surasun") and 2.5e-6."""
    return {"rel": 1e-5} if case["dtype"] == "float32" else {"rel": 0.03}


# ---- the same in 64 bits ----

def _weight(case, seed, name, shape, kind="matrix"):
    """The engine's seeded random weights: every tensor from a generator of its own, seeded by (seed, name)."""
    digest = hashlib.sha256(("%d:%s" % (int(seed), name)).encode()).digest()
    gen = torch.Generator(device="cuda:0")
    gen.manual_seed(int.from_bytes(digest[:8], "little") & 0x7FFFFFFFFFFFFFFF)
    if kind == "scale":
        t = 1.0 + (2.0 * torch.rand(shape, generator=gen, device="cuda:0", dtype=torch.float32) - 1.0) * 0.1
    else:
        t = torch.randn(shape, generator=gen, device="cuda:0", dtype=torch.float32) * _std(case)
    return t.to(torch.bfloat16).double()


def _norm(x, weight, eps):
    return x / torch.sqrt((x * x).mean(dim=-1, keepdim=True) + eps) * weight


def _in_rows(f, x, rows=8192):
    return torch.cat([f(part) for part in x.split(rows)])


def _attended(q, k, v, scale, cap=None):
    """q (heads, T, d), k and v (1, T, .): causal attention, some queries at a time; scores bent to cap tanh(s / cap)."""
    T = q.shape[1]
    at = torch.arange(T, device=q.device)
    out = []
    for first in range(0, T, 2048):
        end = min(T, first + 2048)
        s = torch.matmul(q[:, first:end], k[:, :end].transpose(1, 2)) * scale
        if cap:
            s = cap * torch.tanh(s / cap)
        hidden = at[first:end, None] < at[None, :end]
        out.append(torch.matmul(torch.softmax(s.masked_fill(hidden, float("-inf")), dim=-1), v[:, :end]))
    return torch.cat(out, dim=1)


def _qwen3_rows(case, seed, sequences, wanted):
    c = QWEN3[case["model"]]
    W, D, H, G, I, eps = (c["hidden_size"], c["head_dim"], c["num_attention_heads"], c["num_key_value_heads"],
                          c["intermediate_size"], c["rms_norm_eps"])
    lengths = [len(s) for s in sequences]
    ids = torch.tensor([t for s in sequences for t in s], device="cuda:0")
    x = _weight(case, seed, "model.embed_tokens.weight", (c["vocab_size"], W))[ids]
    exponent = torch.arange(0, D, 2, dtype=torch.float32) / D
    f = (1.0 / (c["rope_theta"] ** exponent)).double().cuda()
    at = torch.cat([torch.arange(n) for n in lengths]).cuda()
    cos, sin = ((at[:, None] * f[None, :]).cos()[:, None, :], (at[:, None] * f[None, :]).sin()[:, None, :])

    def turned(y):
        a, b = y[..., :D // 2], y[..., D // 2:]
        return torch.cat((a * cos - b * sin, b * cos + a * sin), dim=-1)

    for i in range(c["num_hidden_layers"]):
        p = "model.layers.%d." % i
        h = _norm(x, _weight(case, seed, p + "input_layernorm.weight", (W,), "scale"), eps)
        q, k, v = ((h @ _weight(case, seed, p + "self_attn.%s_proj.weight" % n, (heads * D, W)).T).view(-1, heads, D)
                   for n, heads in (("q", H), ("k", G), ("v", G)))
        q = turned(_norm(q, _weight(case, seed, p + "self_attn.q_norm.weight", (D,), "scale"), eps))
        k = turned(_norm(k, _weight(case, seed, p + "self_attn.k_norm.weight", (D,), "scale"), eps))
        o = torch.empty_like(q)
        first = 0
        for n in lengths:
            part = slice(first, first + n)
            for g in range(G):
                heads = slice(g * (H // G), (g + 1) * (H // G))
                o[part, heads] = _attended(q[part, heads].transpose(0, 1), k[part, g][None], v[part, g][None],
                                               D ** -0.5).transpose(0, 1)
            first += n
        x = x + o.reshape(-1, H * D) @ _weight(case, seed, p + "self_attn.o_proj.weight", (W, H * D)).T
        gate, up, down = (_weight(case, seed, p + "mlp.%s_proj.weight" % n, s)
                          for n, s in (("gate", (I, W)), ("up", (I, W)), ("down", (W, I))))
        norm = _weight(case, seed, p + "post_attention_layernorm.weight", (W,), "scale")

        def fed(rows):
            h = _norm(rows, norm, eps)
            a = h @ gate.T
            return (h @ up.T * (a * torch.sigmoid(a))) @ down.T

        x = x + _in_rows(fed, x)
    x = _norm(x[wanted], _weight(case, seed, "model.norm.weight", (W,), "scale"), eps)
    return x @ _weight(case, seed, "lm_head.weight", (c["vocab_size"], W)).T


def _surasun_rows(case, seed, sequences, wanted):
    c = SURASUN
    W, eps, n = c["width"], c["eps"], c["streams"]

    def weight(name, *shape, kind="matrix"):
        return _weight(case, seed, name, shape, kind)

    def layer_norm(x, name):
        x = x - x.mean(dim=-1, keepdim=True)
        return _norm(x, weight(name, W, kind="scale"), eps)

    def silu(z):
        return z * torch.sigmoid(z)

    def conv(x, p, taps):
        channels = x.shape[1]
        w, out = weight(p + "conv", channels, taps), weight(p + "conv.b", channels).expand(x.shape[0], channels).clone()
        for j in range(min(taps, x.shape[0])):
            out[j:] += w[:, taps - 1 - j] * x[:x.shape[0] - j]
        return out

    def angles(T, rot):
        f = torch.tensor([rot["base"] ** (-2.0 * i / rot["dims"]) for i in range(rot["dims"] // 2)]).double().cuda()
        a = torch.arange(T, device="cuda:0")[:, None, None] * f
        return a.cos(), a.sin()

    def decayed(q, k, v, log_decay):
        """sum over j <= i of (q_i . k_j) exp(log_decay_i - log_decay_j) v_j; heads first, log_decay their running sum"""
        back = (log_decay[:, :, None] - log_decay[:, None, :]).tril()
        return torch.matmul((torch.matmul(q, k.transpose(1, 2)) * back.exp()).tril(), v)

    def mamba2(h, p):
        m, T = c["mamba2"], h.shape[0]
        H, P, N = m["heads"], m["vdim"], m["state"]
        inner = H * P
        z, x, dt = (h @ weight(p + "in", 2 * inner + 2 * N + H, W).T).split((inner, inner + 2 * N, H), dim=1)
        x, B, C = silu(conv(x, p, m["conv"])).split((inner, N, N), dim=1)
        x = x.reshape(T, H, P)
        dt = torch.nn.functional.softplus(dt + weight(p + "dt_bias", H))
        log_decay = (-dt * weight(p + "A_log", H).exp()).cumsum(dim=0)
        y = torch.cat([decayed(C[None], B[None], (dt[:, a, None] * x[:, a])[None], log_decay[None, :, a]) for a in range(H)])
        y = (y.transpose(0, 1) + weight(p + "D", H, kind="scale")[:, None] * x).reshape(T, inner) * silu(z)
        return _norm(y, weight(p + "norm", inner, kind="scale"), eps) @ weight(p + "o", W, inner).T

    def rglru(h, p):
        m, T = c["rglru"], h.shape[0]
        width, blocks = m["width"], m["blocks"]
        b = width // blocks
        y = torch.nn.functional.gelu(h @ weight(p + "y", width, W).T + weight(p + "y.b", width), approximate="tanh")
        u = conv(h @ weight(p + "x", width, W).T + weight(p + "x.b", width), p, m["conv"])
        r, i = (torch.sigmoid(torch.matmul(u.view(T, blocks, b).transpose(0, 1), weight(p + g, blocks, b, b).transpose(1, 2)).transpose(0, 1)
                              + weight(p + g + ".b", blocks, b)).reshape(T, width) for g in ("ra", "ri"))
        a = torch.exp(-8.0 * r * torch.nn.functional.softplus(weight(p + "lam", width)))
        out = torch.sqrt(1.0 - a * a) * i * u
        for t in range(1, T):
            out[t].addcmul_(a[t], out[t - 1])
        return (out * y) @ weight(p + "o", W, width).T

    def attention(h, p):
        m, T = c["left"], h.shape[0]
        H, G, d = m["heads"], m["kv_heads"], m["dim"]
        cos, sin = angles(T, m["rot"])

        def turned(x):
            x, kept = x[..., :m["rot"]["dims"]], x[..., m["rot"]["dims"]:]
            x = torch.stack((x[..., 0::2] * cos - x[..., 1::2] * sin, x[..., 1::2] * cos + x[..., 0::2] * sin), dim=-1)
            return torch.cat((x.flatten(-2), kept), dim=-1)

        q, k, v = (h @ weight(p + name, heads * d, W).T + weight(p + name + ".b", heads * d)
                   for name, heads in (("q", H), ("k", G), ("v", G)))
        q = turned(_norm(q, weight(p + "q.norm", H * d, kind="scale"), eps).view(T, H, d)).transpose(0, 1)
        k = turned(_norm(k, weight(p + "k.norm", G * d, kind="scale"), eps).view(T, G, d)).transpose(0, 1)
        v = v.view(T, G, d).transpose(0, 1)
        o = torch.cat([_attended(q[g * (H // G):(g + 1) * (H // G)], k[g][None], v[g][None], m["scale"], m["softcap"])
                       for g in range(G)]).transpose(0, 1)
        o = o * torch.sigmoid(h @ weight(p + "g", H, W).T)[:, :, None]
        return o.reshape(T, H * d) @ weight(p + "o", W, H * d).T

    def retention(h, p):
        m, T = c["right"], h.shape[0]
        H, d, dv = m["heads"], m["dim"], m["vdim"]
        cos, sin = angles(T, m["rot"])

        def turned(x):
            a, b = x[..., :d // 2], x[..., d // 2:]
            return torch.cat((a * cos - b * sin, b * cos + a * sin), dim=-1).transpose(0, 1)

        q, k, v, g = (h @ weight(p + name, H * size, W).T for name, size in (("q", d), ("k", d), ("v", dv), ("g", dv)))
        log_decay = torch.tensor(m["decay"], dtype=torch.float64).log().cuda()[:, None] * torch.arange(T, device="cuda:0")
        o = decayed(turned(q.view(T, H, d)), turned(k.view(T, H, d)) * d ** -0.5, v.view(T, H, dv).transpose(0, 1), log_decay)
        o = _norm(o, 1.0, eps).transpose(0, 1).reshape(T, H * dv)
        return (o * silu(g)) @ weight(p + "o", W, H * dv).T

    def mixed(kind, h, p):
        if kind == "parallel":
            return c["scales"][0] * attention(h, p + "left.") + c["scales"][1] * retention(h, p + "right.")
        return mamba2(h, p) if kind == "mamba2" else rglru(h, p)

    def sublayer(xs, p, number, f):
        hc = p + "hc%d." % number
        read, write, mix = weight(hc + "in", n, kind="scale"), weight(hc + "out", n, kind="scale"), weight(hc + "mix", n, n)
        y = f(layer_norm(sum(read[s] * xs[s] for s in range(n)), p + "norm%d" % number))
        return [sum(mix[s, t] * xs[s] for s in range(n)) + write[t] * y for t in range(n)]

    ids = torch.tensor([t for s in sequences for t in s], device="cuda:0")
    lengths, embed = [len(s) for s in sequences], weight("embed", c["vocab"], W)
    xs = [embed[ids]] * n
    for i, (kind, fed) in enumerate(c["layers"]):
        p = "l%d." % i
        xs = sublayer(xs, p, 1, lambda h: torch.cat([mixed(kind, part, p + "mix.") for part in h.split(lengths)]))
        if fed:
            gate, up, down = (weight(p + "mlp." + name, *shape)
                              for name, shape in (("gate", (c["ff"], W)), ("up", (c["ff"], W)), ("down", (W, c["ff"]))))
            xs = sublayer(xs, p, 2, lambda h: _in_rows(lambda rows: (silu(rows @ gate.T) * (rows @ up.T)) @ down.T, h))
    return layer_norm(sum(xs)[wanted], "final.norm") @ embed.T


def exact(case, seed):
    """The first pass over a prepared state, every sequence whole from its first token on."""
    live, prompts = _tokens(case, seed)
    steps = _plan(case)
    sequences = [tokens[:n + len(steps)] for tokens, n in zip(live, _contexts(case))] + prompts
    if sum(map(len, sequences)) * (15e9 if case["model"] == "8b" else 1e9) > 400e12:
        return None                        # over about 20 seconds
    first, starts = 0, []
    for s in sequences:
        starts.append(first)
        first += len(s)
    wanted, rows = [], []                  # places among all tokens, in the order of the steps' logits
    for i, slices in enumerate(steps):
        here = [starts[j] + n + i for j, n in enumerate(_contexts(case))]
        here += [starts[len(live) + p] + end - 1 for p, _, end in slices if end == len(prompts[p])]
        wanted += here
        rows.append(len(here))
    one = _surasun_rows if case["model"] == "surasun" else _qwen3_rows
    logits = one(case, seed, sequences, torch.tensor(wanted, device="cuda:0"))
    return list(logits.split(rows))
