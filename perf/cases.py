"""What programs have this framework do, as cases that can be timed: decode steps of the Qwen models, attention over prompts through the `hip` attention module, and
the mechanisms of the other models over prompts (attention over pages, experts, lightning attention, time mixing, selective scan, gated recurrence).

    listed() / draw(rng)      cases: dicts of plain values
    prepare(case, seed)       what a program has in hand before the call
    run(state)                one pass, and its outputs
    work(case)                bytes and operations a pass cannot do without
    tolerance(case)           how far two correct implementations may be apart
    exact(case, seed)         the outputs in 64 bits by plain torch

Model shapes are those of models/qwen.py, mechanism sizes those of bench_models.SIZES; everything runs in bfloat16 with 32-bit states, as the engine does.
"""
import math
import os
import random
import sys

import torch
import torch.nn.functional as F

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
PKG = os.path.join(ROOT, "nano-vllm-learn_amd")
if PKG not in sys.path:
    sys.path.insert(0, PKG)

BF16, F32, F64 = torch.bfloat16, torch.float32, torch.float64
EPS = 1e-6
BLOCK = 256                                    # tokens per page of the Qwen models' cache
PAGE = 64                                      # tokens per page of the other models'
# query heads, key heads, width of a head: the attention shapes of Qwen2-0.5B, Qwen3-0.6B, Qwen2-7B and of one of its ranks at four
HEADS = {"14/2/64": (14, 2, 64), "16/8/128": (16, 8, 128), "28/4/128": (28, 4, 128), "7/1/128": (7, 1, 128)}
# width, attention heads, key heads, width of the gated recurrence and its blocks, feed-forward of one of 32 experts
SIZES = {"1k": (1024, 8, 2, 1024, 4, 768), "2k": (2048, 16, 4, 2560, 10, 1536), "4k": (4096, 32, 8, 4096, 16, 3072)}
EXPERTS, TOP = 32, 4
STATES = 16                                    # of a scan channel
RECURRENT = ("lightning", "time_mixing", "scan", "recurrence")


# ------------------------------------------------------------------------------------------------ the cases
def listed():
    return [
        # one chat user: a decode step is about 120 launches that stream the weights once
        dict(name="decode qwen2 0.5b x1", kind="decode", model="Qwen2-0.5B", batch=1, shortest=513, longest=1024),
        # the headline workload: 32 sequences, prompts and answers of 1024 tokens
        dict(name="decode qwen2 0.5b x32", kind="decode", model="Qwen2-0.5B", batch=32, shortest=1025, longest=2048),
        # long answers of many users: the cache outweighs the weights
        dict(name="decode qwen3 0.6b x48", kind="decode", model="Qwen3-0.6B", batch=48, shortest=2049, longest=4096),
        # a batch of prompts of all lengths, as a scheduler packs them
        dict(name="prompts qwen2 0.5b", kind="prompts", heads="14/2/64", tokens=16384, sequences=24, cached=0),
        # prompts whose first half is in the cache already (a shared system prompt), 7B heads
        dict(name="prompts cached qwen2 7b", kind="prompts", heads="28/4/128", tokens=8192, sequences=8, cached=1024),
        # prompts of a layer with a window, kept first tokens and sinks
        dict(name="pages window 2k", kind="pages", size="2k", tokens=16384, sequences=14, mask="window", later=False),
        # feed-forward of experts: prompts, and a decode batch
        dict(name="experts prompts 2k", kind="experts", size="2k", tokens=16384, router="sigmoid"),
        dict(name="experts decode 2k", kind="experts", size="2k", tokens=32, router="softmax"),
        # the recurrent mechanisms over prompts, whole ones and portions of longer ones
        dict(name="lightning 2k", kind="lightning", size="2k", tokens=16384, sequences=16, later=False),
        dict(name="time mixing 2k", kind="time_mixing", size="2k", tokens=12000, sequences=11, later=True),
        dict(name="scan 1k", kind="scan", size="1k", tokens=16384, sequences=5, later=False),
        dict(name="recurrence 2k", kind="recurrence", size="2k", tokens=16384, sequences=16, later=False),
    ]


def draw(rng):
    """Kinds as often as they are listed; sizes spread over their logarithm, odd ones as likely as round ones."""
    def size(lo, hi):
        return round(math.exp(rng.uniform(math.log(lo), math.log(hi))))
    kind = rng.choice(["decode"] * 3 + ["prompts"] * 2 + ["experts"] * 2 + ["pages", *RECURRENT])
    if kind == "decode":
        model = rng.choice(["Qwen2-0.5B", "Qwen2-0.5B", "Qwen3-0.6B"])
        longest = size(64, 4096)
        return dict(kind=kind, model=model, batch=size(1, 48), shortest=max(1, round(longest * rng.uniform(0.3, 1.0))), longest=longest)
    if kind == "prompts":
        tokens = size(2000, 16384)
        return dict(kind=kind, heads=rng.choice(list(HEADS)), tokens=tokens, sequences=max(-(-tokens // 4096), size(1, 64)), cached=rng.choice([0, 0, 0, BLOCK * rng.randint(1, 6)]))
    which = rng.choice(["1k", "2k", "2k"])
    if kind == "experts":
        return dict(kind=kind, size=which, tokens=size(65, 16384) if rng.random() < 0.6 else size(1, 64), router=rng.choice(["sigmoid", "softmax"]))
    tokens = size(2000, 16384)
    case = dict(kind=kind, size=which, tokens=tokens, sequences=max(-(-tokens // 4096), size(1, 40)), later=rng.random() < 0.3)
    if kind == "pages":
        case["mask"] = rng.choice(["window", "all", "chunk"])
    return case


# ------------------------------------------------------------------------------------------------ inputs
class Inputs:
    """Random numbers of one seed, made on the GPU."""

    def __init__(self, seed):
        self.rng = random.Random(seed)
        self.gen = torch.Generator(device="cuda").manual_seed(seed)

    def randn(self, *shape, dtype=BF16, scale=1.0):
        t = torch.randn(*shape, generator=self.gen, device="cuda", dtype=dtype)
        return t if scale == 1.0 else t.mul_(scale)

    def rand(self, *shape, lo=0.0, hi=1.0):
        return torch.rand(*shape, generator=self.gen, device="cuda") * (hi - lo) + lo

    def perm(self, n):
        return torch.randperm(n, generator=self.gen, device="cuda")


def _lengths(rng, total, parts, most=None):
    """`parts` lengths that sum to `total`: between a quarter of their mean and twice it, as prompts differ."""
    w = [rng.uniform(0.25, 2.0) for _ in range(parts)]
    out = [max(1, int(total * x / sum(w))) for x in w]
    out[-1] += total - sum(out)
    while most and max(out) > most:
        i, j = out.index(max(out)), out.index(min(out))
        move = min(out[i] - most, most - out[j])
        out[i], out[j] = out[i] - move, out[j] + move
    return out


def _i32(values):
    return torch.tensor(values, dtype=torch.int32, device="cuda")


def _starts(lengths):
    out = [0]
    for n in lengths:
        out.append(out[-1] + n)
    return out


def _tables(d, counts, pages):
    """Block tables of sequences of these page counts: pages of one pool in random order."""
    order, at, rows, width = d.perm(pages).tolist(), 0, [], max(counts)
    for n in counts:
        rows.append(order[at:at + n] + [0] * (width - n))
        at += n
    return rows


# ------------------------------------------------------------------------------------------------ decode steps
_MODELS = {}


def _model(name):
    """The model with random weights, built once: what a serving program loads when it starts."""
    if name not in _MODELS:
        from nanovllm_hip.models.qwen import QwenForCausalLM, model_config
        with torch.device("cuda"):
            model = QwenForCausalLM(model_config(name)).to(BF16).eval()
        gen = torch.Generator(device="cuda").manual_seed(0)
        with torch.no_grad():
            for key, p in sorted(model.named_parameters()):
                norm = key.endswith("norm.weight")
                # (embeddings as large as a trained stream is beside what one layer adds: else every layer doubles the rounding errors of the one before)
                p.copy_(torch.randn(p.shape, generator=gen, device="cuda") * (0.1 if norm else 0.5 if key.startswith("embed") else 0.02) + (1.0 if norm else 0.0))
        _MODELS[name] = model
    return _MODELS[name]


def _decode_inputs(case, seed):
    cfg, d = _model(case["model"]).cfg, Inputs(seed)
    lengths = [d.rng.randint(case["shortest"], case["longest"]) for _ in range(case["batch"])]
    blocks = len(lengths) * -(-case["longest"] // BLOCK) + 1
    rows = _tables(d, [-(-n // BLOCK) for n in lengths], blocks)
    kv = d.randn(2, cfg.num_hidden_layers, blocks, BLOCK, cfg.num_key_value_heads, cfg.head_dim, scale=0.7)
    tokens = torch.randint(0, 10000, (case["batch"],), generator=d.gen, device="cuda")
    return lengths, rows, kv, tokens


@torch.inference_mode()
def _prepare_decode(case, seed):
    from nanovllm_hip import reset_context, set_context
    model = _model(case["model"])
    lengths, rows, kv, tokens = _decode_inputs(case, seed)
    tables, context = _i32(rows), _i32(lengths)
    slots = _i32([r[(n - 1) // BLOCK] * BLOCK + (n - 1) % BLOCK for r, n in zip(rows, lengths)])
    positions = context.long() - 1
    for i, layer in enumerate(model.layers):
        layer.self_attn.attn.k_cache, layer.self_attn.attn.v_cache = kv[0, i], kv[1, i]
    model.reserve_decode_workspace(len(lengths), tables.shape[1], BLOCK, torch.device("cuda"))

    def step():
        set_context(False, slot_mapping=slots, context_lens=context, block_tables=tables)
        logits = model.compute_logits(model(tokens, positions))
        reset_context()
        return logits
    side = torch.cuda.Stream()
    side.wait_stream(torch.cuda.current_stream())
    with torch.cuda.stream(side):
        step()
    torch.cuda.current_stream().wait_stream(side)
    torch.cuda.synchronize()
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        logits = step()
    return dict(graph=graph, logits=logits, keep=(kv, tables, context, slots, positions, tokens))


def _run_decode(s):
    s["graph"].replay()
    return s["logits"]


@torch.inference_mode()
def _exact_decode(case, seed):
    model = _model(case["model"])
    cfg = model.cfg
    lengths, rows, kv, tokens = _decode_inputs(case, seed)
    b, h, g, d = len(lengths), cfg.num_attention_heads, cfg.num_key_value_heads, cfg.head_dim
    longest = max(lengths)
    ctx = torch.tensor(lengths, device="cuda")
    seen = torch.arange(longest, device="cuda")[None, :] < ctx[:, None]
    at = torch.tensor([[r[t // BLOCK] * BLOCK + t % BLOCK if t < n else 0 for t in range(longest)] for r, n in zip(rows, lengths)], device="cuda")
    angle = (ctx - 1).double()[:, None] * cfg.rope_theta ** (-torch.arange(0, d, 2, device="cuda", dtype=F64) / d)

    def norm(x, w):
        return x / torch.sqrt((x * x).mean(dim=-1, keepdim=True) + cfg.rms_norm_eps) * w.double()

    def turn(x):
        u, v = x.chunk(2, dim=-1)
        c, s = angle.cos()[:, None], angle.sin()[:, None]
        return torch.cat((u * c - v * s, v * c + u * s), dim=-1)

    x = model.embed_tokens.weight[tokens].double()
    last = torch.arange(b, device="cuda")
    for i, layer in enumerate(model.layers):
        a = layer.self_attn
        qkv = F.linear(norm(x, layer.input_layernorm.weight), a.qkv_proj.weight.double(), a.qkv_proj.bias.double() if cfg.qkv_bias else None)
        q, k, v = (t.view(b, -1, d) for t in qkv.split([h * d, g * d, g * d], dim=-1))
        if cfg.qk_norm:
            q, k = norm(q, a.q_norm.weight), norm(k, a.k_norm.weight)
        q, k = turn(q), turn(k)
        keys, values = (kv[n, i].view(-1, g, d)[at].double() for n in (0, 1))                    # [b, longest, g, d]
        keys[last, ctx - 1], values[last, ctx - 1] = k, v
        score = torch.matmul(q.view(b, g, h // g, d), keys.permute(0, 2, 3, 1).contiguous()) * d ** -0.5
        p = torch.softmax(score.masked_fill(~seen[:, None, None], float("-inf")), dim=-1)
        o = torch.matmul(p, values.transpose(1, 2).contiguous()).reshape(b, h * d)
        x = x + o @ a.o_proj.weight.double().t()
        gate, up = F.linear(norm(x, layer.post_attention_layernorm.weight), layer.mlp.gate_up_proj.weight.double()).chunk(2, dim=-1)
        x = x + (F.silu(gate) * up) @ layer.mlp.down_proj.weight.double().t()
        del keys, values
    head = model.embed_tokens.weight if cfg.tie_word_embeddings else model.lm_head.weight
    return torch.cat([norm(x, model.norm.weight) @ w.double().t() for w in head.split(32768)], dim=-1)


def _work_decode(case):
    from nanovllm_hip.models.qwen import model_config
    cfg = model_config(case["model"])
    hid, d, h, g = cfg.hidden_size, cfg.head_dim, cfg.num_attention_heads, cfg.num_key_value_heads
    weights = cfg.num_hidden_layers * hid * (2 * (h + g) * d + 3 * cfg.intermediate_size) + cfg.vocab_size * hid
    b, context = case["batch"], case["batch"] * (case["shortest"] + case["longest"]) / 2
    return dict(bytes=2 * weights + cfg.num_hidden_layers * context * 4 * g * d + 2 * b * cfg.vocab_size,
                flops=2 * b * weights + cfg.num_hidden_layers * context * 4 * h * d)


# ------------------------------------------------------------------------------------------------ prompts through the attention module
def _prompts_inputs(case, seed):
    h, g, d = HEADS[case["heads"]]
    r = Inputs(seed)
    new = _lengths(r.rng, case["tokens"], case["sequences"], 4096)
    old = [case["cached"] if i % 4 < 3 else 0 for i in range(len(new))] if case["cached"] else [0] * len(new)
    blocks = (case["tokens"] + case["sequences"] * case["cached"]) // BLOCK + case["sequences"] + 1
    rows = _tables(r, [-(-(n + o) // BLOCK) for n, o in zip(new, old)], blocks)
    kv = r.randn(2, blocks, BLOCK, g, d)
    qkv = r.randn(sum(new), (h + 2 * g) * d)
    return new, old, rows, kv, qkv


def _prepare_prompts(case, seed):
    from nanovllm_hip.layers.attention_hip import Attention
    h, g, d = HEADS[case["heads"]]
    new, old, rows, kv, qkv = _prompts_inputs(case, seed)
    attn = Attention(h, d, d ** -0.5, g)
    attn.k_cache, attn.v_cache = kv[0], kv[1]
    at = [r[t // BLOCK] * BLOCK + t % BLOCK for r, n, o in zip(rows, new, old) for t in range(o, o + n)]
    total = [n + o for n, o in zip(new, old)]
    context = dict(cu_seqlens_q=_i32(_starts(new)), cu_seqlens_k=_i32(_starts(total)), max_seqlen_q=max(new), max_seqlen_k=max(total), slot_mapping=_i32(at),
                   block_tables=_i32(rows) if case["cached"] else None)
    return dict(attn=attn, kv=kv, context=context, qkv=qkv.split([h * d, g * d, g * d], dim=-1))


def _run_prompts(s):
    from nanovllm_hip import reset_context, set_context
    set_context(True, **s["context"])
    out = s["attn"](*s["qkv"])
    reset_context()
    return out, s["kv"]


def _attend64(q, k, v, scale, ok, sink=None):
    """q [n, h, d], k and v [m, g, d] in bfloat16, ok [n, m] -> [n, h, d] in 64 bits, one key head at a time."""
    h, g = q.shape[1], k.shape[1]
    out = torch.empty(q.shape[0], h, v.shape[2], dtype=F64, device=q.device)
    for j in range(g):
        heads = slice(j * (h // g), (j + 1) * (h // g))
        score = torch.einsum("nhd,md->hnm", q[:, heads].double(), k[:, j].double()).mul_(scale).masked_fill_(~ok, float("-inf"))
        top = score.amax(dim=-1, keepdim=True)
        if sink is not None:
            top = torch.maximum(top, sink[heads].double()[:, None, None])
        p = score.sub_(top).exp_()
        total = p.sum(dim=-1, keepdim=True)
        if sink is not None:
            total = total + torch.exp(sink[heads].double()[:, None, None] - top)
        out[:, heads] = torch.einsum("hnm,md->nhd", p / total, v[:, j].double())
    return out


def _exact_prompts(case, seed):
    h, g, d = HEADS[case["heads"]]
    new, old, rows, kv, qkv = _prompts_inputs(case, seed)
    q, k, v = (t.view(t.shape[0], -1, d) for t in qkv.split([h * d, g * d, g * d], dim=-1))
    flat, out, first = kv.view(2, -1, g, d), [], 0
    for r, n, o in zip(rows, new, old):
        at = torch.tensor([r[t // BLOCK] * BLOCK + t % BLOCK for t in range(n + o)], device="cuda")
        flat[0, at[o:]], flat[1, at[o:]] = k[first:first + n], v[first:first + n]
        i, j = torch.arange(o, o + n, device="cuda")[:, None], torch.arange(n + o, device="cuda")[None, :]
        out.append(_attend64(q[first:first + n], flat[0, at], flat[1, at], d ** -0.5, j <= i))
        first += n
    return torch.cat(out).view(first, h * d), kv


def _work_prompts(case):
    h, g, d = HEADS[case["heads"]]
    t, each = case["tokens"], case["tokens"] / case["sequences"]
    cached = case["cached"] * 0.75
    return dict(bytes=t * (2 * h + 4 * g) * d * 2 + case["sequences"] * cached * 4 * g * d, flops=4 * h * d * t * (1.2 * each / 2 + cached))


# ------------------------------------------------------------------------------------------------ attention of prompts over pages
def _portions(case, r):
    """Lengths of the portions and the tokens that came before each: prompts from their start, or most of them later portions."""
    new = _lengths(r.rng, case["tokens"], case["sequences"], 4096)
    return new, [r.rng.randint(1, 2000) if case["later"] and r.rng.random() < 0.8 else 0 for _ in new]


def _pages_inputs(case, seed):
    _, h, g, *_ = SIZES[case["size"]]
    r, d = Inputs(seed), 128
    new, old = _portions(case, r)
    pages = (case["tokens"] + 2000 * case["sequences"]) // PAGE + case["sequences"]
    rows = _tables(r, [-(-(n + o) // PAGE) for n, o in zip(new, old)], pages)
    cache = r.randn(pages, g, 2, PAGE, d)                       # inside a page: [key head][keys, values]
    return new, old, rows, cache, r.randn(case["tokens"], (h + 2 * g) * d), r.randn(h, dtype=F32)


def _prepare_pages(case, seed):
    from nanovllm_hip.layers.rotary import rotation_table
    _, h, g, *_ = SIZES[case["size"]]
    new, old, rows, cache, qkv, sink = _pages_inputs(case, seed)
    mask = {"window": dict(window=512, keep_first=4, sink=sink), "all": dict(sink=sink), "chunk": dict(chunk=512, turn=rotation_table(128, 10000.0, 8192, "cuda"))}[case["mask"]]
    args = (cache.view(cache.shape[0], PAGE, -1), _i32(rows), _i32(_starts(new)), _i32(_starts([n + o for n, o in zip(new, old)])), max(new), h, g, 128, 128, 128 ** -0.5)
    return dict(q=qkv, args=args, mask=mask)


def _run_pages(s):
    from nanovllm_hip import ops
    return ops.paged_attend_prompt(s["q"], *s["args"], **s["mask"])


def _exact_pages(case, seed):
    _, h, g, *_ = SIZES[case["size"]]
    new, old, rows, cache, qkv, sink = _pages_inputs(case, seed)
    q, out, first = qkv[:, :h * 128].view(-1, h, 128), [], 0
    for r, n, o in zip(rows, new, old):
        kv = cache[torch.tensor(r[:-(-(n + o) // PAGE)], device="cuda")]
        k, v = (kv[:, :, t].transpose(1, 2).reshape(-1, g, 128)[:n + o] for t in (0, 1))
        i, j = torch.arange(o, o + n, device="cuda")[:, None], torch.arange(n + o, device="cuda")[None, :]
        ok = j <= i
        if case["mask"] == "window":
            ok = ok & ((i - j < 512) | (j < 4))
        elif case["mask"] == "chunk":
            ok = ok & (i // 512 == j // 512)
        a = _attend64(q[first:first + n], k, v, 128 ** -0.5, ok, None if case["mask"] == "chunk" else sink)
        if case["mask"] == "chunk":                             # values turn with their position; the output is turned back
            angle = i.double() * 10000.0 ** (-torch.arange(0, 128, 2, device="cuda", dtype=F64) / 128)
            c, s, x, y = angle.cos()[:, None], angle.sin()[:, None], a[..., 0::2], a[..., 1::2]
            a = torch.stack((x * c + y * s, y * c - x * s), dim=-1).flatten(-2)
        out.append(a)
        first += n
    return torch.cat(out).view(first, h * 128)


def _work_pages(case):
    _, h, g, *_ = SIZES[case["size"]]
    t, each = case["tokens"], case["tokens"] / case["sequences"]
    before = 800 if case["later"] else 0
    seen = 0.6 * each + before
    if case["mask"] != "all":
        seen = min(seen, 512 if case["mask"] == "window" else 256)
    return dict(bytes=2 * t * (2 * h + 2 * g) * 128 + case["sequences"] * before * 4 * g * 128, flops=4 * 128 * h * t * seen)


# ------------------------------------------------------------------------------------------------ experts
def _choice(logits, bias, router):
    """[rows, experts] in 64 bits -> (scores to choose by, with closed groups at -inf; how clear the choice is)."""
    if router == "softmax":
        open_to, gap = logits + bias, math.inf
    else:
        score = torch.sigmoid(logits) + bias
        groups = score.view(-1, 8, EXPERTS // 8)
        best = groups.topk(2, dim=-1).values.sum(dim=-1)
        rank = best.sort(dim=-1, descending=True)
        gap = rank.values[:, 3] - rank.values[:, 4]
        kept = torch.zeros_like(best, dtype=torch.bool).scatter_(1, rank.indices[:, :4], True)
        open_to = groups.masked_fill(~kept[..., None], float("-inf")).flatten(1)
    top = open_to.topk(TOP + 1, dim=-1).values
    near = (top[:, :-1] - top[:, 1:]).amin(dim=-1)
    return open_to, near if router == "softmax" else torch.minimum(near, gap)


def _experts_inputs(case, seed):
    width, *_, ff = SIZES[case["size"]]
    r = Inputs(seed)
    router, bias = r.randn(EXPERTS, width, scale=width ** -0.5), r.randn(EXPERTS, dtype=F32, scale=0.1)
    x = r.randn(case["tokens"] + 64, width)
    # rows whose choice hangs on the last bits of a sum have no one right answer: other rows come in their place
    clear = _choice(x.double() @ router.double().t(), bias.double(), case["router"])[1] > 1e-4
    x = x[clear.nonzero()[:case["tokens"], 0]] if int(clear.sum()) >= case["tokens"] else x[clear.nonzero()[:1, 0]].repeat(case["tokens"], 1)
    gate_up, down = r.randn(EXPERTS, 2 * ff, width, scale=width ** -0.5), r.randn(EXPERTS, width, ff, scale=ff ** -0.5)
    return x, router, bias, gate_up, down


def _prepare_experts(case, seed):
    from nanovllm_hip.layers.moe import MixtureOfExperts
    x, router, bias, gate_up, down = _experts_inputs(case, seed)
    width, ff = x.shape[1], down.shape[2]
    how = dict(groups=8, keep=4, scale=2.5) if case["router"] == "sigmoid" else dict(softmax=True, unit=(7.0, 1.702))
    layer = MixtureOfExperts(width, width, ff, EXPERTS, TOP, BF16, **how)

    def get(name):
        if name.startswith("router") or name == "correction":
            return router if name == "router" else bias
        e, part = name[1:].split(".")
        return {"gate": gate_up[int(e), :ff], "up": gate_up[int(e), ff:], "down": down[int(e)]}[part]
    layer.load(get)
    return dict(layer=layer, x=x)


def _run_experts(s):
    return s["layer"](s["x"])


def _exact_experts(case, seed):
    x, router, bias, gate_up, down = _experts_inputs(case, seed)
    logits, ff = x.double() @ router.double().t(), down.shape[2]
    ids = _choice(logits, bias.double(), case["router"])[0].topk(TOP, dim=-1).indices
    if case["router"] == "softmax":
        weights = torch.softmax((logits + bias.double()).gather(1, ids), dim=-1)
    else:
        weights = torch.sigmoid(logits).gather(1, ids)
        weights = weights / (weights.sum(dim=-1, keepdim=True) + 1e-20) * 2.5
    out = torch.empty(ids.numel(), x.shape[1], dtype=F64, device="cuda")
    for e in range(EXPERTS):
        pairs = (ids.flatten() == e).nonzero()[:, 0]
        gate, up = (x[pairs // TOP].double() @ gate_up[e].double().t()).split(ff, dim=1)
        if case["router"] == "softmax":
            gate, up = gate.clamp(max=7.0), up.clamp(-7.0, 7.0) + 1.0
            act = gate * torch.sigmoid(1.702 * gate) * up
        else:
            act = F.silu(gate) * up
        out[pairs] = act @ down[e].double().t()
    return out, weights


def _work_experts(case):
    width, *_, ff = SIZES[case["size"]]
    t = case["tokens"]
    used = EXPERTS * (1 - (1 - TOP / EXPERTS) ** t)
    return dict(bytes=used * 6 * ff * width + 2 * EXPERTS * width + t * width * (2 + 2 * TOP), flops=t * (6 * TOP * ff * width + 2 * EXPERTS * width))


# ------------------------------------------------------------------------------------------------ recurrent mechanisms over prompts
def _segments(units, new):
    """The segment table an engine step makes for these portions."""
    from nanovllm_hip.engine.model_runner import recurrence_chunks
    from nanovllm_hip.layers.rglru import choose_segment
    segment = choose_segment(new, units)
    chunks = [c for i, (first, n) in enumerate(zip(_starts(new), new)) for c in recurrence_chunks(first, n, i, segment)]
    return segment, _i32(chunks), any(k for *_, k in chunks)


def _recurrent_inputs(case, seed):
    width, h, _, rec, blocks, _ = SIZES[case["size"]]
    r, t = Inputs(seed), case["tokens"]
    new, old = _portions(case, r)
    slots = r.perm(len(new) + 2)[:len(new)].int()
    n, kind = len(new) + 2, case["kind"]
    if kind == "lightning":                                   # q | k | v | gate of heads of 128, one decay per head
        x = r.randn(t, 4 * h * 128)
        p = dict(decay=torch.tensor([1 - 2.0 ** -(3 + 6 * i / h) for i in range(h)], device="cuda"))
        state = dict(state=r.randn(n, h, 128, 128, dtype=F32))
    elif kind == "time_mixing":                               # heads of 64, decays from 0.999 to 0.4 per token and channel
        x = [r.randn(t, width) for _ in range(5)]
        x[4].mul_(0.3)
        p = dict(w0=r.rand(width, lo=-6.0, hi=-1.0), u=0.5 + r.randn(width, dtype=F32, scale=0.5), norm=1.0 + r.randn(width, dtype=F32, scale=0.2))
        state = dict(state=r.randn(n, width // 64, 64, 64, dtype=F32))
    elif kind == "scan":                                      # x | gate of twice the width, 16 states per channel
        inner = 2 * width
        x = [r.randn(t, 2 * inner), r.randn(t, inner), r.randn(t, 64)]
        p = dict(a_log2=-r.rand(inner, STATES, lo=0.1, hi=4.0), d=0.8 + r.randn(inner, dtype=F32, scale=0.2), dt_bias=r.rand(inner, lo=-5.0, hi=-1.0))
        state = dict(state=r.randn(n, inner, STATES, dtype=F32))
    else:                                                     # gate | recurrent branch, block-diagonal gates, four taps
        x, s = r.randn(t, 2 * rec), rec // blocks
        p = dict(conv_w=r.randn(4, rec, dtype=F32, scale=0.5), conv_b=r.randn(rec, dtype=F32, scale=0.1), ra=r.randn(blocks, s, s, scale=s ** -0.5),
                 ri=r.randn(blocks, s, s, scale=s ** -0.5), ra_b=r.randn(rec, dtype=F32), ri_b=r.randn(rec, dtype=F32), rate=r.rand(rec, lo=0.01, hi=2.0))
        state = dict(state=r.randn(n, rec, dtype=F32), conv_state=r.randn(n, 4, rec))
    return new, old, slots, x, p, state


def _prepare_recurrent(case, seed):
    width, h, _, rec, blocks, _ = SIZES[case["size"]]
    new, old, slots, x, p, state = _recurrent_inputs(case, seed)
    from nanovllm_hip.layers.lightning import LightningAttention
    from nanovllm_hip.layers.mamba import SelectiveScan
    from nanovllm_hip.layers.rglru import RGLRU
    from nanovllm_hip.layers.wkv import TimeMixing
    layer = {"lightning": lambda: LightningAttention(width, width, h, 128, 128, [0.9] * h, EPS, BF16), "time_mixing": lambda: TimeMixing(width, width, width // 64, 64, EPS, BF16),
             "scan": lambda: SelectiveScan(width, width, 2 * width, STATES, width // 16, 4, BF16), "recurrence": lambda: RGLRU(width, width, rec, blocks, 4, BF16)}[case["kind"]]()
    segment, chunks, more = _segments(getattr(layer, "segment_units", blocks), new)
    positions = torch.cat([torch.arange(o, o + n, device="cuda") for n, o in zip(new, old)])
    return dict(kind=case["kind"], x=x, p=p, at=(positions, slots, chunks), segment=segment, more=more, state=state)


def _run_recurrent(s):
    from nanovllm_hip import ops
    x, p, state = s["x"], s["p"], s["state"]
    if s["kind"] == "lightning":
        out = ops.lightning_chunks(x, p["decay"], *s["at"], s["more"], state["state"])
    elif s["kind"] == "time_mixing":
        out = ops.wkv_chunks(*x, p, EPS, 64, *s["at"], s["more"], state["state"])
    elif s["kind"] == "scan":
        inner = x[1].shape[1]
        out = ops.scan_chunks(x[0][:, :inner], x[1], x[2], x[0][:, inner:], p, *s["at"], s["more"], state["state"])
    else:
        out = ops.rglru_chunks(x, p, *s["at"], s["segment"], s["more"], state["state"], state["conv_state"])
    return dict(out=out, **state)


def _padded(t, new):
    """Rows of the portions side by side, in 64 bits: [longest, portions, ...]."""
    out = t.new_zeros((max(new), len(new), *t.shape[1:]), dtype=F64)
    for i, (first, n) in enumerate(zip(_starts(new), new)):
        out[:n, i] = t[first:first + n].double()
    return out


def _unpadded(t, new):
    return torch.cat([t[:n, i] for i, n in enumerate(new)])


def _walk(new, start, step):
    """step(t, state) -> (state, out) for every token; a portion that has ended keeps its state."""
    s, out = start, []
    length = torch.tensor(new, device="cuda")
    for t in range(max(new)):
        nxt, o = step(t, s)
        s = torch.where((length > t).view(-1, *[1] * (s.dim() - 1)), nxt, s)
        out.append(o)
    return torch.stack(out), s


def _silu(z):
    return z / (1.0 + torch.exp(-z))


def _exact_recurrent(case, seed):
    width, h, _, rec, blocks, _ = SIZES[case["size"]]
    new, old, slots, x, p, state = _recurrent_inputs(case, seed)
    p = {k: v.double() for k, v in p.items()}
    fresh = torch.tensor([o == 0 for o in old], device="cuda")
    start = state["state"][slots.long()].double()
    start = torch.where(fresh.view(-1, *[1] * (start.dim() - 1)), torch.zeros_like(start), start)
    b = len(new)
    if case["kind"] == "lightning":
        q, k, v = (_silu(_padded(x[:, i * h * 128:(i + 1) * h * 128], new)).view(-1, b, h, 128) for i in range(3))
        decay = p["decay"].view(1, h, 1, 1)

        def step(t, s):
            s = s * decay + k[t][..., None] * v[t][..., None, :]
            return s, (s * q[t][..., None]).sum(dim=-2)
        out, last = _walk(new, start, step)
        out = out.flatten(2)
    elif case["kind"] == "time_mixing":
        r, k, v, g, z = (_padded(a, new).view(-1, b, width // 64, 64) for a in x)
        decay = torch.exp(-torch.exp(z + p["w0"].view(-1, 64)))
        u = p["u"].view(1, -1, 64, 1)

        def step(t, s):
            kv = k[t][..., None] * v[t][..., None, :]
            return s * decay[t][..., None] + kv, ((s + u * kv) * r[t][..., None]).sum(dim=-2)
        out, last = _walk(new, start, step)
        out = out / torch.sqrt((out * out).mean(dim=-1, keepdim=True) + EPS) * p["norm"].view(-1, 64) * _silu(g)
        out = out.flatten(2)
    elif case["kind"] == "scan":
        inner = 2 * width
        a, gate, bc = _padded(x[0][:, :inner], new), _padded(x[0][:, inner:], new), _padded(x[2], new)
        dt = _padded(x[1], new) + p["dt_bias"]
        dt = torch.log1p(torch.exp(-dt.abs())) + dt.clamp(min=0.0)

        def step(t, s):
            s = torch.exp2(dt[t][..., None] * p["a_log2"]) * s + (dt[t] * a[t])[..., None] * bc[t][:, None, :STATES]
            return s, (s * bc[t][:, None, STATES:2 * STATES]).sum(dim=-1)
        out, last = _walk(new, start, step)
        out = (out + p["d"] * a) * _silu(gate)
    else:
        y, raw = _padded(x[:, :rec], new), _padded(x[:, rec:], new)
        ring, old_at = state["conv_state"][slots.long()].double(), torch.tensor(old, device="cuda")
        rows, entry = torch.arange(b, device="cuda"), torch.arange(4, device="cuda")
        before = torch.stack([torch.where((old_at >= back)[:, None], ring[rows, (old_at - back) % 4], 0.0) for back in (3, 2, 1)])      # the input at position p lies in entry p mod 4
        line = torch.cat((before, raw))
        u = sum(line[j:j + raw.shape[0]] * p["conv_w"][j] for j in range(4)) + p["conv_b"]
        part = u.view(-1, b, blocks, rec // blocks)
        ra, ri = (torch.sigmoid(torch.einsum("tbks,kos->tbko", part, p[n]).flatten(2) + p[n + "_b"]) for n in ("ra", "ri"))
        log_a = -ra * p["rate"]
        decay, inputs = torch.exp(log_a), torch.sqrt(-torch.expm1(2.0 * log_a)) * ri * u

        def step(t, s):
            s = decay[t] * s + inputs[t]
            return s, s
        out, last = _walk(new, start, step)
        out = out * 0.5 * y * (1.0 + torch.tanh(math.sqrt(2.0 / math.pi) * (y + 0.044715 * y ** 3)))
        conv = state["conv_state"].double()
        for i, (n, o) in enumerate(zip(new, old)):
            for back in range(1, min(4, n) + 1):
                conv[slots[i].long(), (o + n - back) % 4] = raw[n - back, i]
    after = state["state"].double()
    after[slots.long()] = last
    res = dict(out=_unpadded(out, new), state=after)
    return dict(res, conv_state=conv) if case["kind"] == "recurrence" else res


def _work_recurrent(case):
    width, h, _, rec, blocks, _ = SIZES[case["size"]]
    t, n = case["tokens"], case["sequences"]
    per_token, state, flops = {"lightning": (8 * h * 128, 4 * h * 128 * 128, 4 * h * 128 * 128), "time_mixing": (12 * width, 4 * width * 64, 5 * width * 64),
                               "scan": (16 * width + 128, 8 * width * STATES, 2 * width * 5 * STATES), "recurrence": (6 * rec, 12 * rec, 4 * rec * (rec // blocks))}[case["kind"]]
    return dict(bytes=t * per_token + n * state * (2 if case["later"] else 1), flops=t * flops)


# ------------------------------------------------------------------------------------------------ by kind
_KINDS = {"decode": (_prepare_decode, _run_decode, _exact_decode, _work_decode), "prompts": (_prepare_prompts, _run_prompts, _exact_prompts, _work_prompts),
          "pages": (_prepare_pages, _run_pages, _exact_pages, _work_pages), "experts": (_prepare_experts, _run_experts, _exact_experts, _work_experts),
          **{k: (_prepare_recurrent, _run_recurrent, _exact_recurrent, _work_recurrent) for k in RECURRENT}}
# four times the distance from exact() over the listed and some drawn cases (0.0016 to 0.0024: bfloat16 operands and outputs); a decode step is 0.02 off, through 24 and 28 layers
_TOLERANCE = {"decode": 0.03, "prompts": 0.007, "pages": 0.007, "experts": 0.01, "lightning": 0.007, "time_mixing": 0.007, "scan": 0.007, "recurrence": 0.01}


def prepare(case, seed):
    state = _KINDS[case["kind"]][0](case, seed)
    return dict(state, run=_KINDS[case["kind"]][1])


@torch.inference_mode()
def run(state):
    return state["run"](state)


def exact(case, seed):
    return _KINDS[case["kind"]][2](case, seed)


def work(case):
    return _KINDS[case["kind"]][3](case)


def tolerance(case):
    return {"rel": _TOLERANCE[case["kind"]]}
