"""All layers of a decode step in one launch (nvh_decode_layers) against the same layers in 64 bits by plain torch."""
import pytest
import torch
import torch.nn.functional as F

pytestmark = pytest.mark.gpu

BF16, EPS, PAGE = torch.bfloat16, 1e-6, 64


def build(hidden, h, kvh, hd, inter, layers, norm, contexts, slots=None, seed=0):
    gen = torch.Generator(device="cuda").manual_seed(seed)

    def randn(*shape, scale=1.0):
        return (torch.randn(*shape, generator=gen, device="cuda") * scale).to(BF16)
    m, n, pages = len(contexts), (h + 2 * kvh) * hd, [max(1, -(-c // PAGE)) for c in contexts]
    order = torch.randperm(sum(pages) + 2, generator=gen, device="cuda").tolist()
    table = torch.zeros(m, max(pages), dtype=torch.int32)
    at = 0
    for i, p in enumerate(pages):
        table[i, :p] = torch.tensor(order[at:at + p])
        at += p
    if slots is None:
        slots = [int(table[i, (c - 1) // PAGE]) * PAGE + (c - 1) % PAGE if c else -1 for i, c in enumerate(contexts)]
    ws = [dict(qkv_w=randn(n, hidden, scale=hidden ** -0.5), qkv_bias=None if norm else randn(n, scale=0.1), q_norm_w=randn(hd) if norm else None,
               k_norm_w=randn(hd) if norm else None, o_w=randn(hidden, h * hd, scale=(h * hd) ** -0.5), gate_up_w=randn(2 * inter, hidden, scale=hidden ** -0.5),
               down_w=randn(hidden, inter, scale=inter ** -0.5), k_cache=randn(len(order), PAGE, kvh, hd), v_cache=randn(len(order), PAGE, kvh, hd)) for _ in range(layers)]
    angle = torch.outer(torch.arange(8192, device="cuda").float(), 10000.0 ** (-torch.arange(0, hd, 2, device="cuda").float() / hd))
    i32 = lambda v: torch.tensor(v, dtype=torch.int32, device="cuda")
    return dict(x=randn(m, hidden), layers=ws, num_heads=h, num_kv_heads=kvh, head_dim=hd, inter=inter, norm_eps=EPS, post_eps=EPS,
                positions=torch.tensor([max(c - 1, 0) for c in contexts], device="cuda"), cos_sin=torch.cat((angle.cos(), angle.sin()), -1).contiguous(),
                slot_mapping=i32(slots), context_lens=i32(contexts), block_tables=table.cuda())


def exact(s):
    """The stream behind the last layer, and the caches, in 64 bits; rows of the step are stored before any attends."""
    h, g, d = s["num_heads"], s["num_kv_heads"], s["head_dim"]
    x, contexts, slots, table = s["x"].double(), s["context_lens"].tolist(), s["slot_mapping"].tolist(), s["block_tables"].long()
    cos, sin = s["cos_sin"][s["positions"]].double()[:, None].chunk(2, -1)
    rms = lambda t: t / torch.sqrt((t * t).mean(-1, keepdim=True) + EPS)

    def turn(t):
        u, v = t.chunk(2, -1)
        return torch.cat((u * cos - v * sin, v * cos + u * sin), -1)
    caches = []
    for w in s["layers"]:
        qkv = F.linear(rms(x), w["qkv_w"].double(), None if w["qkv_bias"] is None else w["qkv_bias"].double())
        q, k, v = (t.view(len(contexts), -1, d) for t in qkv.split([h * d, g * d, g * d], -1))
        if w["q_norm_w"] is not None:
            q, k = rms(q) * w["q_norm_w"].double(), rms(k) * w["k_norm_w"].double()
        q, k = turn(q), turn(k)
        kc, vc = w["k_cache"].double().view(-1, g, d).clone(), w["v_cache"].double().view(-1, g, d).clone()
        for i, slot in enumerate(slots):
            if slot >= 0:
                kc[slot], vc[slot] = k[i], v[i]
        o = torch.zeros(len(contexts), h, d, dtype=torch.float64, device="cuda")
        for i, c in enumerate(contexts):
            if c:
                t = torch.arange(c, device="cuda")
                at = table[i, t // PAGE] * PAGE + t % PAGE
                kk, vv = kc[at].repeat_interleave(h // g, 1), vc[at].repeat_interleave(h // g, 1)
                p = torch.softmax(torch.einsum("hd,thd->ht", q[i], kk) * d ** -0.5, -1)
                o[i] = torch.einsum("ht,thd->hd", p, vv)
        x = x + o.flatten(1) @ w["o_w"].double().t()
        gate, up = F.linear(rms(x), w["gate_up_w"].double()).chunk(2, -1)
        x = x + (F.silu(gate) * up) @ w["down_w"].double().t()
        caches.append((kc, vc))
    return x, caches


def call(s, ws, **kw):
    from nanovllm_hip import ops
    return ops.decode_layers(s["x"], s["layers"], workspace=ws, **{k: v for k, v in s.items() if k not in ("x", "layers")}, **kw)


def scratch(s):
    from nanovllm_hip import ops
    n = ops.decode_layers_workspace_bytes(s["x"].shape[0], s["x"].shape[1], s["num_heads"], s["num_kv_heads"], s["head_dim"], s["inter"], len(s["layers"]))
    assert n > 0
    return torch.zeros(n, dtype=torch.uint8, device="cuda")


def error(a, b):
    return float((a.double() - b).norm() / b.norm())


# Every residual sum rounds to bf16 (relative 2^-9 at most, a third of it in the mean), as do the inputs of every product: six sums behind one another stay under 6 * 2^-9
BOUND = 6 * 2.0 ** -9
SMALL, WIDE = (256, 4, 2, 64, 512), (384, 4, 4, 128, 640)


@pytest.mark.parametrize("shape,norm", [(SMALL, False), (WIDE, True), ((264, 7, 1, 64, 1000), True), ((896, 14, 2, 64, 4864), False), ((1024, 16, 8, 128, 3072), True), ((512, 16, 1, 128, 256), False)])
@pytest.mark.parametrize("contexts", [[1], [17], [256], [257], [700], [4500], [0], [300, 1], [1030, 2111], [0, 33], [40, 300, 1], [600, 0, 1500]])
def test_layers_against_64_bits(shape, norm, contexts):
    s = build(*shape, 3, norm, contexts)
    ws = scratch(s)
    want, caches = exact(s)
    before = [(w["k_cache"].clone(), w["v_cache"].clone()) for w in s["layers"]]
    packed = torch.zeros(16 * shape[0], dtype=BF16, device="cuda") if shape[0] % 32 == 0 else None
    got = call(s, ws, out_packed=packed)
    assert error(got, want) < BOUND
    slots = [x for x in s["slot_mapping"].tolist() if x >= 0]
    for w, (k0, v0), (kc, vc) in zip(s["layers"], before, caches):
        for new, old, ref in ((w["k_cache"], k0, kc), (w["v_cache"], v0, vc)):
            new, old = new.view(-1, *ref.shape[1:]), old.view(-1, *ref.shape[1:])
            changed = (new != old).flatten(1).any(1).nonzero()[:, 0].tolist()
            assert set(changed) <= set(slots)
            if slots:
                assert error(new[slots], ref[slots]) < BOUND
    if packed is not None:
        from nanovllm_hip import _lib
        at = [[_lib.load().nvh_pack_index(i, c, shape[0]) for c in range(shape[0])] for i in range(len(contexts))]
        assert torch.equal(packed[torch.tensor(at, device="cuda")], got)
    for _ in range(3):                                       # (the same scratch again: nothing of the launch before is taken for this one's)
        assert torch.equal(call(s, ws), got)


def test_rows_of_one_sequence():
    """The second row's last token but one is the first row: its key and value come from this very launch."""
    s = build(*SMALL, 3, False, [40, 41])
    s["block_tables"][0] = s["block_tables"][1]
    first = int(s["block_tables"][1, 0]) * PAGE
    s["slot_mapping"] = torch.tensor([first + 39, first + 40], dtype=torch.int32, device="cuda")
    for w in s["layers"]:                                    # what the cache holds there must not be read
        w["k_cache"].view(-1, 2, 64)[first + 39:first + 64] = float("nan")
        w["v_cache"].view(-1, 2, 64)[first + 39:first + 64] = float("nan")
    want, _ = exact(s)
    assert error(call(s, scratch(s)), want) < BOUND


def test_row_without_a_slot():
    s = build(*SMALL, 2, False, [100, 70], slots=[-1, -1])
    before = [w["k_cache"].clone() for w in s["layers"]]
    want, _ = exact(s)
    assert error(call(s, scratch(s)), want) < BOUND
    assert all(torch.equal(w["k_cache"], b) for w, b in zip(s["layers"], before))


@pytest.mark.parametrize("late_from", [1, 20, 60, 200])
def test_workgroups_that_start_late(late_from):
    """Workgroups that wait for ones that have not started do their shares: the same bits."""
    s = build(896, 14, 2, 64, 4864, 2, False, [500, 300])
    ws = scratch(s)
    want = call(s, ws)
    for _ in range(2):
        assert torch.equal(call(s, ws, spin_limit=16, late_from=late_from, late_for=4000), want)
    assert torch.equal(call(s, ws), want)
    assert ws.view(torch.int32)[[0, 32, 64]].tolist() == [4, 0, 0]           # launches; workgroups started; gave up


@pytest.mark.parametrize("shape,norm", [((896, 14, 2, 64, 4864), False), ((1024, 16, 8, 128, 3072), True), ((512, 16, 1, 128, 256), False)])
@pytest.mark.parametrize("contexts", [[1], [700], [4500], [0, 33], [1030, 2111], [40, 300, 1], [600, 0, 1500]])
@pytest.mark.parametrize("late_from", [1, 20, 250])
def test_help_in_every_form(shape, norm, contexts, late_from):
    """Shares of both widths of heads, with and without q/k norm, of one to three rows, several rounds of tiles and none, done by workgroups that wait, most of which have no share of
    the attention: a wait's end concerns the whole workgroup or nobody."""
    s = build(*shape, 3, norm, contexts)
    ws = scratch(s)
    want = call(s, ws)
    for _ in range(2):
        assert torch.equal(call(s, ws, spin_limit=8, late_from=late_from, late_for=2000), want)
    assert torch.equal(call(s, ws), want)
    assert ws.view(torch.int32)[[0, 32, 64]].tolist() == [4, 0, 0]


def test_two_launches_side_by_side():
    a, b = build(896, 14, 2, 64, 4864, 3, False, [500], seed=1), build(896, 14, 2, 64, 4864, 3, False, [900, 20], seed=2)
    wa, wb = scratch(a), scratch(b)
    want = call(a, wa), call(b, wb)
    sa, sb = torch.cuda.Stream(), torch.cuda.Stream()
    for t in (sa, sb):
        t.wait_stream(torch.cuda.current_stream())
    got = []
    for _ in range(4):
        with torch.cuda.stream(sa):
            got.append((call(a, wa), want[0]))
        with torch.cuda.stream(sb):
            got.append((call(b, wb), want[1]))
    torch.cuda.synchronize()
    assert all(torch.equal(x, y) for x, y in got)


def test_replays():
    s = build(*WIDE, 4, True, [130, 64])
    ws, out = scratch(s), torch.empty(2, 384, dtype=BF16, device="cuda")
    want = call(s, ws).clone()
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        call(s, ws, out=out)
    for i in range(5):
        out.zero_()
        graph.replay()
        assert torch.equal(out, want)
        if i == 2:                                           # other inputs between replays
            s["x"].mul_(0.5)
            want = call(s, ws).clone()


def test_refusals():
    from nanovllm_hip import ops
    assert ops.decode_layers_workspace_bytes(4, 896, 14, 2, 64, 4864, 24) == 0
    assert ops.decode_layers_workspace_bytes(1, 3584, 28, 4, 128, 18944, 28) == 0           # 466 MB a layer
    assert ops.decode_layers_workspace_bytes(1, 896, 14, 2, 64, 4864, 33) == 0
    s = build(*SMALL, 1, False, [5])
    with pytest.raises(Exception, match="workspace"):
        call(s, torch.zeros(256, dtype=torch.uint8, device="cuda"))
    with pytest.raises(Exception, match="out may not be x"):
        call(s, scratch(s), out=s["x"])


@pytest.mark.parametrize("first", [0xfffd, 0xfffffffd])
def test_launch_numbers_come_round(first):
    """Marks are 16 bits of the launch's number beside an activation and 32 beside a share of the attention: past their ends nothing of the launch before is taken for this one's."""
    s = build(*SMALL, 3, False, [700, 90])
    ws = scratch(s)
    head = ws.view(torch.int64)
    head[0] = first
    want = {}
    for n in range(1, 7):
        s["x"].mul_(-1)                                      # (every launch has other results than the one before)
        got = call(s, ws)
        assert torch.equal(got, want.setdefault(n % 2, got.clone()))
        assert head[0].item() == (first + n) % 2 ** 32       # the next launch's number, and no workgroup started
    assert not torch.equal(want[0], want[1]) and error(want[0], exact(s)[0]) < BOUND
