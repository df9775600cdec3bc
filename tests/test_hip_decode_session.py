"""Decode steps of one to three sequences, whose layers are one launch (nvh_decode_layers), as the engine runs them."""
import pytest
import torch

pytestmark = pytest.mark.gpu

FAMILIES = {"qwen2": {}, "qwen3": dict(num_attention_heads=4, num_key_value_heads=2, head_dim=128, hidden_size=512, intermediate_size=1024, qkv_bias=False, qk_norm=True)}


@pytest.fixture(autouse=True)
def one_launch_pays(monkeypatch):
    """Models of three layers are run the way that larger ones are."""
    from nanovllm_hip import ops
    monkeypatch.setattr(ops, "decode_layers_tokens", lambda m, *a, **kw: 2560 if m <= 3 else 0)


def engine(family, **kw):
    from nanovllm_hip.engine.llm_engine import LLMEngine
    from nanovllm_hip.models import qwen
    cfg = qwen.model_config("Qwen2-0.5B", num_hidden_layers=3, vocab_size=2048, **FAMILIES[family])
    return LLMEngine(cfg, num_kvcache_blocks=12, seed=4, **kw)


def prefilled(eng, lengths, new):
    from nanovllm_hip.engine.sequence import Sequence
    gen = torch.Generator().manual_seed(11)
    seqs = [Sequence(torch.randint(0, 2048, (n,), generator=gen).tolist(), max_tokens=new) for n in lengths]
    eng.prefill(seqs, reserve_tokens=new)
    return seqs


@pytest.fixture
def one_launch(monkeypatch):
    """Steps whose layers went in one launch (recorded ones count once)."""
    from nanovllm_hip import ops
    calls, real = [], ops.decode_layers
    monkeypatch.setattr(ops, "decode_layers", lambda *a, **kw: calls.append(1) or real(*a, **kw))
    return calls


@pytest.mark.parametrize("family", ["qwen2", "qwen3"])
@pytest.mark.parametrize("lengths", [(250,), (1,), (511, 40), (250, 300, 7), (250, 300, 7, 40)])
def test_sessions_against_steps_of_the_host(family, lengths, one_launch):
    """Generation over a page's end: a session that replays recorded steps (one and four at a time; embedded rows come from the arg-max launch, positions and slots advance on the
    device), one that runs them, and steps whose metadata the host makes give the same tokens."""
    eng, new = engine(family), 23
    few = len(lengths) <= 3
    tokens = []
    for graph in (True, False):
        seqs = prefilled(eng, lengths, new)
        session = eng.runner.decode_session(seqs, new, use_graph=graph)
        assert session.fuse_embed and (session.graph_multi is not None) == graph
        before = len(one_launch)
        assert not graph or before == (6 if few else 0)      # (a step to warm up, one recorded, four recorded)
        session.step(new)
        assert len(one_launch) - before == (new if few and not graph else 0)
        tokens.append(session.finish())
        for s in seqs:
            eng.block_manager.deallocate(s)
    seqs, host = prefilled(eng, lengths, new), []
    for _ in range(new):
        host.append(eng.runner.run(seqs, False))
        for s, t in zip(seqs, host[-1]):
            s.append_token(t)
    assert tokens[0] == tokens[1] == host


def test_the_one_launch_up_to_its_width_of_tables(one_launch):
    """The choice is by the longest context that the block table holds; launches give the same logits beyond it."""
    from nanovllm_hip import reset_context, set_context
    from nanovllm_hip.engine.model_runner import build_decode_meta
    eng = engine("qwen2")
    seqs, model = prefilled(eng, (40, 300, 7), 4), eng.runner.model
    want = logits(eng, seqs)
    pages = model._decode_bufs[(3, "cuda:0")]["layers_tokens"] // 256
    m = {k: v.cuda() for k, v in build_decode_meta(seqs).items()}
    assert len(one_launch) == 1 and 0 < pages
    for width, count in ((pages, 2), (pages + 1, 2), (pages, 3)):
        table = m["block_tables"].new_zeros(3, width)
        table[:, :m["block_tables"].shape[1]] = m["block_tables"]
        with torch.inference_mode():
            set_context(False, slot_mapping=m["slot_mapping"], context_lens=m["context_lens"], block_tables=table)
            got = model.compute_logits(model(m["input_ids"], m["positions"])).float()
            reset_context()
        assert len(one_launch) == count
        assert torch.equal(got, want) if width == pages else (got - want).abs().max() <= 3e-2 * want.abs().max()


def test_a_step_that_gave_up_is_an_error():
    eng = engine("qwen2")
    seqs = prefilled(eng, (40, 7), 8)
    session = eng.runner.decode_session(seqs, 8, use_graph=False)
    session.step(2)
    eng.runner.raise_if_device_failed()
    held = [b["layers_ws"] for b in eng.runner.model._decode_bufs.values() if b["layers_ws"] is not None]
    assert len(held) == 1 and held[0].view(torch.int32)[0] == 2            # (two launches)
    held[0].view(torch.int32)[64] = 1                                      # what a workgroup leaves that gives up
    with pytest.raises(RuntimeError, match="gave up"):
        eng.runner.raise_if_device_failed()
    with pytest.raises(RuntimeError, match="gave up"):
        session.finish()
    with torch.inference_mode():
        held[0].zero_()
    eng.runner.raise_if_device_failed()


@torch.inference_mode()
def logits(eng, seqs, more=0):
    """One decode step, not kept; positions and slots of `more` rows than there are sequences."""
    from nanovllm_hip import reset_context, set_context
    from nanovllm_hip.engine.model_runner import build_decode_meta
    m, model = {k: v.cuda() for k, v in build_decode_meta(seqs).items()}, eng.runner.model
    slots, positions = (torch.cat([m[k], m[k].new_zeros(more)]) for k in ("slot_mapping", "positions"))
    set_context(False, slot_mapping=slots, context_lens=m["context_lens"], block_tables=m["block_tables"])
    try:
        return model.compute_logits(model(m["input_ids"], positions)).float()
    finally:
        reset_context()


def test_positions_and_slots_of_more_rows():
    """Buffers made for the largest batch, as the projection's launch takes them: the first rows count."""
    eng = engine("qwen2")
    seqs = prefilled(eng, (40, 7), 4)
    want = logits(eng, seqs)
    assert torch.equal(logits(eng, seqs, more=6), want)


@pytest.mark.parametrize("switch,value", [("QKV_ATTEND_MODE", "auto"), ("QKV_ATTEND_MODE", "two_launches_kv_prefetch"), ("PREFETCH_WEIGHTS", False), ("KV_AHEAD", "o_k")])
def test_switches_of_the_launches_are_followed(switch, value, monkeypatch):
    from nanovllm_hip import ops
    from nanovllm_hip.models import qwen
    eng = engine("qwen2")
    seqs = prefilled(eng, (40, 7), 4)
    calls = []
    real = ops.decode_layers
    monkeypatch.setattr(ops, "decode_layers", lambda *a, **kw: calls.append(1) or real(*a, **kw))
    want = logits(eng, seqs)
    assert len(calls) == 1
    monkeypatch.setattr(qwen, switch, value)
    got = logits(eng, seqs)
    assert len(calls) == 1 and (got - want).abs().max() <= 3e-2 * want.abs().max()


@pytest.mark.parametrize("cus", [256, 192])
def test_streams_that_may_not_use_every_cu_get_launches(cus, monkeypatch):
    """Workgroups that wait for each other all want a CU: eager steps and a session that is replayed on such a stream take launches."""
    import ctypes
    from nanovllm_hip import ops
    words = (torch.cuda.get_device_properties(0).multi_processor_count + 31) // 32
    mask = (ctypes.c_uint32 * words)(*[(1 << min(max(cus - 32 * i, 0), 32)) - 1 for i in range(words)])
    hip, handle = ctypes.CDLL("libamdhip64.so"), ctypes.c_void_p()
    assert hip.hipExtStreamCreateWithCUMask(ctypes.byref(handle), words, mask) == 0
    calls, real = [], ops.decode_layers
    monkeypatch.setattr(ops, "decode_layers", lambda *a, **kw: calls.append(1) or real(*a, **kw))
    eng = engine("qwen2")
    seqs = prefilled(eng, (40, 7), 8)
    want = logits(eng, seqs)
    assert len(calls) == 1
    torch.cuda.synchronize()
    with torch.cuda.stream(torch.cuda.ExternalStream(handle.value)):
        got = logits(eng, seqs)
        session = eng.runner.decode_session(seqs, 8)
        session.step(8)
        torch.cuda.synchronize()
    assert (len(calls) > 1) == (cus >= 256) and eng.runner.model.decode_in_one_launch
    assert (got - want).abs().max() <= 3e-2 * want.abs().max()


@pytest.mark.parametrize("hidden,heads", [(256, 16), (512, 32)])
def test_attention_outputs_wider_than_the_stream(hidden, heads, monkeypatch):
    """The output projection's launch splits a long contraction: its scratch is sized by the heads, not by the stream."""
    from nanovllm_hip.models import qwen
    monkeypatch.setitem(FAMILIES, "wide", dict(num_attention_heads=heads, num_key_value_heads=4, head_dim=128, hidden_size=hidden, intermediate_size=512, qkv_bias=False, qk_norm=True))
    eng = engine("wide")
    seqs = prefilled(eng, (40, 300, 7, 5), 4)
    got = logits(eng, seqs)
    monkeypatch.setattr(qwen, "FUSED_DECODE", False)
    want = logits(eng, seqs)
    assert (got - want).abs().max() <= 3e-2 * want.abs().max()
