"""CPU checks of the drop-in boundary: the C-ABI library loads, exports every symbol include/nvh_attn.h
declares, validates arguments without touching a GPU, and the host-side mirror keeps the reference's
interface (names, constructor, attributes, Context fields).  No compute calls here."""
import ctypes
import inspect
import os
import re

import pytest
import torch

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))


@pytest.fixture(scope="module")
def lib():
    from nanovllm_hip import _lib
    return _lib.load()


def test_header_symbols_all_exported(lib):
    from nanovllm_hip import _lib
    header = open(os.path.join(ROOT, "include", "nvh_attn.h")).read()
    declared = set(re.findall(r"\b(nvh_[a-z_0-9]+)\s*\(", header))
    assert declared, "no declarations parsed"
    assert declared == set(_lib.EXPORTS), f"binding/header mismatch: {declared ^ set(_lib.EXPORTS)}"
    for name in declared:
        assert hasattr(lib, name), f"libnvh_attn.so does not export {name}"


def test_version_matches_header(lib):
    header = open(os.path.join(ROOT, "include", "nvh_attn.h")).read()
    assert lib.nvh_version() == int(re.search(r"#define NVH_VERSION (\d+)", header).group(1))


def test_workspace_is_pure_function_of_static_shapes(lib):
    a = lib.nvh_paged_decode_workspace(32, 14, 64, 16, 256)
    assert a == lib.nvh_paged_decode_workspace(32, 14, 64, 16, 256) and a > 0
    hdr = 65536 + 8192                                                       # fixed header (tickets + the fused launch's counters), then the partial records
    assert lib.nvh_paged_decode_workspace(64, 14, 64, 16, 256) - hdr == 2 * (a - hdr)
    assert lib.nvh_paged_decode_workspace(32, 14, 96, 16, 256) == 0          # unsupported head_dim
    # partial = (D + 2) floats per (row, head, split)
    assert (a - hdr) % ((64 + 2) * 4 * 32 * 14) == 0 and (a - hdr) // ((64 + 2) * 4 * 32 * 14) == 2 * 16


def test_argument_validation_without_gpu(lib):
    buf = (ctypes.c_char * 4096)()
    p = ctypes.addressof(buf)
    p = (p + 15) & ~15
    # null pointers
    assert lib.nvh_store_kvcache(None, None, None, None, None, 4, 2, 64, 128, 128, 0, None) == -5
    assert b"null" in lib.nvh_last_error()
    # zero work is a no-op that needs no pointers
    assert lib.nvh_store_kvcache(None, None, None, None, None, 0, 2, 64, 128, 128, 0, None) == 0
    assert lib.nvh_paged_decode(None, None, None, None, None, None, 0, 14, 2, 64, 256, 4, 896, 4, 0.125, 0, 0, None, 0, None) == 0
    # dtype / shape / stride / alignment / workspace checks fire before any launch
    assert lib.nvh_store_kvcache(p, p, p, p, p, 4, 2, 64, 128, 128, 7, None) == -1
    assert lib.nvh_store_kvcache(p, p, p, p, p, 4, 2, 64, 100, 128, 0, None) == -3
    assert lib.nvh_store_kvcache(p + 2, p, p, p, p, 4, 2, 64, 128, 128, 0, None) == -6
    assert lib.nvh_paged_decode(p, p, p, p, p, p, 1, 14, 2, 96, 256, 4, 1344, 4, 0.1, 0, 0, p, 1 << 20, None) == -2
    assert lib.nvh_paged_decode(p, p, p, p, p, p, 1, 14, 3, 64, 256, 4, 896, 4, 0.1, 0, 0, p, 1 << 20, None) == -2
    assert lib.nvh_paged_decode(p, p, p, p, p, p, 1, 14, 2, 64, 100, 4, 896, 4, 0.1, 0, 0, p, 1 << 20, None) == -2
    assert lib.nvh_paged_decode(p, p, p, p, p, p, 1, 14, 2, 64, 256, 4, 896, 4, 0.1, 0, 0, p, 16, None) == -4
    assert b"workspace" in lib.nvh_last_error()
    assert lib.nvh_prefill_varlen(p, p, p, p, p, p, None, 2, 16, 16, 14, 2, 64, 0, 0, 890, 128, 128, 0, 0.1, 0, 0, None) == -3
    # arg-max + advance + next step's embedding lookup: argument errors before any launch
    adv = (p, p, 8, 64, 4, p, p, p, p, p, 4, 256, p, 4, p)
    assert lib.nvh_greedy_advance_candidates_embed(*adv, None, 1000, 896, p, 896, p, 0, None) == -5          # no embedding table
    assert lib.nvh_greedy_advance_candidates_embed(*adv, p, 1000, 896, None, 896, p, 0, None) == -5          # no output rows
    assert lib.nvh_greedy_advance_candidates_embed(*adv, p, 1000, 900, p, 900, None, 0, None) == -2          # hidden % 32
    assert lib.nvh_greedy_advance_candidates_embed(*adv, p, 1000, 896, p, 800, None, 0, None) == -2          # row stride < hidden
    assert lib.nvh_greedy_advance_candidates_embed(*adv, p, 0, 896, p, 896, None, 0, None) == -2             # vocab
    assert lib.nvh_greedy_advance_candidates_embed(*adv, p + 2, 1000, 896, p, 896, None, 0, None) == -6
    assert lib.nvh_greedy_advance_candidates_embed(*adv, p, 1000, 896, p, 896, None, 3, None) == -1
    assert lib.nvh_greedy_advance_candidates_embed(p, p, 8, 64, 0, p, p, p, p, p, 4, 256, p, 4, p, None, 0, 0, None, 0, None, 0, None) == 0   # zero rows
    # the variant entry points validate their selectors
    dec = (p, p, p, p, p, p, 1, 14, 2, 64, 256, 4, 896, 4, 0.1, 0, 0, p, 1 << 20, None)
    assert lib.nvh_paged_decode_variant(6, 0, 0, *dec) == -2 and lib.nvh_paged_decode_variant(0, 5, 0, *dec) == -2
    assert lib.nvh_paged_decode_variant(2, 0, 0, p, p, p, p, p, p, 1, 16, 1, 64, 256, 4, 1024, 4, 0.1, 0, 0, p, 1 << 20, None) == -2   # VALU form: G <= 8
    pre = (p, p, p, p, p, p, None, 2, 16, 16, 14, 2, 64, 0, 0, 896, 128, 128, 0, 0.1, 0, 0, None)
    assert lib.nvh_prefill_varlen_variant(4, 0, *pre) == -2 and lib.nvh_prefill_varlen_variant(2, 4, *pre) == -2
    paged = (p, p, p, p, p, p, p, 2, 16, 16, 14, 2, 64, 256, 4, 896, 128, 128, 4, 0.1, 0, 0, None)
    assert lib.nvh_prefill_varlen_variant(3, 0, *paged) == -2                       # the fp16-V measurement variant never reads a paged cache
    # the fused front of a decode layer and the fp16 row conversion: argument errors before any launch
    assert lib.nvh_qkv_rope_attend(None, p, None, p, p, 256, 4, 4, 0.1, 0, p, 1 << 20, None) == -5
    assert lib.nvh_qkv_rope_attend_status(None, None) == -5
    assert lib.nvh_bf16_rows_to_f16(p, p, 4, 100, 128, 128, None) == -2 and lib.nvh_bf16_rows_to_f16(p, p, 4, 128, 100, 128, None) == -3
    assert lib.nvh_bf16_rows_to_f16(None, None, 0, 128, 128, 128, None) == 0
    # prefill with P V on the fp16 pipe: scratch size is a pure function of the shapes; argument errors before any stream operation
    assert lib.nvh_prefill_pv16_scratch_bytes(100, 2, 64) == 256 + 100 * 2 * 64 * 2 and lib.nvh_prefill_pv16_scratch_bytes(0, 2, 64) == 0
    pv = (p, p, p, p, p, p, 2, 1024, 1024, 2048, 14, 2, 64, 896, 128, 128, 0.125, 0, 0)
    assert lib.nvh_prefill_varlen_pv16(*pv, None, 0, None) == -5                      # no scratch
    assert lib.nvh_prefill_pv16_uses_scratch(2, 1024, 1024, 2, 64) == 1 and lib.nvh_prefill_pv16_uses_scratch(128, 128, 128, 2, 64) == 0
    assert lib.nvh_prefill_pv16_uses_scratch(16, 128, 128, 2, 64) == 1               # few sequences: the tiled kernel
    assert lib.nvh_prefill_varlen_pv16(*pv, p, 4096, None) == -4                      # scratch too small
    assert b"scratch" in lib.nvh_last_error()
    assert lib.nvh_prefill_varlen_pv16(*pv[:9], 0, *pv[10:], p, 1 << 20, None) == -4  # total_k missing
    assert lib.nvh_prefill_varlen_pv16(p, p, p, p, p, p, 0, 0, 0, 0, 14, 2, 64, 896, 128, 128, 0.125, 0, 0, None, 0, None) == 0   # empty batch


def test_decode_layers_status_refuses_null_pointers(lib):
    v = ctypes.c_uint32(5)
    assert lib.nvh_decode_layers_status(None, ctypes.byref(v)) == -5 and b"decode_layers_status" in lib.nvh_last_error()
    assert lib.nvh_decode_layers_status(ctypes.c_void_p(4096), None) == -5


def test_experts_in_one_call_refuse_scratch_that_is_too_small(lib):
    """Scratch is a pure function of the sizes (no tiles up to 64 rows in bf16, always some in fp32); nothing is launched without all of it."""
    from nanovllm_hip import _lib
    p = ctypes.c_void_p(4096)
    assert [lib.nvh_moe_experts_scratch_bytes(*a) for a in ((0, 2, 8, 64, 0), (5, 2, 8, 60, 0), (5, 2, 4096, 64, 0), (5, 0, 8, 64, 0))] == [0] * 4
    assert lib.nvh_moe_experts_scratch_bytes(5, 2, 8, 64, 0) == 4 * (10 * 64 // 2 + 12)
    assert lib.nvh_moe_experts_scratch_bytes(100, 2, 8, 64, 0) == 4 * (200 * 64 // 2 + 2 * 200 + 4 * (200 // 64 + 8) + 8)
    assert lib.nvh_moe_experts_scratch_bytes(5, 2, 8, 64, 1) == 4 * (10 * 64 + 2 * 12 + 4 * 8 + 8)
    d = _lib.MoeExpertsDesc(p, 64, p, p, p, p, 100, 64, 64, 8, 2, 1, 1, 0, 1.0, 0.0, 0.0, p, lib.nvh_moe_experts_scratch_bytes(100, 2, 8, 64, 0) - 4, p, p)
    assert lib.nvh_moe_experts(ctypes.byref(d), 0, None) == -4 and b"scratch" in lib.nvh_last_error()
    d.scratch_bytes, d.scratch = 1 << 20, None
    assert lib.nvh_moe_experts(ctypes.byref(d), 0, None) == -5
    d.scratch, d.scratch_bytes, d.rows = p, 0, 0
    assert lib.nvh_moe_experts(ctypes.byref(d), 0, None) == 0


def test_experts_share_a_launch_where_nothing_read_is_overwritten(lib):
    """Both products in one launch store outputs while rows and weights are still read: not where they overlap (two launches let them).  By the rule of sizes; scratch on whole lines."""
    from nanovllm_hip import _lib
    rows, cols, n, experts, top = 9000, 1024, 64, 24, 4
    out, x, w, scratch = 1 << 40, 1 << 41, 1 << 42, 1 << 43
    size, stride = 2 * rows * top * cols, cols + 64

    def one(dtype=0, **kw):
        d = _lib.MoeExpertsDesc(x, stride, w, w, w, w, rows, cols, n, experts, top, 1, 1, 0, 1.0, 0.0, 0.0, scratch, lib.nvh_moe_experts_scratch_bytes(rows, top, experts, n, 0), out, w)
        for name, value in kw.items():
            setattr(d, name, value)
        return lib.nvh_moe_experts_one_launch(ctypes.byref(d), dtype)
    used, weights = 2 * ((rows - 1) * stride + cols), 2 * experts * 2 * n * cols
    assert one() == 1
    assert [one(x=out + at) for at in (-used, 16 - used, 0, 4096, size - 16, size)] == [1, 0, 0, 0, 0, 1]
    assert [one(gate_up=out + at) for at in (-weights, 16 - weights, 0, size - 16, size)] == [1, 0, 0, 0, 1]
    assert [one(scratch=scratch + at) for at in (16, 64, 128)] == [0, 0, 1]
    full, least = lib.nvh_moe_experts_scratch_bytes(rows, top, experts, n, 0), 4 * (rows * top * n // 2 + 2 * rows * top + 4 * (rows * top // 256 + experts) + 18 * experts)
    assert full == least + 128 * (8 + rows * top // 256 + experts) and [one(scratch_bytes=b) for b in (full, full - 4, least)] == [1, 0, 0]
    d = _lib.MoeExpertsDesc(x, stride, w, w, w, w, rows, cols, n, experts, top, 1, 1, 0, 1.0, 0.0, 0.0, scratch, least - 4, out, None)
    assert lib.nvh_moe_experts(ctypes.byref(d), 0, None) == -4 and str(least).encode() in lib.nvh_last_error()
    d.scratch_bytes = least
    assert lib.nvh_moe_experts(ctypes.byref(d), 0, None) == -5 and b"moe_route" in lib.nvh_last_error()     # (enough: the next check is another one)
    assert one(dtype=1) == 0 and one(rows=60) == 0 and one(rows=700) == 0 and one(rows=0) == 0
    ran_out = ctypes.c_uint32(5)
    assert lib.nvh_moe_experts_status(None, 0, ctypes.byref(ran_out)) == -5 and lib.nvh_moe_experts_status(ctypes.byref(d), 0, None) == -5
    assert lib.nvh_moe_experts_status(ctypes.byref(d), 0, ctypes.byref(ran_out)) == 0 and ran_out.value == 0         # (two launches: none waits)
    assert one(dtype=9) == -1 and lib.nvh_moe_experts_one_launch(None, 0) == -5 and one(n=60) == -2


@pytest.mark.parametrize("experts,rows", [(8, {16: 64, 25: 64, 26: 128, 109: 128, 110: 256, 192: 256, 193: 128, 240: 128, 256: 128, 287: 128, 288: 256}),
                                          (32, {25: 64, 100: 128, 192: 256, 193: 256, 240: 256, 241: 128, 256: 128, 288: 256}),
                                          (64, {16: 64, 17: 128, 25: 128, 100: 128, 240: 256, 241: 128, 255: 128, 256: 256}), (96, {99: 128, 100: 256, 109: 256, 241: 128, 256: 256})])
def test_rows_of_expert_tiles(lib, experts, rows):
    """By the pairs of an expert and by how wide all of them are (1024 columns each); fp32 has one size."""
    assert {mean: lib.nvh_moe_tile_rows(mean * experts, experts, 0) for mean in rows} == rows
    assert all(lib.nvh_moe_tile_rows(mean * experts, experts, 1) == 64 for mean in rows)


def test_asm_of_several_instructions_shares_no_register():
    """An output that is written while inputs are still to be read must not share a register with one: the compiler may give equal values the same unless it is told (&)."""
    seen = 0
    for root, _, names in os.walk(os.path.join(ROOT, "nano-vllm-learn_amd", "csrc")):
        for name in names:
            text = re.sub(r"//.*", "", open(os.path.join(root, name)).read())
            for body in re.findall(r"\basm(?: volatile)?\s*\((.*?)\)\s*;", text, re.S):
                strings = []
                marked = re.sub(r'"((?:[^"\\]|\\.)*)"', lambda m: strings.append(m[1]) or f"#{len(strings) - 1} ", body)
                code, outputs, inputs = ([strings[int(i)] for i in re.findall(r"#(\d+)", part)] for part in (marked.split(":") + ["", ""])[:3])
                lines = [i for i in re.split(r"\\n|\\t|;", "".join(code)) if i.strip()]
                if len(lines) > 1 and any(re.search("[vsa]", i) for i in inputs):
                    seen += 1
                    assert all("&" in o for o in outputs), f"{name}: {lines[0]}"
    assert seen >= 3


def test_ops_refuse_cpu_tensors():
    """No CPU fallback: the product path must fail loudly off-GPU."""
    from nanovllm_hip import ops
    q = torch.zeros(1, 14, 64, dtype=torch.bfloat16)
    kc = torch.zeros(1, 256, 2, 64, dtype=torch.bfloat16)
    with pytest.raises(RuntimeError, match="no CPU path"):
        ops.flash_attn_with_kvcache(q, kc, kc, torch.ones(1, dtype=torch.int32), torch.zeros(1, 1, dtype=torch.int32))
    with pytest.raises(RuntimeError, match="no CPU path"):
        ops.store_kvcache(q[:, :2], q[:, :2], kc, kc, torch.zeros(1, dtype=torch.int32))


def test_missing_library_fails_loudly(monkeypatch, tmp_path):
    from nanovllm_hip import _lib
    monkeypatch.setattr(_lib, "_lib", None)
    monkeypatch.setattr(_lib, "LIB_PATH", str(tmp_path / "libnvh_attn.so"))
    with pytest.raises(_lib.NvhLibraryError, match="no fallback"):
        _lib.load()


def test_product_never_imports_oracle():
    pkg = os.path.join(ROOT, "nano-vllm-learn_amd")
    for dirpath, _, files in os.walk(pkg):
        for f in files:
            if f.endswith((".py", ".hip", ".h")):
                src = open(os.path.join(dirpath, f)).read()
                assert not re.search(r"^\s*(from|import)\s+oracle\b", src, re.M), f"{f} imports the oracle"


def test_attention_module_mirrors_reference_interface():
    from nanovllm_hip import VALID_ATTN_BACKENDS, resolve_attention
    from nanovllm_hip.layers.attention_hip import Attention
    assert "hip" in VALID_ATTN_BACKENDS and not "hip".startswith("sdpa")
    for ref_name in ("flash", "sdpa", "sdpa.math", "triton"):             # config.py:6
        assert ref_name in VALID_ATTN_BACKENDS
    cls, kw = resolve_attention("hip", block_size=256)
    assert cls is Attention and kw == {"block_size": 256}
    with pytest.raises(ValueError):
        resolve_attention("nope")
    params = list(inspect.signature(Attention.__init__).parameters)
    assert params[1:5] == ["num_heads", "head_dim", "scale", "num_kv_heads"]     # attention.py:60-66, positional use qwen3.py:89-95
    m = Attention(14, 64, 0.125, 2, **kw)
    assert m.k_cache.numel() == 0 and m.v_cache.numel() == 0              # attention.py:72, duck-typed by model_runner.py:151
    assert list(inspect.signature(m.forward).parameters) == ["q", "k", "v"]


def test_context_fields_match_reference():
    from nanovllm_hip import Context, get_context, reset_context, set_context
    assert [f for f in Context.__dataclass_fields__] == ["is_prefill", "cu_seqlens_q", "cu_seqlens_k", "max_seqlen_q",
                                                         "max_seqlen_k", "slot_mapping", "context_lens", "block_tables"]
    set_context(False, slot_mapping=1, context_lens=2, block_tables=3)
    c = get_context()
    assert (c.is_prefill, c.slot_mapping, c.context_lens, c.block_tables) == (False, 1, 2, 3)
    reset_context()
    assert get_context() == Context()


def test_pack_index_matches_the_torch_packer():
    """nvh_pack_index (host-callable) is the layout ops.pack_rows / unpack_rows produce."""
    import torch
    from nanovllm_hip import _lib, ops
    lib = _lib.load()
    m, c = 37, 96
    x = torch.arange(m * c, dtype=torch.float32).view(m, c).bfloat16()
    xp = ops.pack_rows(x)
    assert xp.numel() == 48 * c
    for row, col in [(0, 0), (1, 0), (0, 8), (15, 31), (16, 0), (36, 95), (17, 40)]:
        assert xp[lib.nvh_pack_index(row, col, c)] == x[row, col]
    assert torch.equal(ops.unpack_rows(xp, m, c), x)
    assert lib.nvh_linear_small_m_workspace(32, 896, 896, 2) == 0           # K <= 1024: one workgroup per tile, no hand-off
    assert lib.nvh_linear_small_m_workspace(32, 896, 4864, 2) >= 56 * 4 + 56 * 5 * (2 * 256 + 32) * 4


# what the split of a decode step's layers over a chip of 256 CUs says of these sizes (0: not served): in a process of its own, a division by zero would end it
_PLAN = """
import ctypes
from nanovllm_hip import _lib
plan = ctypes.CDLL(_lib.LIB_PATH)["_ZN3nvh18plan_decode_layersERNS_16DecodeLayersArgsEiiiiiiii"]
args = (ctypes.c_char * 8192)()
for m, hidden, h, kvh, hd, inter, layers in {sizes}:
    print(plan(args, 256, m, hidden, h, kvh, hd, inter, layers))
"""


def test_decode_layers_plan_refuses_sizes_without_heads():
    import subprocess
    import sys
    good = (1, 896, 14, 2, 64, 4864, 24)
    bad = [(1, 896, h, kvh, 64, 4864, 24) for h, kvh in ((0, 2), (-2, 2), (-14, 2), (14, 0), (14, -2), (-14, -2))] + [(0, *good[1:]), (1, 0, *good[2:]), (*good[:5], 0, 24), (*good[:6], 0)]
    done = subprocess.run([sys.executable, "-c", _PLAN.format(sizes=[good, *bad])], capture_output=True, text=True, timeout=300, cwd=os.path.join(ROOT, "nano-vllm-learn_amd"))
    assert done.returncode == 0, done.stderr[-500:]
    first, *rest = [int(x) for x in done.stdout.split()]
    assert first > 0 and rest == [0] * len(bad)


def test_a_decode_step_is_one_launch_where_that_is_faster():
    """Contexts up to which it is chosen on 256 CUs, beside steps timed both ways: (m, hidden, heads, key heads, width, inter, layers, q/k norm), a context, launches / one launch."""
    from nanovllm_hip import _lib
    tokens = ctypes.CDLL(_lib.LIB_PATH)["_ZN3nvh20decode_layers_tokensEiiiiiiiib"]
    qwen2, qwen3 = (896, 14, 2, 64, 4864, 24, False), (1024, 16, 8, 128, 3072, 28, True)
    timed = [((1, *qwen2), 4096, 1.54), ((1, *qwen2), 12288, 1.23), ((2, *qwen2), 1024, 1.37), ((2, *qwen2), 4096, 1.11), ((3, *qwen2), 2048, 1.07), ((3, *qwen2), 4096, 0.95),
             ((1, *qwen3), 9216, 1.09), ((2, *qwen3), 2560, 1.03), ((2, *qwen3), 3500, 0.96), ((3, *qwen3), 1024, 1.07),
             ((3, 768, 16, 2, 128, 2368, 16, True), 1115, 0.94), ((3, 768, 16, 2, 128, 2368, 16, True), 5120, 0.76), ((3, 256, 7, 1, 128, 960, 32, False), 59, 0.92),
             ((3, 896, 16, 1, 128, 2944, 32, False), 5120, 0.80), ((2, 256, 16, 2, 128, 4800, 2, False), 1090, 0.85), ((1, 512, 4, 1, 64, 448, 1, False), 3, 0.95),
             ((3, 256, 16, 2, 64, 3776, 1, True), 125, 0.83), ((2, 640, 16, 1, 64, 960, 24, False), 7168, 0.95), ((1, 384, 8, 1, 128, 5056, 16, False), 12288, 1.20)]
    for sizes, context, speed in timed:
        assert (tokens(256, *sizes) >= context) == (speed > 1), (sizes, context, tokens(256, *sizes))
    assert tokens(256, 4, *qwen2) == tokens(32, 1, *qwen2) == tokens(256, 1, 896, 0, 2, 64, 4864, 24, False) == 0
