"""Prompt attention with 128 rows a workgroup (32 x 32 tiles): the bits that 64 rows a workgroup (16 x 16 tiles) give, at the edges of blocks of 32 keys, tiles of 64 and workgroups;
the order of the workgroups of up to three sequences, empty ones and cached keys among them."""
import pytest
import torch

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("lens", [(2079, 0, 33), (2113, 128, 65, 96, 160), (2176,), (2048, 2048)])
@pytest.mark.parametrize("form", ["fp16", "exact", "paged"])
@pytest.mark.parametrize("d", [64, 128])
def test_rows_of_a_workgroup(d, form, lens):
    """All heads fill the GPU with 128 rows a workgroup, those of one key head do not: every head's rows come out the same.  (The heads of one key head are as many as keep a launch
    of theirs from 1.3 on, in the units of launch_d: below, two groups of waves share the keys, whose sums are joined in another order.)"""
    from nanovllm_hip import ops
    kvh, page = 8, 256
    gen = torch.Generator().manual_seed(d + len(lens))
    old = [(0, 257, 64)[i % 3] if form == "paged" else 0 for i in range(len(lens))]
    total, keys = sum(lens), [n + o for n, o in zip(lens, old)]
    fill = 0.5 * max(lens) * (len(lens) + 1) / 16384 * (1.0 - 0.5 * max(lens) / max(keys))
    h = kvh * next(n for n in range(1, 99) if n * fill >= 1.32)
    assert h // kvh * fill < 1.8 and 0.5 * h * total / 16384 >= 3.0
    q = torch.randn(total, h, d, generator=gen).bfloat16().cuda()
    if form == "paged":
        width = -(-max(keys) // page)
        tables = torch.randperm(width * len(lens), generator=gen).view(len(lens), width).int().cuda()
        k, v = (torch.randn(width * len(lens), page, kvh, d, generator=gen).bfloat16().cuda() for _ in range(2))
    else:
        tables, (k, v) = None, (torch.randn(total, kvh, d, generator=gen).bfloat16().cuda() for _ in range(2))

    def cu(n):
        return torch.tensor([0, *n]).cumsum(0).int().cuda()

    def run(heads, of):
        return ops.flash_attn_varlen_func(q[:, heads].contiguous(), k[..., of, :].contiguous(), v[..., of, :].contiguous(), max_seqlen_q=max(lens), cu_seqlens_q=cu(lens), max_seqlen_k=max(keys),
                                          cu_seqlens_k=cu(keys), block_table=tables, pv_fp16=form == "fp16")
    got = run(slice(0, h), slice(0, kvh))
    for j in range(kvh):
        part = slice(j * (h // kvh), (j + 1) * (h // kvh))
        assert torch.equal(got[:, part], run(part, slice(j, j + 1))), j


@pytest.mark.parametrize("portions", [((130, 900), (257, 257)), ((1, 1), (300, 364), (64, 64)), ((0, 5), (513, 600))])
@pytest.mark.parametrize("window,keep,chunk", [(0, 0, 0), (70, 40, 0), (0, 0, 96)])
def test_few_portions_over_pages(portions, window, keep, chunk):
    """Up to three portions against each alone, at heads that make pairs for the XCDs (16 key heads) and one list for all (2)."""
    from nanovllm_hip import ops
    from paged_cases import Pages
    for heads, kvh in ((32, 16), (96, 2)):
        pg = Pages([k for _, k in portions], kvh, 128, 128, torch.bfloat16, seed=4)
        gen = torch.Generator().manual_seed(heads)
        q = torch.randn(sum(r for r, _ in portions), heads, 128, generator=gen).bfloat16()

        def cu(lengths):
            return torch.tensor([0, *lengths]).cumsum(0).int().cuda()

        def run(rows, some, most):
            return pg.unpad(ops.paged_attend_prompt(pg.pad_q(q[rows]), pg.cache(), pg.tables[some].contiguous().cuda(), cu(r for r, _ in portions[some]), cu(k for _, k in portions[some]), most,
                                                    heads, kvh, pg.dk, pg.dv, 0.2, window, keep, None, chunk=chunk), heads)
        got, at = run(slice(None), slice(None), max(r for r, _ in portions)), 0
        for i, (r, _) in enumerate(portions):
            if r:
                assert torch.equal(got[at:at + r], run(slice(at, at + r), slice(i, i + 1), r)), (heads, i)
            at += r


def attend_portions(pg, q, portions, some, most, heads, kvh, chunk=0, turn=None, window=0, keep=0):
    """Rows of the portions `some`, one after the other."""
    from nanovllm_hip import ops
    first = sum(r for r, _ in portions[:some.start or 0])
    rows = slice(first, first + sum(r for r, _ in portions[some]))

    def cu(lengths):
        return torch.tensor([0, *lengths]).cumsum(0).int().cuda()
    return pg.unpad(ops.paged_attend_prompt(pg.pad_q(q[rows]), pg.cache(), pg.tables[some].contiguous().cuda(), cu(r for r, _ in portions[some]), cu(k for _, k in portions[some]), most, heads,
                                            kvh, pg.dk, pg.dv, 0.2, window, keep, None, chunk=chunk, turn=turn), heads)


# 128 rows a workgroup with pairs split over the XCDs and as one list; 64 rows in launches of more workgroups than run at once (no portion of more than 256 rows), and where a CU holds one
@pytest.mark.parametrize("heads,kvh,dim,portions", [
    (96, 16, 128, ((130, 900), (257, 257))), (96, 16, 64, ((1, 1), (300, 364), (364, 400))), (112, 2, 128, ((0, 5), (513, 600))), (112, 16, 128, ((250, 250), (130, 900), (256, 300))),
    (112, 2, 64, ((256, 700), (250, 250), (255, 255))), (8, 8, 256, ((200, 200), (257, 600))), (6, 2, 256, ((1, 300), (140, 140), (65, 700)))])
@pytest.mark.parametrize("window,keep,chunk", [(0, 0, 0), (70, 40, 0), (0, 0, 96)])
def test_portions_in_the_order_of_their_work(heads, kvh, dim, portions, window, keep, chunk):
    from paged_cases import Pages
    pg = Pages([k for _, k in portions], kvh, dim, dim, torch.bfloat16, seed=4)
    q = torch.randn(sum(r for r, _ in portions), heads, dim, generator=torch.Generator().manual_seed(heads)).bfloat16()
    got, at = attend_portions(pg, q, portions, slice(0, len(portions)), max(r for r, _ in portions), heads, kvh, chunk, None, window, keep), 0
    for i, (r, _) in enumerate(portions):
        if r:
            assert torch.equal(got[at:at + r], attend_portions(pg, q, portions, slice(i, i + 1), r, heads, kvh, chunk, None, window, keep)), i
        at += r


@pytest.mark.parametrize("dim,vdim,turned,shift", [(64, 64, 64, 0), (128, 128, 128, 0), (128, 128, 62, 0), (128, 64, 64, 1), (192, 128, 100, 1), (64, 128, 6, 0)])
def test_turned_outputs_of_many_rows(dim, vdim, turned, shift):
    """Outputs turned back by 128 rows a workgroup: all columns and some, pairs that do not come in twos, a table `shift` floats behind a border of 8 bytes; the bits of each portion alone
    (64 rows a workgroup), and rows near the reference."""
    from paged_cases import Pages, close
    from test_hip_zaposun_ops import attend_ref, table_of, turned_back
    heads, kvh, chunk, portions = 48, 2, 100, ((300, 300), (3, 400), (130, 190), (327, 470))
    whole = table_of(turned)
    table = torch.cat([whole.new_zeros(shift), whole.flatten()])[shift:].view_as(whole)
    pg = Pages([k for _, k in portions], kvh, dim, vdim, torch.bfloat16, seed=3)
    q = torch.randn(sum(r for r, _ in portions), heads, dim, generator=torch.Generator().manual_seed(8)).bfloat16()
    got, at = attend_portions(pg, q, portions, slice(0, 4), 327, heads, kvh, chunk, table), 0
    for i, (r, k) in enumerate(portions):
        assert torch.equal(got[at:at + r], attend_portions(pg, q, portions, slice(i, i + 1), r, heads, kvh, chunk, table)), i
        for t in {0, 31, 32, 63, 64, 127, 128, r // 2, r - 1}:
            if t < r:
                want = turned_back(attend_ref(q[at + t], pg.k[i], pg.v[i], k - r + t, 0.2, chunk, 0), k - r + t, table)
                close(got[at + t], want, torch.bfloat16, f"portion {i} row {t}")
        at += r
