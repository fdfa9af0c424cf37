"""The LSE merge at split counts around its batches (four waves, four partials each): the
split path against the fused pass, which merges nothing, over the same selection.

Both hold fp32 sums and round the output to bf16 once: P is rounded to bf16 against
different running maxima, which moves an output by at most 2^-8 of max|V| (the weights sum
to one), and the output's own rounding by 2^-8 of itself on either side."""
import pytest
import torch

from amass.attention import ensure_stage_b_buffers
from amass.attention.decode import ResidentVSource, sparse_paged_decode_batched
from amass.bench.synth import make_case
from helpers import announce

pytestmark = pytest.mark.gpu
DEV = "cuda"


class _St:
    pass


@pytest.mark.parametrize("G", [1, 4, 8])
@pytest.mark.parametrize("splits", [1, 2, 3, 4, 5, 15, 16, 17, 31, 33, 64, 127])
def test_split_counts(splits, G):
    announce(f"merge of {splits} splits, G {G}")
    pages = 4 * splits - (splits % 2)            # one request: at least 4 pages per split
    case = make_case(B=1, ctx=(16 * pages - 3, 16 * pages - 3), n_kv=2, G=G, heavy=0.0,
                     table="perm", seed=splits, device=DEV)
    st = _St()
    st.max_reqs, st.n_kv, st.G, st.D = 1, 2, G, 128
    ensure_stage_b_buffers(st, DEV)
    st.m_part.fill_(float("nan"))                # only what the launch writes may be read
    st.l_part.fill_(float("nan"))
    st.acc_part.fill_(float("nan"))
    st.page_table = torch.arange(case.max_pages, dtype=torch.int32, device=DEV).expand(
        1, 2, -1).contiguous()
    st.page_cnt = torch.tensor([[case.max_pages, max(1, case.max_pages // 2)]],
                               dtype=torch.int32, device=DEV)   # head 1: empty late splits
    outs = {}
    for path in ("split", "fused"):
        out = torch.full((1, 2 * G, 128), 7.0, dtype=torch.bfloat16, device=DEV)
        sparse_paged_decode_batched(case.q, case.kv_cache, case.block_table, case.seq_lens, st,
                                    out, ResidentVSource(case.kv_cache), scale=case.scale,
                                    path=path)
        outs[path] = out.float()
    torch.cuda.synchronize()
    a, b = outs["split"], outs["fused"]
    assert torch.isfinite(a).all()
    tol = 2.0 ** -8 * (case.V.float().abs().max() + a.abs() + b.abs())
    assert ((a - b).abs() <= tol).all(), float((a - b).abs().max())


@pytest.mark.parametrize("pages, n_kv, split, want", [
    (24, 8, 128, 1),      # three steps of a workgroup's eight waves: whole
    (25, 8, 128, 13),     # a fourth: splits of two pages
    (9, 3, 128, 1), (10, 3, 128, 5),      # the same with three waves
    (253, 8, 128, 127), (255, 8, 128, 127),     # every partial slot taken, 2-3 pages each
    (64, 8, 4, 1),        # three slots leave a split more steps than the waves take
    (64, 8, 17, 16),      # as many splits as steps
    (1, 8, 128, 1), (0, 8, 128, 1),
])
def test_auto_plan_few_units(pages, n_kv, split, want):
    """One request of up to a few hundred pages per head under path "auto": the layout on
    either side of the plan's line, the split count it leaves for the merge, and the output
    against the fused pass."""
    announce(f"auto plan: {pages} pages, {n_kv} heads, {split} slots")
    ctx = max(1, 16 * pages - 3)
    case = make_case(B=1, ctx=(ctx, ctx), n_kv=n_kv, G=4, heavy=0.0, table="perm",
                     seed=pages + split, device=DEV)
    st = _St()
    st.max_reqs, st.n_kv, st.G, st.D = 1, n_kv, 4, 128
    ensure_stage_b_buffers(st, DEV, split=split)
    for t in (st.m_part, st.l_part, st.acc_part):
        t.fill_(float("nan"))
    st.page_table = torch.arange(case.max_pages, dtype=torch.int32, device=DEV).expand(
        1, n_kv, -1).contiguous()
    st.page_cnt = torch.full((1, n_kv), pages, dtype=torch.int32, device=DEV)
    st.page_cnt[0, -1] = pages // 2
    outs = {}
    for path in ("auto", "fused"):
        out = torch.full((1, 4 * n_kv, 128), 7.0, dtype=torch.bfloat16, device=DEV)
        sparse_paged_decode_batched(case.q, case.kv_cache, case.block_table, case.seq_lens, st,
                                    out, ResidentVSource(case.kv_cache), scale=case.scale,
                                    path=path)
        outs[path] = out.float()
    torch.cuda.synchronize()
    counts = st.m_part.view(torch.int32)[0, :, split - 1, 0].tolist()
    assert counts == [want] * n_kv
    a, b = outs["auto"], outs["fused"]
    assert torch.isfinite(a).all()
    tol = 2.0 ** -8 * (case.V.float().abs().max() + a.abs() + b.abs())
    assert ((a - b).abs() <= tol).all(), float((a - b).abs().max())
