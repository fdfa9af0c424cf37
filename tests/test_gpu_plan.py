"""The decode's plan under path "auto" (layout and split counts chosen on the device)."""
import pytest
import torch

from amass.attention import ensure_stage_b_buffers
from amass.attention.decode import ResidentVSource, sparse_paged_decode_batched
from amass.bench.synth import make_case
from amass.tier import Tier
from amass.tier.decode_mem import mem_decode
from helpers import announce

pytestmark = pytest.mark.gpu
DEV = "cuda"


class _St:
    pass


def _state(case, cnt, split=128):
    """Random `cnt` (R, n_kv) pages of every unit, ascending."""
    st = _St()
    R, n_kv, MP = case.q.shape[0], case.n_kv, case.max_pages
    st.max_reqs, st.n_kv, st.G, st.D = R, n_kv, case.G, 128
    ensure_stage_b_buffers(st, DEV, split=split)
    for t in (st.m_part, st.l_part, st.acc_part):
        t.fill_(float("nan"))                    # only what the launch writes may be read
    gen = torch.Generator(device=DEV).manual_seed(R + n_kv)
    rank = torch.rand(R, n_kv, MP, generator=gen, device=DEV).argsort(-1).argsort(-1)
    at = torch.arange(MP, device=DEV)
    tab = torch.where(rank < cnt[..., None], at, MP + at).sort(-1).values
    st.page_table = torch.where(tab < MP, tab, -1).to(torch.int32).contiguous()
    st.page_cnt = cnt.to(torch.int32).contiguous()
    return st


def _counts(st):
    """Split counts per unit, as the decode leaves them for the merge."""
    return st.m_part.view(torch.int32)[:, :, st.split - 1, 0]


@pytest.mark.parametrize("n_kv", [2, 3, 4, 5, 6, 8])
def test_tiered_equals_resident_under_auto(n_kv):
    """Both V sources run one plan, so their outputs are equal bit for bit: 32 requests
    keeping about 50 pages, and 6 keeping a third of ragged contexts."""
    for B, ctx, lo, hi in ((32, (2000, 2000), 44, 58), (6, (900, 6000), 15, 20)):
        announce(f"tiered vs resident, auto, {B} requests, {n_kv} kv heads")
        case = make_case(B=B, ctx=ctx, n_kv=n_kv, G=4, heavy=0.0, table="perm", seed=n_kv,
                         device=DEV)
        gen = torch.Generator(device=DEV).manual_seed(B)
        cnt = torch.randint(lo, hi + 1, (B, n_kv), generator=gen, device=DEV)
        st = _state(case, cnt)
        res = torch.full((B, 4 * n_kv, 128), 7.0, dtype=torch.bfloat16, device=DEV)
        tie = torch.full_like(res, 9.0)
        sparse_paged_decode_batched(case.q, case.kv_cache, case.block_table, case.seq_lens, st,
                                    res, ResidentVSource(case.kv_cache), scale=case.scale)
        torch.cuda.synchronize()
        splits = _counts(st).clone()
        tier = Tier(num_layers=1, num_blocks=case.kv_cache.shape[0], n_kv=n_kv, page=16, d=128,
                    hot_slots=256, max_reqs=B, max_pages=case.max_pages, device=DEV,
                    v_blocks=2 * B + 8)
        tier.flush_layer(0, case.kv_cache[:, 1])
        tier.step(0, st.page_table, st.page_cnt, case.block_table, case.seq_lens, B)
        mem_decode(case.q, case.kv_cache, case.block_table, case.seq_lens, st, tie, tier, 0,
                   scale=case.scale)
        torch.cuda.synchronize()
        assert torch.equal(_counts(st), splits)
        assert torch.equal(res.view(torch.int16), tie.view(torch.int16))


@pytest.mark.parametrize("n_kv, B, pages, want", [
    (8, 32, 52, 1),                      # whole: a workgroup per CU, no more steps than a split
    (4, 64, 20, 1), (2, 128, 24, 1),     # narrow workgroups: a step is a page per wave
    (2, 127, 24, 3),                     # ... and one workgroup short of the CUs
    (4, 32, 52, 8), (2, 64, 60, 4),      # split: 256 workgroups
    (1, 64, 52, 8),                      # ... 512 of one wave
    (4, 65, 60, 7), (4, 96, 90, 5),      # past 64 requests 8 waves per CU
    (2, 128, 31, 4),                     # ... and splits of 8 pages or more
])
def test_plan_lines(n_kv, B, pages, want):
    """Uniform batches on either side of the plan's lines on 256 CUs: the split counts it
    leaves for the merge, and the output against the fused pass (which merges nothing; P is
    rounded to bf16 against other running maxima, 2^-8 of max|V|, and the output itself)."""
    announce(f"auto plan: {B} requests of {pages} pages, {n_kv} heads")
    case = make_case(B=B, ctx=(16 * pages, 16 * pages), n_kv=n_kv, G=2, heavy=0.0, table="perm",
                     seed=B + pages, device=DEV)
    st = _state(case, torch.full((B, n_kv), pages, device=DEV))
    outs = {}
    for path in ("fused", "auto"):
        out = torch.full((B, 2 * n_kv, 128), 7.0, dtype=torch.bfloat16, device=DEV)
        sparse_paged_decode_batched(case.q, case.kv_cache, case.block_table, case.seq_lens, st,
                                    out, ResidentVSource(case.kv_cache), scale=case.scale,
                                    path=path)
        outs[path] = out.float()
    torch.cuda.synchronize()
    assert _counts(st).unique().tolist() == [want]
    a, b = outs["auto"], outs["fused"]
    tol = 2.0 ** -8 * (case.V.float().abs().max() + a.abs() + b.abs())
    assert torch.isfinite(a).all() and ((a - b).abs() <= tol).all()
