"""The builder's block lists from the device launches equal the tensor operations: tables of
one to many mark workgroups, block counts around the compaction's loads and its
4096-mark chunks, shared blocks, empty rows, strided tables."""
import pytest
import torch

from amass.selection import build
from amass.selection import QuadState, R8State, quad_build_tail
from amass.selection.build import (_list_rows, _tail_blocks, summary_build_hip,
                                   unique_finalized_blocks)

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("nb", [1, 15, 16, 17, 1000, 4096, 4097, 16385, 32768, 32769, 40001])
@pytest.mark.parametrize("B, W", [(1, 1), (3, 255), (5, 257), (64, 600)])
def test_block_lists(nb, B, W):
    gen = torch.Generator().manual_seed(nb + W)
    bt = torch.randint(0, nb, (B, W + 3), generator=gen, dtype=torch.int32)[:, :W]   # strided
    sl = torch.randint(0, 16 * W + 1, (B,), generator=gen, dtype=torch.int32)
    sl[0] = 16 * W if B < 5 else 0
    dbt = torch.full((B, W + 3), -7, dtype=torch.int32, device="cuda")[:, :W]
    dbt.copy_(bt)
    dsl = sl.cuda()
    assert _list_rows(dbt, dsl, B) and not _list_rows(bt, sl, B)
    for n in {1, B}:
        got = unique_finalized_blocks(dbt, dsl, n, 16, nb)
        want = unique_finalized_blocks(bt, sl, n, 16, nb)
        assert got.dtype == torch.int64 and torch.equal(got.cpu(), want)
        assert torch.equal(_tail_blocks(dbt, dsl, n, 16).cpu(), _tail_blocks(bt, sl, n, 16))


def test_block_lists_refuse():
    bt = torch.zeros(2, 4, dtype=torch.int32, device="cuda")
    sl = torch.tensor([64, 80], dtype=torch.int32, device="cuda")          # 4 and 5 pages
    with pytest.raises(IndexError):
        unique_finalized_blocks(bt, sl, 2, 16, 8)
    for bad in (-1, 8):
        bt[0, 3] = bad
        with pytest.raises(IndexError):
            unique_finalized_blocks(bt, sl, 1, 16, 8)
    sl[0] = 63                                       # the bad entry is not finalised
    assert unique_finalized_blocks(bt, sl, 1, 16, 8).tolist() == [0]


def test_tail_leaves_a_row_longer_than_the_table_alone():
    """Nothing but the other rows' pages is rebuilt: the long row's last page has no block."""
    bt = torch.tensor([[5, 2, 7], [1, 0, 4]], dtype=torch.int32, device="cuda")
    sl = torch.tensor([64, 40], dtype=torch.int32, device="cuda")          # 4 and 2 pages
    assert _tail_blocks(bt, sl, 2, 16).tolist() == [-1, 0]
    gen = torch.Generator(device="cuda").manual_seed(1)
    K = [torch.randn(8, 16, 2, 128, generator=gen, device="cuda").to(torch.bfloat16)] * 2
    st = QuadState("cuda", num_layers=2, num_blocks=8, n_kv=2, G=1, head_dim=128, page=16,
                   max_reqs=2, max_pages=3, rank=4, combine="max")
    st.quad_rec.fill_(77)
    quad_build_tail(st, K, bt, sl, 2)
    torch.cuda.synchronize()
    same = (st.quad_rec == 77).all(-1)                                     # (layer, block)
    assert same.tolist() == [[False] + [True] * 7] * 2


@pytest.mark.parametrize("kind, rank, n_kv", [("quad", 8, 3), ("quad", 2, 1), ("r8", 8, 2),
                                              ("r8", 4, 5), ("clse", 2, 3), ("clse", 8, 1)])
def test_the_builder_skips_negative_blocks(kind, rank, n_kv):
    """In every place of a wave of four items, and whole waves of them."""
    NB = 12
    gen = torch.Generator(device="cuda").manual_seed(rank)
    K = torch.randn(NB, 16, n_kv, 128, generator=gen, device="cuda").to(torch.bfloat16)
    kw = dict(num_layers=1, num_blocks=NB, n_kv=n_kv, G=1, head_dim=128, page=16, max_reqs=1,
              max_pages=NB, rank=rank)

    def build(blocks):
        st = (R8State("cuda", **kw) if kind == "r8" else
              QuadState("cuda", combine="max", coords="lse" if kind == "clse" else "none", **kw))
        rec, tag = (st.r8_rec, st.r8_tag) if kind == "r8" else (st.quad_rec, st.quad_tag)
        rec.fill_(77)
        summary_build_hip(st, 0, K, torch.tensor(blocks, device="cuda"))
        torch.cuda.synchronize()
        return rec, tag.view(torch.int16)

    keep = [3, 8, 1, 6, 0, 9]
    want = build(keep)
    for blocks in ([-1] + keep, keep + [-1], [-1, 3, -1, 8, 1, -1, -1, 6, 0, -7, 9],
                   [-1] * 16 + keep + [-1] * 9):
        for a, b in zip(build(blocks), want):
            assert torch.equal(a, b)
    assert (build([-1] * 5)[0] == 77).all()


@pytest.mark.parametrize("extra, launches", [(0, 1), (1, 0)])
def test_a_pool_too_large_for_the_launches_takes_tensor_operations(monkeypatch, extra, launches):
    nb = build.LIST_MAX_BLOCKS + extra
    bt = torch.tensor([[nb - 1, 0, 9], [4, nb - 1, 7]], dtype=torch.int32, device="cuda")
    sl = torch.tensor([48, 32], dtype=torch.int32, device="cuda")
    calls, real = [], build.block_list
    monkeypatch.setattr(build, "block_list", lambda *a: (calls.append(1), real(*a)))
    assert unique_finalized_blocks(bt, sl, 2, 16, nb).tolist() == [0, 4, 9, nb - 1]
    assert len(calls) == launches
