"""The builder's block lists from the device launches equal the tensor operations: tables of
one to many mark workgroups, block counts around the compaction's loads and its
4096-mark chunks, shared blocks, empty rows, strided tables."""
import pytest
import torch

from amass.selection.build import _list_rows, _tail_blocks, unique_finalized_blocks

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
