"""The host side of the launches: packed argument structs equal field-by-field ones, layer
slabs equal views, the finalised blocks' set equals the sorted unique ids, and a bulk build
equals a forced refresh of every layer."""
import ctypes

import pytest
import torch

from amass import _hip
from amass.selection import QuadState, R8State, quad_build_refresh, r8_build_refresh
from amass.selection.build import finalized_blocks, r8_build_bulk, unique_finalized_blocks
from amass.selection.quad_build import quad_build_bulk


@pytest.mark.parametrize("name", sorted(_hip.STRUCTS))
def test_packed_struct_equals_assigned(name):
    st = _hip.STRUCTS[name][1]
    vals = []
    for i, (_, t) in enumerate(st._fields_):
        vals.append({_hip._F32: 0.5 + i, _hip._F64: 0.25 + i}.get(
            t, (1 << 40) + i if t in (_hip._P, _hip._I64) else -1 - i))
    a = _hip.packer(st)(*vals)
    b = st(**{n: v for (n, _), v in zip(st._fields_, vals)})
    assert bytes(a) == bytes(b) and ctypes.sizeof(a) == ctypes.sizeof(b)


def test_layer_slab_equals_the_view():
    t = torch.arange(3 * 4 * 5, dtype=torch.int16).view(3, 4, 5)[:, ::2]
    for layer in (0, 1, 2, -1, -3):
        at, strides, shape = _hip.layer_slab(t, layer)
        v = t[layer]
        assert (at, strides, shape) == (v.data_ptr(), v.stride(), v.shape)
    for layer in (3, -4):
        with pytest.raises(IndexError):
            _hip.layer_slab(t, layer)


def test_current_stream_refuses_a_host_device(monkeypatch):
    """A launch for tensors in host memory must not get as far as the kernel."""
    monkeypatch.setattr(torch.cuda, "current_device", lambda: 0)
    monkeypatch.setattr(torch._C, "_cuda_getCurrentRawStream", lambda i: 7, raising=False)
    assert _hip.current_stream(torch.device("cuda")) == 7
    with pytest.raises((ValueError, RuntimeError, AssertionError)):
        _hip.current_stream(torch.device("cpu"))


def test_finalised_blocks_refuse_a_row_longer_than_the_table():
    bt = torch.zeros(2, 4, dtype=torch.int32)
    sl = torch.tensor([64, 80], dtype=torch.int32)             # 4 and 5 pages
    for fn in (finalized_blocks, lambda *a: unique_finalized_blocks(*a, 8)):
        with pytest.raises(IndexError):
            fn(bt, sl, 2, 16)
    assert unique_finalized_blocks(bt, sl, 1, 16, 8).tolist() == [0]


@pytest.mark.parametrize("dtype", [torch.int32, torch.int64])
@pytest.mark.parametrize("bad", [-9, -1, 8, 9, 1000])
def test_finalised_blocks_refuse_a_block_outside_the_pool(bad, dtype):
    bt = torch.tensor([[3, bad, 5]], dtype=dtype)
    with pytest.raises(IndexError):
        unique_finalized_blocks(bt, torch.tensor([32], dtype=torch.int32), 1, 16, 8)
    sl = torch.tensor([31], dtype=torch.int32)                 # the bad entry is not finalised
    assert unique_finalized_blocks(bt, sl, 1, 16, 8).tolist() == [3]


@pytest.mark.parametrize("dtype", [torch.int32, torch.int64])
@pytest.mark.parametrize("lens", [[0], [15], [16], [17, 400, 0, 33], [16 * 30] * 5])
def test_finalised_blocks(lens, dtype):
    gen = torch.Generator().manual_seed(len(lens))
    W, nb = 30, 211
    bt = torch.randint(0, nb, (len(lens) + 1, W), generator=gen).to(dtype)   # shared blocks
    sl = torch.tensor(lens + [16 * W], dtype=dtype)                          # one row beyond
    got = unique_finalized_blocks(bt, sl, len(lens), 16, nb)
    assert torch.equal(got, torch.unique(finalized_blocks(bt, sl, len(lens), 16)))
    assert got.dtype == torch.int64
    assert unique_finalized_blocks(bt, sl, 0, 16, nb).numel() == 0


@pytest.mark.parametrize("kind", ["quad", "r8"])
def test_bulk_equals_refresh_of_every_layer(kind):
    gen = torch.Generator().manual_seed(5)
    NB, n_kv, L = 9, 2, 3
    Ks = [torch.randn(NB, 16, n_kv, 128, generator=gen).to(torch.bfloat16) for _ in range(L)]
    bt = torch.tensor([[3, 1, 4, 0], [8, 2, 1, 6]], dtype=torch.int32)
    sl = torch.tensor([50, 64], dtype=torch.int32)
    kw = dict(num_layers=L, num_blocks=NB, n_kv=n_kv, G=1, head_dim=128, page=16, max_reqs=2,
              max_pages=4, rank=2)
    make, bulk, refresh, rec = {
        "quad": (QuadState, quad_build_bulk, quad_build_refresh, "quad_rec"),
        "r8": (R8State, r8_build_bulk, r8_build_refresh, "r8_rec")}[kind]
    a, b = make("cpu", **kw), make("cpu", **kw)
    n = bulk(a, Ks, bt, sl, 2)
    m = sum(refresh(b, layer, K, bt, sl, 2, force=True) for layer, K in enumerate(Ks))
    assert n == m == L * 6
    assert torch.equal(getattr(a, rec), getattr(b, rec))


@pytest.mark.parametrize("missing", ["amass_abi_version", "amass_quad_score",
                                     "amass_binding_block_list", "amass_binding_begin_step"])
def test_a_library_without_a_function_asks_for_a_rebuild(monkeypatch, missing):
    """A library built from other sources of the same ABI version fails with the same message
    as one of another version, not with ctypes' own error, and is not kept."""
    real = ctypes.CDLL(_hip.LIB_PATH)

    class Lib:
        def __getattr__(self, name):
            if name == missing:
                raise AttributeError(f"undefined symbol: {name}")
            return getattr(real, name)

    monkeypatch.setattr(_hip, "_LIB", None)
    monkeypatch.setattr(_hip.C, "CDLL", lambda path: Lib())
    with pytest.raises(_hip.AmassError, match="rebuild"):
        _hip.load_library()
    assert _hip._LIB is None


def test_a_v_source_may_leave_its_tier_fields_none(monkeypatch):
    """NULL in the struct, as ctypes takes None; another source's values arrive as they are."""
    from amass.attention import decode
    monkeypatch.setattr(decode, "require_cuda", lambda *t: None)
    kv = torch.zeros(4, 2, 16, 2, 128, dtype=torch.bfloat16)
    q = torch.zeros(1, 2, 128, dtype=torch.bfloat16)

    class St:
        n_kv, G, max_reqs = 2, 1, 1
        page_table = torch.zeros(1, 2, 4, dtype=torch.int32)
        page_cnt = torch.ones(1, 2, dtype=torch.int32)

    class Source(decode.ResidentVSource):
        fields = {}

        def tier_fields(self):
            return self.fields

    src = Source(kv)
    rows = torch.zeros(1, 4, dtype=torch.int32), torch.full((1,), 16, dtype=torch.int32)

    def args():
        return decode._decode_args(q, kv[:, 0], src, *rows, St, q.clone(), 1.0, 1, dense=False,
                                   path="fused")

    names = ("hot", "page2slot", "vbo", "pool", "t_layer", "t_nb", "t_slots")
    src.fields = dict(hot=None, page2slot=None, vbo=None, pool=None, nb=None)
    a = args()
    assert [getattr(a, x) or 0 for x in names] == [0] * 7
    src.fields = dict(hot=1 << 40, page2slot=2, vbo=3, pool=4, layer=5, nb=6, slots=7)
    a = args()
    assert [getattr(a, x) for x in names] == [1 << 40, 2, 3, 4, 5, 6, 7]
