"""The HIP builder's items are independent: a (block, kv head)'s summary is a function of its
own keys, whatever shares its wave (four items, two of them per accumulator set above rank
4).  Records are compared byte for byte."""
import pytest
import torch

from amass.selection import QuadState, R8State
from amass.selection.build import summary_build_hip
from helpers import announce

pytestmark = pytest.mark.gpu
DEV = "cuda"
KINDS = {"quad": dict(), "r8": dict(), "clse": dict(coords="lse", c_bits=8)}


def _state(kind, n, n_kv, rank):
    kw = dict(num_layers=1, num_blocks=n, n_kv=n_kv, G=1, head_dim=128, page=16, max_reqs=1,
              max_pages=n, rank=rank)
    if kind == "r8":
        return R8State(DEV, **kw)
    return QuadState(DEV, combine="max", **kw, **KINDS[kind])


def _items(kind, st):
    """Per (block, head) tensors that make up the summary."""
    if kind == "r8":
        return dict(mu=st.r8_mu[0], mus=st.mu_scale[0], V=st.reference_Vk(0), Vs=st.Vk_scale[0],
                    c=st.r8_c[0], cs=st.c_scale[0], tag=st.r8_tag[0].view(torch.int16))
    d = dict(mu=st.quad_mu[0], mus=st.mu_scale[0], V=st.reference_V(0), Vs=st.V_scale[0],
             tag=st.quad_tag[0].view(torch.int16))
    if kind == "clse":
        return dict(d, c=st.quad_c[0], cs=st.c_scale[0], resid=st.quad_resid[0])
    return dict(d, sig2=st.quad_sig2[0])


def _build(kind, K, blocks, rank):
    st = _state(kind, K.shape[0], K.shape[2], rank)
    summary_build_hip(st, 0, K, torch.tensor(blocks, device=DEV))
    torch.cuda.synchronize()
    return _items(kind, st)


@pytest.mark.parametrize("value", [float("nan"), float("inf"), 1e30])
@pytest.mark.parametrize("n_kv", [1, 2, 3])
@pytest.mark.parametrize("kind,rank", [("quad", 8), ("quad", 5), ("quad", 4), ("quad", 2),
                                       ("r8", 8), ("clse", 8), ("clse", 2)])
def test_a_non_finite_page_leaves_its_neighbours_alone(kind, rank, n_kv, value):
    """One key value that makes a page's Gram infinite or NaN (1e30 by overflow), in each
    place of a wave in turn."""
    announce(f"builder {kind} rank {rank}, {n_kv} heads, a key of {value}")
    n = 7
    gen = torch.Generator(device=DEV).manual_seed(rank + n_kv)
    K = torch.randn(n, 16, n_kv, 128, generator=gen, device=DEV).to(torch.bfloat16)
    want = _build(kind, K, list(range(n)), rank)
    for blk in range(n - 1):
        head = blk % n_kv
        bad = K.clone()
        bad[blk, 5, head, 77] = value
        got = _build(kind, bad, list(range(n)), rank)
        other = torch.ones(n, n_kv, dtype=torch.bool, device=DEV)
        other[blk, head] = False
        for name in want:
            assert torch.equal(got[name][other], want[name][other]), (name, blk)


@pytest.mark.parametrize("kind,rank", [("quad", 8), ("quad", 4), ("r8", 8), ("clse", 2)])
def test_summaries_do_not_depend_on_the_packing(kind, rank):
    """Ordinary pages alone, reversed, and between pages whose wanted eigenvalues lie close
    (constant, duplicated tokens, equal eigenvalues by construction)."""
    announce(f"builder {kind} rank {rank}: packing")
    n, n_kv = 96, 1
    gen = torch.Generator(device=DEV).manual_seed(rank)
    K = torch.randn(4 * n, 16, n_kv, 128, generator=gen, device=DEV).to(torch.bfloat16)
    K[n:2 * n] = K[n:2 * n, :1]                              # constant pages
    K[2 * n:3 * n, 1::2] = K[2 * n:3 * n, ::2]               # duplicated tokens
    K[3 * n:] = 0                                            # tokens +-4 e_t: equal eigenvalues
    for t in range(16):
        K[3 * n:, t, :, t // 2] = 4.0 if t % 2 else -4.0
    want = _build(kind, K, list(range(n)), rank)
    for extra in (n, 2 * n, 3 * n):
        for at in range(4):                                  # the close page's place in a wave
            order = []
            for i in range(0, n, 3):
                three = list(range(i, i + 3))
                order += three[:at] + [extra + i] + three[at:]
            got = _build(kind, K, order, rank)
            for name in want:
                assert torch.equal(got[name][:n], want[name][:n]), (name, extra, at)
    got = _build(kind, K, list(range(n))[::-1], rank)
    for name in want:
        assert torch.equal(got[name][:n], want[name][:n]), name
