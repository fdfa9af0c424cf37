"""Stage B -- sparse paged decode attention (host side of ``amass_sparse_decode``).

Same contract as the reference ``sparse_paged_decode_batched`` (attention/decode.py:
247-304): consumes st.page_table / st.page_cnt and writes rows [0, n_req) of ``out``
(T, H, d) in place, reading K from the resident paged cache and V through an injected
V source (the fast / mem-v seam, attention/decode.py:44-95).  No allocation, no host
sync.  Units of a few pages get one workgroup per (request, kv
head) whose waves split the head's pages and merge in LDS; otherwise each request gets S
workgroups with one wave per kv head (split s attends pages s, s + S, ...) that write
split-K partials for a second launch, the LSE merge.  ``path``: "auto" (layout and S chosen on the device so the
workgroups fill the GPU), "split" (every request split, at least pps_min pages per
split, S below the partial capacity), "fused" (every request one workgroup per head).
``dense_paged_decode`` attends every page of every request (the dense baseline).
"""
from __future__ import annotations

from typing import Protocol, Tuple

import torch

from .._hip import DecodeArgs, call, current_stream, packer, require_cuda

SPLIT = 128          # split-K width (partial buffers are (R, n_kv, SPLIT, G[, d]))
PATHS = {"auto": 0, "split": 1, "fused": 2}
_pack_decode = packer(DecodeArgs)


class VSource(Protocol):
    SRC_ID: int

    def args(self) -> Tuple[torch.Tensor, int, int, int]:
        ...


def _split_kv(kv_cache: torch.Tensor):
    """(K, V) views (num_blocks, page, n_kv, d) of a (2, NB, ...) or (NB, 2, ...) cache;
    V is None for a K-only (NB, 1, ...) cache."""
    if kv_cache.shape[0] == 2:
        return kv_cache[0], kv_cache[1]
    if kv_cache.shape[1] == 1:
        return kv_cache.select(1, 0), None
    return kv_cache.select(1, 0), kv_cache.select(1, 1)


def _k_view(kv_cache: torch.Tensor):
    """K (num_blocks, page, n_kv, d) of a cache, as _split_kv finds it (the one view)."""
    return kv_cache[0] if kv_cache.shape[0] == 2 else kv_cache.select(1, 0)


class ResidentVSource:
    """V from the resident engine V half (source id 0)."""

    SRC_ID = 0

    def __init__(self, kv_cache: torch.Tensor):
        _, v = _split_kv(kv_cache)
        if v is None:
            raise ValueError("ResidentVSource needs a resident V half; this cache is "
                             "K-only -- use a tier V source")
        self._v = v

    def args(self):
        v = self._v
        return (v, *v.stride()[:3])

    def tier_fields(self) -> dict:
        return {}


def ensure_stage_b_buffers(st, device, split: int = SPLIT) -> None:
    """Allocate the split-K partials on the state once (outside any graph capture):
    m_part / l_part (R, n_kv, split, G), acc_part (R, n_kv, split, G, D) fp32."""
    if getattr(st, "m_part", None) is not None:
        st.split = getattr(st, "split", split)
        return
    R, n_kv, G, D = st.max_reqs, st.n_kv, st.G, getattr(st, "D", getattr(st, "d", 128))
    st.split = split
    st.m_part = torch.empty(R, n_kv, split, G, device=device, dtype=torch.float32)
    st.l_part = torch.empty(R, n_kv, split, G, device=device, dtype=torch.float32)
    st.acc_part = torch.empty(R, n_kv, split, G, D, device=device, dtype=torch.float32)


def _pps_min(n_req: int, path: str) -> int:
    """Minimum pages per split (one wave per head).  "auto": 2, the device's plan takes more
    per split once the batch fills the GPU (8 requests keeping 52 pages each, decode + merge,
    at a minimum of 8 / 4 / 3 / 2: 25.4 / 15.9 / 15.2 / 15.3 us; 4 keeping 20: 14.7 / 14.7 /
    14.7 / 11.2); 8 past 64 requests, where short splits of a few heads only add partials (256
    requests of one kv head keeping 20, at 8 / 6 / 4 / 2: 18.3 / 18.2 / 24.3 / 24.3; 72 of 3
    heads keeping 12: 12.8 / 12.8 / 15.5 / 15.1).  "split" splits at the minimum whatever the
    batch: 4 for one request, 8 for more."""
    if path == "auto":
        return 2 if n_req <= 64 else 8
    return 4 if n_req == 1 else 8


def _decode_args(q, k, vsource, block_table, seq_lens, st, out, scale, n_req, *, dense,
                 path, table=None, cnt=None) -> DecodeArgs:
    require_cuda(q, k, block_table, seq_lens, out)
    if q.dtype != torch.bfloat16 or k.dtype != torch.bfloat16 or out.dtype != torch.bfloat16:
        raise ValueError("q, K and out must be bf16")
    qs, ks, os_ = q.stride(), k.stride(), out.stride()
    if qs[2] != 1 or ks[3] != 1 or os_[2] != 1:
        raise ValueError("q / K / out need unit stride on the head dim")
    _, page, n_kv, d = k.shape
    v, svb, svt, svh = vsource.args()
    T, H = q.shape[:2]
    if H % n_kv:
        raise ValueError(f"{H} query heads are not a multiple of {n_kv} kv heads")
    G = H // n_kv
    # the kernels index the state's partials, page tables and counts with these values
    if n_kv != st.n_kv or G != st.G:
        raise ValueError(f"cache / query geometry (n_kv {n_kv}, G {G}) differs from the "
                         f"state's (n_kv {st.n_kv}, G {st.G})")
    if n_req > st.max_reqs:
        raise ValueError(f"n_req {n_req} exceeds max_reqs {st.max_reqs}")
    o_shape = out.shape
    if T < n_req or o_shape[0] < n_req or o_shape[1:] != (H, d) \
            or block_table.shape[0] < n_req:
        raise ValueError("q, out and block_table need a row per request (out (T, H, d))")
    ts = cs = (0, 0, 0)
    if not dense:
        table = st.page_table if table is None else table
        cnt = st.page_cnt if cnt is None else cnt
    if table is not None and cnt is not None:
        ts, cs = table.stride(), cnt.stride()
    if not dense:
        t_shape, c_shape = table.shape, cnt.shape
        if table.dtype != torch.int32 or cnt.dtype != torch.int32 or \
                t_shape[0] < n_req or t_shape[1] != n_kv or ts[2] != 1 or \
                c_shape[0] < n_req or c_shape[1] != n_kv or cs[1] != 1:
            raise ValueError("page_table (R, n_kv, MP) / page_cnt (R, n_kv) int32 expected")
    m, l, acc = (getattr(st, x, None) for x in ("m_part", "l_part", "acc_part"))
    if path != "fused":
        if m is None:
            raise ValueError("split-K partials missing: call ensure_stage_b_buffers(st, "
                             "device) once before decoding (outside any graph capture)")
        split = getattr(st, "split", SPLIT)
        want = (st.max_reqs, n_kv, split, G)
        if m.shape != want or l.shape != want or acc.shape != want + (d,) or not (
                m.is_contiguous() and l.is_contiguous() and acc.is_contiguous()):
            raise ValueError(f"split-K partials must be contiguous {want}[+(d,)] fp32")
    tf = vsource.tier_fields()
    at = lambda t: 0 if t is None else t.data_ptr()  # noqa: E731
    return _pack_decode(               # in the struct's order
        q.data_ptr(), qs[0], qs[1], k.data_ptr(), ks[0], ks[1], ks[2], at(v), svb, svt, svh,
        block_table.data_ptr(), block_table.stride(0), seq_lens.data_ptr(),
        at(table), ts[0], ts[1], at(cnt), cs[0], at(m), at(l), at(acc),
        out.data_ptr(), os_[0], os_[1], tf.get("hot") or 0, tf.get("page2slot") or 0,
        tf.get("vbo") or 0, tf.get("pool") or 0, tf.get("layer") or 0, tf.get("nb") or 0,
        tf.get("slots") or 0, float(scale), n_req, n_kv, G, d, page,
        getattr(st, "split", SPLIT), _pps_min(n_req, path), PATHS[path], 1 if dense else 0,
        vsource.SRC_ID)


def sparse_paged_decode_batched(q, kv_cache, block_table, seq_lens, st, out, vsource, *,
                                scale: float = None, path: str = "auto") -> None:
    """Attend st.page_table[r, kh, :st.page_cnt[r, kh]] of every (request, kv-head)."""
    if scale is None:
        scale = st.scale
    n_req = seq_lens.shape[0]
    a = _decode_args(q, _k_view(kv_cache), vsource, block_table, seq_lens, st, out, scale, n_req,
                     dense=False, path=path)
    call("amass_tier_decode" if vsource.SRC_ID == 1 else "amass_sparse_decode", a,
         current_stream(q.device))


def dense_paged_decode(q, kv_cache, block_table, seq_lens, st, out, *, scale: float,
                       path: str = "auto") -> None:
    """Dense paged decode over every page 0..ceil(seq_len/page) (the baseline the sparse
    path is measured against; same kernels with the page table bypassed)."""
    k, _ = _split_kv(kv_cache)
    n_req = seq_lens.shape[0]
    a = _decode_args(q, k, ResidentVSource(kv_cache), block_table, seq_lens, st, out,
                     scale, n_req, dense=True, path=path)
    call("amass_dense_paged_decode", a, current_stream(q.device))
