"""r8 page score (Stage A.1, r8 mode) -- host side of ``amass_r8_score``.

Same contract as the reference ``r8_score`` (selection/score.py:123-148): writes
``st.score`` (R, n_kv, MP) fp32, the group max of s*mu.q + logsumexp_t(s * c_t . q~)
over the scored region.  ``comb_out`` (optional int32 (R, n_kv, MP, G, r+1)) receives the
exact integer d-contractions sum_d qi*code (the r columns of Vk, then mu).
"""
from __future__ import annotations

import torch

from .._hip import R8ScoreArgs, call, current_stream, layer_slab, packer, require_cuda

_r8_args = packer(R8ScoreArgs)


def check_rec_span(rec) -> None:
    """The score kernels address a layer's records with 32-bit byte offsets from its base
    (block * rec_sb + head and lane offsets), so the layer's record buffer must span less
    than 4 GiB."""
    _check_span(rec.shape[0], rec.stride(0))


def _check_span(blocks: int, stride: int) -> None:
    if blocks * stride > (1 << 32):
        raise ValueError(f"a layer's summary records span {blocks * stride} "
                         "bytes; the score kernels address at most 4 GiB per layer")


def score_inputs(st, recs, name, layer, q, block_table):
    """The checks that every score launch makes of its query, block table and records, and
    (record address, record block stride, q strides) for the argument struct."""
    require_cuda(q, block_table, recs)
    qs = q.stride()
    if q.dtype != torch.bfloat16 or qs[2] != 1:
        raise ValueError("q must be bf16 (T, H, d) with unit stride on d")
    if block_table.dtype != torch.int32 or block_table.stride(1) != 1:
        raise ValueError("block_table must be int32 with unit column stride")
    rec, rs, shape = layer_slab(recs, layer)
    if rs[1] != 1 or shape[1] != st.n_kv * st.rec_bytes:
        raise ValueError(f"{name} must hold each block's records contiguously")
    _check_span(shape[0], rs[0])
    return rec, rs[0], qs


def r8_score(st, layer: int, q, block_table, seq_lens, n_req: int, scale: float,
             comb_out=None) -> None:
    if n_req > st.max_reqs:
        raise ValueError(f"n_req {n_req} exceeds max_reqs {st.max_reqs}")
    require_cuda(seq_lens)
    if block_table.dtype != torch.int32 or seq_lens.dtype != torch.int32:
        raise ValueError("block_table / seq_lens must be int32")
    rec, rec_sb, qs = score_inputs(st, st.r8_rec, "r8_rec", layer, q, block_table)
    if comb_out is not None and (comb_out.dtype != torch.int32 or not comb_out.is_contiguous()
                                 or tuple(comb_out.shape[1:]) != (st.n_kv, st.max_pages, st.G,
                                                                  st.r + 1)):
        raise ValueError("comb_out must be a contiguous int32 (R, n_kv, MP, G, r+1) tensor")
    sc = st.score
    ss = sc.stride()
    a = _r8_args(                      # in the struct's order
        q.data_ptr(), qs[0], qs[1], rec, rec_sb, block_table.data_ptr(), block_table.stride(0),
        seq_lens.data_ptr(), st.n_sel_hi.data_ptr(), sc.data_ptr(), ss[0], ss[1],
        0 if comb_out is None else comb_out.data_ptr(), float(scale), n_req, st.n_kv, st.G,
        st.d, st.page, st.r, st.vk_bits, st.c_bits, st.max_pages,
        1 if getattr(st, "c_grain", "page") == "page_f32" else 0)
    call("amass_r8_score", a, current_stream(q.device))
