"""Workloads of the decode-time sparse-attention path, as a serving program runs them.

A case is a dict of plain values; ``path`` names what it stands for:

  step    one layer of one decode step: page score, selection and sparse attention over the
          selected pages (what the attention backend calls for every layer)
  select  the page score and the selection alone (a program that attends elsewhere, or the
          longest rows, where the attention would hide them)
  attend  the sparse paged attention over page tables that are there already
  bulk    page summaries of every finalised page of a batch (after a prefill), then the
          page score of the first step that reads them
  tail    the steady-state rebuild of each request's last finalised page in every layer,
          then the page score of one layer
  tier    one layer's decode with V in host memory: residency plan, fetch of the missing
          pages into the hot buffer, tiered attention; the selections of consecutive steps
          are correlated
  write   the write path of that tier for one step: the staging life cycle, then every
          layer's V scatter

Sizes are those of the repository's benchmark configurations (8 kv heads, 4 or 8 query
heads each, 4K to 128K tokens) and generic ragged and odd ones around them.  Inputs come
from the seed alone and from plain torch: queries, keys and values are N(0, 1) in bf16, a
twentieth of each (request, kv head)'s pages hold keys pulled towards the head's mean query
(the pages that a selection is for), block tables are random permutations of one pool.
Summaries of the step and select cases are not built by the framework: the page means are
the keys' own, the other factors are drawn with the scales that 16 random keys of 128
channels have (orthogonal directions of unit length, eigenvalues of 120 to 240).
"""
import math
import os
import random
import sys

import torch

sys.path.insert(0, os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))),
                                "amass-kv_amd"))

DEV = "cuda"
PAGE, D = 16, 128
SCALE = D ** -0.5
HEAVY = 0.05                       # share of pages with boosted keys
BETA = 2.0 * math.sqrt(D)          # their pull, in key norms
STEPS = 64                         # selections that a tier case goes through in turn
DRIFT = 0.04                       # share of a selection that changes from one to the next

COMMON = dict(n_kv=8, G=4, rank=8, bits=8, layers=1, budget=0.0, coverage=0.95)


def _case(name, path, **over):
    return dict(dict(COMMON, path=path, **over), name=name)


def listed():
    return [
        # one user, a short chat, a fixed 5 % of the pages: latency and launches count
        _case("step_quad_1x4k", "step", score="quad", combine="nrm", B=1, lo=4096, hi=4096,
              budget=0.05),
        # the benchmark's batch: 32 users at 16K tokens, coverage nucleus
        _case("step_quad_32x16k", "step", score="quad", combine="nrm", B=32, lo=16384, hi=16384),
        # 64 ragged sequences, the r8 score, a fixed 5 %
        _case("step_r8_64xragged", "step", score="r8", combine="max", B=64, lo=2048, hi=65536,
              budget=0.05),
        # the default configuration's score (rank 2, int4 codes and per-key coordinates)
        _case("step_clse_32x16k", "step", score="clse", combine="nrm", B=32, lo=16384, hi=16384,
              rank=2, bits=4),
        # odd everything: 5 requests of odd lengths, 4 kv heads of 7 queries, rank 4, int4
        _case("step_quad_5xodd_g7", "step", score="quad", combine="max", B=5, lo=777, hi=23001,
              n_kv=4, G=7, rank=4, bits=4, coverage=0.9),
        # the longest rows: 8 requests of 128K tokens, groups of 8
        _case("select_quad_8x128k", "select", score="quad", combine="nrm", B=8, lo=131072,
              hi=131072, G=8),
        # attention where the selection keeps most pages (a flat score): bound by memory
        _case("attend_32x16k_93", "attend", B=32, lo=16384, hi=16384, keep=0.93),
        # attention over a tenth of ragged contexts
        _case("attend_12xragged_10", "attend", B=12, lo=1500, hi=50001, keep=0.1),
        # summaries of a prefilled batch
        _case("bulk_quad_8x16k", "bulk", score="quad", combine="max", B=8, lo=16384, hi=16384),
        # the steady-state rebuild, default configuration, every layer of a 32-layer model
        _case("tail_clse_32x400_l32", "tail", score="clse", combine="max", B=32, lo=401, hi=401,
              rank=2, bits=4, layers=32),
        # V in host memory, a hot buffer of a tenth of the pages, correlated selections
        _case("tier_16x16k", "tier", B=16, lo=16384, hi=16384, keep=HEAVY),
        # its write path in a decode step of 32 requests
        _case("write_32x1", "write", B=32, lo=1024, hi=1024, ql=1, layers=2),
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    path = rng.choice(("step", "step", "step", "step", "select", "attend", "attend", "bulk",
                       "tail", "tier", "write"))
    c = dict(COMMON, path=path)
    if path in ("step", "select", "bulk", "tail"):
        c["score"] = rng.choice(("quad", "quad", "clse", "r8"))
        c["combine"] = "max" if c["score"] == "r8" or path in ("bulk", "tail") else \
            rng.choice(("nrm", "nrm", "max"))
        c["rank"], c["bits"] = rng.choice(((8, 8), (8, 8), (4, 8), (8, 4)) if c["score"] == "r8"
                                          else ((8, 8), (8, 8), (4, 8), (2, 4)))
        c["G"] = rng.choice((1, 2, 4, 4, 8)) if c["score"] != "quad" else rng.choice(
            (1, 3, 4, 4, 5, 7, 8))
        c["n_kv"] = rng.choice((8, 8, 8, 4, 2))
        if rng.random() < 0.4:
            c["budget"] = round(rng.uniform(0.03, 0.2), 3)
        else:
            c["coverage"] = round(rng.uniform(0.85, 0.97), 3)
    if path in ("step", "select", "attend"):
        c["B"] = _log(rng, 1, 64)
        c["hi"] = _log(rng, 600, min(131072, 500000 // c["B"]))
        c["lo"] = c["hi"] if rng.random() < 0.3 else max(64, c["hi"] // rng.choice((2, 4, 16)))
        if path == "attend":
            c["keep"] = round(math.exp(rng.uniform(math.log(0.04), 0.0)), 3)
            c["G"] = rng.choice((1, 2, 4, 4, 6, 8))
            c["n_kv"] = rng.choice((8, 8, 4))
    elif path == "bulk":
        c["B"] = _log(rng, 1, 16)
        c["hi"] = _log(rng, 200, 131072 // c["B"])
        c["lo"] = max(48, c["hi"] // 2)
    elif path == "tail":
        c["B"], c["layers"] = _log(rng, 1, 64), _log(rng, 1, 32)
        c["lo"] = c["hi"] = 16 * rng.randint(4, 60) + 1       # a page has just filled up
    elif path == "tier":
        c["B"] = _log(rng, 1, 16)
        c["hi"] = c["lo"] = _log(rng, 1024, 16384)
        c["keep"] = round(rng.uniform(0.03, 0.08), 3)
    else:
        c["B"], c["ql"] = _log(rng, 1, 32), 1 if rng.random() < 0.6 else _log(rng, 2, 64)
        c["hi"] = c["lo"] = 16 * rng.randint(30, 80)
        c["layers"] = rng.randint(1, 2)
    return c


# ------------------------------------------------------------------ inputs, from the seed
def _gen(seed):
    return torch.Generator(device=DEV).manual_seed(int(seed))


def _lens(c, seed):
    rng = random.Random(int(seed) * 7 + 1)
    return [rng.randint(c["lo"], c["hi"]) for _ in range(c["B"])]


def _max_pages(c):
    return -(-c["hi"] // PAGE)


def _table(lens, MP, gen):
    """(block table (B, MP) int32, blocks): a random permutation of one pool."""
    npg = [-(-n // PAGE) for n in lens]
    NB = sum(npg) + 16
    order = torch.randperm(NB, generator=gen, device=DEV).to(torch.int32)
    bt = torch.zeros(len(lens), MP, dtype=torch.int32, device=DEV)
    at = 0
    for r, n in enumerate(npg):
        bt[r, :n] = order[at:at + n]
        at += n
    return bt, NB


def _randn(shape, gen):
    """bf16 N(0, 1), made in parts (a whole fp32 copy of the largest pool is not needed)."""
    x = torch.empty(shape, dtype=torch.bfloat16, device=DEV)
    flat = x.view(-1)
    for i in range(0, flat.numel(), 1 << 28):
        flat[i:i + (1 << 28)].normal_(generator=gen)
    return x


def _pages(c, seed, layers=1):
    """Queries, paged caches (one per layer), block table and lengths, boosted pages."""
    gen = _gen(seed)
    B, n_kv, G, MP = c["B"], c["n_kv"], c["G"], _max_pages(c)
    lens = _lens(c, seed)
    bt, NB = _table(lens, MP, gen)
    q = _randn((B, n_kv * G, D), gen)
    kvs = []
    u = q.float().view(B, n_kv, G, D).mean(2)
    u = u / u.norm(dim=-1, keepdim=True).clamp_min(1e-12)
    for _ in range(layers):
        kv = _randn((NB, 2, PAGE, n_kv, D), gen)
        heavy = torch.rand(B, MP, n_kv, generator=gen, device=DEV) < HEAVY
        for r, n in enumerate(lens):
            npg = -(-n // PAGE)
            blk = bt[r, :npg].long()
            add = (heavy[r, :npg, :, None] * (BETA * u[r])).to(torch.bfloat16)
            kv[blk, 0] += add[:, None]
        kvs.append(kv)
    sl = torch.tensor(lens, dtype=torch.int32, device=DEV)
    return dict(q=q, kvs=kvs, bt=bt, sl=sl, lens=lens, NB=NB, MP=MP, gen=gen)


def _quant(x, dim, lvl):
    s = (x.abs().amax(dim=dim, keepdim=True) / lvl).clamp_min(1e-8)
    return torch.round(x / s).clamp_(-lvl, lvl).to(torch.int8), s


def _pack(code, bits):
    """int4: two columns to a byte, the even one in the low half."""
    if bits == 8:
        return code
    x = code.to(torch.int32) & 0xF
    return (x[..., 0::2] | (x[..., 1::2] << 4)).to(torch.uint8).view(torch.int8).contiguous()


def _summary(c, inp):
    """Codes and scales of every block, as a program that loads them holds them."""
    NB, n_kv, r, gen = inp["NB"], c["n_kv"], c["rank"], inp["gen"]
    lvl = 127.0 if c["bits"] == 8 else 7.0
    mu = torch.empty(NB, n_kv, D, device=DEV)
    for i in range(0, NB, 8192):
        mu[i:i + 8192] = inp["kvs"][0][i:i + 8192, 0].float().mean(1)
    mu, mus = _quant(mu, -1, 127.0)
    V = torch.randn(NB, n_kv, D, r, generator=gen, device=DEV) / math.sqrt(D)
    V, Vs = _quant(V, -2, lvl)
    sig2 = 120.0 + 15.0 * torch.arange(r, device=DEV) + 5.0 * torch.rand(
        NB, n_kv, r, generator=gen, device=DEV)
    s = dict(mu=mu, mus=mus[..., 0].half(), V=V, Vs=Vs[..., 0, :].half(), sig2=sig2.half())
    if c["score"] != "quad":
        x = 0.25 * sig2.sqrt()[..., None, :] * torch.randn(NB, n_kv, PAGE, r, generator=gen,
                                                           device=DEV)
        s["c"], cs = _quant(x, -1, lvl)
        s["cs"] = cs[..., 0].half()
        s["resid"] = (15.0 * D - sig2.sum(-1)).clamp_min(0).half()
    return s


# ------------------------------------------------------------------ prepare and run
def _state(c, NB, MP, layers=1):
    from amass.attention import ensure_stage_b_buffers
    from amass.selection import QuadState, R8State
    kw = dict(num_layers=layers, num_blocks=NB, n_kv=c["n_kv"], G=c["G"], head_dim=D, page=PAGE,
              max_reqs=c["B"], max_pages=MP, rank=c["rank"], budget=c["budget"] or 0.1)
    score = c.get("score", "quad")
    if score == "r8":
        st = R8State(DEV, vk_bits=c["bits"], c_bits=c["bits"], **kw)
    elif score == "clse":
        st = QuadState(DEV, v_bits=c["bits"], combine=c["combine"], coords="lse",
                       c_bits=c["bits"], **kw)
    else:
        st = QuadState(DEV, v_bits=c["bits"], combine=c.get("combine", "max"), **kw)
    st.coverage = None if c["budget"] else c["coverage"]
    st.scale = SCALE
    ensure_stage_b_buffers(st, DEV)
    st.score.zero_()               # its entries past a row's end are never written
    st.page_table.fill_(-1)
    return st


def _tables(c, inp, gen, n):
    """n page tables (B, n_kv, MP) and their counts: the first and last pages of every row
    and a random `keep` of the others, DRIFT of which moves from one table to the next."""
    B, n_kv, MP = c["B"], c["n_kv"], inp["MP"]
    npg = (inp["sl"].long() + PAGE - 1) // PAGE
    p = torch.arange(MP, device=DEV)
    on = (p[None] < npg[:, None])[:, None].expand(B, n_kv, MP)
    always = ((p[None] == 0) | (p[None] >= npg[:, None] - 2))[:, None]
    pick = torch.rand(B, n_kv, MP, generator=gen, device=DEV) < c["keep"]
    out = []
    for _ in range(n):
        keep = on & (always | pick)
        cnt = keep.sum(-1).to(torch.int32)
        key = torch.where(keep, p, MP + p)                    # kept pages first, ascending
        tab = key.sort(-1).values
        tab = torch.where(tab < MP, tab, -1).to(torch.int32).contiguous()
        out.append((tab, cnt))
        new = torch.rand(B, n_kv, MP, generator=gen, device=DEV) < c["keep"]
        move = torch.rand(B, n_kv, MP, generator=gen, device=DEV) < DRIFT
        pick = torch.where(move, new, pick)
    return out


def prepare(case, seed):
    c = case
    return {"step": _prepare_step, "select": _prepare_step, "attend": _prepare_attend,
            "bulk": _prepare_build, "tail": _prepare_build, "tier": _prepare_tier,
            "write": _prepare_write}[c["path"]](c, seed)


def run(state):
    return state["run"](state)


def _prepare_step(c, seed):
    from amass.attention.decode import ResidentVSource
    from amass.selection import derive_page_params
    inp = _pages(c, seed)
    s = _summary(c, inp)
    st = _state(c, inp["NB"], inp["MP"])
    V = _pack(s["V"], c["bits"])
    if c["score"] == "quad":
        st.load_reference(0, s["mu"], s["mus"], V, s["Vs"], s["sig2"])
    elif c["score"] == "clse":
        st.load_reference(0, s["mu"], s["mus"], V, s["Vs"], c=_pack(s["c"], c["bits"]),
                          c_scale=s["cs"], resid=s["resid"])
    else:
        st.load_reference(0, s["mu"], s["mus"], V, s["Vs"], _pack(s["c"], c["bits"]), s["cs"])
    # an engine derives a step's page counts once for all layers
    derive_page_params(st, inp["sl"], c["B"])
    kv = inp["kvs"][0]
    return dict(run=_run_step, c=c, st=st, q=inp["q"], kv=kv, bt=inp["bt"], sl=inp["sl"],
                out=torch.zeros_like(inp["q"]), vs=ResidentVSource(kv))


def _select(s, st, layer=0):
    from amass.selection import select_pages_clse, select_pages_quad, select_pages_r8
    fn = {"quad": select_pages_quad, "clse": select_pages_clse, "r8": select_pages_r8}
    fn[s["c"]["score"]](st, layer, s["q"], s["bt"], s["sl"], s["c"]["B"], SCALE, derive=False)


def _run_step(s):
    from amass.attention.decode import sparse_paged_decode_batched
    from amass.selection import select_then_attend
    c, st = s["c"], s["st"]
    res = dict(score=st.score, page_cnt=st.page_cnt, page_table=st.page_table)
    if c["path"] == "select":
        _select(s, st)
        return res
    if c["score"] == "quad":
        select_then_attend(st, 0, s["q"], s["kv"], s["bt"], s["sl"], c["B"], SCALE, s["out"],
                           s["vs"])
    else:
        _select(s, st)
        sparse_paged_decode_batched(s["q"], s["kv"], s["bt"], s["sl"], st, s["out"], s["vs"],
                                    scale=SCALE)
    return dict(res, out=s["out"])


def _prepare_attend(c, seed):
    from amass.attention.decode import ResidentVSource
    inp = _pages(c, seed)
    st = _state(c, 1, inp["MP"])
    tab, cnt = _tables(c, inp, inp["gen"], 1)[0]
    st.page_table.copy_(tab)
    st.page_cnt.copy_(cnt)
    kv = inp["kvs"][0]
    return dict(run=_run_attend, c=c, st=st, q=inp["q"], kv=kv, bt=inp["bt"], sl=inp["sl"],
                out=torch.zeros_like(inp["q"]), vs=ResidentVSource(kv))


def _run_attend(s):
    from amass.attention.decode import sparse_paged_decode_batched
    sparse_paged_decode_batched(s["q"], s["kv"], s["bt"], s["sl"], s["st"], s["out"], s["vs"],
                                scale=SCALE)
    return s["out"]


def _build_fns(c):
    from amass import selection as sel
    if c["score"] == "r8":
        return sel.r8_build_bulk, sel.r8_build_tail
    return sel.quad_build_bulk, sel.quad_build_tail


def _prepare_build(c, seed):
    from amass.attention.decode import _split_kv
    from amass.selection import derive_page_params
    inp = _pages(c, seed, c["layers"])
    st = _state(c, inp["NB"], inp["MP"], c["layers"])
    derive_page_params(st, inp["sl"], c["B"])
    Ks = [_split_kv(kv)[0] for kv in inp["kvs"]]
    if c["path"] == "tail":            # everything but the last page is summarised already
        _build_fns(c)[0](st, Ks, inp["bt"], inp["sl"] - PAGE, c["B"])
    return dict(run=_run_build, c=c, st=st, Ks=Ks, q=inp["q"], bt=inp["bt"], sl=inp["sl"],
                kvs=inp["kvs"])


def _run_build(s):
    """Eigenvectors have no sign of their own, so the V codes and coordinates come back as
    the page score that they give; the other parts of the summaries come back whole."""
    from amass.selection import clse_score, quad_score, r8_score
    c, st = s["c"], s["st"]
    bulk, tail = _build_fns(c)
    (tail if c["path"] == "tail" else bulk)(st, s["Ks"], s["bt"], s["sl"], c["B"])
    fn = {"quad": quad_score, "clse": clse_score, "r8": r8_score}[c["score"]]
    fn(st, c["layers"] - 1, s["q"], s["bt"], s["sl"], c["B"], SCALE)
    if c["score"] == "r8":
        return dict(mu=st.r8_mu, mu_scale=st.mu_scale, V_scale=st.Vk_scale, c_scale=st.c_scale,
                    score=st.score)
    res = dict(mu=st.quad_mu, mu_scale=st.mu_scale, V_scale=st.V_scale, score=st.score)
    if c["score"] == "clse":
        return dict(res, c_scale=st.c_scale, resid=st.quad_resid)
    return dict(res, sig2=st.quad_sig2)


def _prepare_tier(c, seed):
    from amass.tier import Tier
    inp = _pages(c, seed)
    st = _state(c, 1, inp["MP"])
    kv = inp["kvs"][0]
    tier = Tier(num_layers=1, num_blocks=inp["NB"], n_kv=c["n_kv"], page=PAGE, d=D,
                hot_slots=max(64, c["B"] * inp["MP"] // 10), max_reqs=c["B"],
                max_pages=inp["MP"], device=DEV, v_blocks=2 * c["B"] + 8)
    tier.flush_layer(0, kv[:, 1])
    tabs = _tables(c, inp, inp["gen"], STEPS)
    # the hot buffer holds the pages of the step before the first
    tier.step(0, tabs[-1][0], tabs[-1][1], inp["bt"], inp["sl"], c["B"])
    return dict(run=_run_tier, c=c, st=st, tier=tier, tabs=tabs, at=0, q=inp["q"], kv=kv,
                bt=inp["bt"], sl=inp["sl"], out=torch.zeros_like(inp["q"]))


def _run_tier(s):
    from amass.tier import mem_dynamic_decode
    st, r5 = s["st"], s["tier"].residency
    st.page_table, st.page_cnt = s["tabs"][s["at"] % STEPS]
    s["at"] += 1
    mem_dynamic_decode(s["q"], s["kv"], s["bt"], s["sl"], st, s["out"], s["tier"], 0,
                       scale=SCALE)
    return dict(out=s["out"], page2slot=r5.page2slot, slot2page=r5.slot2page,
                lru_clock=r5.lru_clock, clock=r5.clock)


def _prepare_write(c, seed):
    """32 consecutive steps of `ql` tokens per request, each request at a phase of its own
    (the requests do not cross page boundaries together), then over again: a request that
    ends gives its blocks to the next one."""
    from amass.tier import Tier
    gen = _gen(seed)
    B, ql, L, n_kv = c["B"], c["ql"], c["layers"], c["n_kv"]
    MP = -(-(c["hi"] + 32 * ql) // PAGE)
    bt, NB = _table([MP * PAGE] * B, MP, gen)
    tier = Tier(num_layers=L, num_blocks=NB, n_kv=n_kv, page=PAGE, d=D, hot_slots=256,
                max_reqs=B, max_pages=MP, device=DEV, max_tokens=B * ql,
                v_blocks=B * (32 * ql // PAGE + 3))
    phase = torch.randint(0, 32, (B,), generator=gen, device=DEV)
    qsl = (ql * torch.arange(B + 1, device=DEV)).to(torch.int32)
    sls = [(c["lo"] + ql * ((phase + k) % 32 + 1)).to(torch.int32) for k in range(32)]
    vals = [_randn((B * ql, n_kv, D), gen) for _ in range(L)]
    return dict(run=_run_write, c=c, tier=tier, bt=bt, qsl=qsl, sls=sls, vals=vals, at=0)


def _run_write(s):
    tier, c = s["tier"], s["c"]
    n = c["B"] * c["ql"]
    tier.begin_step(s["bt"], s["sls"][s["at"] % 32], s["qsl"], n)
    s["at"] += 1
    for layer in range(c["layers"]):
        tier.write_kv(layer, s["vals"][layer], n)
    sg = tier.staging
    return dict(v_pool=sg.v_pool, slots=sg.v_slot_mapping, vbo=sg.vbo, free_top=sg.v_free_top,
                overflow=sg.overflow, pool_valid=tier.residency.pool_valid)


# ------------------------------------------------------------------ what a pass needs
def _record_bytes(c):
    """One (page, kv head)'s summary: V, mu, their scales, and sig2 or the coordinates."""
    r, b = c["rank"], c["bits"]
    n = D * r * b // 8 + D + 2 * r + 2
    if c["score"] == "quad":
        return n + 2 * r
    return n + PAGE * r * b // 8 + 2 * PAGE + (2 if c["score"] == "clse" else 0)


def work(case):
    c = case
    B, n_kv, G = c["B"], c["n_kv"], c["G"]
    pages = B * -(-(c["lo"] + c["hi"]) // (2 * PAGE))       # of the mean length
    units = pages * n_kv
    rec = _record_bytes(c) if "score" in c else 0
    kv = 2 * PAGE * D * 2                                   # K and V of a (page, kv head)
    qo = 2 * B * n_kv * G * D * 2
    att = 4 * G * PAGE * D                                  # flops of attending one
    sc = 2 * G * D * (c["rank"] + 1)                        # ... and of scoring one
    if c["path"] == "tail":
        units, read = B * n_kv * c["layers"], pages * n_kv
        return dict(bytes=units * (kv // 2 + rec) + read * (rec + 4),
                    flops=units * (2 * PAGE * PAGE * D + 2 * PAGE * D * c["rank"]) + read * sc)
    if c["path"] == "bulk":
        return dict(bytes=units * (kv // 2 + 2 * rec + 4),
                    flops=units * (2 * PAGE * PAGE * D + 2 * PAGE * D * c["rank"] + sc))
    if c["path"] == "write":
        n = B * c["ql"] * c["layers"] * n_kv * D * 2
        return dict(bytes=3 * n + 8 * B * c["ql"], flops=0)
    if c["path"] in ("attend", "tier"):
        kept = units * c["keep"] + 3 * B * n_kv
        return dict(bytes=kept * (kv + 8) + qo, flops=kept * att)
    kept = 0.0 if c["path"] == "select" else units * (c["budget"] or HEAVY) + 3 * B * n_kv
    return dict(bytes=units * (rec + 8) + pages * 4 + kept * kv + qo,
                flops=units * sc + kept * att)


def tolerance(case):
    p = case["path"]
    if p == "write":
        return "exact"                              # bf16 rows and tables are copied
    if p in ("attend", "tier"):
        return {"rel": 8e-3, "max": 0.2}            # bf16 outputs: 2e-3 off the 64-bit ones
    if p in ("bulk", "tail"):
        # fp16 scales; a score of int8 or int4 codes whose ties round apart with another
        # eigensolver (32 against 64 bits: 1.4e-4 and 7e-4, at most 0.07 of a score)
        return {"rel": 3e-3, "max": 0.3, "differ": 1e-3}
    # a page at the selection's cut may be the next one; scores are fp32 (1.5e-5 off the
    # 64-bit ones: the query's two int8 limbs)
    if p == "select":
        return {"rel": 6e-5, "max": 4e-3, "differ": 5e-3}
    return {"rel": 8e-3, "max": 0.2, "differ": 5e-3}


# ------------------------------------------------------------------ the same in 64 bits
def _scores64(c, q, mu, V, sig2, coords, resid, bt_r, sl_r, nsel):
    """(n_kv, G, nsel) page scores of one request.  q (n_kv, G, D); mu (NB, n_kv, D), V
    (NB, n_kv, D, r) and the other factors by block, all in 64 bits."""
    blk = bt_r[:nsel].long()
    S = SCALE * torch.matmul(q, mu(blk).permute(1, 2, 0))                    # (n_kv, G, n)
    w = torch.matmul(q[None], V(blk))                                        # (n, n_kv, G, r)
    if c["score"] == "quad":
        quad = (w * w * sig2(blk)[:, :, None, :]).sum(-1) * (SCALE * SCALE / (2 * PAGE))
        return S + quad.permute(1, 2, 0)
    tok = SCALE * torch.matmul(w, coords(blk).transpose(-1, -2))             # (n, n_kv, G, 16)
    at = PAGE * torch.arange(nsel, device=DEV)[:, None] + torch.arange(PAGE, device=DEV)
    tok = tok.masked_fill((at >= sl_r)[:, None, None, :], -math.inf)
    S = S + torch.logsumexp(tok, -1).permute(1, 2, 0)
    if c["score"] == "clse":
        iso = ((q * q).sum(-1)[None] - (w * w).sum(-1)).clamp_min(0) * resid(blk)[..., None]
        S = S + (iso * (SCALE * SCALE / (2 * PAGE * max(D - c["rank"], 1)))).permute(1, 2, 0)
    return S


def _score_rows64(c, inp, **factors):
    """st.score: the group's maximum, or the sum of its heads' normalised masses."""
    B, n_kv, G = c["B"], c["n_kv"], c["G"]
    out = torch.zeros(B, n_kv, inp["MP"], dtype=torch.float64, device=DEV)
    q = inp["q"].double().view(B, n_kv, G, D)
    for r, n in enumerate(inp["lens"]):
        nsel = -(-n // PAGE) - 1
        if nsel <= 0:
            continue
        for h in range(n_kv):          # one kv head at a time: bounded temporaries
            f = {k: (lambda b, v=v, h=h: v(b, h)) for k, v in factors.items()}
            S = _scores64(c, q[r, h:h + 1], f["mu"], f["V"], f["sig2"], f["coords"], f["resid"],
                          inp["bt"][r], n, nsel)[0]
            out[r, h, :nsel] = torch.exp(S - S.amax(-1, keepdim=True)).sum(0) \
                if c["combine"] == "nrm" else S.amax(0)
    return out


def _attend64(c, inp, tab, cnt):
    B, n_kv, G = c["B"], c["n_kv"], c["G"]
    out = torch.zeros(B, n_kv, G, D, dtype=torch.float64, device=DEV)
    q = inp["q"].double().view(B, n_kv, G, D)
    p = torch.arange(inp["MP"], device=DEV)
    for r, n in enumerate(inp["lens"]):
        for h in range(n_kv):
            t = tab[r, h, :int(cnt[r, h])].long()
            kv = inp["kvs"][0][inp["bt"][r, t].long(), :, :, h].double()     # (n, 2, 16, D)
            K, V = kv[:, 0].reshape(-1, D), kv[:, 1].reshape(-1, D)
            pos = (PAGE * t[:, None] + torch.arange(PAGE, device=DEV)).reshape(-1)
            lg = (SCALE * (q[r, h] @ K.T)).masked_fill((pos >= n)[None], -math.inf)
            out[r, h] = torch.softmax(lg, -1) @ V
    return out.view(B, n_kv * G, D)


def exact(case, seed):
    c = case
    if c["path"] == "write":
        return None
    if c["path"] in ("attend", "tier"):
        inp = _pages(c, seed)
        tab, cnt = _tables(c, inp, inp["gen"], STEPS if c["path"] == "tier" else 1)[0]
        out = _attend64(c, inp, tab, cnt)
        if c["path"] == "attend":
            return out
        return dict(out=out, page2slot=None, slot2page=None, lru_clock=None, clock=None)
    if c["path"] in ("bulk", "tail"):
        units = c["B"] * (c["hi"] // PAGE) * c["n_kv"] * c["layers"]
        return _exact_build(c, seed) if units <= 300000 else None   # (an eigh on the host each)
    inp = _pages(c, seed)
    s = _summary(c, inp)
    f = dict(mu=lambda b, h: s["mu"][b, h:h + 1].double() * s["mus"][b, h:h + 1, None].double(),
             V=lambda b, h: (s["V"][b, h:h + 1].double() * s["Vs"][b, h:h + 1, None].double()),
             sig2=lambda b, h: s["sig2"][b, h:h + 1].double(),
             coords=lambda b, h: (s["c"][b, h:h + 1].double()
                                  * s["cs"][b, h:h + 1, :, None].double()),
             resid=lambda b, h: s["resid"][b, h:h + 1].double())
    res = dict(score=_score_rows64(c, inp, **f), page_cnt=None, page_table=None)
    return res if c["path"] == "select" else dict(res, out=None)


def _exact_build(c, seed):
    """Summaries without their quantisation, and the score that they give."""
    L, r, n_kv = c["layers"], c["rank"], c["n_kv"]
    inp = _pages(c, seed, L)
    NB = inp["NB"]
    lvl = 127.0 if c["bits"] == 8 else 7.0
    f64 = dict(dtype=torch.float64, device=DEV)
    mus, Vs = torch.zeros(L, NB, n_kv, **f64), torch.zeros(L, NB, n_kv, r, **f64)
    sig2, cs = torch.zeros(L, NB, n_kv, r, **f64), torch.zeros(L, NB, n_kv, PAGE, **f64)
    resid = torch.zeros(L, NB, n_kv, **f64)
    blocks = torch.cat([inp["bt"][i, :n // PAGE].long() for i, n in enumerate(inp["lens"])])
    for lay in range(L):
        mu, V = torch.zeros(NB, n_kv, D, **f64), torch.zeros(NB, n_kv, D, r, **f64)
        co = torch.zeros(NB, n_kv, PAGE, r, **f64)
        K = inp["kvs"][lay][blocks, 0].permute(0, 2, 1, 3).double()          # (n, n_kv, 16, D)
        m = K.mean(2)
        dc = K - m[:, :, None]
        S2, U = torch.linalg.eigh(torch.matmul(dc, dc.transpose(-1, -2)).cpu())
        S2r, U8 = S2[..., -r:].clamp_min(1e-10).to(DEV), U[..., -r:].to(DEV)
        vk = torch.matmul(dc.transpose(-1, -2), U8) / S2r.sqrt()[..., None, :]
        cc = U8 * S2r.sqrt()[..., None, :]
        mu[blocks], V[blocks], co[blocks] = m, vk, cc
        mus[lay, blocks] = (m.abs().amax(-1) / 127.0).clamp_min(1e-8)
        Vs[lay, blocks] = (vk.abs().amax(-2) / lvl).clamp_min(1e-8)
        sig2[lay, blocks] = S2r
        cs[lay, blocks] = (cc.abs().amax(-1) / lvl).clamp_min(1e-8)
        resid[lay, blocks] = ((dc * dc).sum((-1, -2)) - S2r.sum(-1)).clamp_min(0)
    f = dict(mu=lambda b, h: mu[b, h:h + 1], V=lambda b, h: V[b, h:h + 1],
             sig2=lambda b, h: sig2[L - 1, b, h:h + 1], coords=lambda b, h: co[b, h:h + 1],
             resid=lambda b, h: resid[L - 1, b, h:h + 1])
    res = dict(mu=None, mu_scale=mus, V_scale=Vs, score=_score_rows64(c, inp, **f))
    if c["score"] == "r8":
        return dict(res, c_scale=cs)
    if c["score"] == "clse":
        return dict(res, c_scale=cs, resid=resid)
    return dict(res, sig2=sig2)
