// mem-v write path for gfx950: residency invalidation, the per-step staging lifecycle
// (flushed-bit clear, flush collect, flush copy to the pinned pool, staging-block alloc,
// token slots) and the per-layer V scatter.
//
// Semantics of tier/residency.py:251-278 (_invalidate_kernel) and tier/staging.py:51-232
// (_scatter_kv, _vflush_clear, _flush_collect, _flush_copy, _valloc, _vslot kernels),
// taken in (request, page) order.  The reference serialises collect and alloc in one
// program (grid (1,)) because they share the flush index and the free-stack top; here
// they are one 1024-thread workgroup each that ranks a whole chunk of pages at once with
// block scans, and visits only the 256-page chunks a parallel mark pass found holding a
// staged block (a decode step completes about one page per request every 16 tokens, so
// almost every chunk is skipped).  Shared blocks count once (the first occurrence in
// order), as the reference's atomic claims make them.
//
// Latency-bound: a decode step moves a few pages, so its cost is launches and dependent
// memory rounds.  A step is two launches where the batch's block tables hold at most
// ST_SMALL entries (n_req max_pages, n_req <= ST_REQS): one workgroup that reads every
// table entry's staging block itself (up to 8 per thread, all in flight) and collects, then
// one launch whose first workgroup allocates and maps the tokens while the others copy the
// flushed pages (the copies read the flush list and v_pool, neither of which the alloc
// writes; the scatter that reuses a staging block is a later launch).  Wider batches spread
// the table scan over a mark launch first: one CU gathers 1-2 entries a nanosecond, which
// past the limits costs more than the launch.  Decode steps with the invalidation, us, one
// workgroup / mark launch, in a graph (five launches before: 15.3-16.5 throughout) and eager:
// 32 requests of 192-page tables 10.8 / 12.2 and 12.8 / 19.4, of 256 13.7 / 12.3 and 13.6 / 19.3,
// of 512 20.2 / 12.0 and 20.0 / 15.9; 128 of 32 12.2 / 12.5 and 13.0 / 18.7, of 64 15.8 / 12.8 and
// 16.0 / 18.5; 256 of 64 24.7 / 13.2 and 25.0 / 15.9.  At 32 decode requests
// of 66-page tables the two take 6.1 + 6.0 us (five launches -- mark, collect, copy, alloc,
// token slots -- 3.8 + 5.0 + 4.9 + 4.9 + 2.5), the whole eager step with the invalidation and
// two layers' scatters 46.8 -> 26.6 us, bound by the host's launches; with the invalidation in
// the collect's launch 28.2 -> 23.0 (both sides in one run).
#include "common.h"

namespace amass {

constexpr int ST_SMALL = 8192;     // table entries one workgroup scans: 8 per thread ...
constexpr int ST_REQS = 128;       // ... of at most so many requests
constexpr int ST_TOKENS = 16384;   // tokens the allocating workgroup maps itself
constexpr int ST_CHUNK = 256;      // pages per mark chunk
constexpr int ST_THREADS = 1024;   // collect / alloc workgroup
constexpr int ST_WAVES = ST_THREADS / WAVE;

// exclusive prefix over the workgroup's threads of v; total in `total` (two barriers)
__device__ __forceinline__ int st_excl_scan(int v, int* red, int& total) {
    const int lane = threadIdx.x & 63, w = threadIdx.x >> 6;
    const int nw = blockDim.x >> 6;
    const int x = wave_incl_scan(v);                  // DPP row steps + readlane
    __syncthreads();
    if (lane == 63) red[w] = x;
    __syncthreads();
    int base = 0, tot = 0;
    for (int i = 0; i < nw; ++i) {
        const int t = red[i];
        if (i < w) base += t;
        tot += t;
    }
    total = tot;
    return base + x - v;
}

struct ReqRange {
    bool active;      // sl > 0 and ql > 0
    int ctx;          // settled tokens sl - ql
    int p0, p1;       // written pages
};
__device__ __forceinline__ ReqRange req_range(const int32_t* sl_, const int32_t* qsl, int r,
                                              int page) {
    ReqRange x;
    const int sl = sl_[r];
    const int ql = qsl[r + 1] - qsl[r];
    x.active = sl > 0 && ql > 0 && ql <= sl;
    x.ctx = sl - ql;
    x.p0 = x.ctx >= 0 ? x.ctx / page : 0;
    x.p1 = sl > 0 ? (sl - 1) / page : -1;
    return x;
}

// ------------------------------------------------------------------ invalidate
// every (written page, kv head) of request r in layer l, by 256 threads
constexpr int INV_THREADS = 256;
__device__ __forceinline__ void invalidate_pages(const amass_invalidate_args& a, int r, int l,
                                                 int tid) {
    const int sl = a.seq_lens[r];
    if (sl <= 0) return;
    const int ql = a.query_start_loc[r + 1] - a.query_start_loc[r];
    const int ctx = sl - ql > 0 ? sl - ql : 0;
    const int p0 = ctx / a.page;
    const int p1 = min((sl - 1) / a.page, a.max_pages - 1);
    const int npg = p1 - p0 + 1;
    const int32_t* bt = a.block_table + (int64_t)r * a.bt_st;
    for (int i = tid; i < npg * a.n_kv; i += INV_THREADS) {
        const int p = p0 + i / a.n_kv, kv = i % a.n_kv;
        const int blk = bt[p];
        if (blk < 0 || blk >= a.nb) continue;
        const int64_t lk = (int64_t)l * a.n_kv + kv;
        const int64_t row = lk * a.nb + blk;
        a.pool_valid[row] = 0;
        const int slot = a.page2slot[row];
        if (slot >= 0 && slot < a.slots) {
            a.page2slot[row] = -1;
            a.slot2page[lk * a.slots + slot] = -1;
        }
    }
}

// grid (n_req, L)
__global__ __launch_bounds__(INV_THREADS) void invalidate_kernel(const amass_invalidate_args a) {
    invalidate_pages(a, blockIdx.x, blockIdx.y, threadIdx.x);
}

// ------------------------------------------------------------------ begin_step 1: mark
// grid (n_chunks, n_req): workgroup (c, r) counts the staged complete pages of chunk c of
// request r into mark[r][c]; chunk 0 also clears v_flushed of r's written pages.
__global__ __launch_bounds__(ST_CHUNK) void stage_mark_kernel(const amass_stage_args a,
                                                              int n_chunks) {
    __shared__ int red[ST_CHUNK / WAVE];
    const int c = blockIdx.x, r = blockIdx.y;
    const ReqRange q = req_range(a.seq_lens, a.query_start_loc, r, a.page);
    const int32_t* bt = a.block_table + (int64_t)r * a.bt_st;
    if (q.active && c == 0) {
        for (int p = q.p0 + (int)threadIdx.x; p <= q.p1 && p < a.max_pages; p += blockDim.x) {
            const int blk = bt[p];
            if (blk >= 0 && blk < a.nb) a.v_flushed[blk] = 0;
        }
    }
    const int np = q.active ? min(q.ctx / a.page, a.max_pages) : 0;
    const int p = c * ST_CHUNK + threadIdx.x;
    int cand = 0;
    if (p < np) {
        const int blk = bt[p];
        cand = (blk >= 0 && blk < a.nb && a.vbo[blk] >= 0) ? 1 : 0;
    }
    int tot;
    st_excl_scan(cand, red, tot);
    if (threadIdx.x == 0) a.mark[(int64_t)r * n_chunks + c] = tot;
}

// ------------------------------------------------------------------ begin_step 2: collect
// One workgroup.  Nonzero mark chunks in (request, chunk) order; per chunk one page per
// thread: new claims (not flushed) take flush-list slots while there is room, every
// staged page not left over is freed onto the stack.
__global__ __launch_bounds__(ST_THREADS) void stage_collect_kernel(const amass_stage_args a,
                                                                   int n_chunks) {
    __shared__ int red[ST_WAVES];
    __shared__ int list[ST_THREADS];
    __shared__ int s_fcnt, s_top;
    const int tid = threadIdx.x;
    if (tid == 0) {
        s_fcnt = 0;
        s_top = *a.free_top;
    }
    __syncthreads();
    const int T = a.n_req * n_chunks;
    for (int w0 = 0; w0 < T; w0 += ST_THREADS) {
        const int e = w0 + tid;
        const int nz = (e < T && a.mark[e] > 0) ? 1 : 0;
        int nlist;
        const int pos = st_excl_scan(nz, red, nlist);
        if (nz) list[pos] = e;
        __syncthreads();
        for (int k = 0; k < nlist; ++k) {
            const int ch = list[k];
            const int r = ch / n_chunks, c = ch % n_chunks;
            const ReqRange q = req_range(a.seq_lens, a.query_start_loc, r, a.page);
            const int np = q.active ? min(q.ctx / a.page, a.max_pages) : 0;
            const int p = c * ST_CHUNK + tid;
            int blk = -1, vb = -1;
            bool cand = false, fresh = false;
            if (tid < ST_CHUNK && p < np) {
                blk = a.block_table[(int64_t)r * a.bt_st + p];
                if (blk >= 0 && blk < a.nb) {
                    vb = a.vbo[blk];
                    cand = vb >= 0 && vb < a.nv;
                    fresh = cand && a.v_flushed[blk] == 0;
                }
            }
            const int fc = s_fcnt, top = s_top;
            int nfresh;
            const int rn = st_excl_scan(fresh ? 1 : 0, red, nfresh);
            const int i = fc + rn;
            const bool ok = fresh && i < a.maxf;
            const bool over = fresh && i >= a.maxf;
            const bool fr = cand && !over;
            int nfree;
            const int rf = st_excl_scan(fr ? 1 : 0, red, nfree);
            if (ok) {
                a.flush_list[2 * i] = blk;
                a.flush_list[2 * i + 1] = vb;
                a.v_flushed[blk] = 1;
            }
            if (fr) {
                a.vbo[blk] = -1;
                a.free_stack[top + rf] = vb;
            }
            __syncthreads();
            if (tid == 0) {
                s_fcnt = min(fc + nfresh, max(fc, a.maxf));
                s_top = top + nfree;
            }
            __syncthreads();
        }
    }
    if (tid == 0) {
        *a.flush_cnt = s_fcnt;
        *a.free_top = s_top;
    }
}

// The mark and collect of a batch of few table entries in one workgroup: thread t looks at
// entries K t .. K t + K of the (request, page) grid, the candidates (settled pages with a
// staging block) are compacted into LDS in that order, and each chunk of 1024 of them is
// claimed as above; a block shared by several requests counts at its first candidate
// (atomicMin on `first`, restored).  Workgroups past the first, if any, invalidate the written
// pages of four (request, layer) pairs each: the residency's maps, none of which the collect
// touches, so a step needs no launch of its own for them.
__global__ __launch_bounds__(ST_THREADS) void stage_collect_small_kernel(
        const amass_stage_args a, const amass_invalidate_args inv) {
    constexpr int KMAX = ST_SMALL / ST_THREADS;
    __shared__ int red[ST_WAVES];
    __shared__ int s_np[ST_REQS];                  // settled pages of each request
    __shared__ uint16_t list[ST_SMALL];            // candidates, as grid entries
    __shared__ int s_fcnt, s_top;
    const int tid = threadIdx.x;
    if (blockIdx.x > 0) {
        const int64_t x = (int64_t)(blockIdx.x - 1) * (ST_THREADS / INV_THREADS) + tid / INV_THREADS;
        if (x < (int64_t)inv.n_req * inv.n_layers)
            invalidate_pages(inv, (int)(x % inv.n_req), (int)(x / inv.n_req), tid % INV_THREADS);
        return;
    }
    if (tid == 0) {
        s_fcnt = 0;
        s_top = *a.free_top;
    }
    if (tid < a.n_req) {
        const ReqRange q = req_range(a.seq_lens, a.query_start_loc, tid, a.page);
        s_np[tid] = q.active ? min(q.ctx / a.page, a.max_pages) : 0;
    }
    // v_flushed = 0 for the written pages: half a wave per request
    for (int r = tid >> 5; r < a.n_req; r += ST_THREADS / 32) {
        const ReqRange q = req_range(a.seq_lens, a.query_start_loc, r, a.page);
        if (!q.active) continue;
        const int32_t* bt = a.block_table + (int64_t)r * a.bt_st;
        for (int p = q.p0 + (tid & 31); p <= q.p1 && p < a.max_pages; p += 32) {
            const int blk = bt[p];
            if (blk >= 0 && blk < a.nb) a.v_flushed[blk] = 0;
        }
    }
    __syncthreads();
    const int T = a.n_req * a.max_pages;           // <= ST_SMALL
    const int K = (T + ST_THREADS - 1) / ST_THREADS;
    const int e0 = tid * K;
    int blk[KMAX];
    {
        int r = e0 / a.max_pages, p = e0 - r * a.max_pages;
#pragma unroll
        for (int i = 0; i < KMAX; ++i) {
            blk[i] = -1;
            if (i < K && e0 + i < T) {
                if (p < s_np[r]) blk[i] = a.block_table[(int64_t)r * a.bt_st + p];
                if (++p == a.max_pages) {
                    p = 0;
                    ++r;
                }
            }
        }
    }
    uint32_t cand = 0;
#pragma unroll
    for (int i = 0; i < KMAX; ++i) {
        const int vb = blk[i] >= 0 && blk[i] < a.nb ? a.vbo[blk[i]] : -1;
        if (vb >= 0 && vb < a.nv) cand |= 1u << i;
    }
    int nlist;
    int pos = st_excl_scan(__popc(cand), red, nlist);
#pragma unroll
    for (int i = 0; i < KMAX; ++i)
        if (cand >> i & 1) list[pos++] = (uint16_t)(e0 + i);
    __syncthreads();
    for (int k0 = 0; k0 < nlist; k0 += ST_THREADS) {
        const int idx = k0 + tid;
        int b = -1, vb = -1;
        if (idx < nlist) {
            const int e = list[idx];
            const int r = e / a.max_pages;
            b = a.block_table[(int64_t)r * a.bt_st + (e - r * a.max_pages)];
            vb = a.vbo[b];                         // (-1 if an earlier chunk freed it)
        }
        const bool here = vb >= 0;
        if (here) atomicMin(&a.first[b], idx);
        __syncthreads();
        const bool lead = here && atomicAdd(&a.first[b], 0) == idx;
        const bool fresh = lead && a.v_flushed[b] == 0;
        const int fc = s_fcnt, top = s_top;
        const int room = max(a.maxf - fc, 0);
        // one scan of (fresh | already flushed << 16): fresh ones claim list entries while
        // there is room, those and the already flushed ones are freed
        int tot;
        const int pk = st_excl_scan((fresh ? 1 : 0) | (lead && !fresh ? 1 << 16 : 0), red, tot);
        const int nf = pk & 0xFFFF, no = pk >> 16;
        const int rf = no + min(nf, room);
        if (fresh && nf < room) {
            const int i = fc + nf;
            a.flush_list[2 * i] = b;
            a.flush_list[2 * i + 1] = vb;
            a.v_flushed[b] = 1;
        }
        if (lead && (!fresh || nf < room)) {
            a.vbo[b] = -1;
            a.free_stack[top + rf] = vb;
        }
        if (here) atomicExch(&a.first[b], 0x7FFFFFFF);     // scratch back at rest
        __syncthreads();
        if (tid == 0) {
            const int take = min(tot & 0xFFFF, room);
            s_fcnt = fc + take;
            s_top = top + (tot >> 16) + take;
        }
        __syncthreads();
    }
    if (tid == 0) {
        *a.flush_cnt = s_fcnt;
        *a.free_top = s_top;
    }
}

// ------------------------------------------------------------------ begin_step 3: copy
// List entry i of layer l: v_pool[l, vb] (page, n_kv, d) -> pinned pool [l, blk, kv]
// (page, d) for every kv head, 16-byte copies; then pool_valid = 1.
__device__ __forceinline__ void flush_copy(const amass_stage_args& a, int i, int l) {
    const int blk = a.flush_list[2 * i], vb = a.flush_list[2 * i + 1];
    const int cpr = a.d / 8;                           // 16-byte chunks per row
    const int total = a.n_kv * a.page * cpr;
    const uint16_t* src = (const uint16_t*)a.v_pool + (int64_t)l * a.vp_sl + (int64_t)vb * a.vp_sb;
    uint16_t* dst = (uint16_t*)a.pool + (((int64_t)l * a.nb + blk) * a.n_kv) * a.page * a.d;
    for (int x = threadIdx.x; x < total; x += blockDim.x) {
        const int ch = x % cpr, t = (x / cpr) % a.page, kv = x / (cpr * a.page);
        const uint4 v = *reinterpret_cast<const uint4*>(src + (int64_t)t * a.vp_st +
                                                        (int64_t)kv * a.vp_sh + 8 * ch);
        *reinterpret_cast<uint4*>(dst + ((int64_t)kv * a.page + t) * a.d + 8 * ch) = v;
    }
    for (int kv = threadIdx.x; kv < a.n_kv; kv += blockDim.x)
        a.pool_valid[((int64_t)l * a.n_kv + kv) * a.nb + blk] = 1;
}

// ------------------------------------------------------------------ begin_step 4: alloc
// One workgroup.  The written pages of all active requests, flattened in (request, page)
// order, in chunks of 1024: a page whose block has no staging block pops the stack;
// duplicates of a block inside a chunk defer to the first (atomicMin on `first`).
__device__ __forceinline__ void stage_alloc(const amass_stage_args& a, int* red, int* woff,
                                            int& s_top, int& s_ovf) {
    const int tid = threadIdx.x;
    if (tid == 0) {
        s_top = *a.free_top;
        s_ovf = 0;
    }
    __syncthreads();
    for (int rb = 0; rb < a.n_req; rb += ST_THREADS) {
        const int nr = min(ST_THREADS, a.n_req - rb);
        int nw = 0;
        if (tid < nr) {
            const ReqRange q = req_range(a.seq_lens, a.query_start_loc, rb + tid, a.page);
            if (q.active) nw = max(0, min(q.p1, a.max_pages - 1) - q.p0 + 1);
        }
        int tot;
        const int off = st_excl_scan(nw, red, tot);
        woff[tid] = off;
        __syncthreads();
        for (int e0 = 0; e0 < tot; e0 += ST_THREADS) {
            const int e = e0 + tid;
            int blk = -1;
            bool need = false;
            if (e < tot) {
                int lo = 0, hi = nr - 1;                 // last request with woff <= e
                while (lo < hi) {
                    const int mid = (lo + hi + 1) >> 1;
                    if (woff[mid] <= e) lo = mid;
                    else hi = mid - 1;
                }
                const int r = rb + lo;
                const ReqRange q = req_range(a.seq_lens, a.query_start_loc, r, a.page);
                blk = a.block_table[(int64_t)r * a.bt_st + q.p0 + (e - woff[lo])];
                need = blk >= 0 && blk < a.nb && a.vbo[blk] < 0;
            }
            // (a decode step seldom starts a page: no dedup round then)
            if (__syncthreads_or(need)) {
                if (need) atomicMin(&a.first[blk], e);
                __syncthreads();
                const bool lead = need && atomicAdd(&a.first[blk], 0) == e;
                int nlead;
                const int rk = st_excl_scan(lead ? 1 : 0, red, nlead);
                const int top = s_top;
                if (lead) {
                    if (rk < top) a.vbo[blk] = a.free_stack[top - 1 - rk];
                    else s_ovf = 1;
                }
                __syncthreads();
                if (need) atomicExch(&a.first[blk], 0x7FFFFFFF);   // scratch back at rest
                if (tid == 0) s_top = max(top - nlead, 0);
                __syncthreads();
            }
        }
    }
    if (tid == 0) {
        *a.free_top = s_top;
        if (s_ovf) *a.overflow = 1;
    }
}

// ------------------------------------------------------------------ begin_step 5: slots
// v_slot of token t; qsl = query_start_loc (global, or its copy in LDS)
__device__ __forceinline__ int64_t token_slot(const amass_stage_args& a, const int32_t* qsl,
                                              int t) {
    if (a.n_req <= 0 || t < qsl[0] || t >= qsl[a.n_req]) return -1;
    int lo = 0, hi = a.n_req - 1;                      // last request with qsl <= t
    while (lo < hi) {
        const int mid = (lo + hi + 1) >> 1;
        if (qsl[mid] <= t) lo = mid;
        else hi = mid - 1;
    }
    const ReqRange q = req_range(a.seq_lens, qsl, lo, a.page);
    if (!q.active) return -1;
    const int pos = q.ctx + (t - qsl[lo]);
    const int p = pos / a.page;
    if (p >= a.max_pages) return -1;
    const int blk = a.block_table[(int64_t)lo * a.bt_st + p];
    if (blk < 0 || blk >= a.nb) return -1;
    const int vb = a.vbo[blk];
    return vb >= 0 ? (int64_t)vb * a.page + pos % a.page : -1;
}

__global__ __launch_bounds__(256) void stage_vslot_kernel(const amass_stage_args a) {
    const int t = blockIdx.x * blockDim.x + threadIdx.x;
    if (t < a.n_tokens) a.v_slot[t] = token_slot(a, a.query_start_loc, t);
}

// Steps 3-5 in one launch: workgroup 0 allocates and, with `slots`, maps the tokens (their
// offsets in LDS); the others copy the flushed pages, (entry, layer) by (entry, layer).
__global__ __launch_bounds__(ST_THREADS) void stage_place_kernel(const amass_stage_args a,
                                                                 int slots) {
    __shared__ int red[ST_WAVES];
    __shared__ int woff[ST_THREADS];
    __shared__ int32_t s_qsl[ST_THREADS + 1];
    __shared__ int s_top, s_ovf;
    if (blockIdx.x > 0) {
        const int cnt = *a.flush_cnt;
        for (int64_t x = blockIdx.x - 1; x < (int64_t)cnt * a.n_layers; x += gridDim.x - 1)
            flush_copy(a, (int)(x % cnt), (int)(x / cnt));
        return;
    }
    if (slots)
        for (int i = threadIdx.x; i <= a.n_req; i += ST_THREADS) s_qsl[i] = a.query_start_loc[i];
    stage_alloc(a, red, woff, s_top, s_ovf);
    if (!slots) return;
    __syncthreads();
    for (int t = threadIdx.x; t < a.n_tokens; t += ST_THREADS) a.v_slot[t] = token_slot(a, s_qsl, t);
}

// ------------------------------------------------------------------ scatter
// grid (n_tokens): token t's n_kv x d V row -> its staging slot
__global__ __launch_bounds__(128) void stage_scatter_kernel(const amass_scatter_args a) {
    const int t = blockIdx.x;
    const int64_t vs = a.v_slot[t];
    if (vs < 0) return;
    const int64_t vb = vs / a.page;
    const int off = (int)(vs % a.page);
    if (vb >= a.nv) return;
    const int cpr = a.d / 8;
    const uint16_t* src = (const uint16_t*)a.value + (int64_t)t * a.v_st;
    uint16_t* dst = (uint16_t*)a.v_pool + vb * a.vp_sb + (int64_t)off * a.vp_st;
    for (int x = threadIdx.x; x < a.n_kv * cpr; x += blockDim.x) {
        const int kv = x / cpr, ch = x % cpr;
        *reinterpret_cast<uint4*>(dst + (int64_t)kv * a.vp_sh + 8 * ch) =
            *reinterpret_cast<const uint4*>(src + (int64_t)kv * a.v_sh + 8 * ch);
    }
}

static bool al16(const void* p, int64_t elems) {
    return (((uintptr_t)p) & 15) == 0 && (elems % 8) == 0;
}

static int check_invalidate(const amass_invalidate_args* a) {
    if (!a) return AMASS_ERR_NULL;
    if (!a->block_table || !a->seq_lens || !a->query_start_loc || !a->page2slot ||
        !a->slot2page || !a->pool_valid)
        return AMASS_ERR_NULL;
    if (a->n_req < 0 || a->n_layers < 1 || a->nb < 1 || a->n_kv < 1 || a->slots < 1 ||
        a->page < 1 || a->max_pages < 1)
        return AMASS_ERR_GEOMETRY;
    return AMASS_OK;
}

static int launch_invalidate(const amass_invalidate_args& a, hipStream_t s) {
    if (a.n_req == 0) return AMASS_OK;
    hipLaunchKernelGGL(invalidate_kernel, dim3(a.n_req, a.n_layers), dim3(INV_THREADS), 0, s, a);
    return check_launch();
}

// inv: the invalidation of the same step's written pages, or null
static int begin_step(const amass_invalidate_args* inv, const amass_stage_args* a,
                      hipStream_t s) {
    if (!a) return AMASS_ERR_NULL;
    if (!a->block_table || !a->seq_lens || !a->query_start_loc || !a->vbo || !a->v_flushed ||
        !a->free_stack || !a->free_top || !a->v_slot || !a->flush_list || !a->flush_cnt ||
        !a->overflow || !a->mark || !a->first || !a->v_pool || !a->pool || !a->pool_valid)
        return AMASS_ERR_NULL;
    if (a->n_req < 0 || a->n_tokens < 0 || a->max_pages < 1 || a->n_layers < 1 || a->nb < 1 ||
        a->nv < 1 || a->n_kv < 1 || a->page < 1 || a->maxf < 1 || a->d < 8 || a->d % 8)
        return AMASS_ERR_GEOMETRY;
    if (!al16(a->v_pool, a->vp_sl) || a->vp_sb % 8 || a->vp_st % 8 || a->vp_sh % 8 ||
        !al16(a->pool, a->d))
        return AMASS_ERR_GEOMETRY;
    const int n_chunks = (a->max_pages + ST_CHUNK - 1) / ST_CHUNK;
    int rc;
    if (a->n_req <= ST_REQS && (int64_t)a->n_req * a->max_pages <= ST_SMALL) {
        constexpr int per = ST_THREADS / INV_THREADS;
        const int64_t pairs = inv ? (int64_t)inv->n_req * inv->n_layers : 0;
        const amass_invalidate_args none = {};
        hipLaunchKernelGGL(stage_collect_small_kernel, dim3(1 + (uint32_t)((pairs + per - 1) / per)),
                           dim3(ST_THREADS), 0, s, *a, inv ? *inv : none);
    } else {
        if (inv && (rc = launch_invalidate(*inv, s))) return rc;
        hipLaunchKernelGGL(stage_mark_kernel, dim3(n_chunks, a->n_req), dim3(ST_CHUNK), 0, s,
                           *a, n_chunks);
        if ((rc = check_launch())) return rc;
        hipLaunchKernelGGL(stage_collect_kernel, dim3(1), dim3(ST_THREADS), 0, s, *a, n_chunks);
    }
    if ((rc = check_launch())) return rc;
    const int slots = a->n_req <= ST_THREADS && a->n_tokens <= ST_TOKENS;
    const int64_t copies = (int64_t)a->maxf * a->n_layers;
    hipLaunchKernelGGL(stage_place_kernel, dim3(1 + (int)(copies < 255 ? copies : 255)),
                       dim3(ST_THREADS), 0, s, *a, slots);
    if ((rc = check_launch())) return rc;
    if (!slots && a->n_tokens > 0) {
        hipLaunchKernelGGL(stage_vslot_kernel, dim3((a->n_tokens + 255) / 256), dim3(256), 0,
                           s, *a);
        rc = check_launch();
    }
    return rc;
}

}  // namespace amass

using namespace amass;

extern "C" int amass_tier_invalidate(const amass_invalidate_args* a, void* stream) {
    const int rc = check_invalidate(a);
    return rc ? rc : launch_invalidate(*a, (hipStream_t)stream);
}

extern "C" int amass_stage_begin_step(const amass_stage_args* a, void* stream) {
    return begin_step(nullptr, a, (hipStream_t)stream);
}

// amass_tier_invalidate and amass_stage_begin_step of one step (a helper of the Python
// binding, not part of the C-ABI): batches of few table entries invalidate in the collect's
// launch.
extern "C" int amass_binding_begin_step(const amass_invalidate_args* inv,
                                        const amass_stage_args* a, void* stream) {
    const int rc = check_invalidate(inv);
    return rc ? rc : begin_step(inv, a, (hipStream_t)stream);
}

extern "C" int amass_stage_scatter(const amass_scatter_args* a, void* stream) {
    if (!a) return AMASS_ERR_NULL;
    if (!a->value || !a->v_slot || !a->v_pool) return AMASS_ERR_NULL;
    if (a->n_tokens < 0 || a->n_kv < 1 || a->d < 8 || a->d % 8 || a->page < 1 || a->nv < 1)
        return AMASS_ERR_GEOMETRY;
    if (!al16(a->value, a->v_st) || a->v_sh % 8 || !al16(a->v_pool, a->vp_sb) ||
        a->vp_st % 8 || a->vp_sh % 8)
        return AMASS_ERR_GEOMETRY;
    if (a->n_tokens == 0) return AMASS_OK;
    hipLaunchKernelGGL(stage_scatter_kernel, dim3(a->n_tokens), dim3(128), 0,
                       (hipStream_t)stream, *a);
    return check_launch();
}
