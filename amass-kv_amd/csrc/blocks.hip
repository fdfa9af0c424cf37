// Block lists of the summary builder for gfx950: the distinct physical blocks of a batch's
// finalised pages, and each request's last finalised page.
//
// Both are a few KB, so their cost is launches and dependent rounds, on the host above all:
// as tensor operations the first took ten launches and the second seven, at ~5 us of host
// time each beside a 31-us build.  Here the first is a mark launch over the table, a compaction
// in ascending block order and one 12-byte copy, the second one launch without a sync: a bulk
// build of 8 x 16K tokens with its first score 278 -> 237 us, the 32-layer tail rebuild of 32
// requests, all of them, with a score 68 -> 42 (now the kernels' own time).  A tail of named
// rows takes the tensor operations.
//
// A helper of the Python binding, not part of the C-ABI in include/amass_hip.h.
#include "common.h"

namespace amass {

struct BlockListArgs {
    const int32_t* block_table;     // (n_req, max_pages), unit column stride
    int64_t bt_st;
    const int32_t* seq_lens;        // (n_req,)
    uint8_t* mark;                  // nb bytes padded to 16, zero; null: tail blocks
    int32_t* info;                  // three, zero: {longest row, bad block, count}
    int64_t* blocks;                // min(nb, n_req max_pages) entries; tail blocks: n_req
    int32_t n_req, max_pages, nb, page;
};

constexpr int BL_COLS = 256;       // table columns per mark workgroup
constexpr int BL_THREADS = 1024;   // compaction workgroup
constexpr int BL_CHUNK = 4 * BL_THREADS;
constexpr int BL_MAX = 1 << 22;    // blocks: the compaction's counting is quadratic in them

// grid (column chunk, request): mark[blk] = 1 for every finalised page; info[0] the longest
// row's pages, info[1] != 0 if a page's block is not in [0, nb).
__global__ __launch_bounds__(BL_COLS) void block_mark_kernel(const BlockListArgs a) {
    const int r = blockIdx.y, p = blockIdx.x * BL_COLS + threadIdx.x;
    const int nfin = a.seq_lens[r] / a.page;
    if (p == 0) atomicMax(&a.info[0], nfin);
    if (p < nfin && p < a.max_pages) {
        const int blk = a.block_table[(int64_t)r * a.bt_st + p];
        if (blk >= 0 && blk < a.nb) a.mark[blk] = 1;
        else a.info[1] = 1;
    }
}

// grid (chunks of BL_CHUNK marks): workgroup c writes its chunk's marked blocks behind those of
// the chunks before it, which it counts itself (16-byte loads of up to nb marks, from the L2
// in the main, instead of a pass of its own or a wait for its neighbours); the last one's end is the
// number of blocks, info[2].  mark is padded to whole 16 bytes.  One workgroup for the whole
// pool was bound by its stores: all blocks marked, with the mark launch, 8208 blocks 8.4 -> 7.1
// us, 32768 21.8 -> 7.7, 262144 156.5 -> 11.5.
__global__ __launch_bounds__(BL_THREADS) void block_compact_kernel(const BlockListArgs a) {
    __shared__ int red[BL_THREADS / WAVE], red2[BL_THREADS / WAVE];
    const int tid = threadIdx.x, lane = tid & 63, w = tid >> 6;
    const int c0 = blockIdx.x * BL_CHUNK;
    const int id0 = c0 + 4 * tid;
    const uint32_t m = id0 < a.nb ? *reinterpret_cast<const uint32_t*>(a.mark + id0) : 0u;
    int pre = 0;
    for (int i = 16 * tid; i < c0; i += 16 * BL_THREADS) {
        const uint4 v = *reinterpret_cast<const uint4*>(a.mark + i);
        pre += __popc(v.x) + __popc(v.y) + __popc(v.z) + __popc(v.w);     // bytes 0 | 1
    }
    const int cnt = __popc(m);
    const int incl = wave_incl_scan(cnt), psum = wave_incl_scan(pre);
    if (lane == 63) {
        red[w] = incl;
        red2[w] = psum;
    }
    __syncthreads();
    int at = incl - cnt, end = 0;
#pragma unroll
    for (int x = 0; x < BL_THREADS / WAVE; ++x) {
        at += red2[x] + (x < w ? red[x] : 0);
        end += red2[x] + red[x];
    }
#pragma unroll
    for (int b = 0; b < 4; ++b)
        if (m >> (8 * b) & 1u) a.blocks[at++] = id0 + b;
    if (blockIdx.x == gridDim.x - 1 && tid == 0) a.info[2] = end;
}

// blocks[r]: the block of request r's last finalised page (its first page if it has none), -1
// (which the builder skips) for a row longer than the table
__global__ __launch_bounds__(256) void block_tail_kernel(const BlockListArgs a) {
    const int r = blockIdx.x * blockDim.x + threadIdx.x;
    if (r >= a.n_req) return;
    const int p = max(a.seq_lens[r] / a.page - 1, 0);
    a.blocks[r] = p < a.max_pages ? a.block_table[(int64_t)r * a.bt_st + p] : -1;
}

}  // namespace amass

using namespace amass;

// mark != null: the distinct blocks of every finalised page (page p of request r with p <
// seq_lens[r] / page) in ascending order, and info; null: blocks[r] = the block of request r's
// last finalised page (-1 for a row longer than the table).
extern "C" int amass_binding_block_list(const int32_t* block_table, int64_t bt_st,
                                        const int32_t* seq_lens, uint8_t* mark, int32_t* info,
                                        int64_t* blocks, int32_t n_req, int32_t max_pages,
                                        int32_t nb, int32_t page, void* stream) {
    if (!block_table || !seq_lens || !blocks || (mark && !info)) return AMASS_ERR_NULL;
    if (n_req < 0 || n_req > 65535 || max_pages < 1 || nb < 1 || nb > BL_MAX || page < 1)
        return AMASS_ERR_GEOMETRY;
    if (((uintptr_t)mark & 15) != 0) return AMASS_ERR_GEOMETRY;
    if (n_req == 0) return AMASS_OK;
    const BlockListArgs a = {block_table, bt_st, seq_lens, mark,      info,
                             blocks,      n_req, max_pages, nb,       page};
    hipStream_t s = (hipStream_t)stream;
    if (!mark) {
        hipLaunchKernelGGL(block_tail_kernel, dim3((n_req + 255) / 256), dim3(256), 0, s, a);
        return check_launch();
    }
    hipLaunchKernelGGL(block_mark_kernel, dim3((max_pages + BL_COLS - 1) / BL_COLS, n_req),
                       dim3(BL_COLS), 0, s, a);
    const int rc = check_launch();
    if (rc) return rc;
    hipLaunchKernelGGL(block_compact_kernel, dim3((nb - 1) / BL_CHUNK + 1), dim3(BL_THREADS), 0, s,
                       a);
    return check_launch();
}
