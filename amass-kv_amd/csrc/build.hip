// Page-summary builder for gfx950: the quad and r8 summaries of finalised K pages.
//
// Math per (block, kv-head) of a 16-token page (reference selection/quad_build.py:1-25,
// 124-198 and selection/build.py:297-348,396-412):
//   mu  = mean_t K[t]                       dc = K - mu            (16, d) fp32
//   Gm  = dc dc^T (16 x 16)                 S2, U = eigh(Gm), eigenvalues ascending
//   S2r = clamp(top-r eigenvalues, 1e-10)   U8 = their eigenvectors, S8 = sqrt(S2r)
//   Vk  = dc^T U8 / S8 (d, r)               c = U8 * S8 (16, r)    (r8 only)
//   quant: lvl = 127 | 7, s = max(amax / lvl, 1e-8) fp32, code = clamp(rint(x / s), +-lvl)
//          (V and c: rint(x (1 / s)), which |x| <= lvl s keeps in range; a code may differ
//          where x / s lies within 1e-7 of a half), stored scale fp16(s); mu per (block, head), Vk per column ("col") or per
//          (block, head) ("tensor"), c per token ("page") or per (block, head) ("tensor")
//   quad stores sig2 = fp16(S2r); r8 stores c; both the content tag K[15][:TAGW].
// Output goes straight into the packed records the score kernels read
// (AMASS_QUAD_REC_BYTES / AMASS_R8_REC_BYTES / AMASS_CLSE_REC_BYTES).
//
// One wave summarises four (block, kv-head) items of one layer; a DPP row of 16 lanes owns
// one item in the eigen step.  Phases:
//   1  per item: the K page in 16-byte loads (lane (g, n): tokens 4g + u, channels 8n ..
//      + 8, whole 256-byte rows), mu over registers and the two lane-row swaps, dc through
//      LDS into token-major order, and the Gram on 32 v_mfma_f32_16x16x4f32 whose A and B
//      operands are the same register (any split of d over the K steps gives the same sum)
//   2  the four Grams through LDS into one column per lane; the top-r eigenpairs of all
//      four at once (eigh16.h)
//   3  Vk = dc^T U8 / S8 (the items' K re-read, 4 KB each from a near cache): for r > 4 on the
//      matrix cores, two items per accumulator set (A = the items' scaled eigenvectors in
//      their own 8 rows, zero elsewhere, B = dc as phase 1 loaded it); for r <= 4 as plain
//      products of each lane's four tokens, summed over the lane rows by two swap steps that
//      leave item p in row p.  Then scales and codes in registers, 8 code bytes per store
//   4  mu codes, c rows, scale blocks, tags: row p serves item p
// Bound by instruction issue (~6 thousand per four items; an f32 matrix instruction holds the
// SIMD for its 8 passes, which is why few columns are cheaper as plain products: CLSE r' = 2
// 174 -> 154 us with them).  Back to back, 65 536 items (8192 blocks of 8 heads): quad r = 8
// int8 197 us (347 MB moved, 1.8 TB/s), r8 r = 8 200, CLSE r' = 2 int4 155; 262 144 items 748 us;
// one layer's tail of 256 items 20.6 us, the latency of one wave.  The one-item-per-wave
// round-robin Jacobi in LDS before it: 1645 us, 6.4 ms, 76 us.  Three waves per SIMD (157-160
// VGPRs, none spilled); four spill (207 us), two took 247 us on an earlier build that ran 202
// with three.
#include "common.h"
#include "eigh16.h"

namespace amass {

constexpr int BP = 16;           // tokens per page
constexpr int BD = 128;          // head dim
constexpr int BI = 4;            // items per wave
constexpr int BMS = BP + 4;      // padded fp32 column of a 16 x 16 matrix

// 10 KB per wave: sixteen waves per CU.
struct BuildLds {
    union {
        // phase 1: dc of one item, token-major; 16-byte chunk c of row t at c ^ t (the 16
        // tokens' reads of one chunk index then spread over the banks)
        float4 t[BP][BD / 4];
        float hv[14][WAVE];                // phase 2: the reflections
        struct {
            float m[BI][BP][BMS];          // phases 2-4: column n of item p's Gram, then
                                           // eigenvector k (m[p][k][token])
            float vsc[BI][8], s2[BI][8];   // V scales and clamped eigenvalues
            float meta[BI][32];            // scale block halves before their rounding
        };
    };
    float mu[BI][BD];
};
static_assert(sizeof(BuildLds) <= 10240, "sixteen waves per CU");

__device__ __forceinline__ float quant_scale(float amax, float lvl) {
    return fmaxf(__fdiv_rn(amax, lvl), 1e-8f);
}
__device__ __forceinline__ int quant_code(float x, float s, float lvl) {
    return (int)fminf(fmaxf(rintf(__fdiv_rn(x, s)), -lvl), lvl);
}
__device__ __forceinline__ uint16_t f2h_bits(float f) {
    return __half_as_ushort(__float2half_rn(f));
}
// The code of x as the low byte of the result: |x| <= lvl / inv, so rounding x * inv to an
// integer in the mantissa of 1.5 * 2^23 is the rint and the conversion in one instruction.
__device__ __forceinline__ uint32_t code_byte(float x, float inv) {
    return __float_as_uint(__builtin_fmaf(x, inv, 12582912.f));
}
__device__ __forceinline__ uint32_t pack4(uint32_t a, uint32_t b, uint32_t c, uint32_t d) {
    return perm(perm(d, c, 0x0C0C0400u), perm(b, a, 0x0C0C0400u), 0x05040100u);
}

// dc of one item in the phase-1 layout: x[u][e] = K[4g + u][8n + e] - mu[8n + e]
typedef uint32_t u32x4_t __attribute__((ext_vector_type(4)));
typedef const __attribute__((address_space(1))) uint16_t* gk_ptr;    // K is in global memory
struct Raw {
    u32x4_t q[4];
};
__device__ __forceinline__ void load_item(gk_ptr kp, int64_t k_st, int g, int n, Raw& w) {
#pragma unroll
    for (int u = 0; u < 4; ++u)
        w.q[u] = *(const __attribute__((address_space(1))) u32x4_t*)(
            kp + (int64_t)(4 * g + u) * k_st + 8 * n);
}
__device__ __forceinline__ void unpack_item(const Raw& w, float (&x)[4][8]) {
#pragma unroll
    for (int u = 0; u < 4; ++u) {
#pragma unroll
        for (int j = 0; j < 4; ++j) {
            x[u][2 * j] = bf16lo(w.q[u][j]);
            x[u][2 * j + 1] = bf16hi(w.q[u][j]);
        }
    }
}

__device__ __forceinline__ void centre_item(const Raw& w, const float* mu, int n, float (&x)[4][8]) {
    unpack_item(w, x);
    const float4 m0 = *reinterpret_cast<const float4*>(mu + 8 * n);
    const float4 m1 = *reinterpret_cast<const float4*>(mu + 8 * n + 4);
    const float m[8] = {m0.x, m0.y, m0.z, m0.w, m1.x, m1.y, m1.z, m1.w};
#pragma unroll
    for (int u = 0; u < 4; ++u)
#pragma unroll
        for (int e = 0; e < 8; ++e) x[u][e] -= m[e];
}
// v[k][e]: the part of tokens 4g .. 4g + 3 in column k, channel 8n + e of item p's Vk
template <int NK>
__device__ __forceinline__ void item_columns(const Raw& w, const BuildLds& L, int p, int g, int n,
                                             int r, float (&v)[NK][8]) {
    float x[4][8];
    centre_item(w, L.mu[p], n, x);
#pragma unroll
    for (int k = 0; k < NK; ++k) {
        const float is8 = k < r ? __builtin_amdgcn_rsqf(L.s2[p][k]) : 0.f;
        const float4 uv = *reinterpret_cast<const float4*>(&L.m[p][k][4 * g]);
        const float us[4] = {uv.x * is8, uv.y * is8, uv.z * is8, uv.w * is8};
#pragma unroll
        for (int e = 0; e < 8; ++e)
            v[k][e] = __builtin_fmaf(us[3], x[3][e], __builtin_fmaf(us[2], x[2][e],
                      __builtin_fmaf(us[1], x[1][e], us[0] * x[0][e])));
    }
}

// KIND 0: quad record; 1: r8 record; 2: CLSE (quad_V / mu, c rows and the residual energy).
// RP: the power of two at or above the rank.
template <int KIND, int RP>
__global__ __launch_bounds__(WAVE, 3) void summary_build_kernel(const amass_build_args a,
                                                             int64_t items) {
    constexpr bool COORD = KIND >= 1;
    constexpr bool CLSE = KIND == 2;
    constexpr int RW = RP == 8 ? 8 : 4;          // accumulator rows per item
    constexpr int PG = 16 / RW;                  // items per accumulator set
    constexpr int NJ = RP < 4 ? RP : 4;          // accumulator registers in use per tile
    __shared__ BuildLds L;
    const int lane = threadIdx.x;
    const int g = lane >> 4, n = lane & 15;
    const int layer = blockIdx.z;
    const int r = a.rank;
    const gk_ptr kbase = (gk_ptr)(a.k_layers ? a.k_layers[layer] : (uint64_t)a.k);
    // items past the end repeat the last one and those of a negative block read block 0;
    // only the items in `ok` are stored
    const int64_t i0 = (int64_t)blockIdx.x * BI;
    const int live = (int)(items - i0 < BI ? items - i0 : BI);
    int64_t blk[BI];
    int head[BI];
    gk_ptr kp[BI];
    uint32_t ok = 0;
    {
        int64_t bi = i0 / a.n_kv;
        int h = (int)(i0 - bi * a.n_kv);
#pragma unroll
        for (int p = 0; p < BI; ++p) {
            const int64_t b = a.blocks[bi];
            if (b >= 0 && p < live) ok |= 1u << p;
            blk[p] = b >= 0 ? b : 0;
            head[p] = h;
            kp[p] = kbase + blk[p] * a.k_sb + (int64_t)h * a.k_sh;
            if (p + 1 < live && ++h == a.n_kv) {
                h = 0;
                ++bi;
            }
        }
    }

    // ---- 1: mu, dc, Gram -----------------------------------------------------------------
    f32x4_t gram[BI];
    Raw raw[BI];
#pragma unroll
    for (int p = 0; p < BI; ++p) load_item(kp[p], a.k_st, g, n, raw[p]);
#pragma unroll
    for (int p = 0; p < BI; ++p) {
        float x[4][8];
        unpack_item(raw[p], x);
        float mu[8];
#pragma unroll
        for (int e = 0; e < 8; ++e) {
            const float s = (x[0][e] + x[1][e]) + (x[2][e] + x[3][e]);
            mu[e] = xor32_sumf(xor16_sumf(s)) * (1.0f / BP);
        }
        if (g == 0) {
            *reinterpret_cast<float4*>(&L.mu[p][8 * n]) = make_float4(mu[0], mu[1], mu[2], mu[3]);
            *reinterpret_cast<float4*>(&L.mu[p][8 * n + 4]) = make_float4(mu[4], mu[5], mu[6], mu[7]);
        }
#pragma unroll
        for (int u = 0; u < 4; ++u) {
            const int t = 4 * g + u;
            L.t[t][(2 * n) ^ t] =
                make_float4(x[u][0] - mu[0], x[u][1] - mu[1], x[u][2] - mu[2], x[u][3] - mu[3]);
            L.t[t][(2 * n + 1) ^ t] =
                make_float4(x[u][4] - mu[4], x[u][5] - mu[5], x[u][6] - mu[6], x[u][7] - mu[7]);
        }
        __syncthreads();
        float4 y[8];
#pragma unroll
        for (int i = 0; i < 8; ++i) y[i] = L.t[n][(8 * g + i) ^ n];
        __syncthreads();
        f32x4_t acc = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
        for (int i = 0; i < 8; ++i) {
            acc = __builtin_amdgcn_mfma_f32_16x16x4f32(y[i].x, y[i].x, acc, 0, 0, 0);
            acc = __builtin_amdgcn_mfma_f32_16x16x4f32(y[i].y, y[i].y, acc, 0, 0, 0);
            acc = __builtin_amdgcn_mfma_f32_16x16x4f32(y[i].z, y[i].z, acc, 0, 0, 0);
            acc = __builtin_amdgcn_mfma_f32_16x16x4f32(y[i].w, y[i].w, acc, 0, 0, 0);
        }
        gram[p] = acc;                           // rows 4g + j, column n
    }

    // ---- 2: eigenpairs -----------------------------------------------------------------------
#pragma unroll
    for (int p = 0; p < BI; ++p)
        *reinterpret_cast<f32x4_t*>(&L.m[p][n][4 * g]) = gram[p];
    __syncthreads();
    float trace = 0.f;
    {
        float am[16], x[16], lam;
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            const float4 v = *reinterpret_cast<const float4*>(&L.m[g][n][4 * i]);
            am[4 * i] = v.x; am[4 * i + 1] = v.y; am[4 * i + 2] = v.z; am[4 * i + 3] = v.w;
        }
        static_for<0, 16>([&](auto I) {
            constexpr int i = I;
            trace += row_bcast<i>(am[i]);
        });
        __syncthreads();
        eigh16_top<RP>(am, r, trace, lam, x, L.hv);
        __syncthreads();
        // eigenvector k of item g: m[g][k][token] (lanes past the rank hold copies)
#pragma unroll
        for (int i = 0; i < 4; ++i)
            *reinterpret_cast<float4*>(&L.m[g][n][4 * i]) =
                make_float4(x[4 * i], x[4 * i + 1], x[4 * i + 2], x[4 * i + 3]);
        if (n < 8) L.s2[g][n] = n < r ? fmaxf(lam, 1e-10f) : 0.f;
        L.meta[g][n] = 0.f;
        L.meta[g][n + 16] = 0.f;
    }
#pragma unroll
    for (int p = 0; p < BI; ++p) load_item(kp[p], a.k_st, g, n, raw[p]);
    __syncthreads();

    // ---- record addressing ---------------------------------------------------------------
    // quad / r8: head h's record [V | mu (| c rows)] at h VM, its scale block (quad 48,
    // r8 64 bytes) at n_kv VM + TB h.  CLSE: [V | mu] at h VM, its tail of TB bytes
    // [c rows | scale part] at n_kv VM + TB h (AMASS_CLSE_REC_BYTES).
    const int CB = a.v_bits == 8 ? BD : BD / 2;
    const int crow = COORD ? r * a.c_bits / 8 : 0;
    const int VM = r * CB + BD + (CLSE ? 0 : 16 * crow);
    const int TB = CLSE ? 16 * crow + 16 * ((36 + 2 * r + 15) / 16) : (COORD ? 64 : 48);
    int8_t* lrec = a.rec + layer * a.rec_lsb;
    const float vlvl = a.v_bits == 8 ? 127.f : 7.f;

    // ---- 3: Vk = dc^T U8 / S8, per-column (or per-head) int8 / int4 ----------------------
#pragma unroll
    for (int set = 0; set < BI / PG; ++set) {
        f32x4_t acc[8];
        if constexpr (RP == 8) {
#pragma unroll
            for (int e = 0; e < 8; ++e) acc[e] = f32x4_t{0.f, 0.f, 0.f, 0.f};
#pragma unroll
            for (int q = 0; q < PG; ++q) {
                const int p = set * PG + q;
                // (a key that is not finite, or overflows the Gram: 0 * NaN would reach the
                // other item's rows, so this item's products stay out and its codes are zero)
                const float tr = __int_as_float(
                    __builtin_amdgcn_readlane(__float_as_int(trace), 16 * p));
                if (!(tr < EIGH16_MAX_TRACE)) continue;
                float x[4][8];
                centre_item(raw[p], L.mu[p], n, x);
                // A rows RW q .. + RW: column k = n mod RW of U8 / S8, tokens 4g ..; others 0
                const int k = n & (RW - 1);
                const bool mine = n / RW == q && k < r;
                const float is8 = mine ? __builtin_amdgcn_rsqf(L.s2[p][k & 7]) : 0.f;
                const float4 uv = *reinterpret_cast<const float4*>(&L.m[p][k][4 * g]);
                const float us[4] = {mine ? uv.x * is8 : 0.f, mine ? uv.y * is8 : 0.f,
                                     mine ? uv.z * is8 : 0.f, mine ? uv.w * is8 : 0.f};
#pragma unroll
                for (int u = 0; u < 4; ++u)
#pragma unroll
                    for (int e = 0; e < 8; ++e)
                        acc[e] = __builtin_amdgcn_mfma_f32_16x16x4f32(us[u], x[u][e], acc[e],
                                                                      0, 0, 0);
            }
        } else {
            // few columns: products of the lane's four tokens, then the four lane rows' sums,
            // item p's into row p (two swap steps, each halving the registers)
            float even[NJ][8], odd[NJ][8];             // items (0 | 2) and (1 | 3)
#pragma unroll
            for (int h = 0; h < 2; ++h) {
                float lo[NJ][8], hi[NJ][8];
                item_columns<NJ>(raw[h], L, h, g, n, r, lo);
                item_columns<NJ>(raw[h + 2], L, h + 2, g, n, r, hi);
#pragma unroll
                for (int k = 0; k < NJ; ++k)
#pragma unroll
                    for (int e = 0; e < 8; ++e) {
                        const auto w = __builtin_amdgcn_permlane32_swap(
                            __float_as_uint(lo[k][e]), __float_as_uint(hi[k][e]), false, false);
                        (h ? odd : even)[k][e] = __uint_as_float(w[0]) + __uint_as_float(w[1]);
                    }
            }
#pragma unroll
            for (int k = 0; k < NJ; ++k)
#pragma unroll
                for (int e = 0; e < 8; ++e) {
                    const auto w = __builtin_amdgcn_permlane16_swap(
                        __float_as_uint(even[k][e]), __float_as_uint(odd[k][e]), false, false);
                    acc[e][k] = __uint_as_float(w[0]) + __uint_as_float(w[1]);
                }
        }
        // lane (g, n): item pi, columns k0 + j, channels 8n + e
        const int pi = RW == 8 ? set * PG + (g >> 1) : g;
        const int k0 = RW == 8 ? 4 * (g & 1) : 0;
        float sc[NJ];
        float all = 0.f;
#pragma unroll
        for (int j = 0; j < NJ; ++j) {
            float m = 0.f;
#pragma unroll
            for (int e = 0; e < 8; ++e) m = fmaxf(m, fabsf(acc[e][j]));
            sc[j] = row16_maxf(m);
            all = fmaxf(all, sc[j]);
        }
        if (a.v_grain == 1) {                    // one scale per (block, head)
            if constexpr (RW == 8) all = xor16_maxf(all);
#pragma unroll
            for (int j = 0; j < NJ; ++j) sc[j] = all;
        }
        // (the columns of an item are rank wide: this lane's item and its record)
        int64_t bo = blk[0];
        int ho = head[0];
#pragma unroll
        for (int p = 1; p < BI; ++p) {
            bo = pi == p ? blk[p] : bo;
            ho = pi == p ? head[p] : ho;
        }
        int8_t* rec = lrec + bo * a.rec_sb + (int64_t)ho * VM;
#pragma unroll
        for (int j = 0; j < NJ; ++j) {
            const int k = k0 + j;
            sc[j] = quant_scale(sc[j], vlvl);
            if (n == 0) L.vsc[pi][k] = sc[j];
            const float inv = __fdiv_rn(1.f, sc[j]);
            uint32_t w0 = pack4(code_byte(acc[0][j], inv), code_byte(acc[1][j], inv),
                                code_byte(acc[2][j], inv), code_byte(acc[3][j], inv));
            uint32_t w1 = pack4(code_byte(acc[4][j], inv), code_byte(acc[5][j], inv),
                                code_byte(acc[6][j], inv), code_byte(acc[7][j], inv));
            // the tiled layout of the score kernels' column groups: 16 bytes per (K-step t,
            // d group kg, column k) at ((t * 4 + kg) * r + k) * 16, t * 4 + kg = n / 2 here
            // (int4: t folded into the nibbles, channels d and d + 64 in lanes n and n + 8)
            bool st = (ok >> pi & 1) && k < r;
            if (a.v_bits == 4) {
                w0 = (w0 & 0x0F0F0F0Fu) | ((dpp_u<DPP_ROW_ROR + 8>(w0) & 0x0F0F0F0Fu) << 4);
                w1 = (w1 & 0x0F0F0F0Fu) | ((dpp_u<DPP_ROW_ROR + 8>(w1) & 0x0F0F0F0Fu) << 4);
                st = st && n < 8;
            }
            if (st) {
                const uint2 w = make_uint2(w0, w1);
                __builtin_memcpy(rec + ((n >> 1) * r + k) * 16 + 8 * (n & 1), &w, 8);
            }
        }
    }
    __syncthreads();

    // ---- 4: row g serves item g: mu codes, c rows, the scale block, the tag -------------
    {
        const bool mine = ok >> g & 1;
        int64_t bo = blk[0];
        int ho = head[0];
        gk_ptr ko = kp[0];
#pragma unroll
        for (int p = 1; p < BI; ++p) {
            bo = g == p ? blk[p] : bo;
            ho = g == p ? head[p] : ho;
            ko = g == p ? kp[p] : ko;
        }
        int8_t* brec = lrec + bo * a.rec_sb;
        int8_t* rec = brec + (int64_t)ho * VM;
        int8_t* tail = brec + (int64_t)a.n_kv * VM + (int64_t)TB * ho;
        int8_t* crows = CLSE ? tail : rec + r * CB + BD;
        uint16_t* meta = (uint16_t*)(CLSE ? tail + 16 * crow : tail);

        float mu[8];
        float mm = 0.f;
#pragma unroll
        for (int e = 0; e < 8; ++e) {
            mu[e] = L.mu[g][8 * n + e];
            mm = fmaxf(mm, fabsf(mu[e]));
        }
        const float msc = quant_scale(row16_maxf(mm), 127.f);
        uint32_t mc[2] = {0u, 0u};
#pragma unroll
        for (int e = 0; e < 8; ++e)
            mc[e >> 2] |= (uint32_t)(quant_code(mu[e], msc, 127.f) & 0xFF) << (8 * (e & 3));
        if (mine) __builtin_memcpy(rec + r * CB + 8 * n, mc, 8);

        float csc = 0.f;                         // token n's coordinate scale
        if constexpr (COORD) {
            const float clvl = a.c_bits == 8 ? 127.f : 7.f;
            float cv[RP];
            float m = 0.f;
#pragma unroll
            for (int k = 0; k < RP; ++k) {
                cv[k] = k < r ? L.m[g][k][n] * __builtin_amdgcn_sqrtf(L.s2[g][k]) : 0.f;
                m = fmaxf(m, fabsf(cv[k]));
            }
            if (a.c_grain >= 1) m = row16_maxf(m);      // one scale per (block, head)
            csc = quant_scale(m, clvl);
            const float inv = __fdiv_rn(1.f, csc);
            unsigned long long row = 0ull;
#pragma unroll
            for (int k = 0; k < RP; ++k) {
                const uint32_t b = code_byte(cv[k], inv);
                if (a.c_bits == 8) row |= (unsigned long long)(b & 0xFFu) << (8 * k);
                else row |= (unsigned long long)(b & 0xFu) << (4 * k);
            }
            if (mine) {
                int8_t* cr = crows + n * crow;
                if (crow == 8) {
                    __builtin_memcpy(cr, &row, 8);
                } else if (crow == 4) {
                    const uint32_t x = (uint32_t)row;
                    __builtin_memcpy(cr, &x, 4);
                } else {
                    for (int i = 0; i < crow; ++i) cr[i] = (int8_t)(row >> (8 * i));
                }
            }
        }

        // the fp16 scale block (CLSE: the tail's scale part), gathered half by half
        constexpr int VH = CLSE ? 16 : 0;        // V scales from this half on
        if (n < r) L.meta[g][VH + n] = L.vsc[g][n & 7];
        if constexpr (CLSE) {
            L.meta[g][n] = csc;
            if (n == 0) {
                L.meta[g][16 + r] = msc;
                float top = 0.f;
                for (int k = 0; k < r; ++k) top += L.s2[g][k];
                L.meta[g][17 + r] = fmaxf(trace - top, 0.f);
            }
        } else if constexpr (COORD) {
            if (a.c_grain != 2) L.meta[g][8 + n] = csc;
            if (n == 0) L.meta[g][24] = msc;
        } else {
            if (n < r) L.meta[g][8 + n] = L.s2[g][n & 7];
            if (n == 0) L.meta[g][16] = msc;
        }
        __syncthreads();
        const int halves = (TB - (CLSE ? 16 * crow : 0)) / 2;
        if (mine && 2 * n < halves) {
            uint32_t w = (uint32_t)f2h_bits(L.meta[g][2 * n]) |
                         ((uint32_t)f2h_bits(L.meta[g][2 * n + 1]) << 16);
            if constexpr (KIND == 1) {
                if (a.c_grain == 2 && n == 4) w = __float_as_uint(csc);   // the fp32 c scale
            }
            __builtin_memcpy(meta + 2 * n, &w, 4);
        }
        if (a.tag != nullptr && mine) {
            uint16_t* tg = (uint16_t*)a.tag + layer * a.tag_lsb + bo * a.tag_sb +
                           (int64_t)ho * a.tag_sh;
            for (int i = n; i < a.tagw; i += 16) tg[i] = ko[(int64_t)(BP - 1) * a.k_st + i];
        }
    }
}

template <int KIND>
static void launch_build(const amass_build_args& a, hipStream_t s) {
    const int64_t items = (int64_t)a.n * a.n_kv;
    const dim3 grid((uint32_t)((items + BI - 1) / BI), 1, a.n_layers), blk(WAVE);
    if (a.rank > 4)
        hipLaunchKernelGGL((summary_build_kernel<KIND, 8>), grid, blk, 0, s, a, items);
    else if (a.rank > 2)
        hipLaunchKernelGGL((summary_build_kernel<KIND, 4>), grid, blk, 0, s, a, items);
    else if (a.rank > 1)
        hipLaunchKernelGGL((summary_build_kernel<KIND, 2>), grid, blk, 0, s, a, items);
    else
        hipLaunchKernelGGL((summary_build_kernel<KIND, 1>), grid, blk, 0, s, a, items);
}

}  // namespace amass

using namespace amass;

extern "C" int amass_summary_build(const amass_build_args* a, void* stream) {
    if (!a) return AMASS_ERR_NULL;
    if ((!a->k && !a->k_layers) || !a->blocks || !a->rec) return AMASS_ERR_NULL;
    if (a->d != BD || a->page != BP || a->n < 0 || a->n_kv < 1) return AMASS_ERR_GEOMETRY;
    if (a->kind < 0 || a->kind > 2) return AMASS_ERR_GEOMETRY;
    if (a->rank < 1 || a->rank > 8) return AMASS_ERR_UNSUPPORTED;
    if (a->v_bits != 8 && a->v_bits != 4) return AMASS_ERR_GEOMETRY;
    if (a->kind >= 1 && a->c_bits != 8 && a->c_bits != 4) return AMASS_ERR_GEOMETRY;
    if (a->c_grain < 0 || a->c_grain > (a->kind == 1 ? 2 : 1)) return AMASS_ERR_GEOMETRY;
    if ((a->v_bits == 4 || (a->kind >= 1 && a->c_bits == 4)) && (a->rank & 1))
        return AMASS_ERR_GEOMETRY;
    if (a->tag && (a->tagw < 0 || a->tagw > 64)) return AMASS_ERR_GEOMETRY;
    const int crow = a->kind >= 1 ? a->rank * a->c_bits / 8 : 0;
    const int vm = a->rank * (a->v_bits == 8 ? BD : BD / 2) + BD + 16 * crow;
    const int64_t rec_bytes = a->kind == 2 ? AMASS_CLSE_REC_BYTES(a->rank, a->v_bits, a->c_bits)
                              : (a->kind == 1 ? vm + 64 : AMASS_QUAD_REC_BYTES(a->rank, a->v_bits));
    if (a->rec_sb < (int64_t)a->n_kv * rec_bytes) return AMASS_ERR_GEOMETRY;
    if (a->n_layers < 1 || (a->n_layers > 1 && !a->k_layers)) return AMASS_ERR_GEOMETRY;
    if (a->n == 0) return AMASS_OK;
    hipStream_t s = (hipStream_t)stream;
    if (a->kind == 2) launch_build<2>(*a, s);
    else if (a->kind == 1) launch_build<1>(*a, s);
    else launch_build<0>(*a, s);
    return check_launch();
}
