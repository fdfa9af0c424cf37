// The top eigenpairs of four 16 x 16 symmetric positive semi-definite matrices per wave.
//
// Row p of 16 lanes (a DPP row) holds matrix p, lane n its column n in 16 registers, so the
// broadcasts and sums of every step are DPP row operands (row_newbcast, row steps): no LDS,
// no barriers.  Steps (fp32 throughout, the matrix scaled to mean eigenvalue 1):
//   tridiagonalise   14 Householder reflections; a row's scaled vector v~ (H = 1 - v~ v~^T)
//                    stays in LDS, a float per lane and step, for the back transform
//   eigenvalues      Sturm counts of the tridiagonal matrix by the determinant recurrence
//                    (rescaled every 4 steps, sign bits gathered with alignbit): one round of
//                    16 points over the spectrum, then 16 / RP lanes section each of the RP
//                    wanted intervals together; the Rayleigh quotient finishes
//   eigenvectors     inverse iteration, two solves with a pivoted LU per lane, followed by
//                    modified Gram-Schmidt (after the first solve only where two wanted
//                    eigenvalues lie close)
//   back transform   x <- H_0 .. H_13 x
// Clusters and zero blocks: clamped pivots, start vectors that differ per eigenvector and
// the orthogonalisation give an orthonormal basis of the cluster's space.  Eigenvalues come
// out within ~1e-6 of the largest one, residuals ~3e-7 (mean) of it, orthogonality ~1e-6.
//
// Why not Jacobi: the two-sided round-robin Jacobi this replaced took ~6 sweeps of 15
// rounds, each with three LDS passes over both matrices, for all 16 pairs; the reduction to
// tridiagonal form is one pass and only the wanted pairs are computed after it.
#pragma once
#include <type_traits>

#include "common.h"

namespace amass {

template <int B, int E, typename F>
__device__ __forceinline__ void static_for(F&& f) {
    if constexpr (B < E) {
        f(std::integral_constant<int, B>{});
        static_for<B + 1, E>(f);
    }
}

// lane I of the row's value, in every lane of the row
template <int I>
__device__ __forceinline__ float row_bcast(float v) {
    return __int_as_float(__builtin_amdgcn_update_dpp(0, __float_as_int(v), 0x150 + I, 0xF, 0xF, true));
}
template <int CTRL>
__device__ __forceinline__ float dpp_full(float v) {
    return __int_as_float(__builtin_amdgcn_update_dpp(0, __float_as_int(v), CTRL, 0xF, 0xF, true));
}
__device__ __forceinline__ float row16_sumf(float v) {
    v += dpp_full<DPP_HALF_MIRROR>(v);
    v += dpp_full<DPP_XOR2>(v);
    v += dpp_full<DPP_XOR1>(v);
    v += dpp_full<DPP_ROW_MIRROR>(v);
    return v;
}
constexpr int DPP_ROW_ROR = 0x120;

// Fused multiply-adds with a row_newbcast operand.  The compiler does not fold the DPP move
// into v_fmac_f32 (a move and its wait states for every product: 710 moves and 690 waits in
// this solver), so these are written out, up to five rows to a block.  A DPP operand may
// not have been written by the two VALU cycles before it, and the compiler does not look
// into the blocks: each begins and ends with s_nop 1, inside a block no DPP operand is
// written.  All 64 lanes must be active.
#define AMASS_FMAC_DPP(acc, src, mul, l) \
    "v_fmac_f32_dpp " acc ", " src ", " mul " row_newbcast:" l " row_mask:0xf bank_mask:0xf\n"
__device__ __forceinline__ float sel(bool c, float x, float y) { return c ? x : y; }

// p += sum over i in [I, 16) of (lane i's v) a[i]
template <int I>
__device__ __forceinline__ void bcast_dot(float& p, float v, const float (&a)[16]) {
    if constexpr (I + 5 <= 16) {
        asm("s_nop 1\n"
            AMASS_FMAC_DPP("%0", "%1", "%2", "%7")
            AMASS_FMAC_DPP("%0", "%1", "%3", "%8")
            AMASS_FMAC_DPP("%0", "%1", "%4", "%9")
            AMASS_FMAC_DPP("%0", "%1", "%5", "%10")
            AMASS_FMAC_DPP("%0", "%1", "%6", "%11")
            "s_nop 1" : "+&v"(p) : "v"(v), "v"(a[I + 0]), "v"(a[I + 1]), "v"(a[I + 2]), "v"(a[I + 3]), "v"(a[I + 4]), "n"(I + 0), "n"(I + 1), "n"(I + 2), "n"(I + 3), "n"(I + 4));
        bcast_dot<I + 5>(p, v, a);
    } else if constexpr (I + 4 == 16) {
        asm("s_nop 1\n"
            AMASS_FMAC_DPP("%0", "%1", "%2", "%6")
            AMASS_FMAC_DPP("%0", "%1", "%3", "%7")
            AMASS_FMAC_DPP("%0", "%1", "%4", "%8")
            AMASS_FMAC_DPP("%0", "%1", "%5", "%9")
            "s_nop 1" : "+&v"(p) : "v"(v), "v"(a[I + 0]), "v"(a[I + 1]), "v"(a[I + 2]), "v"(a[I + 3]), "n"(I + 0), "n"(I + 1), "n"(I + 2), "n"(I + 3));
    } else if constexpr (I + 3 == 16) {
        asm("s_nop 1\n"
            AMASS_FMAC_DPP("%0", "%1", "%2", "%5")
            AMASS_FMAC_DPP("%0", "%1", "%3", "%6")
            AMASS_FMAC_DPP("%0", "%1", "%4", "%7")
            "s_nop 1" : "+&v"(p) : "v"(v), "v"(a[I + 0]), "v"(a[I + 1]), "v"(a[I + 2]), "n"(I + 0), "n"(I + 1), "n"(I + 2));
    } else if constexpr (I + 2 == 16) {
        asm("s_nop 1\n"
            AMASS_FMAC_DPP("%0", "%1", "%2", "%4")
            AMASS_FMAC_DPP("%0", "%1", "%3", "%5")
            "s_nop 1" : "+&v"(p) : "v"(v), "v"(a[I + 0]), "v"(a[I + 1]), "n"(I + 0), "n"(I + 1));
    } else if constexpr (I + 1 == 16) {
        asm("s_nop 1\n"
            AMASS_FMAC_DPP("%0", "%1", "%2", "%3")
            "s_nop 1" : "+&v"(p) : "v"(v), "v"(a[I + 0]), "n"(I + 0));
    }
}
// a[i] += (lane i's v) c, i in [I, 16)
template <int I>
__device__ __forceinline__ void bcast_axpy(float (&a)[16], float v, float c) {
    if constexpr (I + 5 <= 16) {
        asm("s_nop 1\n"
            AMASS_FMAC_DPP("%0", "%5", "%6", "%7")
            AMASS_FMAC_DPP("%1", "%5", "%6", "%8")
            AMASS_FMAC_DPP("%2", "%5", "%6", "%9")
            AMASS_FMAC_DPP("%3", "%5", "%6", "%10")
            AMASS_FMAC_DPP("%4", "%5", "%6", "%11")
            "s_nop 1" : "+&v"(a[I + 0]), "+&v"(a[I + 1]), "+&v"(a[I + 2]), "+&v"(a[I + 3]), "+&v"(a[I + 4]) : "v"(v), "v"(c), "n"(I + 0), "n"(I + 1), "n"(I + 2), "n"(I + 3), "n"(I + 4));
        bcast_axpy<I + 5>(a, v, c);
    } else if constexpr (I + 4 == 16) {
        asm("s_nop 1\n"
            AMASS_FMAC_DPP("%0", "%4", "%5", "%6")
            AMASS_FMAC_DPP("%1", "%4", "%5", "%7")
            AMASS_FMAC_DPP("%2", "%4", "%5", "%8")
            AMASS_FMAC_DPP("%3", "%4", "%5", "%9")
            "s_nop 1" : "+&v"(a[I + 0]), "+&v"(a[I + 1]), "+&v"(a[I + 2]), "+&v"(a[I + 3]) : "v"(v), "v"(c), "n"(I + 0), "n"(I + 1), "n"(I + 2), "n"(I + 3));
    } else if constexpr (I + 3 == 16) {
        asm("s_nop 1\n"
            AMASS_FMAC_DPP("%0", "%3", "%4", "%5")
            AMASS_FMAC_DPP("%1", "%3", "%4", "%6")
            AMASS_FMAC_DPP("%2", "%3", "%4", "%7")
            "s_nop 1" : "+&v"(a[I + 0]), "+&v"(a[I + 1]), "+&v"(a[I + 2]) : "v"(v), "v"(c), "n"(I + 0), "n"(I + 1), "n"(I + 2));
    } else if constexpr (I + 2 == 16) {
        asm("s_nop 1\n"
            AMASS_FMAC_DPP("%0", "%2", "%3", "%4")
            AMASS_FMAC_DPP("%1", "%2", "%3", "%5")
            "s_nop 1" : "+&v"(a[I + 0]), "+&v"(a[I + 1]) : "v"(v), "v"(c), "n"(I + 0), "n"(I + 1));
    } else if constexpr (I + 1 == 16) {
        asm("s_nop 1\n"
            AMASS_FMAC_DPP("%0", "%1", "%2", "%3")
            "s_nop 1" : "+&v"(a[I + 0]) : "v"(v), "v"(c), "n"(I + 0));
    }
}
// a[i] += (lane i's v) nw + (lane i's w) nv, i in [I, 16)
template <int I>
__device__ __forceinline__ void bcast_rank2(float (&a)[16], float v, float w, float nv, float nw) {
    if constexpr (I + 5 <= 16) {
        asm("s_nop 1\n"
            AMASS_FMAC_DPP("%0", "%5", "%8", "%9")
            AMASS_FMAC_DPP("%0", "%6", "%7", "%9")
            AMASS_FMAC_DPP("%1", "%5", "%8", "%10")
            AMASS_FMAC_DPP("%1", "%6", "%7", "%10")
            AMASS_FMAC_DPP("%2", "%5", "%8", "%11")
            AMASS_FMAC_DPP("%2", "%6", "%7", "%11")
            AMASS_FMAC_DPP("%3", "%5", "%8", "%12")
            AMASS_FMAC_DPP("%3", "%6", "%7", "%12")
            AMASS_FMAC_DPP("%4", "%5", "%8", "%13")
            AMASS_FMAC_DPP("%4", "%6", "%7", "%13")
            "s_nop 1" : "+&v"(a[I + 0]), "+&v"(a[I + 1]), "+&v"(a[I + 2]), "+&v"(a[I + 3]), "+&v"(a[I + 4]) : "v"(v), "v"(w), "v"(nv), "v"(nw), "n"(I + 0), "n"(I + 1), "n"(I + 2), "n"(I + 3), "n"(I + 4));
        bcast_rank2<I + 5>(a, v, w, nv, nw);
    } else if constexpr (I + 4 == 16) {
        asm("s_nop 1\n"
            AMASS_FMAC_DPP("%0", "%4", "%7", "%8")
            AMASS_FMAC_DPP("%0", "%5", "%6", "%8")
            AMASS_FMAC_DPP("%1", "%4", "%7", "%9")
            AMASS_FMAC_DPP("%1", "%5", "%6", "%9")
            AMASS_FMAC_DPP("%2", "%4", "%7", "%10")
            AMASS_FMAC_DPP("%2", "%5", "%6", "%10")
            AMASS_FMAC_DPP("%3", "%4", "%7", "%11")
            AMASS_FMAC_DPP("%3", "%5", "%6", "%11")
            "s_nop 1" : "+&v"(a[I + 0]), "+&v"(a[I + 1]), "+&v"(a[I + 2]), "+&v"(a[I + 3]) : "v"(v), "v"(w), "v"(nv), "v"(nw), "n"(I + 0), "n"(I + 1), "n"(I + 2), "n"(I + 3));
    } else if constexpr (I + 3 == 16) {
        asm("s_nop 1\n"
            AMASS_FMAC_DPP("%0", "%3", "%6", "%7")
            AMASS_FMAC_DPP("%0", "%4", "%5", "%7")
            AMASS_FMAC_DPP("%1", "%3", "%6", "%8")
            AMASS_FMAC_DPP("%1", "%4", "%5", "%8")
            AMASS_FMAC_DPP("%2", "%3", "%6", "%9")
            AMASS_FMAC_DPP("%2", "%4", "%5", "%9")
            "s_nop 1" : "+&v"(a[I + 0]), "+&v"(a[I + 1]), "+&v"(a[I + 2]) : "v"(v), "v"(w), "v"(nv), "v"(nw), "n"(I + 0), "n"(I + 1), "n"(I + 2));
    } else if constexpr (I + 2 == 16) {
        asm("s_nop 1\n"
            AMASS_FMAC_DPP("%0", "%2", "%5", "%6")
            AMASS_FMAC_DPP("%0", "%3", "%4", "%6")
            AMASS_FMAC_DPP("%1", "%2", "%5", "%7")
            AMASS_FMAC_DPP("%1", "%3", "%4", "%7")
            "s_nop 1" : "+&v"(a[I + 0]), "+&v"(a[I + 1]) : "v"(v), "v"(w), "v"(nv), "v"(nw), "n"(I + 0), "n"(I + 1));
    } else if constexpr (I + 1 == 16) {
        asm("s_nop 1\n"
            AMASS_FMAC_DPP("%0", "%1", "%4", "%5")
            AMASS_FMAC_DPP("%0", "%2", "%3", "%5")
            "s_nop 1" : "+&v"(a[I + 0]) : "v"(v), "v"(w), "v"(nv), "v"(nw), "n"(I + 0));
    }
}
// s += x . (lane K's x)
template <int K, int I = 0>
__device__ __forceinline__ void lane_dot(float& s, const float (&x)[16]) {
    if constexpr (I < 15) {
        asm("s_nop 1\n"
            AMASS_FMAC_DPP("%0", "%1", "%1", "%6")
            AMASS_FMAC_DPP("%0", "%2", "%2", "%6")
            AMASS_FMAC_DPP("%0", "%3", "%3", "%6")
            AMASS_FMAC_DPP("%0", "%4", "%4", "%6")
            AMASS_FMAC_DPP("%0", "%5", "%5", "%6")
            "s_nop 1" : "+&v"(s) : "v"(x[I + 0]), "v"(x[I + 1]), "v"(x[I + 2]), "v"(x[I + 3]), "v"(x[I + 4]), "n"(K));
        lane_dot<K, I + 5>(s, x);
    } else {
        asm("s_nop 1\n"
            AMASS_FMAC_DPP("%0", "%1", "%1", "%2")
            "s_nop 1" : "+&v"(s) : "v"(x[I + 0]), "n"(K));
    }
}
// x += (lane K's x) c
template <int K, int I = 0>
__device__ __forceinline__ void lane_axpy(float (&x)[16], float c) {
    if constexpr (I < 15) {
        asm("s_nop 1\n"
            AMASS_FMAC_DPP("%0", "%0", "%5", "%6")
            AMASS_FMAC_DPP("%1", "%1", "%5", "%6")
            AMASS_FMAC_DPP("%2", "%2", "%5", "%6")
            AMASS_FMAC_DPP("%3", "%3", "%5", "%6")
            AMASS_FMAC_DPP("%4", "%4", "%5", "%6")
            "s_nop 1" : "+&v"(x[I + 0]), "+&v"(x[I + 1]), "+&v"(x[I + 2]), "+&v"(x[I + 3]), "+&v"(x[I + 4]) : "v"(c), "n"(K));
        lane_axpy<K, I + 5>(x, c);
    } else {
        asm("s_nop 1\n"
            AMASS_FMAC_DPP("%0", "%0", "%1", "%2")
            "s_nop 1" : "+&v"(x[I + 0]) : "v"(c), "n"(K));
    }
}
#undef AMASS_FMAC_DPP

// Rounds of the section search after the shared one (16 points over the whole spectrum):
// 16 / RP lanes per interval cut it into 16 / RP + 1 parts per round, until it is narrower than
// SECT_REL of the eigenvalue or SECT_ABS of the mean one (what fp32 counts resolve).  The
// Rayleigh quotient would forgive a wider one for the eigenvalue, the two solves do not for
// the vector: on pages with one outlier token, whose mean eigenvalue is far above the other
// fifteen, 9 / 7 / 5 / 4 rounds (5e-5 .. 1e-5 of the mean) took the error of the r8 factors'
// product from 2.80e-3, as with Jacobi, to 4.61e-3 (rank 8, an outlier of 100 in units of the
// keys' spread; rank 2 2.42e-3 to 2.59e-3).  NIT rounds reach SECT_ABS from any spectrum;
// ordinary pages stop after 9 / 7 / 5 / 4.
constexpr float SECT_REL = 1e-5f, SECT_ABS = 7e-7f;
template <int RP>
struct Sections {
    static constexpr int M = 16 / RP;
    static constexpr int NIT = RP == 8 ? 13 : (RP == 4 ? 9 : (RP == 2 ? 7 : 5));
};

// Number of eigenvalues of the tridiagonal matrix (d, e^2) below x.
__device__ __forceinline__ int sturm_count(const float (&d)[16], const float (&e2)[15], float x) {
    float p0 = 1.f, p1 = d[0] - x;
    uint32_t m = __builtin_amdgcn_alignbit(0u, __float_as_uint(p1), 31);
    static_for<1, 16>([&](auto I) {
        constexpr int i = I;
        const float p2 = __builtin_fmaf(d[i] - x, p1, -(e2[i - 1] * p0));
        m = __builtin_amdgcn_alignbit(m, __float_as_uint(p2), 31);
        p0 = p1;
        p1 = p2;
        if constexpr (i % 4 == 0) {
            const int ex = -__builtin_amdgcn_frexp_expf(fmaxf(fabsf(p0), fabsf(p1)));
            p0 = __builtin_amdgcn_ldexpf(p0, ex);
            p1 = __builtin_amdgcn_ldexpf(p1, ex);
        }
    });
    return __popc((m ^ (m >> 1)) & 0xFFFFu);
}

// x <- x minus its projections on the vectors of higher k (lanes with k' < k lose vector
// k's part), in the rows with `on`; vector k sits in the lanes with kl == k.  Vectors keep
// their lengths.
template <int RP>
__device__ __forceinline__ void gram_schmidt(float (&x)[16], int r, int kl, bool on) {
    static_for<0, RP - 1>([&](auto K) {
        constexpr int k = RP - 1 - K;                  // RP-1 .. 1
        if (k < r) {
            float s = 0.f;
            lane_dot<k>(s, x);                         // (in lane k: its squared length)
            const float t = s * __builtin_amdgcn_rcpf(fmaxf(row_bcast<k>(s), 1e-30f));
            lane_axpy<k>(x, on && kl < k ? -t : 0.f);
        }
    });
}

__device__ __forceinline__ void unit_length(float (&x)[16]) {
    float mx = 0.f;
#pragma unroll
    for (int i = 0; i < 16; ++i) mx = fmaxf(mx, fabsf(x[i]));
    const float s = __builtin_amdgcn_rcpf(fmaxf(mx, 1e-30f));
    float nn = 0.f;
#pragma unroll
    for (int i = 0; i < 16; ++i) {
        x[i] *= s;
        nn = __builtin_fmaf(x[i], x[i], nn);
    }
    const float u = __builtin_amdgcn_rsqf(fmaxf(nn, 1e-30f));
#pragma unroll
    for (int i = 0; i < 16; ++i) x[i] *= u;
}

constexpr float EIGH16_MAX_TRACE = 3e38f;              // a matrix of this trace is not solved

// a: column n (lane n of the row) of the row's matrix, destroyed.  Lane k < r gets the
// k-th of the top r eigenvalues in ascending order (unclamped) and its eigenvector x; lanes
// k + RP, k + 2 RP, ... get copies.  tr: the matrix's trace.  hv: 14 x 64 floats of LDS for
// the reflections (each lane reads what it wrote), which frees their registers for the LU.
template <int RP>
__device__ __forceinline__ void eigh16_top(float (&a)[16], int r, float tr, float& lam,
                                           float (&x)[16], float (*hv)[WAVE]) {
    using S = Sections<RP>;
    const int lane = threadIdx.x & 63, n = lane & 15;
    const int kl = n & (RP - 1);
    const bool live = tr > 1e-30f && tr < EIGH16_MAX_TRACE;    // else zero, infinite or NaN
    const float sc = live ? 16.f / tr : 0.f;
#pragma unroll
    for (int i = 0; i < 16; ++i) a[i] *= sc;

    // ---- Householder ---------------------------------------------------------------------
    float d[16], e[15];
    static_for<0, 14>([&](auto K) {
        constexpr int k = K;
        const float t = n > k + 1 ? a[k] : 0.f;        // row k = column k: x_j in lane j
        const float tail = row16_sumf(t * t);
        const float al = row_bcast<k + 1>(a[k]);
        const float sig = __builtin_fmaf(al, al, tail);
        const float sq = __builtin_amdgcn_sqrtf(sig);
        const float beta = al < 0.f ? sq : -sq;
        const float h = __builtin_fmaf(fabsf(al), sq, sig);
        const bool on = h > 1e-30f;
        const float rs = on ? __builtin_amdgcn_rsqf(h) : 0.f;
        const float v = (n == k + 1 ? al - beta : t) * rs;
        hv[k][lane] = v;
        e[k] = on ? beta : al;
        float p = 0.f;
        bcast_dot<k + 1>(p, v, a);
        const float kk = 0.5f * row16_sumf(v * p);
        const float w = __builtin_fmaf(-kk, v, p);
        bcast_rank2<k + 1>(a, v, w, -v, -w);
    });
    static_for<0, 16>([&](auto I) {
        constexpr int i = I;
        d[i] = row_bcast<i>(a[i]);
    });
    e[14] = row_bcast<15>(a[14]);

    // ---- eigenvalues -----------------------------------------------------------------------
    float lo, hi;
    {
        float e2[15];
        float top = d[0] + fabsf(e[0]);                // Gershgorin's upper bound
#pragma unroll
        for (int i = 0; i < 15; ++i) {
            e2[i] = e[i] * e[i];
            top = fmaxf(top, d[i + 1] + fabsf(e[i]) + (i < 14 ? fabsf(e[i < 14 ? i + 1 : 14]) : 0.f));
        }
        const int target = 16 - r + kl;                // its index, ascending
        {
            const float l0 = -1e-4f;
            const float w = __builtin_fmaf(top, 1.00001f, 2e-4f) * (1.f / 17.f);
            const int c = sturm_count(d, e2, __builtin_fmaf(w, (float)(n + 1), l0));
            int at = 0;                                // points at or below the eigenvalue
            static_for<0, 16>([&](auto I) {
                constexpr int i = I;
                at += __float_as_int(row_bcast<i>(__int_as_float(c))) <= target ? 1 : 0;
            });
            lo = __builtin_fmaf(w, (float)at, l0 - 2e-6f);
            hi = lo + w + 4e-6f;
        }
        const float fr = (float)(n / RP + 1) * (1.f / (S::M + 1));
#pragma unroll 1
        for (int it = 0; it < S::NIT; ++it) {
            // (an interval's lanes agree, and each stops by itself whatever the others need)
            const bool wide = hi - lo > fmaxf(SECT_ABS, SECT_REL * lo);
            if (__ballot(wide) == 0) break;
            const float xs = __builtin_fmaf(hi - lo, fr, lo);
            const bool above = sturm_count(d, e2, xs) <= target;   // eigenvalue >= xs
            float nl = above ? xs : lo, nh = above ? hi : xs;
            if constexpr (RP <= 8) {
                nl = fmaxf(nl, dpp_full<DPP_ROW_ROR + 8>(nl));
                nh = fminf(nh, dpp_full<DPP_ROW_ROR + 8>(nh));
            }
            if constexpr (RP <= 4) {
                nl = fmaxf(nl, dpp_full<DPP_ROW_ROR + 4>(nl));
                nh = fminf(nh, dpp_full<DPP_ROW_ROR + 4>(nh));
            }
            if constexpr (RP <= 2) {
                nl = fmaxf(nl, dpp_full<DPP_ROW_ROR + 2>(nl));
                nh = fminf(nh, dpp_full<DPP_ROW_ROR + 2>(nh));
            }
            if constexpr (RP <= 1) {
                nl = fmaxf(nl, dpp_full<DPP_ROW_ROR + 1>(nl));
                nh = fminf(nh, dpp_full<DPP_ROW_ROR + 1>(nh));
            }
            lo = wide ? nl : lo;
            hi = wide ? nh : hi;
        }
    }
    const float lm = 0.5f * (lo + hi);

    // ---- LU of T - lam with partial pivoting (row i and i + 1), per lane ---------------
    constexpr float PIV = 2e-6f;                       // a pivot's least magnitude
    float rp[16], s1[15], s2[15], mm[15];
    bool sw[15];
    {
        float u = d[0] - lm, v = e[0];
        static_for<1, 16>([&](auto I) {
            constexpr int i = I;
            const float ee = e[i - 1], dd = d[i] - lm;
            const float en = i < 15 ? e[i < 15 ? i : 14] : 0.f;
            const bool s = fabsf(ee) > fabsf(u);
            float pv = sel(s, ee, u);
            pv = fabsf(pv) < PIV ? __builtin_copysignf(PIV, pv) : pv;
            const float q = __builtin_amdgcn_rcpf(pv);
            rp[i - 1] = q;
            const float m = sel(s, u, ee) * q;
            mm[i - 1] = m;
            sw[i - 1] = s;
            s1[i - 1] = sel(s, dd, v);
            s2[i - 1] = s ? en : 0.f;
            u = __builtin_fmaf(-m, s1[i - 1], sel(s, v, dd));
            v = sel(s, -m * en, en);
        });
        const float pv = fabsf(u) < PIV ? __builtin_copysignf(PIV, u) : u;
        rp[15] = __builtin_amdgcn_rcpf(pv);
    }
    auto back = [&]() {                                // x <- U^-1 x
        x[15] *= rp[15];
        x[14] = __builtin_fmaf(-s1[14], x[15], x[14]) * rp[14];
#pragma unroll
        for (int i = 13; i >= 0; --i)
            x[i] = __builtin_fmaf(-s2[i], x[i + 2], __builtin_fmaf(-s1[i], x[i + 1], x[i])) * rp[i];
    };
    // start vectors: magnitudes 1 .. 2 and signs from rotations of a word per k
    const uint32_t word = ((uint32_t)kl + 1u) * 0x9E3779B1u ^ 0x5F356495u;
#pragma unroll
    for (int i = 0; i < 16; ++i) {
        const uint32_t w = __builtin_amdgcn_alignbit(word, word, (2 * i + 1) & 31);
        x[i] = __uint_as_float((w & 0x807FFFFFu) | 0x3F800000u);
    }
    back();
    unit_length(x);
    // wanted eigenvalues closer than 1e-3 of the mean: separate the vectors before the
    // second solve, or both would converge to the same one
    // (row by row: a page's summary is a function of its own keys, not of its wave's others)
    const float up = dpp_full<DPP_ROW_SHR1>(lm);       // lane n - 1's
    const unsigned long long near = __ballot(kl > 0 && n < r && !(lm - up > 1e-3f));
    if (near) gram_schmidt<RP>(x, r, kl, (near >> (lane & 48) & 0xFFFF) != 0);
#pragma unroll
    for (int i = 1; i < 16; ++i) {                     // x <- L^-1 P x
        const float xa = x[i - 1], xb = x[i];
        x[i - 1] = sel(sw[i - 1], xb, xa);
        x[i] = __builtin_fmaf(-mm[i - 1], x[i - 1], sel(sw[i - 1], xa, xb));
    }
    back();
    unit_length(x);
    gram_schmidt<RP>(x, r, kl, true);
    unit_length(x);

    {   // the eigenvalue: lm + x^T (T - lm) x
        float s = 0.f, t = 0.f;
#pragma unroll
        for (int i = 0; i < 16; ++i) {
            s = __builtin_fmaf(d[i] - lm, x[i] * x[i], s);
            if (i < 15) t = __builtin_fmaf(e[i < 15 ? i : 14], x[i] * x[i < 15 ? i + 1 : 15], t);
        }
        lam = live ? (lm + __builtin_fmaf(2.f, t, s)) * (tr * 0.0625f) : 0.f;
    }

    // ---- back transform --------------------------------------------------------------------
    static_for<0, 14>([&](auto K) {
        constexpr int k = 13 - K;
        float s = 0.f;
        const float v = hv[k][lane];
        bcast_dot<k + 1>(s, v, x);
        bcast_axpy<k + 1>(x, v, -s);
    });
}

}  // namespace amass
