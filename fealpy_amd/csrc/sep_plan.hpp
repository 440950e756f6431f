// Evaluation of a separable coefficient (fa_sep_t) that forms each distinct
// factor once a point.  A sum of products repeats its factors (the source
// -div(k grad u) + u of two three-factor functions has 29 factors, 11 of them
// distinct), and the sine and cosine of one argument share its reduction and
// both polynomials.  A block lists the distinct arguments once (`SepPlan`);
// each thread evaluates them into its own column of an LDS table, and the
// terms multiply table entries, four a step.  The values are those of
// sep_value, bit for bit: the same reductions, polynomials, products and
// order (a step is filled up with factors of exactly 1).
#pragma once
#include "cell.hpp"

namespace fa {

constexpr int SEP_COLS = 18;  // table columns a thread (column 0 holds 1.0); an expression that needs more is evaluated factor by factor
constexpr int SEP_WORDS = FA_SEP_MAX_TERMS + FA_SEP_MAX_FACTORS / 4;  // steps of four factors, at least one a term

struct SepPlan {
    int fits;                          // 0: more distinct factors than columns
    int nargs;
    int cls[SEP_COLS], dim[SEP_COLS];  // 0: sin/cos(a s + b), 1: sin/cos(pi (a s + b)), 2: exp, 3: a s + b, 4: s^a
    int cols[SEP_COLS], colc[SEP_COLS];  // columns of the value (sine) and of the cosine, -1: not used
    double a[SEP_COLS], b[SEP_COLS];
    int nterms, fields;                // bit t of fields: term t has a per-cell field
    int wend[FA_SEP_MAX_TERMS];        // one past the term's last word
    double coef[FA_SEP_MAX_TERMS];
    uint32_t word[SEP_WORDS + 1];      // four column indices each
};

// the block's plan in LDS, built by its first wave, a factor per lane; the
// caller synchronises before use
__device__ inline void sep_plan(const fa_sep_t* __restrict__ e, SepPlan& p) {
    static_assert(FA_SEP_MAX_FACTORS <= WAVE && SEP_WORDS < WAVE, "one factor or word per lane of a wave");
    if (threadIdx.x >= WAVE) return;
    const int k = threadIdx.x, nf = e->nfactors;
    const int kind = k < nf ? e->kind[k] : -1;
    const int cls = kind < 0                                         ? -1
                    : kind == FA_SEP_SIN || kind == FA_SEP_COS       ? 0
                    : kind == FA_SEP_SINPI || kind == FA_SEP_COSPI   ? 1
                    : kind == FA_SEP_EXP                             ? 2
                    : kind == FA_SEP_AFFINE                          ? 3
                                                                     : 4;
    const int cosine = kind == FA_SEP_COS || kind == FA_SEP_COSPI;
    const int dim = k < nf ? e->dim[k] : 0;
    const double a = k < nf ? e->a[k] : 0.0, b = k < nf ? e->b[k] : 0.0;
    int first = k, us = 0, uc = 0;  // the argument's first factor; whether its value / cosine is used
    for (int j = nf - 1; j >= 0; --j) {
        const int cj = __shfl(cls, j), dj = __shfl(dim, j), oj = __shfl(cosine, j);
        const double aj = __shfl(a, j), bj = __shfl(b, j);
        // a factor matches itself whatever its numbers: a NaN equals nothing
        if (j == k || (cj == cls && dj == dim && aj == a && bj == b)) {
            if (j < k) first = j;
            us |= !oj;
            uc |= oj;
        }
    }
    const bool rep = cls >= 0 && first == k;
    const unsigned long long args = __ballot(rep), sines = __ballot(rep && us), cosines = __ballot(rep && uc);
    const unsigned long long below = (1ull << first) - 1;
    const int col = 1 + __popcll(sines & below) + __popcll(cosines & below);
    const bool fits = 1 + __popcll(sines) + __popcll(cosines) <= SEP_COLS;
    if (k == 0) {
        p.fits = fits;
        p.nargs = __popcll(args);
    }
    if (!fits) return;
    if (rep) {
        const int u = __popcll(args & below);
        p.cls[u] = cls;
        p.dim[u] = dim;
        p.a[u] = a;
        p.b[u] = b;
        p.cols[u] = us ? col : -1;
        p.colc[u] = uc ? col + us : -1;
    }
    if (k <= SEP_WORDS) p.word[k] = 0;
    __builtin_amdgcn_wave_barrier();
    __builtin_amdgcn_fence(__ATOMIC_SEQ_CST, "wavefront");
    const int nt = e->nterms;
    const bool field = k < nt && e->field[k] != nullptr;
    const unsigned long long fields = __ballot(field);
    if (k < nt) p.coef[k] = e->coef[k];
    if (k == 0) {
        p.nterms = nt;
        p.fields = static_cast<int>(fields);
    }
    int start = 0, words = 0;
    for (int t = 0; t < nt; ++t) {
        const int end = e->term_end[t];
        if (k >= start && k < end)
            reinterpret_cast<uint8_t*>(p.word)[4 * words + (k - start)] = static_cast<uint8_t>(cosine ? col + us : col);
        words += max(1, (end - start + 3) / 4);
        if (k == 0) p.wend[t] = words;
        start = end;
    }
}

// column 0 of the calling thread
template <int STRIDE>
__device__ inline void sep_ones(double* __restrict__ val) {
    val[threadIdx.x] = 1.0;
}

// f at the point x of cell c for a plan that fits; `val` is the block's
// [SEP_COLS][STRIDE] table, of which a thread uses column threadIdx.x only
template <int TD, int STRIDE>
__device__ inline double sep_value_planned(const fa_sep_t* __restrict__ e, const SepPlan& p, const double (&x)[TD],
                                           int64_t c, double* __restrict__ val) {
    double* mine = val + threadIdx.x;
    const int na = __builtin_amdgcn_readfirstlane(p.nargs);
    for (int u = 0; u < na; ++u) {
        const int d = __builtin_amdgcn_readfirstlane(p.dim[u]), cls = __builtin_amdgcn_readfirstlane(p.cls[u]);
        const int cs = __builtin_amdgcn_readfirstlane(p.cols[u]), cc = __builtin_amdgcn_readfirstlane(p.colc[u]);
        const double s = d == 0 ? x[0] : (d == 1 ? x[1] : x[TD - 1]);
        const double t = p.a[u] * s + p.b[u];
        if (cls <= 1) {
            const double arg = cls == 0 ? t * INV_PI : t;
            const double k = rint(2.0 * arg);
            double sn, co;
            sincospi_quarter(fma(-0.5, k, arg), sn, co);
            const int q = static_cast<int>(fma(-4.0, floor(0.25 * k), k));  // k mod 4, exact
            const double vs = (q & 1) ? co : sn, vc = (q & 1) ? sn : co;
            if (cs >= 0) mine[cs * STRIDE] = (q & 2) ? -vs : vs;
            if (cc >= 0) mine[cc * STRIDE] = ((q + 1) & 2) ? -vc : vc;
        } else {
            double v;
            if (cls == 2) {
                v = exp_reduced(t);
            } else if (cls == 3) {
                v = t;
            } else {
                v = 1.0;
                for (int i = 0; i < static_cast<int>(p.a[u]); ++i) v *= s;
            }
            mine[cs * STRIDE] = v;
        }
    }
    double acc = 0.0;
    int w = 0;
    uint32_t cur = __builtin_amdgcn_readfirstlane(p.word[0]);
    const int nt = __builtin_amdgcn_readfirstlane(p.nterms), fields = __builtin_amdgcn_readfirstlane(p.fields);
    for (int t = 0; t < nt; ++t) {
        double v = p.coef[t];
        if ((fields >> t) & 1) v *= e->field[t][c];
        const int we = __builtin_amdgcn_readfirstlane(p.wend[t]);
        for (; w < we; ++w) {
            const uint32_t next = p.word[w + 1];
            const double f0 = mine[(cur & 255) * STRIDE], f1 = mine[((cur >> 8) & 255) * STRIDE];
            const double f2 = mine[((cur >> 16) & 255) * STRIDE], f3 = mine[(cur >> 24) * STRIDE];
            v = v * f0 * f1 * f2 * f3;
            cur = __builtin_amdgcn_readfirstlane(next);
        }
        acc += v;
    }
    return acc;
}

}  // namespace fa
