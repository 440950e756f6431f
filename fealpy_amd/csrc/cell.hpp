// Cell geometry and coefficient values shared by the element and assembly
// kernels.
#pragma once
#include "common.hpp"

namespace fa {

// ---- cell geometry ---------------------------------------------------------
// Triangle: grad lambda as numpy_backend.py:586-598, |T| = det(p1-p0, p2-p1)/2
// (simplex_measure, numpy_backend.py:413-421).
// Tetrahedron: grad lambda = cross(v_jm, v_jk) / (6 vol) over localFace
// (numpy_backend.py:619-629, tetrahedron_mesh.py:23-24), |T| by the triple
// product of tetrahedron_mesh.py:165-175.
template <int TD>
struct Geom;

template <>
struct Geom<2> {
    double gl[3][2];
    double meas;
    __device__ void compute(const double p[3][2]) {
        double e[3][2];
        for (int d = 0; d < 2; ++d) {
            e[0][d] = p[2][d] - p[1][d];
            e[1][d] = p[0][d] - p[2][d];
            e[2][d] = p[1][d] - p[0][d];
        }
        const double nv = e[0][0] * e[1][1] - e[0][1] * e[1][0];
        for (int i = 0; i < 3; ++i) {
            gl[i][0] = -e[i][1] / nv;
            gl[i][1] = e[i][0] / nv;
        }
        const double a0 = p[1][0] - p[0][0], a1 = p[1][1] - p[0][1];
        const double b0 = p[2][0] - p[1][0], b1 = p[2][1] - p[1][1];
        meas = (a0 * b1 - a1 * b0) / 2.0;
    }
};

__device__ inline void cross3(const double a[3], const double b[3], double c[3]) {
    c[0] = a[1] * b[2] - a[2] * b[1];
    c[1] = a[2] * b[0] - a[0] * b[2];
    c[2] = a[0] * b[1] - a[1] * b[0];
}

template <>
struct Geom<3> {
    double gl[4][3];
    double meas;
    __device__ void compute(const double p[4][3]) {
        // simplex_measure: det of consecutive edge vectors / 6
        double a[3], b[3], c[3], t[3];
        for (int d = 0; d < 3; ++d) {
            a[d] = p[1][d] - p[0][d];
            b[d] = p[2][d] - p[1][d];
            c[d] = p[3][d] - p[2][d];
        }
        cross3(b, c, t);
        const double vol6 = a[0] * t[0] + a[1] * t[1] + a[2] * t[2];  // 6 * simplex_measure
        const int lf[4][3] = {{1, 2, 3}, {0, 3, 2}, {0, 1, 3}, {0, 2, 1}};
        for (int i = 0; i < 4; ++i) {
            double vjk[3], vjm[3], n[3];
            for (int d = 0; d < 3; ++d) {
                vjk[d] = p[lf[i][1]][d] - p[lf[i][0]][d];
                vjm[d] = p[lf[i][2]][d] - p[lf[i][0]][d];
            }
            cross3(vjm, vjk, n);
            for (int d = 0; d < 3; ++d) gl[i][d] = n[d] / vol6;
        }
        double v01[3], v02[3], v03[3], x[3];
        for (int d = 0; d < 3; ++d) {
            v01[d] = p[1][d] - p[0][d];
            v02[d] = p[2][d] - p[0][d];
            v03[d] = p[3][d] - p[0][d];
        }
        cross3(v01, v02, x);
        meas = (v03[0] * x[0] + v03[1] * x[1] + v03[2] * x[2]) / 6.0;
    }
};

template <int TD>
__device__ inline void load_cell(const double* __restrict__ node, const int32_t* __restrict__ cell, int64_t c,
                                 double p[TD + 1][TD]) {
#pragma unroll
    for (int v = 0; v < TD + 1; ++v) {
        const int64_t n = cell[c * (TD + 1) + v];
#pragma unroll
        for (int d = 0; d < TD; ++d) p[v][d] = node[n * TD + d];
    }
}

__device__ inline double coef_value(int kind, double scale, const double* __restrict__ coef, int64_t c, int q,
                                    int nq) {
    switch (kind) {
        case FA_COEF_CONST: return scale;
        case FA_COEF_CELL: return scale * coef[c];
        case FA_COEF_CELLQ: return scale * coef[c * nq + q];
        default: return 0.0;
    }
}

// ---- separable coefficients (FA_COEF_SEP) -----------------------------------
// sin(pi x) and cos(pi x): x = k/2 + r with k = rint(2x), |r| <= 1/4 (r = x - k/2
// is exact for |x| < 2^51), then the Taylor series of sin(pi r) and cos(pi r)
// at 0 (coefficients (-1)^n pi^(2n+1)/(2n+1)! and (-1)^n pi^(2n)/(2n)!, through
// r^17 and r^18: the remainder is below 1e-19 for |r| <= 1/4) by Horner's rule,
// and the quadrant k mod 4.  Few registers, unlike the general library sin.
__device__ inline void sincospi_quarter(double r, double& s, double& c) {
    const double z = r * r;
    double ps = 7.952054001475513e-07;
    ps = fma(ps, z, -2.1915353447830217e-05);
    ps = fma(ps, z, 0.00046630280576761255);
    ps = fma(ps, z, -0.0073704309457143504);
    ps = fma(ps, z, 0.08214588661112823);
    ps = fma(ps, z, -0.5992645293207921);
    ps = fma(ps, z, 2.5501640398773455);
    ps = fma(ps, z, -5.16771278004997);
    ps = fma(ps, z, 3.141592653589793);
    s = r * ps;
    double pc = -1.3878952462213771e-07;
    pc = fma(pc, z, 4.303069587032947e-06);
    pc = fma(pc, z, -0.0001046381049248457);
    pc = fma(pc, z, 0.0019295743094039231);
    pc = fma(pc, z, -0.02580689139001406);
    pc = fma(pc, z, 0.2353306303588932);
    pc = fma(pc, z, -1.3352627688545895);
    pc = fma(pc, z, 4.0587121264167685);
    pc = fma(pc, z, -4.934802200544679);
    c = fma(pc, z, 1.0);
}

// sin(pi x) for shift 0, cos(pi x) for shift 1
__device__ inline double sinpi_shift(double x, int shift) {
    const double k = rint(2.0 * x);
    const double r = fma(-0.5, k, x);
    double s, c;
    sincospi_quarter(r, s, c);
    const int q = (static_cast<int>(static_cast<long long>(k) & 3) + shift) & 3;
    const double v = (q & 1) ? c : s;
    return (q & 2) ? -v : v;
}

constexpr double INV_PI = 0.31830988618379067154;

// exp(x) = 2^k e^r: k = rint(x / ln 2), r = x - k ln 2 with ln 2 split in two
// doubles (Cody and Waite's reduction, the second part applied by FMA), so
// |r| <= ln(2)/2; e^r from its Taylor series through r^14 (remainder below
// 1e-19), by Horner's rule; then the exponent is scaled in by ldexp.
__device__ inline double exp_reduced(double x) {
    if (x > 709.78) return HUGE_VAL;
    if (x < -745.2) return 0.0;
    const double k = rint(x * 1.4426950408889634);
    double r = fma(-k, 0.6931471805599453, x);
    r = fma(-k, 2.3190468138462996e-17, r);
    double e = 1.1470745597729725e-11;
    e = fma(e, r, 1.6059043836821613e-10);
    e = fma(e, r, 2.08767569878681e-09);
    e = fma(e, r, 2.505210838544172e-08);
    e = fma(e, r, 2.755731922398589e-07);
    e = fma(e, r, 2.7557319223985893e-06);
    e = fma(e, r, 2.48015873015873e-05);
    e = fma(e, r, 0.0001984126984126984);
    e = fma(e, r, 0.001388888888888889);
    e = fma(e, r, 0.008333333333333333);
    e = fma(e, r, 0.041666666666666664);
    e = fma(e, r, 0.16666666666666666);
    e = fma(e, r, 0.5);
    e = fma(e, r, 1.0);
    e = fma(e, r, 1.0);
    return ldexp(e, static_cast<int>(k));
}

// One factor g(s) of a term; every lane runs the same program (the struct is
// read through uniform loads), so the switch does not diverge.
__device__ inline double sep_factor(int kind, double a, double b, double s) {
    switch (kind) {
        case FA_SEP_SIN: return sinpi_shift((a * s + b) * INV_PI, 0);
        case FA_SEP_COS: return sinpi_shift((a * s + b) * INV_PI, 1);
        case FA_SEP_EXP: return exp_reduced(a * s + b);
        case FA_SEP_AFFINE: return a * s + b;
        case FA_SEP_SINPI: return sinpi_shift(a * s + b, 0);
        case FA_SEP_COSPI: return sinpi_shift(a * s + b, 1);
        default: {  // FA_SEP_POW: s^a, a a whole number
            const int k = static_cast<int>(a);
            double r = 1.0;
            for (int i = 0; i < k; ++i) r *= s;
            return r;
        }
    }
}

// f(x) at quadrature point q of cell c with vertices p: x = sum_v bcs[q][v] p_v
// (the order of bc_to_point), then the sum of the terms in order
template <int TD>
__device__ inline double sep_value(const fa_sep_t* __restrict__ e, int q, const double p[TD + 1][TD], int64_t c) {
    double x[TD];
#pragma unroll
    for (int d = 0; d < TD; ++d) x[d] = 0.0;
#pragma unroll
    for (int v = 0; v < TD + 1; ++v) {
        const double w = e->bcs[q * (TD + 1) + v];
#pragma unroll
        for (int d = 0; d < TD; ++d) x[d] += w * p[v][d];
    }
    double acc = 0.0;
    int k = 0;
    const int nt = e->nterms;
    for (int t = 0; t < nt; ++t) {
        double v = e->coef[t];
        const double* fld = e->field[t];
        if (fld) v *= fld[c];
        const int kend = e->term_end[t];
        for (; k < kend; ++k) {
            const int d = e->dim[k];
            const double s = (TD == 2) ? (d == 0 ? x[0] : x[TD - 1]) : (d == 0 ? x[0] : (d == 1 ? x[1] : x[TD - 1]));
            v *= sep_factor(e->kind[k], e->a[k], e->b[k], s);
        }
        acc += v;
    }
    return acc;
}

// coefficient at quadrature point q of cell c: `ci` indexes the per-cell /
// per-point arrays (which may be a block's staged copy), `cg` is the global
// cell id (fields of a separable coefficient)
// SEP: the kernel was instantiated for a separable coefficient; kernels
// without one do not carry the transcendental code (it costs registers).
template <int TD, bool SEP>
__device__ inline double coef_at(int kind, double scale, const double* __restrict__ coef, int64_t ci, int64_t cg,
                                 int q, int nq, const double p[TD + 1][TD]) {
    if constexpr (SEP) {
        if (kind == FA_COEF_SEP) return scale * sep_value<TD>(reinterpret_cast<const fa_sep_t*>(coef), q, p, cg);
    }
    return coef_value(kind, scale, coef, ci, q, nq);
}

}  // namespace fa
