// FP64 element matrices of scalar diffusion and mass on simplices, on the FP64
// matrix instruction v_mfma_f64_16x16x4_f64.
#include "cell.hpp"
#include "common.hpp"

#include <algorithm>

namespace fa {

// K[c][a][b] = sum_q w_q k_cq |T| grad phi_a . grad phi_b + sum_q w_q m_cq |T| phi_a phi_b.
// With the reduced reference gradients R'_m = R_m - R_0 (sum_m grad lambda_m = 0)
// the first term is sum_{q,s} (w_q k_cq G_cs) B_qs[ab], G_cs = |T| grad
// lambda_m . grad lambda_n for the NS = TD (TD + 1) / 2 pairs s = (m, n) and
// B_qs = R'_am R'_bn (+ R'_an R'_bm for m != n): a product of a (cells x NQ NS)
// matrix by a (NQ NS x pairs) one that every cell shares.  Only the pairs
// a <= b are formed; the result is symmetric.
//
// A wave takes 16 cells (rows of the instruction) and up to NT tiles of 16
// pairs; both operands are formed in registers: w k from LDS times the lane's
// cell's G_cs, and the reference gradients of the lane's pair from LDS
// (NS products a point, used by NS instructions).  What bounds it is the FP64
// rate (the matrix and vector rates are the same on this chip): a kernel with
// a thread per (cell, row) spent its FP64 instructions on forming grad phi_b
// again for every row a and point.  A constant or per-cell coefficient needs
// no sum over points per cell: B is summed over q once a block (`cst`).  The
// results leave through LDS, CS cells at a time, as whole contiguous matrices.
// Tetrahedra P3, 663,552 cells, 35 points, k(x) and mass 1: 10.5 -> 1.56 ms (59
// GFLOP with the symmetry: 0.75 ms at the FP64 peak; 2.1 GB out: 0.4 ms).
// A separable coefficient is formed here too, but the caller does better to
// sample it first (fa_sep_sample, 0.28 ms): its registers crowd the
// accumulators' (1.88 ms).
using d4 = double __attribute__((ext_vector_type(4)));

template <int TD, int LDOF>
struct Em {
    static constexpr int NS = TD * (TD + 1) / 2;
    static constexpr int NP = LDOF * (LDOF + 1) / 2;
    static constexpr int TILES = (NP + 15) / 16;
    static constexpr int NW = TILES > 14 ? 3 : 1;  // waves that share 16 cells: 14 tiles of accumulators are 112 registers
    static constexpr int NT = (TILES + NW - 1) / NW;
    static constexpr int MT = LDOF > 20 ? 2 : 4;    // groups of 16 cells a block works on
    static constexpr int THREADS = 64 * NW * MT;
    static constexpr int CS = LDOF > 20 ? 2 : 4;   // matrices staged at a time (39 KB of LDS at P4)
    static constexpr int PADDED = NT * NW * 16;
    // LDS record of a cell: G, |T| and, to evaluate a separable coefficient, its vertices
    static constexpr int geo_doubles(bool sep) { return NS + 1 + (sep ? TD * (TD + 1) : 0); }
    static constexpr int QMAX = LDOF > 20 ? 56 : 64;  // points whose tables a block holds at once
};

// pair p of a <= b in row order: row a starts at a (2 LDOF + 1 - a) / 2
template <int LDOF>
__device__ inline void pair_of(int p, int& a, int& b) {
    const float m = 2 * LDOF + 1;
    a = static_cast<int>(0.5f * (m - sqrtf(m * m - 8.0f * static_cast<float>(p))));
    if (a * (2 * LDOF + 1 - a) / 2 > p) --a;  // the root rounded across a row's start
    if ((a + 1) * (2 * LDOF - a) / 2 <= p) ++a;
    b = a + p - a * (2 * LDOF + 1 - a) / 2;
}

// the pair's two indices, unpacked where they are used: kept apart over the
// point loop, the offsets of NT tiles would not fit the registers
__device__ inline void unpack(uint32_t ab, int& a, int& b) {
    asm volatile("" : "+v"(ab));
    a = static_cast<int>(ab & 0xffff);
    b = static_cast<int>(ab >> 16);
}

// reference gradient of basis function a at point q, reduced to lambda_1..
template <int TD, int LDOF>
__device__ inline double reduced(const double* __restrict__ gphi, int q, int a, int m) {
    const double* r = gphi + ((int64_t)q * LDOF + a) * (TD + 1);
    return r[m + 1] - r[0];
}

template <int TD, int LDOF, class T, bool SEP>
__global__ void __launch_bounds__((Em<TD, LDOF>::THREADS)) __attribute__((amdgpu_waves_per_eu(2))) k_element_matrices(
    const double* __restrict__ node, const int32_t* __restrict__ cell, int64_t nc, int nq, int qc,
    const double* __restrict__ qw, const double* __restrict__ phi, const double* __restrict__ gphi, int dk, double ds,
    const double* __restrict__ dc, int mk, double ms, const double* __restrict__ mc, T* __restrict__ elem) {
    using E = Em<TD, LDOF>;
    constexpr int NS = E::NS, NT = E::NT, NN = LDOF * LDOF;
    constexpr int GS = E::geo_doubles(SEP);
    extern __shared__ double lds[];
    const bool dpoint = dk >= FA_COEF_CELLQ, mpoint = mk >= FA_COEF_CELLQ;
    const bool dcell = dk && !dpoint, mcell = mk && !mpoint;
    const int kst = qc + 1;  // odd row stride of the point coefficients: qc is a multiple of 4
    double* rq = lds;                                          // [qc][LDOF][TD]
    double* ph = rq + (dpoint ? qc * LDOF * TD : 0);           // [qc][LDOF]
    double* cst = ph + (mpoint ? qc * LDOF : 0);               // [NS + 1][PADDED]
    double* geo = cst + ((dcell ? NS : 0) + (mcell ? 1 : 0)) * E::PADDED;  // [MT][16][GS]
    double* tile0 = geo + E::MT * 16 * GS;
    const int region = max(16 * kst * ((dpoint ? 1 : 0) + (mpoint ? 1 : 0)), E::CS * NN);
    const int wave = threadIdx.x / 64, lane = threadIdx.x % 64;
    const int mt = wave / E::NW, wn = wave % E::NW;
    const int tl = wn * 64 + lane;                             // thread within the 16 cells' waves
    double* mine = tile0 + mt * region;                        // point coefficients, then staged matrices
    double* kd = mine;
    double* km = mine + (dpoint ? 16 * kst : 0);
    double* g = geo + mt * 16 * GS;
    double* cstm = cst + (dcell ? NS * E::PADDED : 0);
    const int row = lane % 16, kq = lane / 16;                 // the lane's cell (A operand), k index and pair column

    uint32_t ab[NT];
#pragma unroll
    for (int t = 0; t < NT; ++t) {
        int a, b;
        pair_of<LDOF>(min((wn * NT + t) * 16 + row, E::NP - 1), a, b);
        ab[t] = static_cast<uint32_t>(a | (b << 16));
    }
    // tables of the first chunk of points, and the sums over all points of a per-cell coefficient
    auto stage = [&](int q0) {
        if (dpoint)
            for (int e = threadIdx.x; e < qc * LDOF * TD; e += E::THREADS) {
                const int q = q0 + e / (LDOF * TD), r = e % (LDOF * TD);
                rq[e] = q < nq ? reduced<TD, LDOF>(gphi, q, r / TD, r % TD) : 0.0;
            }
        if (mpoint)
            for (int e = threadIdx.x; e < qc * LDOF; e += E::THREADS)
                ph[e] = q0 + e / LDOF < nq ? phi[(int64_t)q0 * LDOF + e] : 0.0;
    };
    stage(0);
    if (dcell || mcell) {
        for (int p = threadIdx.x; p < E::PADDED; p += E::THREADS) {
            int a, b;
            pair_of<LDOF>(min(p, E::NP - 1), a, b);
            if (dcell) {
                // four points at a time, then added with what the last addition's
                // rounding left out: every cell multiplies the same sums, whose
                // errors would not average out (P2 tetrahedra 20^3, against 64
                // bits: 4.5e-16 -> 3.5e-16; 3.3e-16 summed cell by cell)
                double s[NS], r[NS];
#pragma unroll
                for (int u = 0; u < NS; ++u) s[u] = r[u] = 0.0;
                auto point = [&](int q) {
                    int u = 0;
#pragma unroll
                    for (int m = 0; m < TD; ++m)
#pragma unroll
                        for (int n = m; n < TD; ++n, ++u) {
                            const double x = reduced<TD, LDOF>(gphi, q, a, m) * reduced<TD, LDOF>(gphi, q, b, n);
                            const double y = reduced<TD, LDOF>(gphi, q, a, n) * reduced<TD, LDOF>(gphi, q, b, m);
                            r[u] += qw[q] * (m == n ? x : x + y);
                        }
                };
                int q = 0;
                for (; q + 4 <= nq; q += 4) {
#pragma unroll
                    for (int k = 0; k < 4; ++k) point(q + k);
#pragma unroll
                    for (int u = 0; u < NS; ++u) {
                        const double sum = s[u] + r[u];
                        r[u] -= sum - s[u];
                        s[u] = sum;
                    }
                }
                for (; q < nq; ++q) point(q);
#pragma unroll
                for (int u = 0; u < NS; ++u) s[u] += r[u];
#pragma unroll
                for (int u = 0; u < NS; ++u) cst[u * E::PADDED + p] = s[u];
            }
            if (mcell) {
                double s = 0.0, r = 0.0;
                for (int q = 0; q < nq; ++q) {
                    r += qw[q] * phi[(int64_t)q * LDOF + a] * phi[(int64_t)q * LDOF + b];
                    if (q % 4 == 3) {
                        const double sum = s + r;
                        r -= sum - s;
                        s = sum;
                    }
                }
                s += r;
                cstm[p] = s;
            }
        }
    }
    __syncthreads();
    // the waves of one group of cells wait for each other; a lone wave only for its own LDS traffic
    auto group_sync = [&]() {
        if constexpr (E::NW > 1) {
            __syncthreads();
        } else {
            __builtin_amdgcn_wave_barrier();
            __builtin_amdgcn_fence(__ATOMIC_SEQ_CST, "wavefront");
        }
    };
    const int64_t groups = (nc + 16 * E::MT - 1) / (16 * E::MT);
    for (int64_t gr = blockIdx.x; gr < groups; gr += gridDim.x) {
        const int64_t c0 = (gr * E::MT + mt) * 16;
        const int nb = static_cast<int>(c0 >= nc ? 0 : (nc - c0 < 16 ? nc - c0 : 16));
        group_sync();
        if (tl < 16) {
            double p[TD + 1][TD];
            load_cell<TD>(node, cell, c0 + tl < nc ? c0 + tl : nc - 1, p);
            Geom<TD> ge;
            ge.compute(p);
            int u = 0;
#pragma unroll
            for (int m = 0; m < TD; ++m)
#pragma unroll
                for (int n = m; n < TD; ++n, ++u) {
                    double s = 0.0;
#pragma unroll
                    for (int d = 0; d < TD; ++d) s += ge.gl[m + 1][d] * ge.gl[n + 1][d];
                    g[tl * GS + u] = ge.meas * s;
                }
            g[tl * GS + NS] = ge.meas;
            if constexpr (SEP) {
#pragma unroll
                for (int v = 0; v < TD + 1; ++v)
#pragma unroll
                    for (int d = 0; d < TD; ++d) g[tl * GS + NS + 1 + v * TD + d] = p[v][d];
            }
        }
        group_sync();
        double G[NS];
#pragma unroll
        for (int u = 0; u < NS; ++u) G[u] = g[row * GS + u];
        const double meas = g[row * GS + NS];
        // w k and w m of the cells' points from q0 on, 0 past the rule's end
        auto fill = [&](int q0) {
            for (int e = tl; e < 16 * qc; e += 64 * E::NW) {
                const int cl = e / qc, q = q0 + e - cl * qc;
                const int64_t c = c0 + cl < nc ? c0 + cl : nc - 1;
                double vd = 0.0, vm = 0.0;
                if (q < nq) {
                    double p[TD + 1][TD];
                    if constexpr (SEP) {
#pragma unroll
                        for (int v = 0; v < TD + 1; ++v)
#pragma unroll
                            for (int d = 0; d < TD; ++d) p[v][d] = g[cl * GS + NS + 1 + v * TD + d];
                    }
                    const double w = qw[q];
                    if (dpoint) vd = w * coef_at<TD, SEP>(dk, ds, dc, c, c, q, nq, p);
                    if (mpoint) vm = w * coef_at<TD, SEP>(mk, ms, mc, c, c, q, nq, p);
                }
                if (dpoint) kd[cl * kst + q - q0] = vd;
                if (mpoint) km[cl * kst + q - q0] = vm;
            }
            group_sync();
        };
        // the first points before the accumulators are live (evaluating a
        // separable coefficient takes most of the registers)
        if (dpoint || mpoint) {
            if (nq > qc && gr != (int64_t)blockIdx.x) {  // uniform over the block
                __syncthreads();
                stage(0);
                __syncthreads();
            }
            fill(0);
        }
        d4 acc[NT];
#pragma unroll
        for (int t = 0; t < NT; ++t) acc[t] = d4{0.0, 0.0, 0.0, 0.0};
        if (dpoint || mpoint) {
            for (int q0 = 0; q0 < nq; q0 += qc) {
                if (q0 > 0) {  // uniform over the block
                    __syncthreads();
                    stage(q0);
                    __syncthreads();
                    fill(q0);
                }
                const int steps = (min(qc, nq - q0) + 3) / 4;
                if (dpoint) {
                    for (int j = 0; j < steps; ++j) {
                        const double k = kd[row * kst + 4 * j + kq];
                        double A[NS];
#pragma unroll
                        for (int u = 0; u < NS; ++u) A[u] = k * G[u];
                        const double* r = rq + (4 * j + kq) * LDOF * TD;
                        // the next tile's gradients are read before this tile's products, no
                        // further ahead (all tiles' at once would not fit the registers)
                        double x[2][TD], y[2][TD];
                        int a, b;
                        unpack(ab[0], a, b);
#pragma unroll
                        for (int m = 0; m < TD; ++m) {
                            x[0][m] = r[a * TD + m];
                            y[0][m] = r[b * TD + m];
                        }
#pragma unroll
                        for (int t = 0; t < NT; ++t) {
                            if (t + 1 < NT) {
                                unpack(ab[t + 1 < NT ? t + 1 : t], a, b);
#pragma unroll
                                for (int m = 0; m < TD; ++m) {
                                    x[(t + 1) & 1][m] = r[a * TD + m];
                                    y[(t + 1) & 1][m] = r[b * TD + m];
                                }
                            }
                            const double(&xt)[TD] = x[t & 1];
                            const double(&yt)[TD] = y[t & 1];
                            int u = 0;
#pragma unroll
                            for (int m = 0; m < TD; ++m)
#pragma unroll
                                for (int n = m; n < TD; ++n, ++u) {
                                    const double B = m == n ? xt[m] * yt[m] : xt[m] * yt[n] + xt[n] * yt[m];
                                    acc[t] = __builtin_amdgcn_mfma_f64_16x16x4f64(A[u], B, acc[t], 0, 0, 0);
                                }
                            __builtin_amdgcn_sched_barrier(0);
                        }
                    }
                }
                if (mpoint) {
                    for (int j = 0; j < steps; ++j) {
                        const double A = km[row * kst + 4 * j + kq] * meas;
                        const double* r = ph + (4 * j + kq) * LDOF;
#pragma unroll
                        for (int t = 0; t < NT; ++t) {
                            int a, b;
                            unpack(ab[t], a, b);
                            acc[t] = __builtin_amdgcn_mfma_f64_16x16x4f64(A, r[a] * r[b], acc[t], 0, 0, 0);
                            if (t % 4 == 3) __builtin_amdgcn_sched_barrier(0);
                        }
                    }
                }
                group_sync();  // kd, km are written again (or staged over)
            }
        }
        // register r of a lane holds cell 4 r + lane / 16
#pragma unroll
        for (int r = 0; r < 4; ++r) {
            const int cl = 4 * r + kq;
            if (dcell || mcell) {
                const int64_t c = c0 + cl < nc ? c0 + cl : nc - 1;
                const double kc = dcell ? coef_value(dk, ds, dc, c, 0, nq) : 0.0;
                const double mcv = mcell ? coef_value(mk, ms, mc, c, 0, nq) * g[cl * GS + NS] : 0.0;
                double H[NS];
#pragma unroll
                for (int u = 0; u < NS; ++u) H[u] = kc * g[cl * GS + u];
#pragma unroll
                for (int t = 0; t < NT; ++t) {
                    const int p = (wn * NT + t) * 16 + row;
                    double v = acc[t][r];
                    if (dcell) {
#pragma unroll
                        for (int u = 0; u < NS; ++u) v += H[u] * cst[u * E::PADDED + p];
                    }
                    if (mcell) v += mcv * cstm[p];
                    acc[t][r] = v;
                    __builtin_amdgcn_sched_barrier(0);
                }
            }
#pragma unroll
            for (int h = 0; h < 4 / E::CS; ++h) {
                if (kq / E::CS == h) {
#pragma unroll
                    for (int t = 0; t < NT; ++t) {
                        if ((wn * NT + t) * 16 + row < E::NP) {
                            int a, b;
                            unpack(ab[t], a, b);
                            double* o = mine + (kq % E::CS) * NN;
                            o[a * LDOF + b] = acc[t][r];
                            o[b * LDOF + a] = acc[t][r];
                        }
                    }
                }
                group_sync();
                const int first = 4 * r + h * E::CS;
                const int cnt = max(0, min(E::CS, nb - first)) * NN;
                T* o = elem + (c0 + first) * NN;
                for (int e = tl; e < cnt; e += 64 * E::NW) o[e] = static_cast<T>(mine[e]);
                group_sync();
            }
        }
    }
}

template <int TD, int LDOF, class T>
static int launch_elem(const double* node, const int32_t* cell, int64_t nc, int nq, const double* qw,
                       const double* phi, const double* gphi, int dk, double ds, const double* dc, int mk, double ms,
                       const double* mc, void* elem, hipStream_t s) {
    using E = Em<TD, LDOF>;
    const bool dpoint = dk >= FA_COEF_CELLQ, mpoint = mk >= FA_COEF_CELLQ;
    const int qc = dpoint || mpoint ? std::min(E::QMAX, (nq + 3) / 4 * 4) : 0;
    const size_t region = std::max<size_t>(16 * (qc + 1) * ((dpoint ? 1 : 0) + (mpoint ? 1 : 0)), E::CS * LDOF * LDOF);
    const size_t lds = sizeof(double) * ((dpoint ? qc * LDOF * TD : 0) + (mpoint ? qc * LDOF : 0) +
                                         ((dk && !dpoint ? E::NS : 0) + (mk && !mpoint ? 1 : 0)) * E::PADDED +
                                         E::MT * 16 * E::geo_doubles(dk == FA_COEF_SEP || mk == FA_COEF_SEP) + E::MT * region);
    // a block keeps its tables over its groups of cells: no more blocks than stay resident
    const int resident = std::max<int>(1, std::min<int>(static_cast<int>(160 * 1024 / lds), 2048 / E::THREADS));
    const unsigned grid = grid_for(nc, 16 * E::MT, 256 * resident);
    if (dk == FA_COEF_SEP || mk == FA_COEF_SEP) {
        auto k = k_element_matrices<TD, LDOF, T, true>;
        if (lds > 64 * 1024) FA_HIP(hipFuncSetAttribute(reinterpret_cast<const void*>(k), hipFuncAttributeMaxDynamicSharedMemorySize,
                                   static_cast<int>(lds)));
        hipLaunchKernelGGL(k, dim3(grid), dim3(E::THREADS), lds, s, node, cell, nc, nq, qc, qw, phi, gphi, dk, ds, dc,
                           mk, ms, mc, static_cast<T*>(elem));
    } else {
        auto k = k_element_matrices<TD, LDOF, T, false>;
        if (lds > 64 * 1024) FA_HIP(hipFuncSetAttribute(reinterpret_cast<const void*>(k), hipFuncAttributeMaxDynamicSharedMemorySize,
                                   static_cast<int>(lds)));
        hipLaunchKernelGGL(k, dim3(grid), dim3(E::THREADS), lds, s, node, cell, nc, nq, qc, qw, phi, gphi, dk, ds, dc,
                           mk, ms, mc, static_cast<T*>(elem));
    }
    FA_LAUNCH("k_element_matrices");
    return FA_OK;
}

template <class T>
static int dispatch_elem(int td, int ldof, const double* node, const int32_t* cell, int64_t nc, int nq,
                         const double* qw, const double* phi, const double* gphi, int dk, double ds, const double* dc,
                         int mk, double ms, const double* mc, void* elem, hipStream_t s) {
#define FA_ELEM_CASE(TD_, L_)         \
    if (td == TD_ && ldof == L_)      \
        return launch_elem<TD_, L_, T>(node, cell, nc, nq, qw, phi, gphi, dk, ds, dc, mk, ms, mc, elem, s)
    FA_ELEM_CASE(2, 3);
    FA_ELEM_CASE(2, 6);
    FA_ELEM_CASE(2, 10);
    FA_ELEM_CASE(2, 15);
    FA_ELEM_CASE(3, 4);
    FA_ELEM_CASE(3, 10);
    FA_ELEM_CASE(3, 20);
    FA_ELEM_CASE(3, 35);
#undef FA_ELEM_CASE
    set_error("fa_element_matrices: unsupported (td=%d, ldof=%d); p must be 1..4", td, ldof);
    return FA_EINVAL;
}

}  // namespace fa

using namespace fa;

extern "C" int fa_element_matrices(int dtype, int td, int ldof, int nq, const double* node, const int32_t* cell,
                                   int64_t nc, const double* qw, const double* phi, const double* gphi_u,
                                   int diff_kind, double diff_scale, const double* diff_coef, int mass_kind,
                                   double mass_scale, const double* mass_coef, void* elem, fa_stream_t stream) {
    FA_REQUIRE(dtype == FA_F64 || dtype == FA_F32, "fa_element_matrices: bad dtype %d", dtype);
    FA_REQUIRE(nq > 0 && nc >= 0, "fa_element_matrices: bad sizes");
    FA_REQUIRE(!diff_kind || gphi_u, "fa_element_matrices: diffusion needs gphi_u");
    FA_REQUIRE(!mass_kind || phi, "fa_element_matrices: mass needs phi");
    FA_REQUIRE(!(diff_kind >= FA_COEF_CELL && !diff_coef) && !(mass_kind >= FA_COEF_CELL && !mass_coef),
               "fa_element_matrices: coefficient array missing");
    if (nc == 0) return FA_OK;
    if (dtype == FA_F64)
        return dispatch_elem<double>(td, ldof, node, cell, nc, nq, qw, phi, gphi_u, diff_kind, diff_scale, diff_coef,
                                     mass_kind, mass_scale, mass_coef, elem, S(stream));
    return dispatch_elem<float>(td, ldof, node, cell, nc, nq, qw, phi, gphi_u, diff_kind, diff_scale, diff_coef,
                                mass_kind, mass_scale, mass_coef, elem, S(stream));
}
