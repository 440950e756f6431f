// Element vectors of a scalar source on simplices, and their fixed-order sum.
#include "cell.hpp"
#include "common.hpp"
#include "sep_plan.hpp"

#include <algorithm>

namespace fa {

// Element vectors: out[c][i] = sum_q (w_q |T| f(x_cq)) phi_i(q), q ascending.
// A block takes `cb` cells at a time.  Phase 1, a thread per (cell, point):
// w_q |T| f into LDS.  Phase 2, a thread per (row i, EV_ACC cells): the sums
// over the points, one phi load for the EV_ACC cells.  What bounds it is the
// source: a kernel with a thread per (cell, i) evaluated every point once per
// row (20 times at P3, 35 at P4) and every repeated factor of a term again.
// Tetrahedra P3, 663,552 cells, 35 points, six-term source: 21.9 -> 0.91 ms,
// 0.37 ms of it VALU issue (618 instructions a point wave), the rest latency
// at 3 waves a SIMD (the table of factor values takes 36 KB of LDS a block).
constexpr int EV_ACC = 4;        // cells a thread sums in phase 2
constexpr int EV_CELLS = 64;     // most cells a block takes at once
constexpr int EV_POINTS = 1280;  // (cell, point) values staged at once: five rounds of the block

template <int TD, class T, bool SEP>
__global__ void __launch_bounds__(256) k_element_vectors(const double* __restrict__ node, const int32_t* __restrict__ cell,
                                                        int64_t nc, int ldof, int nq, int cb, int qc,
                                                        const double* __restrict__ qw, const double* __restrict__ phi,
                                                        int sk, double ss, const double* __restrict__ src,
                                                        T* __restrict__ elem) {
    __shared__ double sp[EV_CELLS][TD + 1][TD];
    __shared__ double smeas[EV_CELLS];
    __shared__ double sf[EV_POINTS];
    __shared__ double sval[SEP ? SEP_COLS * 256 : 1];
    __shared__ SepPlan plan;
    const fa_sep_t* se = reinterpret_cast<const fa_sep_t*>(src);
    if constexpr (SEP) {
        sep_plan(se, plan);
        sep_ones<256>(sval);
    }
    const int width = min(ldof, 256), groups = 256 / width;
    const int lane_i = threadIdx.x % width, g = threadIdx.x / width;
    for (int64_t c0 = (int64_t)blockIdx.x * cb; c0 < nc; c0 += (int64_t)gridDim.x * cb) {
        const int nb = static_cast<int>(nc - c0 < cb ? nc - c0 : cb);
        __syncthreads();  // the previous batch's sums (and the plan)
        if (threadIdx.x < nb) {
            double p[TD + 1][TD];
            load_cell<TD>(node, cell, c0 + threadIdx.x, p);
            Geom<TD> geo;
            geo.compute(p);
#pragma unroll
            for (int v = 0; v < TD + 1; ++v)
#pragma unroll
                for (int d = 0; d < TD; ++d) sp[threadIdx.x][v][d] = p[v][d];
            smeas[threadIdx.x] = geo.meas;
        }
        for (int i0 = 0; i0 < ldof; i0 += 256) {
            const int i = i0 + lane_i;
            const bool act = i < ldof && g < groups;
            double acc[EV_ACC];
#pragma unroll
            for (int u = 0; u < EV_ACC; ++u) acc[u] = 0.0;
            for (int q0 = 0; q0 < nq; q0 += qc) {
                const int nqc = min(qc, nq - q0);
                __syncthreads();  // the cells' geometry, or the previous points' sums
                for (int t = threadIdx.x; t < nb * nqc; t += 256) {
                    const int cl = t / nqc, q = q0 + t - cl * nqc;
                    double f;
                    if constexpr (SEP) {
                        double x[TD];
#pragma unroll
                        for (int d = 0; d < TD; ++d) x[d] = 0.0;
#pragma unroll
                        for (int v = 0; v < TD + 1; ++v) {
                            const double w = se->bcs[q * (TD + 1) + v];
#pragma unroll
                            for (int d = 0; d < TD; ++d) x[d] += w * sp[cl][v][d];
                        }
                        f = ss * (plan.fits ? sep_value_planned<TD, 256>(se, plan, x, c0 + cl, sval)
                                            : sep_value<TD>(se, q, sp[cl], c0 + cl));
                    } else {
                        f = coef_value(sk, ss, src, c0 + cl, q, nq);
                    }
                    sf[t] = qw[q] * smeas[cl] * f;
                }
                __syncthreads();
                if (act) {
#pragma unroll 5
                    for (int q = 0; q < nqc; ++q) {
                        const double ph = phi[(int64_t)(q0 + q) * ldof + i];
#pragma unroll
                        for (int u = 0; u < EV_ACC; ++u) {
                            const int cl = min(g + u * groups, nb - 1);
                            acc[u] += sf[cl * nqc + q] * ph;
                        }
                    }
                }
            }
            if (act) {
#pragma unroll
                for (int u = 0; u < EV_ACC; ++u) {
                    const int cl = g + u * groups;
                    if (cl < nb) elem[(c0 + cl) * ldof + i] = static_cast<T>(acc[u]);
                }
            }
        }
    }
}

// out[c][q] = f(x_cq): a thread per point, the block's cells' vertices in LDS
template <int TD>
__global__ void __launch_bounds__(256) k_sep_sample(const double* __restrict__ node, const int32_t* __restrict__ cell,
                                                   int64_t nc, int nq, int cb, const fa_sep_t* __restrict__ se,
                                                   double* __restrict__ out) {
    __shared__ double sp[EV_CELLS][TD + 1][TD];
    __shared__ double sval[SEP_COLS * 256];
    __shared__ SepPlan plan;
    sep_plan(se, plan);
    sep_ones<256>(sval);
    for (int64_t c0 = (int64_t)blockIdx.x * cb; c0 < nc; c0 += (int64_t)gridDim.x * cb) {
        const int nb = static_cast<int>(nc - c0 < cb ? nc - c0 : cb);
        __syncthreads();
        if (threadIdx.x < nb) {
            double p[TD + 1][TD];
            load_cell<TD>(node, cell, c0 + threadIdx.x, p);
#pragma unroll
            for (int v = 0; v < TD + 1; ++v)
#pragma unroll
                for (int d = 0; d < TD; ++d) sp[threadIdx.x][v][d] = p[v][d];
        }
        __syncthreads();
        for (int t = threadIdx.x; t < nb * nq; t += 256) {
            const int cl = t / nq, q = t - cl * nq;
            double f;
            if (plan.fits) {
                double x[TD];
#pragma unroll
                for (int d = 0; d < TD; ++d) x[d] = 0.0;
#pragma unroll
                for (int v = 0; v < TD + 1; ++v) {
                    const double w = se->bcs[q * (TD + 1) + v];
#pragma unroll
                    for (int d = 0; d < TD; ++d) x[d] += w * sp[cl][v][d];
                }
                f = sep_value_planned<TD, 256>(se, plan, x, c0 + cl, sval);
            } else {
                f = sep_value<TD>(se, q, sp[cl], c0 + cl);
            }
            out[c0 * nq + t] = f;
        }
    }
}

// 4 lanes per DOF, lane l adds incidences l, l+4, ...; the lane partials are
// combined by a fixed tree (deterministic).  A P2-P4 row has 4 to 8
// incidences on average (an interior DOF of a cell has one), so 16 lanes a
// row left three in four idle: 164 -> 117 us at 3.05M P3 rows.
template <class T>
__global__ void __launch_bounds__(256) k_gather_vector(int64_t gdof, const int32_t* __restrict__ ptr,
                                                      const int32_t* __restrict__ adj, const T* __restrict__ elem,
                                                      T* __restrict__ out) {
    constexpr int G = 4;
    const int lane = threadIdx.x % G;
    for (int64_t r = (blockIdx.x * (int64_t)blockDim.x + threadIdx.x) / G; r < gdof;
         r += (int64_t)gridDim.x * blockDim.x / G) {
        T s = T(0);
        const int32_t k1 = ptr[r + 1];
        for (int32_t k = ptr[r] + lane; k < k1; k += G) s += elem[adj[k]];
        s = group_sum<G>(s);
        if (lane == 0) out[r] = s;
    }
}

template <int TD, class T>
static void launch_vectors(const double* node, const int32_t* cell, int64_t nc, int ldof, int nq, const double* qw,
                           const double* phi, int sk, double ss, const double* src, void* elem, hipStream_t s) {
    const int groups = 256 / std::min(ldof, 256);
    const int cb = std::max(1, std::min({EV_CELLS, EV_ACC * groups, EV_POINTS / std::min(nq, EV_POINTS)}));
    const int qc = std::min(nq, EV_POINTS / cb);
    // a block keeps its plan over its batches: no more blocks than stay resident
    const unsigned grid = grid_for(nc, cb, sk == FA_COEF_SEP ? 256 * 6 : 1 << 20);
    if (sk == FA_COEF_SEP)
        hipLaunchKernelGGL((k_element_vectors<TD, T, true>), dim3(grid), dim3(256), 0, s, node, cell, nc, ldof, nq, cb,
                           qc, qw, phi, sk, ss, src, static_cast<T*>(elem));
    else
        hipLaunchKernelGGL((k_element_vectors<TD, T, false>), dim3(grid), dim3(256), 0, s, node, cell, nc, ldof, nq,
                           cb, qc, qw, phi, sk, ss, src, static_cast<T*>(elem));
}

}  // namespace fa

using namespace fa;

extern "C" int fa_element_vectors(int dtype, int td, int ldof, int nq, const double* node, const int32_t* cell,
                                  int64_t nc, const double* qw, const double* phi, int src_kind, double src_scale,
                                  const double* src, void* elem, fa_stream_t stream) {
    FA_REQUIRE(dtype == FA_F64 || dtype == FA_F32, "fa_element_vectors: bad dtype %d", dtype);
    FA_REQUIRE(td == 2 || td == 3, "fa_element_vectors: td must be 2 or 3");
    FA_REQUIRE(ldof > 0 && nq > 0 && nc >= 0, "fa_element_vectors: bad sizes");
    FA_REQUIRE(src_kind < FA_COEF_CELL || src, "fa_element_vectors: source array missing");
    if (nc == 0) return FA_OK;
    hipStream_t s = S(stream);
    if (dtype == FA_F64) {
        if (td == 2) launch_vectors<2, double>(node, cell, nc, ldof, nq, qw, phi, src_kind, src_scale, src, elem, s);
        else launch_vectors<3, double>(node, cell, nc, ldof, nq, qw, phi, src_kind, src_scale, src, elem, s);
    } else {
        if (td == 2) launch_vectors<2, float>(node, cell, nc, ldof, nq, qw, phi, src_kind, src_scale, src, elem, s);
        else launch_vectors<3, float>(node, cell, nc, ldof, nq, qw, phi, src_kind, src_scale, src, elem, s);
    }
    FA_LAUNCH("k_element_vectors");
    return FA_OK;
}

extern "C" int fa_sep_sample(int td, int nq, const double* node, const int32_t* cell, int64_t nc, const void* sep,
                             double* out, fa_stream_t stream) {
    FA_REQUIRE(td == 2 || td == 3, "fa_sep_sample: td must be 2 or 3");
    FA_REQUIRE(nq > 0 && nc >= 0, "fa_sep_sample: bad sizes");
    if (nc == 0) return FA_OK;  // an empty array may have no address
    FA_REQUIRE(sep && out, "fa_sep_sample: bad arguments");
    const int cb = std::max(1, std::min(EV_CELLS, EV_POINTS / nq));
    const unsigned grid = grid_for(nc, cb, 256 * 8);
    const auto* se = static_cast<const fa_sep_t*>(sep);
    if (td == 2)
        hipLaunchKernelGGL(k_sep_sample<2>, dim3(grid), dim3(256), 0, S(stream), node, cell, nc, nq, cb, se, out);
    else
        hipLaunchKernelGGL(k_sep_sample<3>, dim3(grid), dim3(256), 0, S(stream), node, cell, nc, nq, cb, se, out);
    FA_LAUNCH("k_sep_sample");
    return FA_OK;
}

extern "C" int fa_gather_vector(int dtype, int64_t gdof, int32_t ldof, const int32_t* adj_ptr, const int32_t* adj,
                                const void* elem, void* out, fa_stream_t stream) {
    (void)ldof;
    FA_REQUIRE(dtype == FA_F64 || dtype == FA_F32, "fa_gather_vector: bad dtype %d", dtype);
    hipStream_t s = S(stream);
    const unsigned grid = grid_for(gdof * 4, 256, 1 << 20);
    if (dtype == FA_F64)
        hipLaunchKernelGGL(k_gather_vector<double>, dim3(grid), dim3(256), 0, s, gdof, adj_ptr, adj,
                           static_cast<const double*>(elem), static_cast<double*>(out));
    else
        hipLaunchKernelGGL(k_gather_vector<float>, dim3(grid), dim3(256), 0, s, gdof, adj_ptr, adj,
                           static_cast<const float*>(elem), static_cast<float*>(out));
    FA_LAUNCH("k_gather_vector");
    return FA_OK;
}
