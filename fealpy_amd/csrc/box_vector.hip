// P1 load vector of a separable source on a from_box tensor grid, one pass.
#include "box.hpp"
#include "common.hpp"

#include <algorithm>

namespace fa {

// A block takes a BV_Y x BV_Z tile of cubes and marches along x.  At each plane
// a thread forms the element vectors of its cube's 6 tetrahedra into LDS (24
// values, cube index fastest), then the sums of its node: the plane's cubes are
// the last four of the eight around the nodes at its low side and the first
// four of those at its high side, in ascending cell order, so a node's partial
// sum waits one plane in a register.  What bounds it is the field, read once
// (100 MB at 128^3): the form with a pass per cube and a pass per node moved
// the element vectors through memory as well (403 MB, twice).  Tiles overlap by
// one cube (8 x 32 cubes: 18% of them formed twice), chunks of the march by one
// plane.  128^3, field times three factors: 332 us in two passes -> 76 us
// (117 MB: 1.5 TB/s).
constexpr int BV_Y = 8, BV_Z = 32;

// a node's cells in one plane of cubes (A = 1: the plane on its low side)
template <int A>
__device__ inline double node_sum(const double (*v)[BV_Y * BV_Z], int at, double acc) {
    // cubes (b, c) = (1,1), (1,0), (0,1), (0,0) below the node at (y + b, z + c) of the tile
#pragma unroll
    for (int bc = 0; bc < 4; ++bc) {
        const int b = bc < 2 ? 1 : 0, c = bc % 2 ? 0 : 1;
        const int cube = at + (1 - b) * BV_Z + (1 - c);
#pragma unroll
        for (int t = 0; t < 6; ++t) {
            const int i = box_local(t, box_corner_of(A, b, c));
            if (i >= 0) acc += v[4 * t + i][cube];
        }
    }
    return acc;
}

template <class T>
__global__ void __launch_bounds__(256) k_p1_box_vector(int nx, int ny, int nz, int span, const double* __restrict__ axes,
                                                       int nq, const double* __restrict__ qw,
                                                       const double* __restrict__ phi, double ss,
                                                       const fa_sep_t* __restrict__ e, const double* __restrict__ tab,
                                                       int nmax, T* __restrict__ out) {
    __shared__ double vec[24][BV_Y * BV_Z];
    const int ly = threadIdx.x / BV_Z, lz = threadIdx.x % BV_Z, gz = nz / (BV_Z - 1) + 1;
    const int by = static_cast<int>(blockIdx.x) / gz, bz = static_cast<int>(blockIdx.x) - by * gz;
    const int iy = by * (BV_Y - 1) + ly, iz = bz * (BV_Z - 1) + lz;  // the thread's node
    const int cy = iy - 1, cz = iz - 1;                                              // the thread's cube
    const bool cube = cy >= 0 && cy < ny && cz >= 0 && cz < nz;
    const bool owns = ly < BV_Y - 1 && lz < BV_Z - 1 && iy <= ny && iz <= nz;
    const int x0 = blockIdx.y * span, x1 = min(x0 + span, nx + 1);
    const double hy = cube ? axes[nx + 2 + cy] - axes[nx + 1 + cy] : 0.0;
    const double hz = cube ? axes[nx + ny + 3 + cz] - axes[nx + ny + 2 + cz] : 0.0;
    const int nt = e->nterms;
    // one term at the four-point rule (the usual source): the factors along y
    // and z stay in registers over the march, those along x are the block's
    const bool one = nt == 1 && nq == 4;
    double yz[24];
    if (one && cube) {
#pragma unroll
        for (int u = 0; u < 24; ++u) yz[u] = e->coef[0];
        for (int k = 0; k < e->term_end[0]; ++k) {
            const int d = e->dim[k];
            if (d == 0) continue;
            const double4* r = reinterpret_cast<const double4*>(tab + ((int64_t)k * nmax + (d == 1 ? cy : cz)) * 24);
#pragma unroll
            for (int t = 0; t < 6; ++t) {
                const double4 w = r[t];
                yz[4 * t] *= w.x;
                yz[4 * t + 1] *= w.y;
                yz[4 * t + 2] *= w.z;
                yz[4 * t + 3] *= w.w;
            }
        }
    }
    double part = 0.0;
    for (int cx = x0 - 1; cx < x1; ++cx) {
        if (cube && cx >= 0 && cx < nx) {
            const double vol = (axes[cx + 1] - axes[cx]) * hy * hz / 6.0;
            const int64_t c0 = 6 * (((int64_t)cx * ny + cy) * nz + cz);
            if (one) {
                double f[24];
                const double* fld = e->field[0];
                double fc[6];
#pragma unroll
                for (int t = 0; t < 6; ++t) fc[t] = fld ? fld[c0 + t] : 1.0;
#pragma unroll
                for (int u = 0; u < 24; ++u) f[u] = yz[u];
                for (int k = 0; k < e->term_end[0]; ++k) {
                    if (e->dim[k] != 0) continue;
                    const double* r = tab + ((int64_t)k * nmax + cx) * 24;  // the same for the whole block
#pragma unroll
                    for (int u = 0; u < 24; ++u) f[u] *= r[u];
                }
#pragma unroll
                for (int t = 0; t < 6; ++t) {
                    const double m = box_sign(t) * vol * (ss * fc[t]);
                    double v[4] = {0.0, 0.0, 0.0, 0.0};
#pragma unroll
                    for (int q = 0; q < 4; ++q) {
                        const double fq = qw[q] * m * f[4 * t + q];
#pragma unroll
                        for (int i = 0; i < 4; ++i) v[i] += fq * phi[q * 4 + i];
                    }
#pragma unroll
                    for (int i = 0; i < 4; ++i) vec[4 * t + i][threadIdx.x] = v[i];
                }
            } else {
#pragma unroll
                for (int t = 0; t < 6; ++t) {
                    const double m = box_sign(t) * vol;
                    double v[4] = {0.0, 0.0, 0.0, 0.0};
                    for (int q = 0; q < nq; ++q) {
                        double f = 0.0;
                        int k = 0;
                        for (int s = 0; s < nt; ++s) {
                            double p = e->coef[s];
                            const double* fld = e->field[s];
                            if (fld) p *= fld[c0 + t];
                            const int kend = e->term_end[s];
                            for (; k < kend; ++k) {
                                const int d = e->dim[k];
                                const int i = d == 0 ? cx : (d == 1 ? cy : cz);
                                p *= tab[(((int64_t)k * nmax + i) * 6 + t) * nq + q];
                            }
                            f += p;
                        }
                        const double fq = qw[q] * m * (ss * f);
#pragma unroll
                        for (int i = 0; i < 4; ++i) v[i] += fq * phi[q * 4 + i];
                    }
#pragma unroll
                    for (int i = 0; i < 4; ++i) vec[4 * t + i][threadIdx.x] = v[i];
                }
            }
        } else {
#pragma unroll
            for (int u = 0; u < 24; ++u) vec[u][threadIdx.x] = 0.0;
        }
        __syncthreads();
        if (owns) {
            const double sum = node_sum<0>(vec, threadIdx.x, part);
            if (cx >= x0) out[((int64_t)cx * (ny + 1) + iy) * (nz + 1) + iz] = static_cast<T>(sum);
            part = node_sum<1>(vec, threadIdx.x, 0.0);
        }
        __syncthreads();
    }
}

static size_t table_offset(int nx, int ny, int nz) {
    return align_up(sizeof(double) * (static_cast<size_t>(nx) + ny + nz + 3), 32);
}

}  // namespace fa

using namespace fa;

extern "C" size_t fa_p1_box_vector_tensor_work_bytes(int nx, int ny, int nz, int nq) {
    const size_t nmax = static_cast<size_t>(std::max(nx, std::max(ny, nz)));
    return table_offset(nx, ny, nz) + sizeof(double) * FA_SEP_MAX_FACTORS * nmax * 6 * static_cast<size_t>(std::max(nq, 0));
}

extern "C" int fa_p1_box_vector_tensor(int dtype, int nx, int ny, int nz, const double* node_wide, const double* axes,
                                       int nq, const double* qw, const double* phi, double scale, const void* sep,
                                       void* out, void* work, size_t work_bytes, fa_stream_t stream) {
    FA_REQUIRE(dtype == FA_F64 || dtype == FA_F32, "fa_p1_box_vector_tensor: bad dtype %d", dtype);
    FA_REQUIRE(nx >= 1 && ny >= 1 && nz >= 1 && nq > 0 && node_wide && axes && qw && phi && sep && out && work,
               "fa_p1_box_vector_tensor: bad arguments");
    const int64_t nn = static_cast<int64_t>(nx + 1) * (ny + 1) * (nz + 1), nc = 6 * static_cast<int64_t>(nx) * ny * nz;
    FA_REQUIRE(nn < INT32_MAX && nc < INT32_MAX, "fa_p1_box_vector_tensor: grid too large for int32 indices");
    const size_t need = fa_p1_box_vector_tensor_work_bytes(nx, ny, nz, nq);
    FA_REQUIRE(work_bytes >= need && (reinterpret_cast<uintptr_t>(work) & 31) == 0,
               "fa_p1_box_vector_tensor: workspace of %zu bytes (32-byte aligned) too small, %zu needed", work_bytes,
               need);
    // tiles along one grid dimension, which takes 2^24 blocks of 256 threads: a
    // grid with more has over 2^31 nodes or 270 GB of factor tables
    const int64_t tiles = static_cast<int64_t>(ny / (BV_Y - 1) + 1) * (nz / (BV_Z - 1) + 1);
    FA_REQUIRE(tiles <= (1 << 24), "fa_p1_box_vector_tensor: grid too large");
    // about three blocks a CU, each at least four planes long
    const int64_t chunks = std::max<int64_t>(1, std::min<int64_t>((nx + 4) / 4, 3 * 256 / tiles));
    const int span = static_cast<int>((nx + chunks) / chunks);
    const dim3 grid(static_cast<unsigned>(tiles), static_cast<unsigned>((nx + span) / span));
    double* lines = static_cast<double*>(work);
    double* tab = reinterpret_cast<double*>(static_cast<char*>(work) + table_offset(nx, ny, nz));
    hipStream_t s = S(stream);
    timer_begin(FA_TIMER_P1_VECTORS, s);
    const int st = launch_box_sep_table(nx, ny, nz, node_wide, sep, nq, lines, tab, s);
    if (st != FA_OK) return st;
    const int nmax = std::max(nx, std::max(ny, nz));
    const auto* e = static_cast<const fa_sep_t*>(sep);
    if (dtype == FA_F64)
        hipLaunchKernelGGL(k_p1_box_vector<double>, grid, dim3(256), 0, s, nx, ny, nz, span, axes, nq, qw, phi, scale, e,
                           tab, nmax, static_cast<double*>(out));
    else
        hipLaunchKernelGGL(k_p1_box_vector<float>, grid, dim3(256), 0, s, nx, ny, nz, span, axes, nq, qw, phi, scale, e,
                           tab, nmax, static_cast<float*>(out));
    timer_end(FA_TIMER_P1_VECTORS, s);
    FA_LAUNCH("k_p1_box_vector");
    return FA_OK;
}
