// Dirichlet BC, CSR SpMV and vector kernels (kernel "d" building blocks).
#include <algorithm>
#include <cmath>

#include "common.hpp"
#include "reduce.hpp"

namespace fa {

// ---- SpMV -------------------------------------------------------------------
// A block takes 256 / G consecutive rows, whose entries are one contiguous
// range: it reads that range whole lines at a time whatever the rows' lengths,
// four entries a thread in flight, leaves the products in LDS, and G lanes a
// row add the row's.  What bounds it is HBM: 12 (8 in FP32) bytes an entry, so
// the sums can afford to lose nothing: FP32 products are kept exact in FP64, and
// the additions keep what they round off (RowSum).  An FP64 product is rounded
// once, where lanes that read a row themselves rounded every partial sum.  Off 64
// bits, 40^3 P2 tetrahedra: FP64 3.9e-16 with 32 lanes a row, 4.8e-16 with 4 that
// add plainly, 3.8e-16 so; FP32 8.0e-8, 7.2e-8, 4.1e-8.
// The form with G lanes reading each row themselves lost them in the rows'
// remainders and waited for one entry at a time: a P2 tetrahedral matrix
// (885k rows of 18 to 65 entries, FP64) 141 -> 73 us, 4.4 TB/s.
constexpr int STREAM = 2048;  // products held at once; no index passes the range's end, which may be near 2^31

template <class T, int G>
__global__ void __launch_bounds__(256) k_spmv(int64_t n, const int32_t* __restrict__ indptr,
                                             const int32_t* __restrict__ indices, const T* __restrict__ vals,
                                             const T* __restrict__ x, T* __restrict__ y) {
    constexpr int RB = 256 / G;
    __shared__ double prod[STREAM];
    const int lane = threadIdx.x % G;
    for (int64_t r0 = (int64_t)xcd_window_block() * RB; r0 < n; r0 += (int64_t)gridDim.x * RB) {
        const int64_t end = min(r0 + RB, n), r = min(r0 + threadIdx.x / G, end);
        const int32_t e0 = indptr[r0], e1 = indptr[end];
        const int32_t k0 = indptr[r], k1 = indptr[min(r + 1, end)];
        RowSum<T> s;
        for (int32_t e = e0, m; (m = min(STREAM, e1 - e)) > 0; e += m) {
            for (int b = 0; b < m; b += 1024) {
                int32_t c[4];
                T v[4];
#pragma unroll
                for (int u = 0; u < 4; ++u) {
                    const int32_t k = e + min(b + u * 256 + (int)threadIdx.x, m - 1);
                    c[u] = indices[k];
                    v[u] = vals[k];
                }
                T w[4];
#pragma unroll
                for (int u = 0; u < 4; ++u) w[u] = x[c[u]];
#pragma unroll
                for (int u = 0; u < 4; ++u)
                    if (b + u * 256 + (int)threadIdx.x < m) prod[b + u * 256 + threadIdx.x] = static_cast<double>(v[u]) * w[u];
            }
            __syncthreads();
            for (int i = max(k0 - e, 0) + lane; i < min(k1 - e, m); i += G) s.add(prod[i]);
            __syncthreads();
        }
        const double t = s.template group<G>();
        if (lane == 0 && r < end) y[r] = static_cast<T>(t);
    }
}

template <class T>
static int spmv_launch(int64_t n, const int32_t* indptr, const int32_t* indices, const T* vals, const T* x, T* y,
                       int G, hipStream_t s) {
    const unsigned grid = xcd_window_grid(grid_for(n * G, 256, 1 << 20));
    auto k = k_spmv<T, 64>;
    switch (G) {
        case 1: k = k_spmv<T, 1>; break;
        case 2: k = k_spmv<T, 2>; break;
        case 4: k = k_spmv<T, 4>; break;
        case 8: k = k_spmv<T, 8>; break;
        case 16: k = k_spmv<T, 16>; break;
        case 32: k = k_spmv<T, 32>; break;
        default: break;
    }
    hipLaunchKernelGGL(k, dim3(grid), dim3(256), 0, s, n, indptr, indices, vals, x, y);
    FA_LAUNCH("k_spmv");
    return FA_OK;
}

// Y = A X for nv right-hand sides stored row-major (X[col*nv + v]), the
// layout of SciPy's csr_matvecs; G lanes per row, each entry's columns of X
// read by one lane, vectors taken VB at a time
template <class T, int G, int VB>
__global__ void __launch_bounds__(256) k_spmm(int64_t n, int64_t nv, const int32_t* __restrict__ indptr,
                                             const int32_t* __restrict__ indices, const T* __restrict__ vals,
                                             const T* __restrict__ x, T* __restrict__ y) {
    const int lane = threadIdx.x % G;
    for (int64_t r = (blockIdx.x * (int64_t)blockDim.x + threadIdx.x) / G; r < n;
         r += (int64_t)gridDim.x * blockDim.x / G) {
        const int32_t k0 = indptr[r], k1 = indptr[r + 1];
        for (int64_t v0 = 0; v0 < nv; v0 += VB) {
            T s[VB];
#pragma unroll
            for (int u = 0; u < VB; ++u) s[u] = T(0);
            for (int32_t k = k0 + lane; k < k1; k += G) {
                const T a = vals[k];
                const T* xr = x + static_cast<int64_t>(indices[k]) * nv + v0;
#pragma unroll
                for (int u = 0; u < VB; ++u)
                    if (v0 + u < nv) s[u] += a * xr[u];
            }
#pragma unroll
            for (int u = 0; u < VB; ++u) {
                const T t = group_sum<G>(s[u]);
                if (lane == 0 && v0 + u < nv) y[r * nv + v0 + u] = t;
            }
        }
    }
}

// lanes per row: so many that a block's 256 / G rows hold one to two
// thousand entries on average.  Against 4 lanes and more a row, each row read by
// its own (1000^2 P1 33.6 -> 21 us, 400^2 P2 34 -> 26, 60^3 P1 14.1 -> 10.2, 128^3
// 149 -> 84); matrices of a few blocks (20^2 to 300^2) take a launch either way
static int lanes_for(int64_t n, int64_t nnz) {
    const double avg = n > 0 ? double(nnz) / double(n) : 1.0;
    int g = 1;
    while (g < 64 && 8.0 * g < avg) g <<= 1;
    return g;
}

// ---- Dirichlet BC (G lanes per row) ------------------------------------------------
constexpr int BCG = 16;

__global__ void __launch_bounds__(256) k_bc_count(int64_t n, const int32_t* __restrict__ indptr,
                                                 const int32_t* __restrict__ indices, const uint8_t* __restrict__ bd,
                                                 int32_t* __restrict__ cnt) {
    const int lane = threadIdx.x % BCG;
    for (int64_t r = (blockIdx.x * (int64_t)blockDim.x + threadIdx.x) / BCG; r < n;
         r += (int64_t)gridDim.x * blockDim.x / BCG) {
        int c = 0;
        if (!bd[r])
            for (int32_t k = indptr[r] + lane; k < indptr[r + 1]; k += BCG) c += bd[indices[k]] ? 0 : 1;
        c = group_sum<BCG>(c);
        if (lane == 0) cnt[r] = bd[r] ? 1 : c;
    }
}

// The Dirichlet condition on a CSR matrix.  VAL 1: the filtered matrix (a unit
// row on boundary rows, boundary columns left out; kept entries keep their
// order); VAL 2: the values on A's own pattern (boundary rows 1 on the diagonal
// and 0 elsewhere, boundary columns 0; nval may be vals itself: a chunk is read
// before any of it is written); VAL 0: none.  RHS: out = f - A uh, uh on
// boundary rows, summed in one order whatever VAL and as precisely as k_spmv's.
// As there a block streams the contiguous entries of 256 / G rows; the kept ones'
// new places are contiguous too: the first row's, plus the kept entries before
// (ballots, a prefix over the block's waves), so values leave in order.  Of a
// boundary row the first entry keeps a place, for the row's thread to fill; a
// boundary row without entries has none, and the block that sees its count fall
// short places its rows one by one.  nidx == NULL refills values only; U: the
// type of the filtered values (an FP32 copy of an FP64 matrix is rounded once).  Both directions of HBM bound it: 20 bytes an entry.
// 15.0M entries (100 x 113 x 90 cells, P1): 16 lanes a row 128 -> 75 us.
template <class T, class U, int G, int VAL, bool RHS>
__global__ void __launch_bounds__(256) k_bc_rows(int64_t n, const int32_t* __restrict__ indptr,
                                                const int32_t* __restrict__ indices, const T* vals,
                                                const uint8_t* __restrict__ bd, const int32_t* __restrict__ nptr,
                                                int32_t* __restrict__ nidx, U* nval,
                                                const T* __restrict__ uh, const T* __restrict__ f,
                                                T* __restrict__ out) {
    constexpr int RB = 256 / G, CH = STREAM / 2, PER = CH / 256, WAVES = 256 / WAVE;
    __shared__ double prod[RHS ? CH : 1];
    __shared__ alignas(4) uint8_t mark[CH];  // 1: entry of a boundary row, 2: its first
    __shared__ int cnt[PER * WAVES];
    const int lane = threadIdx.x % G, wave = threadIdx.x / WAVE;
    const unsigned long long below = (1ull << (threadIdx.x % WAVE)) - 1;
    for (int64_t r0 = (int64_t)xcd_window_block() * RB; r0 < n; r0 += (int64_t)gridDim.x * RB) {
        const int64_t end = min(r0 + RB, n), r = min(r0 + threadIdx.x / G, end);
        const int32_t e0 = indptr[r0], e1 = indptr[end];
        const int32_t k0 = indptr[r], k1 = indptr[min(r + 1, end)];
        const int32_t o0 = VAL == 1 ? nptr[r0] : 0, o1 = VAL == 1 ? nptr[end] : 0;
        const bool fixed = r < end && bd[r] != 0;
        int32_t at = o0;
        RowSum<T> s;
        for (int32_t e = e0, m; (m = min(CH, e1 - e)) > 0; e += m) {
            reinterpret_cast<uint32_t*>(mark)[threadIdx.x] = 0;
            int32_t c[PER];
            T v[PER], w[PER];
            bool cb[PER];
#pragma unroll
            for (int u = 0; u < PER; ++u) {
                const int32_t k = e + min(u * 256 + (int)threadIdx.x, m - 1);
                c[u] = indices[k];
                v[u] = vals[k];
            }
            __syncthreads();
            if (fixed)
                for (int i = max(k0 - e, 0) + lane; i < min(k1 - e, m); i += G) mark[i] = e + i == k0 ? 2 : 1;
#pragma unroll
            for (int u = 0; u < PER; ++u) {
                cb[u] = bd[c[u]] != 0;
                if constexpr (RHS) w[u] = uh[c[u]];
            }
            __syncthreads();
            if constexpr (VAL == 2) {
                if (fixed)
                    for (int i = max(k0 - e, 0) + lane; i < min(k1 - e, m); i += G)
                        nval[e + i] = indices[e + i] == r ? U(1) : U(0);
            }
            bool keep[PER];
            int rank[PER];
#pragma unroll
            for (int u = 0; u < PER; ++u) {
                const int i = u * 256 + threadIdx.x;
                const int mk = i < m ? mark[i] : 1;
                if constexpr (VAL == 1) {
                    const bool place = mk == 2 || (mk == 0 && !cb[u]);
                    keep[u] = mk == 0 && place;
                    const unsigned long long b = __ballot(place);
                    rank[u] = __popcll(b & below);
                    if (threadIdx.x % WAVE == 0) cnt[u * WAVES + wave] = __popcll(b);
                }
                if constexpr (VAL == 2) {
                    if (mk == 0) nval[e + i] = cb[u] ? U(0) : static_cast<U>(v[u]);
                }
                if constexpr (RHS) {
                    if (i < m) prod[i] = static_cast<double>(v[u]) * w[u];
                }
            }
            __syncthreads();
            if constexpr (VAL == 1) {
#pragma unroll
                for (int u = 0; u < PER; ++u)
#pragma unroll
                    for (int q = 0; q < WAVES; ++q) {
                        if (q == wave && keep[u] && at + rank[u] < o1) {
                            if (nidx) nidx[at + rank[u]] = c[u];
                            nval[at + rank[u]] = static_cast<U>(v[u]);
                        }
                        at += cnt[u * WAVES + q];
                    }
            }
            if constexpr (RHS)
                for (int i = max(k0 - e, 0) + lane; i < min(k1 - e, m); i += G) s.add(prod[i]);
            __syncthreads();
        }
        if (at != o1) {  // a boundary row without entries, the same for the whole block
            if (lane == 0 && r < end && !fixed) {
                int32_t o = nptr[r];
                for (int32_t k = k0; k < k1; ++k)
                    if (!bd[indices[k]]) {
                        if (nidx) nidx[o] = indices[k];
                        nval[o++] = static_cast<U>(vals[k]);
                    }
            }
            __syncthreads();
        }
        double Auh = 0.0;
        if constexpr (RHS) Auh = s.template group<G>();
        if (lane == 0 && r < end) {
            if (VAL == 1 && fixed) {
                const int32_t o = nptr[r];
                if (nidx) nidx[o] = static_cast<int32_t>(r);
                nval[o] = U(1);
            }
            if constexpr (RHS) out[r] = fixed ? uh[r] : static_cast<T>(f[r] - Auh);
        }
    }
}

template <class T, class U, int VAL, bool RHS>
static int bc_launch(int64_t n, const int32_t* indptr, const int32_t* indices, const void* vals, const uint8_t* bd,
                     const int32_t* nptr, int32_t* nidx, void* nval, const void* uh, const void* f, void* out,
                     hipStream_t s) {
    // 64 rows a block: 960 entries of a P1 tetrahedral matrix, a chunk; also faster
    // than 16 lanes a row where a block fills half a chunk or takes two (whole
    // boundary condition, 1000^2 P1 127 -> 72 us, 400^2 P2 98 -> 64, 40^3 P2
    // 123 -> 91; at 300^2 and below the launches take it all)
    constexpr int G = 4;
    hipLaunchKernelGGL((k_bc_rows<T, U, G, VAL, RHS>), dim3(xcd_window_grid(grid_for(n * G, 256, 1 << 20))), dim3(256), 0, s,
                       n, indptr, indices, static_cast<const T*>(vals), bd, nptr, nidx, static_cast<U*>(nval),
                       static_cast<const T*>(uh), static_cast<const T*>(f), static_cast<T*>(out));
    FA_LAUNCH("k_bc_rows");
    return FA_OK;
}

// ---- vector kernels --------------------------------------------------------------
template <class T>
__global__ void __launch_bounds__(RED_BLOCK) k_dot(int64_t n, const T* __restrict__ x, const T* __restrict__ y,
                                                  double* __restrict__ partials) {
    double s = 0.0;
    for (int64_t i = blockIdx.x * (int64_t)blockDim.x + threadIdx.x; i < n; i += (int64_t)gridDim.x * blockDim.x)
        s += double(x[i]) * double(y[i]);
    store_partial(block_sum(s), partials);
}

__global__ void __launch_bounds__(RED_BLOCK) k_dot_finish(const double* __restrict__ partials, int nparts,
                                                         double* __restrict__ out) {
    const double t = finish_sum(partials, nparts);
    if (threadIdx.x == 0) *out = t;
}

template <class T>
__global__ void k_axpby(int64_t n, double a, const T* __restrict__ x, double b, T* __restrict__ y) {
    for (int64_t i = blockIdx.x * (int64_t)blockDim.x + threadIdx.x; i < n; i += (int64_t)gridDim.x * blockDim.x)
        y[i] = static_cast<T>(a * double(x[i]) + b * double(y[i]));
}

// x += d off the Dirichlet rows (the correction step of iterative refinement:
// boundary values stay exactly those of the boundary condition)
template <class D>
__global__ void k_refine_update(int64_t n, double* __restrict__ x, const D* __restrict__ d,
                                const uint8_t* __restrict__ bd) {
    for (int64_t i = blockIdx.x * (int64_t)blockDim.x + threadIdx.x; i < n; i += (int64_t)gridDim.x * blockDim.x)
        if (!bd[i]) x[i] += static_cast<double>(d[i]);
}

template <class A, class B>
__global__ void k_cast(int64_t n, const A* __restrict__ x, B* __restrict__ y) {
    for (int64_t i = blockIdx.x * (int64_t)blockDim.x + threadIdx.x; i < n; i += (int64_t)gridDim.x * blockDim.x)
        y[i] = static_cast<B>(x[i]);
}

}  // namespace fa

using namespace fa;

extern "C" int fa_spmv(int dtype, int64_t n, int64_t nnz, const int32_t* indptr, const int32_t* indices,
                       const void* values, const void* x, void* y, fa_stream_t stream) {
    FA_REQUIRE(dtype == FA_F64 || dtype == FA_F32, "fa_spmv: bad dtype %d", dtype);
    if (n == 0) return FA_OK;
    const int G = tuned(FA_TUNE_SPMV_LANES, fa_tune_key(FA_TUNE_SPMV_LANES, n, nnz), lanes_for(n, nnz));
    if (dtype == FA_F64)
        return spmv_launch<double>(n, indptr, indices, static_cast<const double*>(values),
                                   static_cast<const double*>(x), static_cast<double*>(y), G, S(stream));
    return spmv_launch<float>(n, indptr, indices, static_cast<const float*>(values), static_cast<const float*>(x),
                              static_cast<float*>(y), G, S(stream));
}

extern "C" int fa_spmm(int dtype, int64_t n, int64_t nnz, int64_t nvec, const int32_t* indptr, const int32_t* indices,
                       const void* values, const void* x, void* y, fa_stream_t stream) {
    FA_REQUIRE(dtype == FA_F64 || dtype == FA_F32, "fa_spmm: bad dtype %d", dtype);
    FA_REQUIRE(nvec >= 1, "fa_spmm: nvec must be >= 1");
    if (n == 0) return FA_OK;
    const unsigned grid = grid_for(n * 8, 256, 1 << 20);
    if (dtype == FA_F64)
        hipLaunchKernelGGL((k_spmm<double, 8, 4>), dim3(grid), dim3(256), 0, S(stream), n, nvec, indptr, indices,
                           static_cast<const double*>(values), static_cast<const double*>(x), static_cast<double*>(y));
    else
        hipLaunchKernelGGL((k_spmm<float, 8, 4>), dim3(grid), dim3(256), 0, S(stream), n, nvec, indptr, indices,
                           static_cast<const float*>(values), static_cast<const float*>(x), static_cast<float*>(y));
    FA_LAUNCH("k_spmm");
    return FA_OK;
}

extern "C" size_t fa_dirichlet_work_bytes(int64_t n) {
    return align_up((n + 1) * sizeof(int32_t)) + exclusive_scan_work_bytes(n) + 1024;
}

extern "C" int fa_dirichlet_count(int64_t n, const int32_t* indptr, const int32_t* indices, const uint8_t* is_bd,
                                  int32_t* new_indptr, int64_t* new_nnz_host, void* work, size_t work_bytes,
                                  fa_stream_t stream) {
    FA_REQUIRE(n > 0, "fa_dirichlet_count: empty matrix");
    hipStream_t s = S(stream);
    Arena ar(work, work_bytes);
    int32_t* cnt = ar.take<int32_t>(n + 1);
    size_t sb = exclusive_scan_work_bytes(n);
    void* sw = ar.take<char>(sb);
    if (!cnt || !sw) {
        set_error("fa_dirichlet_count: workspace too small");
        return FA_ENOMEM;
    }
    hipLaunchKernelGGL(k_bc_count, dim3(grid_for(n * BCG, 256, 1 << 16)), dim3(256), 0, s, n, indptr, indices, is_bd,
                       cnt);
    FA_LAUNCH("k_bc_count");
    int st = exclusive_scan_i32(cnt, new_indptr, n, sw, sb, s);
    if (st != FA_OK) return st;
    int32_t nnz = 0;
    FA_HIP(hipMemcpyAsync(&nnz, new_indptr + n, sizeof(int32_t), hipMemcpyDeviceToHost, s));
    FA_HIP(hipStreamSynchronize(s));
    if (new_nnz_host) *new_nnz_host = nnz;
    return FA_OK;
}

extern "C" int fa_dirichlet_fill(int dtype, int dtype_out, int64_t n, const int32_t* indptr, const int32_t* indices,
                                 const void* values, const uint8_t* is_bd, const int32_t* new_indptr,
                                 int32_t* new_indices, void* new_values, fa_stream_t stream) {
    FA_REQUIRE(dtype == FA_F64 || dtype == FA_F32, "fa_dirichlet_fill: bad dtype %d", dtype);
    FA_REQUIRE(dtype_out == dtype || (dtype == FA_F64 && dtype_out == FA_F32),
               "fa_dirichlet_fill: values of dtype %d cannot be stored as dtype %d", dtype, dtype_out);
    hipStream_t s = S(stream);
    if (n == 0) return FA_OK;
    auto fill = dtype == FA_F32       ? bc_launch<float, float, 1, false>
                : dtype_out == FA_F64 ? bc_launch<double, double, 1, false>
                                      : bc_launch<double, float, 1, false>;
    return fill(n, indptr, indices, values, is_bd, new_indptr, new_indices, new_values, nullptr, nullptr, nullptr, s);
}

extern "C" int fa_dirichlet_rhs(int dtype, int64_t n, const int32_t* indptr, const int32_t* indices,
                                const void* values, const uint8_t* is_bd, const void* uh, const void* f, void* f_out,
                                fa_stream_t stream) {
    FA_REQUIRE(dtype == FA_F64 || dtype == FA_F32, "fa_dirichlet_rhs: bad dtype %d", dtype);
    hipStream_t s = S(stream);
    if (n == 0) return FA_OK;
    auto rhs = dtype == FA_F64 ? bc_launch<double, double, 0, true> : bc_launch<float, float, 0, true>;
    return rhs(n, indptr, indices, values, is_bd, nullptr, nullptr, nullptr, uh, f, f_out, s);
}

extern "C" int fa_dirichlet_apply(int dtype, int64_t n, const int32_t* indptr, const int32_t* indices,
                                  const void* values, const uint8_t* is_bd, const int32_t* new_indptr,
                                  void* new_values, const void* uh, const void* f, void* f_out, fa_stream_t stream) {
    FA_REQUIRE(dtype == FA_F64 || dtype == FA_F32, "fa_dirichlet_apply: bad dtype %d", dtype);
    hipStream_t s = S(stream);
    if (n == 0) return FA_OK;
    timer_begin(FA_TIMER_BC_APPLY, s);
    auto apply = dtype == FA_F64 ? bc_launch<double, double, 1, true> : bc_launch<float, float, 1, true>;
    const int st = apply(n, indptr, indices, values, is_bd, new_indptr, nullptr, new_values, uh, f, f_out, s);
    timer_end(FA_TIMER_BC_APPLY, s);
    return st;
}

extern "C" size_t fa_reduce_work_bytes(void) { return 3 * align_up(RED_GRID * sizeof(double)) + 1024; }

extern "C" int fa_dot(int dtype, int64_t n, const void* x, const void* y, double* out, void* work,
                      size_t work_bytes, fa_stream_t stream) {
    FA_REQUIRE(dtype == FA_F64 || dtype == FA_F32, "fa_dot: bad dtype %d", dtype);
    Arena ar(work, work_bytes);
    double* partials = ar.take<double>(RED_GRID);
    if (!partials) {
        set_error("fa_dot: workspace too small");
        return FA_ENOMEM;
    }
    hipStream_t s = S(stream);
    const unsigned g = red_grid(n);
    if (dtype == FA_F64)
        hipLaunchKernelGGL(k_dot<double>, dim3(g), dim3(RED_BLOCK), 0, s, n, static_cast<const double*>(x),
                           static_cast<const double*>(y), partials);
    else
        hipLaunchKernelGGL(k_dot<float>, dim3(g), dim3(RED_BLOCK), 0, s, n, static_cast<const float*>(x),
                           static_cast<const float*>(y), partials);
    hipLaunchKernelGGL(k_dot_finish, dim3(1), dim3(RED_BLOCK), 0, s, partials, (int)g, out);
    FA_LAUNCH("k_dot");
    return FA_OK;
}

extern "C" int fa_axpby(int dtype, int64_t n, double a, const void* x, double b, void* y, fa_stream_t stream) {
    FA_REQUIRE(dtype == FA_F64 || dtype == FA_F32, "fa_axpby: bad dtype %d", dtype);
    hipStream_t s = S(stream);
    const unsigned grid = grid_for(n, 256, 1 << 16);
    if (dtype == FA_F64)
        hipLaunchKernelGGL(k_axpby<double>, dim3(grid), dim3(256), 0, s, n, a, static_cast<const double*>(x), b,
                           static_cast<double*>(y));
    else
        hipLaunchKernelGGL(k_axpby<float>, dim3(grid), dim3(256), 0, s, n, a, static_cast<const float*>(x), b,
                           static_cast<float*>(y));
    FA_LAUNCH("k_axpby");
    return FA_OK;
}

extern "C" int fa_cast(int dtype_in, int dtype_out, int64_t n, const void* x, void* y, fa_stream_t stream) {
    hipStream_t s = S(stream);
    const unsigned grid = grid_for(n, 256, 1 << 16);
    if (dtype_in == FA_F64 && dtype_out == FA_F32)
        hipLaunchKernelGGL((k_cast<double, float>), dim3(grid), dim3(256), 0, s, n, static_cast<const double*>(x),
                           static_cast<float*>(y));
    else if (dtype_in == FA_F32 && dtype_out == FA_F64)
        hipLaunchKernelGGL((k_cast<float, double>), dim3(grid), dim3(256), 0, s, n, static_cast<const float*>(x),
                           static_cast<double*>(y));
    else {
        set_error("fa_cast: unsupported dtypes %d -> %d", dtype_in, dtype_out);
        return FA_EINVAL;
    }
    FA_LAUNCH("k_cast");
    return FA_OK;
}


extern "C" int fa_refine_update(int dtype_d, int64_t n, double* x, const void* d, const uint8_t* is_bd,
                                fa_stream_t stream) {
    FA_REQUIRE(dtype_d == FA_F64 || dtype_d == FA_F32, "fa_refine_update: bad dtype %d", dtype_d);
    FA_REQUIRE(n >= 0 && (n == 0 || (x && d && is_bd)), "fa_refine_update: bad arguments");
    if (n == 0) return FA_OK;
    hipStream_t s = S(stream);
    const unsigned grid = grid_for(n, 256, 1 << 16);
    if (dtype_d == FA_F64)
        hipLaunchKernelGGL(k_refine_update<double>, dim3(grid), dim3(256), 0, s, n, x, static_cast<const double*>(d),
                           is_bd);
    else
        hipLaunchKernelGGL(k_refine_update<float>, dim3(grid), dim3(256), 0, s, n, x, static_cast<const float*>(d),
                           is_bd);
    FA_LAUNCH("k_refine_update");
    return FA_OK;
}

// r = b - A x off the Dirichlet rows, 0 on them, stored as Y, and the
// workgroup partial sums of r^2 (a grid fixed by n): the FP64 residual of
// iterative refinement on an assembled FP64 matrix.  Streams the rows' entries
// as k_spmv does; the grid is capped (one partial a block), so a block walks
// many groups of 256 / G rows.  30.4M entries (128^3 P1): 125 us with G lanes
// reading each row -> 104 us (4.0 TB/s) with 4 lanes adding a row; 2 lanes 103 us.
template <int G, class Y>
__global__ void __launch_bounds__(256) k_csr_residual(int64_t n, const int32_t* __restrict__ indptr,
                                                     const int32_t* __restrict__ indices,
                                                     const double* __restrict__ vals, const double* __restrict__ x,
                                                     const double* __restrict__ b, const uint8_t* __restrict__ bd,
                                                     Y* __restrict__ y, double* __restrict__ part) {
    constexpr int RB = 256 / G;
    __shared__ double prod[STREAM];
    const int lane = threadIdx.x % G;
    double nrm = 0.0;
    for (int64_t r0 = (int64_t)blockIdx.x * RB; r0 < n; r0 += (int64_t)gridDim.x * RB) {
        const int64_t end = min(r0 + RB, n), r = min(r0 + threadIdx.x / G, end);
        const int32_t e0 = indptr[r0], e1 = indptr[end];
        const int32_t k0 = indptr[r], k1 = indptr[min(r + 1, end)];
        const int64_t rr = min(r, n - 1);
        const double bv = b[rr];
        const bool fixed = bd[rr] != 0;
        RowSum<double> s;
        for (int32_t e = e0, m; (m = min(STREAM, e1 - e)) > 0; e += m) {
            for (int q = 0; q < m; q += 1024) {
                int32_t c[4];
                double v[4], w[4];
#pragma unroll
                for (int u = 0; u < 4; ++u) {
                    const int32_t k = e + min(q + u * 256 + (int)threadIdx.x, m - 1);
                    c[u] = indices[k];
                    v[u] = vals[k];
                }
#pragma unroll
                for (int u = 0; u < 4; ++u) w[u] = x[c[u]];
#pragma unroll
                for (int u = 0; u < 4; ++u)
                    if (q + u * 256 + (int)threadIdx.x < m) prod[q + u * 256 + threadIdx.x] = v[u] * w[u];
            }
            __syncthreads();
            for (int i = max(k0 - e, 0) + lane; i < min(k1 - e, m); i += G) s.add(prod[i]);
            __syncthreads();
        }
        const double Ax = s.template group<G>();
        const double t = fixed ? 0.0 : bv - Ax;
        if (lane == 0 && r < end) {
            y[r] = static_cast<Y>(t);
            nrm += t * t;
        }
    }
    store_partial(block_sum(nrm), part);
}

__global__ void k_residual_finish(const double* __restrict__ part, int n, double* __restrict__ out) {
    const double s = finish_sum(part, n);
    if (threadIdx.x == 0) *out = s;
}

extern "C" size_t fa_csr_residual_work_bytes(void) { return align_up(RED_GRID * sizeof(double)) + 256; }

extern "C" int fa_csr_residual(int dtype_y, int64_t n, const int32_t* indptr, const int32_t* indices,
                               const double* values, const double* x, const double* b, const uint8_t* is_bd, void* y,
                               double* norm2, void* work, size_t work_bytes, fa_stream_t stream) {
    FA_REQUIRE(dtype_y == FA_F64 || dtype_y == FA_F32, "fa_csr_residual: bad dtype %d", dtype_y);
    FA_REQUIRE(n > 0 && indptr && indices && values && x && b && is_bd && y && norm2, "fa_csr_residual: bad arguments");
    Arena ar(work, work_bytes);
    double* part = ar.take<double>(RED_GRID);
    if (!part) {
        set_error("fa_csr_residual: workspace too small");
        return FA_ENOMEM;
    }
    hipStream_t s = S(stream);
    constexpr int G = 4;
    const unsigned grid = static_cast<unsigned>(std::min<int64_t>((n * G + 255) / 256, RED_GRID));
    if (dtype_y == FA_F64)
        hipLaunchKernelGGL((k_csr_residual<G, double>), dim3(grid), dim3(256), 0, s, n, indptr, indices, values, x, b,
                           is_bd, static_cast<double*>(y), part);
    else
        hipLaunchKernelGGL((k_csr_residual<G, float>), dim3(grid), dim3(256), 0, s, n, indptr, indices, values, x, b,
                           is_bd, static_cast<float*>(y), part);
    FA_LAUNCH("k_csr_residual");
    hipLaunchKernelGGL(k_residual_finish, dim3(1), dim3(RED_BLOCK), 0, s, part, static_cast<int>(grid), norm2);
    FA_LAUNCH("k_residual_finish");
    return FA_OK;
}

extern "C" int fa_dirichlet_apply_keep(int dtype, int64_t n, const int32_t* indptr, const int32_t* indices,
                                       const void* values, const uint8_t* is_bd, void* new_values, const void* uh,
                                       const void* f, void* f_out, fa_stream_t stream) {
    FA_REQUIRE(dtype == FA_F64 || dtype == FA_F32, "fa_dirichlet_apply_keep: bad dtype %d", dtype);
    FA_REQUIRE(n >= 0 && indptr && indices && values && is_bd && new_values && uh && f && f_out,
               "fa_dirichlet_apply_keep: bad arguments");
    if (n == 0) return FA_OK;
    hipStream_t s = S(stream);
    timer_begin(FA_TIMER_BC_APPLY, s);
    auto keep = dtype == FA_F64 ? bc_launch<double, double, 2, true> : bc_launch<float, float, 2, true>;
    const int st = keep(n, indptr, indices, values, is_bd, nullptr, nullptr, new_values, uh, f, f_out, s);
    timer_end(FA_TIMER_BC_APPLY, s);
    return st;
}
