// Fixed-order (ascending cell) sum of element matrices into CSR rows.
#include "common.hpp"

#include <algorithm>

namespace fa {

__device__ inline int lower_bound_lds(const int32_t* a, int n, int32_t v) {
    int lo = 0, hi = n;
    while (lo < hi) {
        int mid = (lo + hi) >> 1;
        if (a[mid] < v) lo = mid + 1;
        else hi = mid;
    }
    return lo;
}

// G lanes per global row (G >= ldof); each row's columns and FP64 accumulators
// live in LDS (the sums of k_sum_rows, bit for bit: a pattern's first assembly
// takes this kernel, the next ones that).  The incident cells of a row are visited in ascending order
// and lane j adds element entry (i, j) of the current cell, so every CSR entry
// is summed in ascending cell order -- the order of the reference's stable
// lexsort + sequential np.add.at.  Distinct columns of one cell never collide.
template <class T, int G>
__global__ void k_gather_matrix(int64_t gdof, int ldof, const int32_t* __restrict__ c2d,
                                const int32_t* __restrict__ ptr, const int32_t* __restrict__ adj,
                                const int32_t* __restrict__ indptr, const int32_t* __restrict__ indices, int lmax,
                                const T* __restrict__ elem, int64_t cstride, T* __restrict__ values) {
    extern __shared__ char smem[];
    const int rpb = blockDim.x / G;
    const int sub = threadIdx.x / G;
    const int lane = threadIdx.x % G;
    int32_t* cols = reinterpret_cast<int32_t*>(smem) + sub * lmax;
    double* acc = reinterpret_cast<double*>(smem + align_up(sizeof(int32_t) * rpb * lmax, 16)) + sub * lmax;
    for (int64_t r = (int64_t)blockIdx.x * rpb + sub; r < gdof; r += (int64_t)gridDim.x * rpb) {
        const int32_t r0 = indptr[r];
        const int L = indptr[r + 1] - r0;
        for (int t = lane; t < L; t += G) {
            cols[t] = indices[r0 + t];
            acc[t] = 0.0;
        }
        __builtin_amdgcn_wave_barrier();
        __builtin_amdgcn_fence(__ATOMIC_SEQ_CST, "wavefront");
        const int32_t k1 = ptr[r + 1];
        if (ldof <= G) {
            // the row's incidences G at a time in one load, handed out by
            // shuffles; the next incidence's column and value loads are issued
            // before the current one's search and add (same adds, same order)
            for (int32_t kb = ptr[r]; kb < k1; kb += G) {
                const int32_t mine = kb + lane < k1 ? adj[kb + lane] : 0;
                const int nk = min(G, k1 - kb);
                const bool act = lane < ldof;
                int32_t e = __shfl(mine, 0, G);
                int32_t c = e / ldof;
                int32_t col = act ? c2d[(int64_t)c * ldof + lane] : 0;
                T v = act ? elem[(int64_t)c * cstride + (e - c * ldof) * ldof + lane] : T(0);
                for (int u = 0; u < nk; ++u) {
                    int32_t col_n = 0;
                    T v_n = T(0);
                    if (u + 1 < nk) {
                        const int32_t en = __shfl(mine, u + 1, G);
                        const int32_t cn = en / ldof;
                        if (act) {
                            col_n = c2d[(int64_t)cn * ldof + lane];
                            v_n = elem[(int64_t)cn * cstride + (en - cn * ldof) * ldof + lane];
                        }
                    }
                    if (act) {
                        const int pos = lower_bound_lds(cols, L, col);
                        if (pos < L && cols[pos] == col) acc[pos] += v;
                    }
                    __builtin_amdgcn_wave_barrier();
                    __builtin_amdgcn_fence(__ATOMIC_SEQ_CST, "wavefront");
                    col = col_n;
                    v = v_n;
                }
            }
        } else {
            for (int32_t k = ptr[r]; k < k1; ++k) {
                const int32_t e = adj[k];
                const int32_t c = e / ldof;
                for (int j = lane; j < ldof; j += G) {
                    const int32_t col = c2d[(int64_t)c * ldof + j];
                    const T v = elem[(int64_t)c * cstride + (e - c * ldof) * ldof + j];
                    const int pos = lower_bound_lds(cols, L, col);
                    if (pos < L && cols[pos] == col) acc[pos] += v;
                }
                __builtin_amdgcn_wave_barrier();
                __builtin_amdgcn_fence(__ATOMIC_SEQ_CST, "wavefront");
            }
        }
        for (int t = lane; t < L; t += G) values[r0 + t] = static_cast<T>(acc[t]);
        __builtin_amdgcn_wave_barrier();
        __builtin_amdgcn_fence(__ATOMIC_SEQ_CST, "wavefront");
    }
}

// ---- with the positions known ------------------------------------------------
// pos[k * ldof + j]: where column j of incidence k's cell lies in its row
// (rows of at most 8192 entries).  They depend on the pattern only.
__global__ void __launch_bounds__(256) k_row_positions(int64_t gdof, int ldof, const int32_t* __restrict__ c2d,
                                                       const int32_t* __restrict__ ptr, const int32_t* __restrict__ adj,
                                                       const int32_t* __restrict__ indptr,
                                                       const int32_t* __restrict__ indices, int lmax,
                                                       uint16_t* __restrict__ pos) {
    extern __shared__ int32_t cols_lds[];
    const int rpb = blockDim.x / WAVE, lane = threadIdx.x % WAVE;
    int32_t* cols = cols_lds + threadIdx.x / WAVE * lmax;
    for (int64_t r = (int64_t)blockIdx.x * rpb + threadIdx.x / WAVE; r < gdof; r += (int64_t)gridDim.x * rpb) {
        const int32_t r0 = indptr[r];
        const int L = indptr[r + 1] - r0;
        for (int t = lane; t < L; t += WAVE) cols[t] = indices[r0 + t];
        __builtin_amdgcn_wave_barrier();
        __builtin_amdgcn_fence(__ATOMIC_SEQ_CST, "wavefront");
        const int64_t k0 = ptr[r];
        const int n = (ptr[r + 1] - ptr[r]) * ldof;
        for (int t = lane; t < n; t += WAVE) {
            const int u = t / ldof;
            const int32_t c = adj[k0 + u] / ldof;
            pos[k0 * ldof + t] = static_cast<uint16_t>(lower_bound_lds(cols, L, c2d[(int64_t)c * ldof + (t - u * ldof)]));
        }
        __builtin_amdgcn_wave_barrier();
        __builtin_amdgcn_fence(__ATOMIC_SEQ_CST, "wavefront");
    }
}

__device__ inline void wave_lds_fence() {
    __builtin_amdgcn_wave_barrier();
    __builtin_amdgcn_fence(__ATOMIC_SEQ_CST, "wavefront");
}

__device__ inline void lds_add(double* p, double v) {
    __hip_atomic_fetch_add(p, v, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
}

// ldof lanes per row, up to 64 / ldof rows per wave (one, and ldof / 64 rounds,
// past 64; fewer where the longest row's sums would not fit otherwise); a row's
// FP64 sums live in LDS.  Lane j adds entry (i, j) of the row's
// incident cells in ascending order, which is the order of the reference's
// stable lexsort + sequential np.add.at.  The additions of one wave to LDS are
// done in the order it issues them, so they are LDS adds without a result
// (ds_add_f64) and nothing waits for them; the columns of one cell never
// collide.  What bounds it is the chain row pointer -> incidence -> element row
// (SUM_U incidences' loads are in flight together) and the bytes: ldof^2
// values a cell in, the row values out.  The form that searches each column in
// the row's column list (k_gather_matrix) spends its time in those searches:
// 3.05M P3 rows 1.71 -> 0.96 ms, 149k P2 triangle rows 18 -> 14 us.
constexpr int SUM_U = 4;

template <int LDOF, class T>
__global__ void __launch_bounds__(256) k_sum_rows(int64_t gdof, int ld, int rows, const int32_t* __restrict__ ptr,
                                                  const int32_t* __restrict__ adj, const int32_t* __restrict__ indptr,
                                                  const uint16_t* __restrict__ pos, int lmax,
                                                  const T* __restrict__ elem, int64_t cpad, T* __restrict__ values) {
    extern __shared__ double sums[];
    const int ldof = LDOF ? LDOF : ld;  // LDOF 0: any width, known at run time
    const int lane = threadIdx.x % WAVE, wave = threadIdx.x / WAVE;
    const int width = min(ldof, WAVE);
    const int sub = lane / width, j0 = lane - sub * width;
    double* acc = sums + (wave * rows + min(sub, rows - 1)) * lmax;
    const int64_t per_block = (int64_t)(blockDim.x / WAVE) * rows;
    const int64_t r = (int64_t)xcd_window_block() * per_block + wave * rows + sub;
    if (sub >= rows || r >= gdof) return;  // no block-wide wait below
    const int32_t r0 = indptr[r];
    const int L = indptr[r + 1] - r0;
    const int32_t k0 = ptr[r], deg = ptr[r + 1] - k0;
    for (int t = j0; t < L; t += width) acc[t] = 0.0;
    wave_lds_fence();
    const int32_t* ad = adj + k0;
    if (ldof <= WAVE) {
        const uint16_t* pr = pos + (int64_t)k0 * ldof + j0;
        const T* el = elem + j0;
        for (int k = 0; k < deg; k += SUM_U) {
            // straight-line loads (the last incidence again past the end): a
            // test around each would wait for one before issuing the next
            uint32_t e[SUM_U];
            int p[SUM_U];
            T v[SUM_U];
#pragma unroll
            for (int u = 0; u < SUM_U; ++u) e[u] = ad[min(k + u, deg - 1)];
#pragma unroll
            for (int u = 0; u < SUM_U; ++u) p[u] = pr[min(k + u, deg - 1) * ldof];
            if (cpad) {
#pragma unroll
                for (int u = 0; u < SUM_U; ++u)
                    v[u] = el[(uint64_t)e[u] * (uint32_t)ldof + e[u] / (uint32_t)ldof * cpad];
            } else {
#pragma unroll
                for (int u = 0; u < SUM_U; ++u) v[u] = el[(uint64_t)e[u] * (uint32_t)ldof];
            }
#pragma unroll
            for (int u = 0; u < SUM_U; ++u)
                if (k + u < deg) lds_add(acc + p[u], v[u]);
        }
    } else {
        // all rounds of one incidence before the next incidence's: with the
        // rounds outermost an entry met in two of them would not be summed in
        // cell order
        for (int k = 0; k < deg; ++k) {
            const uint32_t e = ad[k];
            const uint16_t* pr = pos + (int64_t)(k0 + k) * ldof;
            const T* el = elem + (uint64_t)e * (uint32_t)ldof + e / (uint32_t)ldof * cpad;
            for (int j = j0; j < ldof; j += 2 * WAVE) {
                const int j1 = min(j + WAVE, ldof - 1);
                const int p0 = pr[j], p1 = pr[j1];
                const T v0 = el[j], v1 = el[j1];
                lds_add(acc + p0, v0);
                if (j + WAVE < ldof) lds_add(acc + p1, v1);
            }
        }
    }
    wave_lds_fence();
    for (int t = j0; t < L; t += width) values[r0 + t] = static_cast<T>(acc[t]);
}

template <int LDOF, class T>
static int launch_sum_rows(int64_t gdof, int ldof, const int32_t* ptr, const int32_t* adj, const int32_t* indptr,
                           const uint16_t* pos, int lmax, const void* elem, int64_t cpad, void* values, hipStream_t s) {
    // a wave's sums take 64 KB at most: every row that a pattern can hold (8192
    // entries) fits, and two waves share a CU beside one long row
    int rows = WAVE / std::min(ldof, WAVE);
    while (rows > 1 && sizeof(double) * rows * lmax > 64 * 1024) rows >>= 1;
    const size_t per_wave = sizeof(double) * rows * lmax;
    int waves = 4;
    while (waves > 1 && waves * per_wave > 32 * 1024) waves >>= 1;
    const size_t lds = waves * per_wave;
    if (lds > 160 * 1024) {
        set_error("fa_sum_rows: row length %d exceeds the LDS capacity", lmax);
        return FA_ECAPACITY;
    }
    auto k = k_sum_rows<LDOF, T>;
    if (lds > 64 * 1024)
        FA_HIP(hipFuncSetAttribute(reinterpret_cast<const void*>(k), hipFuncAttributeMaxDynamicSharedMemorySize,
                                   static_cast<int>(lds)));
    const unsigned grid = xcd_window_grid(static_cast<unsigned>((gdof + waves * rows - 1) / (waves * rows)));
    hipLaunchKernelGGL(k, dim3(grid), dim3(waves * WAVE), lds, s, gdof, ldof, rows, ptr, adj, indptr, pos, lmax,
                       static_cast<const T*>(elem), cpad, static_cast<T*>(values));
    FA_LAUNCH("k_sum_rows");
    return FA_OK;
}

template <class T>
static int dispatch_sum_rows(int64_t gdof, int ldof, const int32_t* ptr, const int32_t* adj, const int32_t* indptr,
                             const uint16_t* pos, int lmax, const void* elem, int64_t cpad, void* values,
                             hipStream_t s) {
    switch (ldof) {  // the widths of the scalar spaces; vector spaces and user integrators take the general one
#define FA_CASE(L_) \
    case L_: return launch_sum_rows<L_, T>(gdof, ldof, ptr, adj, indptr, pos, lmax, elem, cpad, values, s)
        FA_CASE(6);
        FA_CASE(10);
        FA_CASE(15);
        FA_CASE(20);
        FA_CASE(35);
#undef FA_CASE
        default: return launch_sum_rows<0, T>(gdof, ldof, ptr, adj, indptr, pos, lmax, elem, cpad, values, s);
    }
}

template <class T, int G>
static int launch_gather(int64_t gdof, int ldof, const int32_t* c2d, const int32_t* ptr, const int32_t* adj,
                         const int32_t* indptr, const int32_t* indices, int lmax, const void* elem, int64_t cstride,
                         void* values, hipStream_t s) {
    const size_t per_row = (sizeof(int32_t) + sizeof(double)) * lmax;
    int rpb = 256 / G;
    while (rpb > 1 && rpb * per_row + 16 > 48 * 1024) rpb >>= 1;
    const size_t lds = align_up(sizeof(int32_t) * rpb * lmax, 16) + sizeof(double) * rpb * lmax;
    if (lds > 160 * 1024) {
        set_error("fa_gather_matrix: row length %d exceeds the LDS capacity", lmax);
        return FA_ECAPACITY;
    }
    auto k = k_gather_matrix<T, G>;
    if (lds > 64 * 1024)
        FA_HIP(hipFuncSetAttribute(reinterpret_cast<const void*>(k), hipFuncAttributeMaxDynamicSharedMemorySize,
                                   static_cast<int>(lds)));
    const unsigned grid = grid_for(gdof, rpb, 1 << 20);
    hipLaunchKernelGGL(k, dim3(grid), dim3(rpb * G), lds, s, gdof, ldof, c2d, ptr, adj, indptr,
                       indices, lmax, static_cast<const T*>(elem), cstride, static_cast<T*>(values));
    FA_LAUNCH("k_gather_matrix");
    return FA_OK;
}

template <class T>
static int dispatch_gather(int64_t gdof, int ldof, const int32_t* c2d, const int32_t* ptr, const int32_t* adj,
                           const int32_t* indptr, const int32_t* indices, int lmax, const void* elem, int64_t cs,
                           void* values, hipStream_t s) {
    if (ldof <= 4) return launch_gather<T, 4>(gdof, ldof, c2d, ptr, adj, indptr, indices, lmax, elem, cs, values, s);
    if (ldof <= 8) return launch_gather<T, 8>(gdof, ldof, c2d, ptr, adj, indptr, indices, lmax, elem, cs, values, s);
    if (ldof <= 16)
        return launch_gather<T, 16>(gdof, ldof, c2d, ptr, adj, indptr, indices, lmax, elem, cs, values, s);
    if (ldof <= 32)
        return launch_gather<T, 32>(gdof, ldof, c2d, ptr, adj, indptr, indices, lmax, elem, cs, values, s);
    return launch_gather<T, 64>(gdof, ldof, c2d, ptr, adj, indptr, indices, lmax, elem, cs, values, s);
}

}  // namespace fa

using namespace fa;

extern "C" int fa_gather_matrix(int dtype, int64_t gdof, int32_t ldof, const int32_t* cell2dof,
                                const int32_t* adj_ptr, const int32_t* adj, const int32_t* indptr,
                                const int32_t* indices, int32_t max_row, const void* elem, int64_t elem_stride,
                                void* values, fa_stream_t stream) {
    FA_REQUIRE(dtype == FA_F64 || dtype == FA_F32, "fa_gather_matrix: bad dtype %d", dtype);
    FA_REQUIRE(gdof > 0 && ldof > 0 && max_row > 0, "fa_gather_matrix: bad sizes");
    const int64_t cs = elem_stride > 0 ? elem_stride : (int64_t)ldof * ldof;
    FA_REQUIRE(cs >= (int64_t)ldof * ldof, "fa_gather_matrix: element stride %lld < ldof^2", (long long)cs);
    if (dtype == FA_F64)
        return dispatch_gather<double>(gdof, ldof, cell2dof, adj_ptr, adj, indptr, indices, max_row, elem, cs, values,
                                       S(stream));
    return dispatch_gather<float>(gdof, ldof, cell2dof, adj_ptr, adj, indptr, indices, max_row, elem, cs, values,
                                  S(stream));
}

extern "C" int fa_row_positions(int64_t gdof, int32_t ldof, const int32_t* cell2dof, const int32_t* adj_ptr,
                                const int32_t* adj, const int32_t* indptr, const int32_t* indices, int32_t max_row,
                                uint16_t* pos, fa_stream_t stream) {
    FA_REQUIRE(gdof > 0 && ldof > 0 && max_row > 0, "fa_row_positions: bad sizes");
    int waves = 4;
    while (waves > 1 && waves * sizeof(int32_t) * max_row > 64 * 1024) waves >>= 1;
    const size_t lds = waves * sizeof(int32_t) * max_row;
    if (lds > 64 * 1024) {
        set_error("fa_row_positions: row length %d exceeds the LDS capacity", max_row);
        return FA_ECAPACITY;
    }
    hipLaunchKernelGGL(k_row_positions, dim3(grid_for(gdof, waves, 1 << 20)), dim3(waves * WAVE), lds, S(stream), gdof,
                       ldof, cell2dof, adj_ptr, adj, indptr, indices, max_row, pos);
    FA_LAUNCH("k_row_positions");
    return FA_OK;
}

extern "C" int fa_sum_rows(int dtype, int64_t gdof, int32_t ldof, const int32_t* adj_ptr, const int32_t* adj,
                           const int32_t* indptr, const uint16_t* pos, int32_t max_row, const void* elem,
                           int64_t elem_stride, void* values, fa_stream_t stream) {
    FA_REQUIRE(dtype == FA_F64 || dtype == FA_F32, "fa_sum_rows: bad dtype %d", dtype);
    FA_REQUIRE(gdof > 0 && ldof > 0 && max_row > 0, "fa_sum_rows: bad sizes");
    const int64_t dense = (int64_t)ldof * ldof, cpad = elem_stride > 0 ? elem_stride - dense : 0;
    FA_REQUIRE(cpad >= 0, "fa_sum_rows: element stride %lld < ldof^2", (long long)elem_stride);
    if (dtype == FA_F64)
        return dispatch_sum_rows<double>(gdof, ldof, adj_ptr, adj, indptr, pos, max_row, elem, cpad, values, S(stream));
    return dispatch_sum_rows<float>(gdof, ldof, adj_ptr, adj, indptr, pos, max_row, elem, cpad, values, S(stream));
}
