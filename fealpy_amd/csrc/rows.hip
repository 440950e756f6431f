// Assembly of CSR rows straight from a record per cell, with no element
// matrices in between: scalar diffusion + mass whose coefficient is constant on
// each cell, and isotropic linear elasticity.
#include "cell.hpp"
#include "common.hpp"

#include <algorithm>

namespace fa {

// Where an element matrix is the same for every cell up to the cell's metric
// (a coefficient constant on each cell), a record per cell says all of it:
//   P1 diffusion + mass: the matrix itself, the (TD + 1)(TD + 2) / 2 entries
//     i <= j (80 bytes in 3D), an 8-byte read an entry;
//   elasticity: grad lambda_1.. and |T| (80 bytes in 3D), about 100 FP64
//     operations a TD x TD block, against 30 x 30 doubles a P2 tetrahedron
//     written and read as an element matrix.
//
// The sum: ldof lanes (P1: four) per row, consecutive rows at a time in a wave,
// whose CSR entries are one contiguous range, held in LDS as it is stored
// (FP64).  Lane j adds entry (i, j) of the row's incident cells in ascending
// order, the order of the reference's stable lexsort + sequential np.add.at.
// The additions of one wave to LDS are done in the order it issues them, so
// they are LDS adds without a result (ds_add_f64) and nothing waits for them;
// the columns of one cell never collide.  What bounds it is the chain incidence
// -> record: incidences are read two steps ahead and records one.
// Workgroups go to the XCDs in windows (xcd_window_block): one contiguous range
// an XCD took twice as long, vertex rows having most of the incidences.
// 40^3 P2 elasticity: element matrices + sum 2.46 ms -> 0.62 ms (1.1 GB in and
// out, 1.8 TB/s); P1 on 2.26M shuffled tetrahedra: 292 -> 217 us.
__device__ inline void lds_add(double* p, double v) {
    __hip_atomic_fetch_add(p, v, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
}

__device__ inline void wave_lds_fence() {
    __builtin_amdgcn_wave_barrier();
    __builtin_amdgcn_fence(__ATOMIC_SEQ_CST, "wavefront");
}

template <int TD>
__device__ inline void load_cell_wide(const double* __restrict__ nodew, const int32_t* __restrict__ cell, int64_t c,
                                      double p[TD + 1][TD]) {
    int32_t v[TD + 1];
#pragma unroll
    for (int a = 0; a < TD + 1; ++a) v[a] = cell[c * (TD + 1) + a];
#pragma unroll
    for (int a = 0; a < TD + 1; ++a) {
        if constexpr (TD == 3) {
            const double4 t = reinterpret_cast<const double4*>(nodew)[v[a]];
            p[a][0] = t.x;
            p[a][1] = t.y;
            p[a][2] = t.z;
        } else {
            const double2 t = reinterpret_cast<const double2*>(nodew)[v[a]];
            p[a][0] = t.x;
            p[a][1] = t.y;
        }
    }
}

// The P1 record: the element matrix, entries i <= j in row order.  Records
// leave through LDS, so that a wave's stores are contiguous.
template <int TD>
struct P1Rec {
    static constexpr int SIZE = (TD + 1) * (TD + 2) / 2;
};

template <int TD>
__global__ void __launch_bounds__(256) k_p1_records(int64_t nc, const double* __restrict__ nodew,
                                                    const int32_t* __restrict__ cell, const double* __restrict__ tab,
                                                    int dk, double ds, const double* __restrict__ dc, int mk, double ms,
                                                    const double* __restrict__ mc, double* __restrict__ rec) {
    constexpr int NS = TD * (TD + 1) / 2, NV = TD + 1, SIZE = P1Rec<TD>::SIZE;
    __shared__ double stage[256 * SIZE];
    const int64_t c0 = blockIdx.x * (int64_t)256, c = c0 + threadIdx.x;
    if (c < nc) {
        double p[TD + 1][TD];
        load_cell_wide<TD>(nodew, cell, c, p);
        const double kd = coef_value(dk, ds, dc, c, 0, 1), km = coef_value(mk, ms, mc, c, 0, 1);
        Geom<TD> g;
        g.compute(p);
        double h[NS];
        int u = 0;
#pragma unroll
        for (int a = 0; a < TD; ++a)
#pragma unroll
            for (int b = a; b < TD; ++b, ++u) {
                double s = 0.0;
#pragma unroll
                for (int d = 0; d < TD; ++d) s += g.gl[a + 1][d] * g.gl[b + 1][d];
                h[u] = kd * g.meas * s;
            }
        const double m = km * g.meas;
        int e = 0;
#pragma unroll
        for (int i = 0; i < NV; ++i)
#pragma unroll
            for (int j = i; j < NV; ++j, ++e) {
                const double* t = tab + i * NV + j;
                double v = 0.0;
                if (dk) {
#pragma unroll
                    for (int s = 0; s < NS; ++s) v += h[s] * t[s * NV * NV];
                }
                if (mk) v += m * t[NS * NV * NV];
                stage[threadIdx.x * SIZE + e] = v;
            }
    }
    __syncthreads();
    const int n = static_cast<int>(nc - c0 < 256 ? nc - c0 : 256) * SIZE;
    for (int t = threadIdx.x; t < n; t += 256) rec[c0 * SIZE + t] = stage[t];
}

// P1 rows: four lanes per row, 16 rows at a time in a wave.  Lane j of a quad
// reads incidence and positions of one of four incidences for all (quad
// broadcasts hand them out: a load an incidence less 3 in 4), then entry (i, j)
// of each.
template <int U>
__device__ inline int quad(int v) {  // lane U of the quad's value
    return __builtin_amdgcn_update_dpp(0, v, U * 0x55, 0xf, 0xf, true);
}

template <int TD, class T>
__global__ void __launch_bounds__(256) k_p1_rows(int64_t gdof, const int32_t* __restrict__ ptr,
                                                 const int32_t* __restrict__ adj, const int32_t* __restrict__ indptr,
                                                 const uint16_t* __restrict__ pos, int cap,
                                                 const double* __restrict__ rec, T* __restrict__ values) {
    constexpr int NV = TD + 1, SIZE = P1Rec<TD>::SIZE;
    extern __shared__ double lds[];
    const int lane = threadIdx.x % WAVE, wave = threadIdx.x / WAVE;
    double* acc = lds + wave * cap;
    const int sub = lane / 4, j = lane % 4;
    const int64_t base = ((int64_t)xcd_window_block() * (blockDim.x / WAVE) + wave) * 16;
    if (base >= gdof) return;  // no block-wide wait below
    const int64_t r = min(base + sub, gdof), r1 = min(r + 1, gdof);
    const int32_t r0 = indptr[r], k0 = ptr[r], k1 = ptr[r1];
    const int32_t first = indptr[base], n = indptr[min(base + 16, gdof)] - first;
    for (int t = lane; t < n; t += WAVE) acc[t] = 0.0;
    wave_lds_fence();
    if (k0 < k1) {
        double* a = acc + (r0 - first);
        int32_t e;
        uint2 w;  // the four positions of the lane's incidence
        auto incidence = [&](int32_t k) {
            const int32_t ku = min(k + j, k1 - 1);
            e = adj[ku];
            const uint16_t* q = pos + (int64_t)ku * NV;
            if constexpr (TD == 3) {
                w = *reinterpret_cast<const uint2*>(q);
            } else {
                w.x = q[0] | (uint32_t)q[1] << 16;
                w.y = q[2];
            }
        };
        auto entries = [&](double (&x)[4], int (&p)[4]) {
            const int32_t c = e / NV, i = e - c * NV;
            const int jj = min(j, NV - 1);
            auto one = [&](int32_t cu, int iu, uint32_t lo, uint32_t hi, double& v, int& at) {
                const int l = min(iu, jj), h = max(iu, jj);
                v = rec[(int64_t)cu * SIZE + l * (2 * NV - 1 - l) / 2 + h];
                at = ((jj < 2 ? lo : hi) >> (16 * (jj & 1))) & 0xffff;
            };
            one(quad<0>(c), quad<0>(i), quad<0>(w.x), quad<0>(w.y), x[0], p[0]);
            one(quad<1>(c), quad<1>(i), quad<1>(w.x), quad<1>(w.y), x[1], p[1]);
            one(quad<2>(c), quad<2>(i), quad<2>(w.x), quad<2>(w.y), x[2], p[2]);
            one(quad<3>(c), quad<3>(i), quad<3>(w.x), quad<3>(w.y), x[3], p[3]);
        };
        auto add = [&](int32_t k, const double (&x)[4], const int (&p)[4]) {
#pragma unroll
            for (int u = 0; u < 4; ++u)
                if (k + u < k1 && j < NV) lds_add(a + p[u], x[u]);
        };
        double h[4], hn[4];
        int p[4], pn[4];
        incidence(k0);
        entries(h, p);
        incidence(k0 + 4);
        for (int32_t k = k0; k < k1; k += 8) {  // two steps a turn: one's loads beside the other's adds
            entries(hn, pn);
            incidence(k + 8);
            add(k, h, p);
            entries(h, p);
            incidence(k + 12);
            add(k + 4, hn, pn);
        }
    }
    wave_lds_fence();
    for (int t = lane; t < n; t += WAVE) values[first + t] = static_cast<T>(acc[t]);
}

// A wave's chunk of up to ROWS_CHUNK rows: lane l holds the entry and incidence
// pointers of row l (and, past the last row, their ends).
constexpr int ROWS_CHUNK = 32;
static_assert(ROWS_CHUNK < WAVE, "a lane per row of a chunk, and one for the end");

// one round: the rows [s0, s1) of a chunk of n that fit the lanes and `cap`
// doubles, B of them per CSR entry of the row pointers `ip`
template <int LDOF, int B>
__device__ inline int round_end(int32_t ip, int s0, int n, int cap) {
    constexpr int NR = WAVE / LDOF;
    const int lane = threadIdx.x % WAVE;
    const int32_t first = __shfl(ip, s0);  // before the tests: every lane takes part
    const bool fits = lane > s0 && lane <= min(s0 + NR, n) && (ip - first) * B <= cap;
    // row pointers ascend, so the fitting rows are the first; `cap` takes the longest row, so there is one
    return s0 + max(1, static_cast<int>(__popcll(__ballot(fits))));
}

// The elasticity record: grad lambda_1.. and |T| (10 doubles in 3D, 5 in 2D, padded to 6)
template <int TD>
struct ElRec {
    static constexpr int SIZE = TD == 3 ? 10 : 6;
};

template <int TD>
__global__ void __launch_bounds__(256) k_elasticity_records(int64_t nc, const double* __restrict__ nodew,
                                                            const int32_t* __restrict__ cell,
                                                            double* __restrict__ rec) {
    constexpr int SIZE = ElRec<TD>::SIZE;
    const int64_t c = blockIdx.x * (int64_t)blockDim.x + threadIdx.x;
    if (c >= nc) return;
    double p[TD + 1][TD];
    load_cell_wide<TD>(nodew, cell, c, p);
    Geom<TD> g;
    g.compute(p);
    double out[SIZE];
#pragma unroll
    for (int e = 0; e < SIZE; ++e) out[e] = 0.0;
#pragma unroll
    for (int a = 0; a < TD; ++a)
#pragma unroll
        for (int d = 0; d < TD; ++d) out[a * TD + d] = g.gl[a + 1][d];
    out[TD * TD] = g.meas;
    double2* o = reinterpret_cast<double2*>(rec + c * SIZE);
#pragma unroll
    for (int e = 0; e < SIZE / 2; ++e) o[e] = double2{out[2 * e], out[2 * e + 1]};
}

// A vector space's scalar structure from its own lists: scalar row s has the
// TD rows `vrow(s, a)`, whose columns are the scalar row's, a component each.
// Component-interleaved (PRIO false): rows TD s + a, columns TD t + b;
// component blocks (PRIO true): rows a n + s, columns b L + t.
template <int TD, bool PRIO>
struct Vec {
    static __device__ int64_t first(int64_t s) { return PRIO ? s : TD * s; }
    static __device__ int64_t incidence(int64_t k) { return PRIO ? k : k / TD; }  // scalar incidence number
    static __device__ void split(int32_t e, int ldof, int32_t& c, int& i) {
        const int n = TD * ldof;
        c = e / n;
        i = e - c * n;
        if (!PRIO) i /= TD;
    }
};

// pos[k * ldof + j]: place of scalar column j of scalar incidence k in its scalar row
template <int TD, bool PRIO>
__global__ void __launch_bounds__(256) k_vector_positions(int64_t ns, int ldof, const int32_t* __restrict__ c2d,
                                                          const int32_t* __restrict__ ptr,
                                                          const int32_t* __restrict__ adj,
                                                          const int32_t* __restrict__ indptr,
                                                          const int32_t* __restrict__ indices, int lmax,
                                                          uint16_t* __restrict__ pos) {
    using V = Vec<TD, PRIO>;
    extern __shared__ int32_t cols_lds[];
    const int rpb = blockDim.x / WAVE, lane = threadIdx.x % WAVE;
    int32_t* cols = cols_lds + threadIdx.x / WAVE * lmax;
    for (int64_t s = (int64_t)blockIdx.x * rpb + threadIdx.x / WAVE; s < ns; s += (int64_t)gridDim.x * rpb) {
        const int64_t r = V::first(s);
        const int32_t r0 = indptr[r];
        const int L = (indptr[r + 1] - r0) / TD;
        for (int t = lane; t < L; t += WAVE) cols[t] = indices[r0 + (PRIO ? t : TD * t)];
        wave_lds_fence();
        const int64_t k0 = ptr[r], ks = V::incidence(k0);
        const int n = (ptr[r + 1] - ptr[r]) * ldof;
        for (int t = lane; t < n; t += WAVE) {
            const int u = t / ldof, j = t - u * ldof;
            int32_t c;
            int i;
            V::split(adj[k0 + u], ldof, c, i);
            const int32_t v = c2d[(int64_t)c * TD * ldof + (PRIO ? j : TD * j)];
            int lo = 0, hi = L;
            while (lo < hi) {
                const int mid = (lo + hi) >> 1;
                if (cols[mid] < v) lo = mid + 1;
                else hi = mid;
            }
            pos[ks * ldof + t] = static_cast<uint16_t>(lo);
        }
        wave_lds_fence();
    }
}

// Elasticity rows: ldof lanes per scalar row, lane j forms the TD x TD block
// of (i, j) of each incident cell,
//   A_de = |T| sum_{a,b >= 1} grad lambda_a[d] grad lambda_b[e] M[i][j][a][b]
// (M reduced as R'), combines it as the element kernel does (d == e: cA A_dd +
// cB of the others; else cC A_de + cD A_ed) and adds it to the scalar row's TD
// rows, all in LDS.
template <int TD, int LDOF, bool PRIO, class T>
__global__ void __launch_bounds__(512) k_elasticity_rows(int64_t ns, int chunk, const int32_t* __restrict__ ptr,
                                                         const int32_t* __restrict__ adj,
                                                         const int32_t* __restrict__ indptr,
                                                         const uint16_t* __restrict__ pos, int cap,
                                                         const double* __restrict__ tab, double cA, double cB,
                                                         double cC, double cD, const double* __restrict__ rec,
                                                         T* __restrict__ values) {
    using V = Vec<TD, PRIO>;
    constexpr int SIZE = ElRec<TD>::SIZE, B = TD * TD, NN = LDOF * LDOF;
    extern __shared__ double lds[];
    for (int e = threadIdx.x; e < B * NN; e += blockDim.x) lds[e] = tab[e];
    __syncthreads();
    const int lane = threadIdx.x % WAVE, wave = threadIdx.x / WAVE;
    double* acc = lds + B * NN + wave * cap;
    const int sub = lane / LDOF, j = lane - sub * LDOF;
    const int64_t base = ((int64_t)xcd_window_block() * (blockDim.x / WAVE) + wave) * chunk;
    if (base >= ns) return;  // no block-wide wait below
    const int rows = static_cast<int>(min((int64_t)chunk, ns - base));
    const int64_t r = V::first(base + min(lane, rows));
    const int32_t ip = indptr[r] / (PRIO ? TD : B), pp = ptr[r];  // scalar entry pointer; the first component's incidences
    for (int s0 = 0; s0 < rows;) {
        const int s1 = round_end<LDOF, B>(ip, s0, rows, cap);
        const int32_t first = __shfl(ip, s0), n = __shfl(ip, s1) - first;
        for (int t = lane; t < n * B; t += WAVE) acc[t] = 0.0;
        const int mine = min(s0 + sub, rows), next = min(mine + 1, rows);
        const int32_t q0 = __shfl(ip, mine) - first, L = __shfl(ip, next) - first - q0;
        const int32_t k0 = __shfl(pp, mine);
        // incidences of one component's row: the next row's first less the other components'
        const int32_t deg = PRIO ? __shfl(pp, next) - k0 : (__shfl(pp, next) - k0) / TD;
        wave_lds_fence();
        if (s0 + sub < s1 && deg > 0) {
            const uint16_t* pr = pos + V::incidence(k0) * LDOF + j;
            double* a = acc + (PRIO ? TD * q0 : B * q0);
            const int drow = PRIO ? TD * n : TD * L, dcol = PRIO ? L : 1, dpos = PRIO ? 1 : TD;
            // incidences are read two steps ahead, records one
            int32_t e = adj[k0];
            int p = pr[0], pn;
            int i, in;
            double h[SIZE], hn[SIZE];
            auto record = [&](double (&x)[SIZE], int& at) {
                int32_t c;
                V::split(e, LDOF, c, at);
                const double2* q = reinterpret_cast<const double2*>(rec + (int64_t)c * SIZE);
#pragma unroll
                for (int d = 0; d < SIZE / 2; ++d) {
                    const double2 y = q[d];
                    x[2 * d] = y.x;
                    x[2 * d + 1] = y.y;
                }
            };
            record(h, i);
            e = adj[k0 + min(1, deg - 1)];
            pn = pr[min(1, deg - 1) * LDOF];
            auto add = [&](const double (&h)[SIZE], int i, int p) {
                const double* m = lds + i * LDOF + j;
                double tm[TD][TD];
#pragma unroll
                for (int x = 0; x < TD; ++x)
#pragma unroll
                    for (int y = 0; y < TD; ++y) {
                        double t = 0.0;
#pragma unroll
                        for (int b = 0; b < TD; ++b) t += m[(x * TD + b) * NN] * h[b * TD + y];
                        tm[x][y] = t;
                    }
                double A[TD][TD];
#pragma unroll
                for (int x = 0; x < TD; ++x)
#pragma unroll
                    for (int y = 0; y < TD; ++y) {
                        double t = 0.0;
#pragma unroll
                        for (int b = 0; b < TD; ++b) t += h[b * TD + x] * tm[b][y];
                        A[x][y] = h[B] * t;
                    }
                double* o = a + dpos * p;
#pragma unroll
                for (int x = 0; x < TD; ++x)
#pragma unroll
                    for (int y = 0; y < TD; ++y) {
                        double v;
                        if (x == y) {
                            double others = 0.0;
#pragma unroll
                            for (int f = 0; f < TD; ++f)
                                if (f != x) others += A[f][f];
                            v = cA * A[x][x] + cB * others;
                        } else {
                            v = cC * A[x][y] + cD * A[y][x];
                        }
                        lds_add(o + x * drow + y * dcol, v);
                    }
            };
            // two steps a turn: the registers of one step are loaded while the other's are added
            for (int32_t k = 0; k < deg; k += 2) {
                int q = p;
                record(hn, in);
                int32_t kn = min(k + 2, deg - 1);
                e = adj[k0 + kn];
                p = pr[kn * LDOF];
                add(h, i, q);
                if (k + 1 >= deg) break;
                q = pn;
                record(h, i);
                kn = min(k + 3, deg - 1);
                e = adj[k0 + kn];
                pn = pr[kn * LDOF];
                add(hn, in, q);
            }
        }
        wave_lds_fence();
        if constexpr (PRIO) {
#pragma unroll
            for (int d = 0; d < TD; ++d) {
                const int64_t o = indptr[d * ns + base + s0];
                for (int t = lane; t < TD * n; t += WAVE) values[o + t] = static_cast<T>(acc[d * TD * n + t]);
            }
        } else {
            for (int t = lane; t < B * n; t += WAVE) values[(int64_t)first * B + t] = static_cast<T>(acc[t]);
        }
        wave_lds_fence();
        s0 = s1;
    }
}

// A launch: the block's LDS holds the table and `cap` doubles per wave -- the
// longest row's entries at least, else what a wave's rows take on average and a
// quarter more, up to 16 KB -- and the block size is the one that puts the most
// waves on a CU.  Short chunks where there are few rows, so that they still
// spread over the chip.
struct RowsLaunch {
    int waves = 0, cap = 0, chunk = 0;
    size_t lds = 0;
    unsigned grid = 0;
};

inline bool rows_launch(size_t table_doubles, int64_t longest, int64_t entries, int64_t rows, int at_once, RowsLaunch& o) {
    const int64_t mean = entries * at_once * 5 / (4 * rows) + 1;
    o.cap = static_cast<int>(std::max(longest, std::min<int64_t>({2048, mean, longest * at_once})));
    int best = 0;
    for (int w = 1; w <= 8; w <<= 1) {
        const size_t lds = sizeof(double) * (table_doubles + (size_t)w * o.cap);
        if (lds > 160 * 1024) break;
        const int resident = w * std::min<int>(static_cast<int>(160 * 1024 / lds), 32 / w);
        if (resident >= best) {
            best = resident;
            o.waves = w;
            o.lds = lds;
        }
    }
    if (!o.waves) return false;
    const int64_t even = (rows + 256 * 16 - 1) / (256 * 16);
    o.chunk = static_cast<int>(std::min<int64_t>(ROWS_CHUNK, std::max<int64_t>(at_once, even)));
    o.grid = xcd_window_grid(static_cast<unsigned>((rows + (int64_t)o.waves * o.chunk - 1) / ((int64_t)o.waves * o.chunk)));
    return true;
}

template <class K>
static int lds_limit(K k, size_t lds) {
    if (lds > 64 * 1024)
        FA_HIP(hipFuncSetAttribute(reinterpret_cast<const void*>(k), hipFuncAttributeMaxDynamicSharedMemorySize,
                                   static_cast<int>(lds)));
    return FA_OK;
}

template <int TD, class T>
static int launch_p1_rows(int64_t gdof, int64_t nc, const double* nodew, const int32_t* cell, const double* tab, int dk,
                          double ds, const double* dc, int mk, double ms, const double* mc, const int32_t* ptr,
                          const int32_t* adj, const int32_t* indptr, const uint16_t* pos, int max_row, double* rec,
                          void* values, hipStream_t s) {
    const int cap = 16 * max_row;  // 16 rows, whatever their lengths
    int waves = 4;
    while (waves > 1 && sizeof(double) * waves * cap > 40 * 1024) waves >>= 1;
    const size_t lds = sizeof(double) * waves * cap;
    if (lds > 160 * 1024) {
        set_error("fa_assemble_p1_rows: row length %d exceeds the LDS capacity", max_row);
        return FA_ECAPACITY;
    }
    timer_begin(FA_TIMER_P1_ROWS, s);
    hipLaunchKernelGGL(k_p1_records<TD>, dim3(static_cast<unsigned>((nc + 255) / 256)), dim3(256), 0, s, nc, nodew, cell,
                       tab, dk, ds, dc, mk, ms, mc, rec);
    timer_end(FA_TIMER_P1_ROWS, s);
    FA_LAUNCH("k_p1_records");
    auto k = k_p1_rows<TD, T>;
    if (const int st = lds_limit(k, lds)) return st;
    const unsigned grid = xcd_window_grid(static_cast<unsigned>((gdof + 16 * waves - 1) / (16 * waves)));
    timer_begin(FA_TIMER_P1_SUM_ROWS, s);
    hipLaunchKernelGGL(k, dim3(grid), dim3(waves * WAVE), lds, s, gdof, ptr, adj, indptr, pos, cap, rec,
                       static_cast<T*>(values));
    timer_end(FA_TIMER_P1_SUM_ROWS, s);
    FA_LAUNCH("k_p1_rows");
    return FA_OK;
}

template <int TD, int LDOF, bool PRIO, class T>
static int launch_elasticity_rows(int64_t ns, int64_t nnz, const double* tab, double cA, double cB, double cC,
                                  double cD, const int32_t* ptr, const int32_t* adj, const int32_t* indptr,
                                  const uint16_t* pos, int max_row, const double* rec, void* values, hipStream_t s) {
    RowsLaunch l;
    if (!rows_launch(TD * TD * LDOF * LDOF, (int64_t)TD * max_row, nnz, ns, WAVE / LDOF, l)) {
        set_error("fa_assemble_elasticity_rows: row length %d exceeds the LDS capacity", max_row);
        return FA_ECAPACITY;
    }
    auto k = k_elasticity_rows<TD, LDOF, PRIO, T>;
    if (const int st = lds_limit(k, l.lds)) return st;
    hipLaunchKernelGGL(k, dim3(l.grid), dim3(l.waves * WAVE), l.lds, s, ns, l.chunk, ptr, adj, indptr, pos, l.cap, tab,
                       cA, cB, cC, cD, rec, static_cast<T*>(values));
    FA_LAUNCH("k_elasticity_rows");
    return FA_OK;
}

}  // namespace fa

using namespace fa;

extern "C" size_t fa_p1_records_bytes(int td, int64_t nc) { return sizeof(double) * (td == 3 ? 10 : 6) * nc; }

extern "C" int fa_assemble_p1_rows(int dtype, int td, int64_t gdof, int64_t nc, const double* node_wide,
                                   const int32_t* cell, const double* table, int diff_kind, double diff_scale,
                                   const double* diff_coef, int mass_kind, double mass_scale, const double* mass_coef,
                                   const int32_t* adj_ptr, const int32_t* adj, const int32_t* indptr,
                                   const uint16_t* pos, int32_t max_row, void* records, size_t records_bytes,
                                   void* values, fa_stream_t stream) {
    FA_REQUIRE(dtype == FA_F64 || dtype == FA_F32, "fa_assemble_p1_rows: bad dtype %d", dtype);
    FA_REQUIRE(td == 2 || td == 3, "fa_assemble_p1_rows: td must be 2 or 3");
    FA_REQUIRE(gdof > 0 && nc > 0 && max_row > 0, "fa_assemble_p1_rows: bad sizes");
    FA_REQUIRE(mass_kind <= FA_COEF_CELL && diff_kind <= FA_COEF_CELL,
               "fa_assemble_p1_rows: a coefficient that varies on a cell");
    FA_REQUIRE((diff_kind < FA_COEF_CELL || diff_coef) && (mass_kind < FA_COEF_CELL || mass_coef),
               "fa_assemble_p1_rows: coefficient array missing");
    if (!records || records_bytes < fa_p1_records_bytes(td, nc)) {
        set_error("fa_assemble_p1_rows: records of %zu bytes, %zu needed", records_bytes, fa_p1_records_bytes(td, nc));
        return FA_ENOMEM;
    }
    auto f = td == 2 ? (dtype == FA_F64 ? launch_p1_rows<2, double> : launch_p1_rows<2, float>)
                     : (dtype == FA_F64 ? launch_p1_rows<3, double> : launch_p1_rows<3, float>);
    return f(gdof, nc, node_wide, cell, table, diff_kind, diff_scale, diff_coef, mass_kind, mass_scale, mass_coef,
             adj_ptr, adj, indptr, pos, max_row, static_cast<double*>(records), values, S(stream));
}

extern "C" int fa_vector_positions(int td, int dof_priority, int64_t ndof, int32_t ldof, const int32_t* cell2dof,
                                   const int32_t* adj_ptr, const int32_t* adj, const int32_t* indptr,
                                   const int32_t* indices, int32_t max_row, uint16_t* pos, fa_stream_t stream) {
    FA_REQUIRE(td == 2 || td == 3, "fa_vector_positions: td must be 2 or 3");
    FA_REQUIRE(ndof > 0 && ldof > 0 && max_row > 0 && max_row % td == 0, "fa_vector_positions: bad sizes");
    const int lmax = max_row / td;
    int waves = 4;
    while (waves > 1 && waves * sizeof(int32_t) * lmax > 64 * 1024) waves >>= 1;
    const size_t lds = waves * sizeof(int32_t) * lmax;
    if (lds > 64 * 1024) {
        set_error("fa_vector_positions: row length %d exceeds the LDS capacity", lmax);
        return FA_ECAPACITY;
    }
    const unsigned grid = grid_for(ndof, waves, 1 << 20);
#define FA_VP(TD_, PR_)                                                                                          \
    hipLaunchKernelGGL((k_vector_positions<TD_, PR_>), dim3(grid), dim3(waves * WAVE), lds, S(stream), ndof, ldof, \
                       cell2dof, adj_ptr, adj, indptr, indices, lmax, pos)
    if (td == 2) {
        if (dof_priority) FA_VP(2, true);
        else FA_VP(2, false);
    } else {
        if (dof_priority) FA_VP(3, true);
        else FA_VP(3, false);
    }
#undef FA_VP
    FA_LAUNCH("k_vector_positions");
    return FA_OK;
}

extern "C" size_t fa_elasticity_records_bytes(int td, int64_t nc) { return sizeof(double) * (td == 3 ? 10 : 6) * nc; }

extern "C" int fa_assemble_elasticity_rows(int dtype, int td, int dof_priority, int64_t ndof, int64_t nc, int32_t ldof,
                                           const double* node_wide, const int32_t* cell, const double* table, double cA,
                                           double cB, double cC, double cD, const int32_t* adj_ptr,
                                           const int32_t* adj, const int32_t* indptr, int64_t nnz, const uint16_t* pos,
                                           int32_t max_row, void* records, size_t records_bytes, void* values,
                                           fa_stream_t stream) {
    FA_REQUIRE(dtype == FA_F64 || dtype == FA_F32, "fa_assemble_elasticity_rows: bad dtype %d", dtype);
    FA_REQUIRE(td == 2 || td == 3, "fa_assemble_elasticity_rows: td must be 2 or 3");
    FA_REQUIRE(ndof > 0 && nc > 0 && nnz > 0 && max_row > 0 && max_row % td == 0,
               "fa_assemble_elasticity_rows: bad sizes");
    if (!records || records_bytes < fa_elasticity_records_bytes(td, nc)) {
        set_error("fa_assemble_elasticity_rows: records of %zu bytes, %zu needed", records_bytes,
                  fa_elasticity_records_bytes(td, nc));
        return FA_ENOMEM;
    }
    hipStream_t s = S(stream);
    double* rec = static_cast<double*>(records);
    const unsigned rgrid = static_cast<unsigned>((nc + 255) / 256);
    if (td == 2)
        hipLaunchKernelGGL(k_elasticity_records<2>, dim3(rgrid), dim3(256), 0, s, nc, node_wide, cell, rec);
    else
        hipLaunchKernelGGL(k_elasticity_records<3>, dim3(rgrid), dim3(256), 0, s, nc, node_wide, cell, rec);
    FA_LAUNCH("k_elasticity_records");
#define FA_CASE(TD_, L_)                                                                                         \
    if (td == TD_ && ldof == L_) {                                                                               \
        auto f = dof_priority ? (dtype == FA_F64 ? launch_elasticity_rows<TD_, L_, true, double>                 \
                                                 : launch_elasticity_rows<TD_, L_, true, float>)                 \
                              : (dtype == FA_F64 ? launch_elasticity_rows<TD_, L_, false, double>                \
                                                 : launch_elasticity_rows<TD_, L_, false, float>);               \
        return f(ndof, nnz, table, cA, cB, cC, cD, adj_ptr, adj, indptr, pos, max_row, rec, values, s);          \
    }
    FA_CASE(2, 3) FA_CASE(2, 6) FA_CASE(2, 10) FA_CASE(2, 15) FA_CASE(3, 4) FA_CASE(3, 10) FA_CASE(3, 20)
#undef FA_CASE
    set_error("fa_assemble_elasticity_rows: unsupported (td=%d, ldof=%d); p must be 1..4 (1..3 in 3D)", td, ldof);
    return FA_EINVAL;
}
