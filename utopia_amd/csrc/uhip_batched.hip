// Batched, multi-right-hand-side kernels: many independent SPD systems stored
// as one block-diagonal CSR matrix (segments of rows), K right-hand sides per
// system stored row-major (entry (i, j) at i*K + j).
//
//   SpMM      a few lanes per row share its K right-hand sides, 16 bytes of
//             them each.
//   segdot    per (segment, column) dot products, two fixed-order stages.
//   batched CG / Chebyshev steps with per-(segment, column) step lengths.
#include <algorithm>

#include "uhip_common.hpp"

namespace uhip {

// A kernel of the batched family returns at once when the context's gate (a device
// counter, uhip_ctx_set_gate) reads 0: a captured run of CG iterations then costs
// only its launches once every (system, rhs) pair has converged.
#define UHIP_GATE() \
    if (gate && *gate == 0) return

// SpMM: the lanes of a row hold V of its K columns each, V * sizeof(TX) being 16 bytes where K is large
// enough (2 FP64, 4 FP32), so the gathered x entries of a column index are one contiguous load across
// the row's lanes. (One thread per row for all K columns reads them 64 bytes apart.) It is bound by the chain of
// dependent loads and by memory: FP64 A p on 3.57M rows of 5 entries with 8 columns moves 683 MB in 175 us, its dot
// included (3.9 TB/s; before, 220 us and 86 for the dot). EB entries' loads are issued before their
// products are added, in entry order, so each column's sum is the sequential CSR sum.
template <int K, typename TX>
constexpr int spmm_cols() {
    return K * (int)sizeof(TX) >= 16 ? 16 / (int)sizeof(TX) : K;
}

// V entries of a row-major [n x K] array at (r, j0): 16-byte aligned where they span 16 bytes or more
// (hipMalloc'd base)
template <int K, int V, typename T>
__device__ __forceinline__ T *kcols(T *base, int32_t r, int j0) {
    T *p = base + (int64_t)r * K + j0;
    if constexpr (V * sizeof(T) >= 16) return (T *)__builtin_assume_aligned(p, 16);
    return p;
}

template <int K, int EB, typename TAcc, class Epi, typename TA, typename TX>
__device__ __forceinline__ void spmm_row(int32_t r, int j0, const int32_t *__restrict__ rowptr,
                                         const int32_t *__restrict__ col, const TA *__restrict__ val,
                                         const TX *__restrict__ X, const Epi &epi, double *part) {
    constexpr int V = spmm_cols<K, TX>();
    TAcc acc[V];
#pragma unroll
    for (int j = 0; j < V; ++j) acc[j] = TAcc(0);
    const int32_t e1 = rowptr[r + 1];
    for (int32_t e = rowptr[r]; e < e1; e += EB) {
        int32_t c[EB];
        TA v[EB];
        TX xv[EB][V];
#pragma unroll
        for (int u = 0; u < EB; ++u) {  // past the row's end: its last entry and x row 0, not added
            c[u] = col[min(e + u, e1 - 1)];
            v[u] = val[min(e + u, e1 - 1)];
            c[u] = e + u < e1 ? c[u] : 0;
        }
#pragma unroll
        for (int u = 0; u < EB; ++u) {
            const TX *xr = kcols<K, V>(X, c[u], j0);
#pragma unroll
            for (int j = 0; j < V; ++j) xv[u][j] = xr[j];
        }
#pragma unroll
        for (int u = 0; u < EB; ++u)
#pragma unroll
            for (int j = 0; j < V; ++j) {
                const TAcc t = acc[j] + (TAcc)v[u] * (TAcc)xv[u][j];
                acc[j] = e + u < e1 ? t : acc[j];
            }
    }
    epi.template apply<K, V>(r, j0, acc, part);
}

template <int K, int EB, typename TAcc, class Epi, typename TA, typename TX>
__global__ __launch_bounds__(256) void k_spmm_csr(const int32_t *__restrict__ gate, int32_t first, int32_t n,
                                                  const int32_t *__restrict__ rowptr,
                                                  const int32_t *__restrict__ col, const TA *__restrict__ val,
                                                  const TX *__restrict__ X, Epi epi) {
    UHIP_GATE();
    constexpr int V = spmm_cols<K, TX>(), L = K / V;
    const int b = xcd_remap(blockIdx.x, gridDim.x);
    const int32_t r = first + b * (256 / L) + (int32_t)threadIdx.x / L;
    if (r >= n) return;
    spmm_row<K, EB, TAcc, Epi, TA, TX>(r, (int)(threadIdx.x % L) * V, rowptr, col, val, X, epi, nullptr);
}

// Entries of a row taken at once, by the matrix' mean row length: whole rows up to 9 entries, equal parts of longer
// ones, so a row is one chain of loads (rowptr, entries, x) and few loads are spent on entries past its end. A mean of
// 2 to 2.5 is taken for a bilinear interpolation's rows of 1, 2 and 4. us a product of 2M rows, K = 8 FP64 / 1 FP32, one
// thread a row with 4 at once against this: rows of 2 78 / 10.9 -> 61 / 9.9 (4 at once 77 / 14.5), of 3 93 / 14.9 -> 69 /
// 13.2 (4: 76 / 15.9), of 5 121 / 21.3 -> 96 / 16.2, of 8 175 / 42.8 -> 136 / 34.8 (9: 139 / 39.1), bilinear 54.6 / 12.8
// -> 46.6 / 13.3 (3: 51.2 / 14.6); 300,000 rows of 12 43 / 12.9 -> 23 / 9.5 (9: 28 / 13.1).
#define UHIP_EB_SWITCH(A, ...)                                                   \
    switch (spmm_entries(A)) {                                                   \
        case 2: { constexpr int EB = 2; __VA_ARGS__; } break;                    \
        case 3: { constexpr int EB = 3; __VA_ARGS__; } break;                    \
        case 4: { constexpr int EB = 4; __VA_ARGS__; } break;                    \
        case 5: { constexpr int EB = 5; __VA_ARGS__; } break;                    \
        case 6: { constexpr int EB = 6; __VA_ARGS__; } break;                    \
        case 7: { constexpr int EB = 7; __VA_ARGS__; } break;                    \
        case 8: { constexpr int EB = 8; __VA_ARGS__; } break;                    \
        default: { constexpr int EB = 9; __VA_ARGS__; } break;                   \
    }
inline int spmm_entries(const uhip_csr *A) {
    const int64_t mean = (A->nnz + A->nrows - 1) / A->nrows;
    if (mean <= 2) return 2;
    if (2 * A->nnz <= 5 * (int64_t)A->nrows) return 4;
    const int64_t parts = (mean + 8) / 9;
    return (int)((mean + parts - 1) / parts);
}

// Sums over the workgroup's threads with the same column: thread t holds V columns from (t % L) * V. Fixed
// order; the K sums go to out.
template <int K, int V>
__device__ __forceinline__ void block_column_sums(double (&v)[V], double *__restrict__ out) {
    constexpr int L = K / V;
    __shared__ double red[4][K];
#pragma unroll
    for (int j = 0; j < V; ++j)
#pragma unroll
        for (int d = L; d < 64; d <<= 1) v[j] += __shfl_xor(v[j], d, 64);
    const int lane = threadIdx.x & 63;
    if (lane < L)
#pragma unroll
        for (int j = 0; j < V; ++j) red[threadIdx.x >> 6][lane * V + j] = v[j];
    __syncthreads();
    if (threadIdx.x < K) out[threadIdx.x] = ((red[0][threadIdx.x] + red[1][threadIdx.x]) + red[2][threadIdx.x]) + red[3][threadIdx.x];
}

// Rows of a reduction chunk (at most 1024 rows of one system) that a workgroup of the kernels with a dot takes:
// their partial sums, K per workgroup, need no look at where systems end.
constexpr int kChunkRows = 1024, kDotRows = 256, kDotGroups = kChunkRows / kDotRows;

// SpMM whose epilogue also adds a dot per column: workgroup 4 c + q takes rows 256 q .. of chunk c.
template <int K, int EB, typename TAcc, class Epi, typename TA, typename TX>
__global__ __launch_bounds__(256) void k_spmm_csr_dot(const int32_t *__restrict__ gate, const int32_t *__restrict__ c_row0,
                                                      const int32_t *__restrict__ c_row1,
                                                      const int32_t *__restrict__ rowptr,
                                                      const int32_t *__restrict__ col, const TA *__restrict__ val,
                                                      const TX *__restrict__ X, Epi epi,
                                                      double *__restrict__ partials) {
    UHIP_GATE();
    constexpr int V = spmm_cols<K, TX>(), L = K / V, ROWS = 256 / L;
    const int b = xcd_remap(blockIdx.x, gridDim.x);
    const int c = b / kDotGroups;
    const int32_t r0 = c_row0[c] + b % kDotGroups * kDotRows, r1 = min(c_row1[c], r0 + kDotRows);
    double part[V];
#pragma unroll
    for (int j = 0; j < V; ++j) part[j] = 0.0;
    for (int32_t r = r0 + (int32_t)threadIdx.x / L; r < r1; r += ROWS)
        spmm_row<K, EB, TAcc, Epi, TA, TX>(r, (int)(threadIdx.x % L) * V, rowptr, col, val, X, epi, part);
    block_column_sums<K, V>(part, partials + (int64_t)b * K);
}

// Epilogues on V columns of a row from j0 (all K of them for the wavefront kernel). They read all inputs
// before writing any output, so an output may alias an input of the same row (in-place updates).
template <typename TAcc, typename TY>
struct EpiKStore {
    TY *y;
    template <int K, int V>
    __device__ void apply(int32_t r, int j0, const TAcc *s, double *) const {
        TY *yr = kcols<K, V>(y, r, j0);
#pragma unroll
        for (int j = 0; j < V; ++j) yr[j] = (TY)s[j];
    }
};

// y = s with the dot of the product's input and its result
template <typename TAcc, typename TX, typename TY>
struct EpiKStoreDot {
    const TX *x;
    TY *y;
    template <int K, int V>
    __device__ void apply(int32_t r, int j0, const TAcc *s, double *part) const {
        const TX *xr = kcols<K, V>(x, r, j0);
        TY *yr = kcols<K, V>(y, r, j0);
#pragma unroll
        for (int j = 0; j < V; ++j) part[j] += (double)xr[j] * (double)s[j];
#pragma unroll
        for (int j = 0; j < V; ++j) yr[j] = (TY)s[j];
    }
};

template <typename TAcc, typename TY>
struct EpiKAdd {
    TY *y;
    template <int K, int V>
    __device__ void apply(int32_t r, int j0, const TAcc *s, double *) const {
        TY *yr = kcols<K, V>(y, r, j0);
        TY t[V];
#pragma unroll
        for (int j = 0; j < V; ++j) t[j] = yr[j];
#pragma unroll
        for (int j = 0; j < V; ++j) yr[j] = (TY)((TAcc)t[j] + s[j]);
    }
};

template <typename TAcc, typename TB, typename TY>
struct EpiKResidual {
    const TB *b;
    TY *y;
    template <int K, int V>
    __device__ void apply(int32_t r, int j0, const TAcc *s, double *) const {
        const TB *br = kcols<K, V>(b, r, j0);
        TB t[V];
#pragma unroll
        for (int j = 0; j < V; ++j) t[j] = br[j];
        TY *yr = kcols<K, V>(y, r, j0);
#pragma unroll
        for (int j = 0; j < V; ++j) yr[j] = (TY)((TAcc)t[j] - s[j]);
    }
};

// Chebyshev step (same algebra as the single-vector EpiCheb) with per-segment
// coefficients coef[3*seg + {0,1,2}] = (a_prev, beta, a_cur). DOT: xout . with (FP64), the z.r of the CG step that
// follows a preconditioner, while z is written.
template <typename TAcc, typename TP, typename TXO, bool DOT = false>
struct EpiKCheb {
    const TP *pprev;
    const TAcc *rprev;
    const TAcc *xin;
    TXO *xout;
    TAcc *rout;
    TAcc *pout;
    const int32_t *rowseg;
    const double *coef;
    int last;
    const double *with;
    template <int K, int V>
    __device__ void apply(int32_t r, int j0, const TAcc *s, double *part) const {
        const int32_t g = rowseg[r];
        const TAcc a_prev = (TAcc)coef[3 * g], beta = (TAcc)coef[3 * g + 1], a_cur = (TAcc)coef[3 * g + 2];
        TAcc pp[V], rp[V], xv[V];
        const TP *ppr = kcols<K, V>(pprev, r, j0);
#pragma unroll
        for (int j = 0; j < V; ++j) pp[j] = (TAcc)ppr[j];
        if (rprev) {
            const TAcc *rpr = kcols<K, V>(rprev, r, j0);
#pragma unroll
            for (int j = 0; j < V; ++j) rp[j] = rpr[j];
        } else {
#pragma unroll
            for (int j = 0; j < V; ++j) rp[j] = -pp[j];
        }
        if (xin) {
            const TAcc *xr = kcols<K, V>(xin, r, j0);
#pragma unroll
            for (int j = 0; j < V; ++j) xv[j] = xr[j];
        } else {
#pragma unroll
            for (int j = 0; j < V; ++j) xv[j] = TAcc(0);
        }
        TAcc rk[V], pk[V];
#pragma unroll
        for (int j = 0; j < V; ++j) {
            rk[j] = rp[j] + a_prev * s[j];
            pk[j] = -rk[j] + beta * pp[j];
            xv[j] = xv[j] + a_prev * pp[j];
        }
        if (last) {
#pragma unroll
            for (int j = 0; j < V; ++j) xv[j] = xv[j] + a_cur * pk[j];
        } else {
            TAcc *ro = kcols<K, V>(rout, r, j0), *po = kcols<K, V>(pout, r, j0);
#pragma unroll
            for (int j = 0; j < V; ++j) ro[j] = rk[j];
#pragma unroll
            for (int j = 0; j < V; ++j) po[j] = pk[j];
        }
        TXO *xo = kcols<K, V>(xout, r, j0);
        if constexpr (DOT) {
            const double *w = kcols<K, V>(with, r, j0);
#pragma unroll
            for (int j = 0; j < V; ++j) part[j] += (double)(TXO)xv[j] * w[j];
        }
#pragma unroll
        for (int j = 0; j < V; ++j) xo[j] = (TXO)xv[j];
    }
};

// Long rows (dense coarse blocks): one wavefront per row, lane l takes entries
// l, l+64, ... in order, and a fixed butterfly combines the lanes.
template <int K, typename TAcc, class Epi, typename TA, typename TX>
__global__ __launch_bounds__(256) void k_spmm_wave(const int32_t *__restrict__ gate, int32_t n, const int32_t *__restrict__ rowptr,
                                                   const int32_t *__restrict__ col, const TA *__restrict__ val,
                                                   const TX *__restrict__ X, Epi epi) {
    UHIP_GATE();
    const int b = xcd_remap(blockIdx.x, gridDim.x);
    const int32_t r = b * 4 + (int32_t)(threadIdx.x >> 6);
    const int l = threadIdx.x & 63;
    if (r >= n) return;
    TAcc acc[K];
#pragma unroll
    for (int j = 0; j < K; ++j) acc[j] = TAcc(0);
    const int32_t e1 = rowptr[r + 1];
    for (int32_t e = rowptr[r] + l; e < e1; e += 64) {
        const TAcc v = (TAcc)val[e];
        const TX *xr = kcols<K, K>(X, col[e], 0);
#pragma unroll
        for (int j = 0; j < K; ++j) acc[j] += v * (TAcc)xr[j];
    }
#pragma unroll
    for (int j = 0; j < K; ++j) acc[j] = wave_sum(acc[j]);
    if (l == 0) epi.template apply<K, K>(r, 0, acc, nullptr);
}

// Rows averaging >= 32 entries take the wavefront-per-row kernel (its sums are
// tree-ordered); all others the row-per-thread kernel (sequential CSR order),
// unless the matrix carries an autotuned choice (spmm_kernel 1 or 2).
template <int K, typename TAcc, class Epi, typename TA, typename TX>
int launch_spmm(uhip_ctx ctx, const uhip_csr *A, const TX *X, const Epi &e) {
    const int32_t n = A->nrows;
    if (n == 0) return UHIP_OK;
    if (uhip_spmm_by_wave(A)) {
        hipLaunchKernelGGL((k_spmm_wave<K, TAcc, Epi, TA, TX>), dim3((n + 3) / 4), dim3(256), 0, ctx->stream,
                           ctx->gate, n, A->rowptr, A->col, (const TA *)A->val, X, e);
    } else {
        constexpr int rows = 256 / (K / spmm_cols<K, TX>());
        // a launch has fewer than 2^32 threads: at 8 lanes a row (16 FP64 columns) less than 2^29 rows
        constexpr int64_t piece = (int64_t(1) << 23) * rows;
        for (int64_t first = 0; first < n; first += piece) {
            const unsigned g = (unsigned)((std::min<int64_t>(piece, n - first) + rows - 1) / rows);
            UHIP_EB_SWITCH(A, hipLaunchKernelGGL((k_spmm_csr<K, EB, TAcc, Epi, TA, TX>), dim3(g), dim3(256), 0, ctx->stream,
                                                 ctx->gate, (int32_t)first, n, A->rowptr, A->col, (const TA *)A->val, X, e));
        }
    }
    UHIP_CHECK_LAUNCH();
    return UHIP_OK;
}

// ---- segmented dots: out[s*K + j] = sum_{i in seg s} x[i,j] * y[i,j] ----
// Chunks of rows never straddle a segment; chunk c covers [c_row0[c], c_row1[c]).
template <int K, typename TX, typename TY>
__global__ __launch_bounds__(256) void k_segdot_chunk(const int32_t *__restrict__ gate, const int32_t *__restrict__ c_row0,
                                                      const int32_t *__restrict__ c_row1, const TX *__restrict__ x,
                                                      const TY *__restrict__ y, double *__restrict__ partials) {
    UHIP_GATE();
    constexpr int RPB = 256 / K;
    __shared__ double red[256];
    const int c = blockIdx.x;
    const int32_t r0 = c_row0[c], r1 = c_row1[c];
    const int j = threadIdx.x % K, ro = threadIdx.x / K;
    double acc = 0.0;
    for (int32_t r = r0 + ro; r < r1; r += RPB) {
        const int64_t i = (int64_t)r * K + j;
        acc += (double)x[i] * (double)y[i];
    }
    red[threadIdx.x] = acc;
    __syncthreads();
    for (int s = RPB / 2; s > 0; s >>= 1) {  // fixed tree over row offsets, per column
        if (ro < s) red[threadIdx.x] += red[threadIdx.x + s * K];
        __syncthreads();
    }
    if (ro == 0) partials[(int64_t)c * K + j] = red[j];
}

// One workgroup per segment over its chunks' partial sums (per_chunk groups of K a chunk): thread t adds the
// elements t, t + 256, .. in order, all of the column t % K, then the threads of a column are combined in a fixed
// order. Consecutive threads read consecutive sums: one system of 14k groups is 56 loads a thread.
template <int K>
__global__ __launch_bounds__(256) void k_segdot_finish(const int32_t *__restrict__ gate, const int32_t *__restrict__ seg_c0,
                                                       const double *__restrict__ partials, double *__restrict__ out,
                                                       int take_sqrt, int per_chunk) {
    UHIP_GATE();
    const int s = blockIdx.x;
    const int64_t i1 = (int64_t)seg_c0[s + 1] * per_chunk * K;
    int64_t i = (int64_t)seg_c0[s] * per_chunk * K + threadIdx.x;
    double acc[1] = {0.0};
    for (; i + 768 < i1; i += 1024) {
        double v[4];
#pragma unroll
        for (int u = 0; u < 4; ++u) v[u] = partials[i + 256 * u];
#pragma unroll
        for (int u = 0; u < 4; ++u) acc[0] += v[u];
    }
    for (; i < i1; i += 256) acc[0] += partials[i];
    __shared__ double sum[K];
    block_column_sums<K, 1>(acc, sum);
    // thread t < K has written sum[t] itself
    if (threadIdx.x < K) out[(int64_t)s * K + threadIdx.x] = take_sqrt ? sqrt(sum[threadIdx.x]) : sum[threadIdx.x];
}

// ---- batched CG on per-(segment, column) scalars ----
// state: rz, pap, alpha, beta, rznew, rr, atol, flags (0 active, 1 converged, 2 stopped on a
// non-finite step), conv_it.
struct BCGState {
    double *rz, *pap, *alpha, *beta, *rznew, *rr, *atol;
    int32_t *flags, *conv_it;
};

__global__ __launch_bounds__(256) void k_bcg_alpha(const int32_t *__restrict__ gate, int32_t m, BCGState st) {
    UHIP_GATE();
    const int t = blockIdx.x * 256 + threadIdx.x;
    if (t >= m) return;
    double a = st.rz[t] / st.pap[t];
    if (st.flags[t] != 0) {
        a = 0.0;
    } else if (!isfinite(a)) {  // utopia_ConjugateGradient_impl.hpp:241-244: stop without updating x
        st.flags[t] = 2;
        a = 0.0;
    }
    st.alpha[t] = a;
}

template <int K>
__global__ __launch_bounds__(256) void k_bcg_update(const int32_t *__restrict__ gate, int32_t n, const int32_t *__restrict__ rowseg,
                                                    const double *__restrict__ alpha, double *__restrict__ x,
                                                    const double *__restrict__ p, double *__restrict__ r,
                                                    const double *__restrict__ Ap) {
    UHIP_GATE();
    const int64_t i = (int64_t)blockIdx.x * 256 + threadIdx.x;
    if (i >= (int64_t)n * K) return;
    const int32_t row = (int32_t)(i / K);
    const double a = alpha[rowseg[row] * K + (int)(i % K)];
    if (a == 0.0) return;
    x[i] = x[i] + a * p[i];
    r[i] = r[i] - a * Ap[i];
}

// after |r| is known: converge (flag 1) where |r| <= atol; count the still active ones
// iter (device) counts the iterations done; it is advanced here so that a
// captured iteration replays with the right count.
__global__ __launch_bounds__(256) void k_bcg_check(const int32_t *__restrict__ gate, int32_t m, BCGState st, int32_t *__restrict__ iter,
                                                   int32_t *__restrict__ active_count) {
    UHIP_GATE();
    __shared__ int32_t cnt[256];
    const int32_t it = *iter + 1;
    int32_t c = 0;
    for (int t = threadIdx.x; t < m; t += 256) {
        if (st.flags[t] == 0) {
            if (st.rr[t] <= st.atol[t]) {
                st.flags[t] = 1;
                st.conv_it[t] = it;
            } else {
                ++c;
            }
        }
    }
    cnt[threadIdx.x] = c;
    __syncthreads();
    for (int s = 128; s > 0; s >>= 1) {
        if (threadIdx.x < s) cnt[threadIdx.x] += cnt[threadIdx.x + s];
        __syncthreads();
    }
    if (threadIdx.x == 0) {
        *active_count = cnt[0];
        *iter = it;
    }
}

__global__ __launch_bounds__(256) void k_bcg_beta(const int32_t *__restrict__ gate, int32_t m, BCGState st) {
    UHIP_GATE();
    const int t = blockIdx.x * 256 + threadIdx.x;
    if (t >= m) return;
    st.beta[t] = (st.flags[t] == 0) ? st.rznew[t] / st.rz[t] : 0.0;
    st.rz[t] = st.rznew[t];
}

template <int K>
__global__ __launch_bounds__(256) void k_bcg_pupdate(const int32_t *__restrict__ gate, int32_t n, const int32_t *__restrict__ rowseg,
                                                     const double *__restrict__ beta, double *__restrict__ p,
                                                     const double *__restrict__ z) {
    UHIP_GATE();
    const int64_t i = (int64_t)blockIdx.x * 256 + threadIdx.x;
    if (i >= (int64_t)n * K) return;
    const int32_t row = (int32_t)(i / K);
    p[i] = z[i] + beta[rowseg[row] * K + (int)(i % K)] * p[i];
}

// The iteration of the fused loop (uhip_bcg_alpha / _residual / _xpupdate): x moves with p at the end (one pass over
// p instead of two) and the dots come from the kernels that write their operands; with 3.57M rows x 8 an iteration of
// the mixed solve moves 4970 MB instead of 6570.
// alpha as in k_bcg_alpha, run at the start of every iteration, gate or not: *pending says whether the iteration is
// under way, as the x update at its end must still happen when the check in between has found the last pair
// converged (the gate then reads 0).
__global__ __launch_bounds__(256) void k_bcg_alpha_pending(const int32_t *__restrict__ gate, int32_t m, BCGState st,
                                                           int32_t *__restrict__ pending) {
    const bool run = !gate || *gate != 0;
    const int t = blockIdx.x * 256 + threadIdx.x;
    if (t == 0) *pending = run ? 1 : 0;
    if (!run || t >= m) return;
    double a = st.rz[t] / st.pap[t];
    if (st.flags[t] != 0) {
        a = 0.0;
    } else if (!isfinite(a)) {
        st.flags[t] = 2;
        a = 0.0;
    }
    st.alpha[t] = a;
}

// r -= alpha Ap and its FP32 copy (the FP32 cycle's right-hand side: three of its kernels read it), with the
// partial sums of r.r; two columns a thread.
template <int K>
__global__ __launch_bounds__(256) void k_bcg_residual(const int32_t *__restrict__ gate, const int32_t *__restrict__ c_row0,
                                                      const int32_t *__restrict__ c_row1,
                                                      const int32_t *__restrict__ rowseg,
                                                      const double *__restrict__ alpha, double *__restrict__ r,
                                                      const double *__restrict__ Ap, float *__restrict__ r32,
                                                      double *__restrict__ partials) {
    UHIP_GATE();
    constexpr int V = K >= 2 ? 2 : 1, L = K / V, ROWS = 256 / L;
    const int c = blockIdx.x / kDotGroups;
    const int32_t r0 = c_row0[c] + blockIdx.x % kDotGroups * kDotRows, r1 = min(c_row1[c], r0 + kDotRows);
    const int j0 = (int)(threadIdx.x % L) * V;
    double part[V], a[V];
    const int32_t g = r0 < r1 ? rowseg[r0] : 0;  // a chunk lies in one system
#pragma unroll
    for (int j = 0; j < V; ++j) {
        part[j] = 0.0;
        a[j] = alpha[g * K + j0 + j];
    }
    for (int32_t i = r0 + (int32_t)threadIdx.x / L; i < r1; i += ROWS) {
        double *rr = kcols<K, V>(r, i, j0);
        const double *ar = kcols<K, V>(Ap, i, j0);
        double rv[V], av[V];
#pragma unroll
        for (int j = 0; j < V; ++j) {
            rv[j] = rr[j];
            av[j] = ar[j];
        }
#pragma unroll
        for (int j = 0; j < V; ++j) {
            if (a[j] != 0.0) rv[j] = rv[j] - a[j] * av[j];
            part[j] += rv[j] * rv[j];
        }
#pragma unroll
        for (int j = 0; j < V; ++j) rr[j] = rv[j];
        if (r32) {
            float *fr = r32 + (int64_t)i * K + j0;
#pragma unroll
            for (int j = 0; j < V; ++j) fr[j] = (float)rv[j];
        }
    }
    block_column_sums<K, V>(part, partials + (int64_t)blockIdx.x * K);
}

// x += alpha p; p = z + beta p (z of either precision). *pending == 0: the iteration did not run; *active == 0:
// it was the last, there is no z.
template <int K, typename TZ>
__global__ __launch_bounds__(256) void k_bcg_xpupdate(const int32_t *__restrict__ pending,
                                                      const int32_t *__restrict__ active, int32_t n,
                                                      const int32_t *__restrict__ rowseg,
                                                      const double *__restrict__ alpha,
                                                      const double *__restrict__ beta, double *__restrict__ x,
                                                      double *__restrict__ p, const TZ *__restrict__ z) {
    if (*pending == 0) return;
    constexpr int V = K >= 2 ? 2 : 1, L = K / V;
    const int64_t t = (int64_t)blockIdx.x * 256 + threadIdx.x;
    const int32_t i = (int32_t)(t / L);
    if (i >= n) return;
    const bool more = *active != 0;
    const int j0 = (int)(t % L) * V;
    const int32_t g = rowseg[i];
    double *xr = kcols<K, V>(x, i, j0), *pr = kcols<K, V>(p, i, j0);
    double pv[V], xv[V];
#pragma unroll
    for (int j = 0; j < V; ++j) {
        pv[j] = pr[j];
        xv[j] = xr[j];
    }
#pragma unroll
    for (int j = 0; j < V; ++j) {
        const double a = alpha[g * K + j0 + j];
        if (a != 0.0) xv[j] = xv[j] + a * pv[j];
    }
#pragma unroll
    for (int j = 0; j < V; ++j) xr[j] = xv[j];
    if (!more) return;
    const TZ *zr = z + (int64_t)i * K + j0;
    double zv[V];
#pragma unroll
    for (int j = 0; j < V; ++j) zv[j] = (double)zr[j];
#pragma unroll
    for (int j = 0; j < V; ++j) pr[j] = zv[j] + beta[g * K + j0 + j] * pv[j];
}

// x_i = xin_i + a[seg]*p_i (Chebyshev with one sweep), dtype conversions
template <int K, typename TP, typename TX, typename TO, typename TAcc>
__global__ __launch_bounds__(256) void k_axpy_seg(const int32_t *__restrict__ gate, int32_t n, const int32_t *__restrict__ rowseg,
                                                  const double *__restrict__ coef, const TP *__restrict__ p,
                                                  const TX *__restrict__ xin, TO *__restrict__ out) {
    UHIP_GATE();
    const int64_t i = (int64_t)blockIdx.x * 256 + threadIdx.x;
    if (i >= (int64_t)n * K) return;
    const TAcc a = (TAcc)coef[3 * rowseg[i / K]];
    TAcc v = xin ? (TAcc)xin[i] : TAcc(0);
    out[i] = (TO)(v + a * (TAcc)p[i]);
}

// per segment power-method helpers (single column)
__global__ __launch_bounds__(256) void k_seg_scale(int32_t n, const int32_t *__restrict__ rowseg,
                                                   const double *__restrict__ norm, const int32_t *__restrict__ done,
                                                   const double *__restrict__ w, double *__restrict__ v) {
    const int32_t i = blockIdx.x * 256 + threadIdx.x;
    if (i >= n) return;
    const int32_t s = rowseg[i];
    if (done && done[s]) return;
    v[i] = (1. / norm[s]) * w[i];
}

// grad_e = -sum_j lambda[i, j] * x[col_e, j] over the pattern (dL/dA_ij = -lambda_i x_j)
template <int K>
__global__ __launch_bounds__(256) void k_pattern_grad(int32_t n, const int32_t *__restrict__ rowptr,
                                                      const int32_t *__restrict__ col,
                                                      const double *__restrict__ lam, const double *__restrict__ x,
                                                      double *__restrict__ grad) {
    const int32_t r = blockIdx.x * 256 + threadIdx.x;
    if (r >= n) return;
    double l[K];
#pragma unroll
    for (int j = 0; j < K; ++j) l[j] = lam[(int64_t)r * K + j];
    for (int32_t e = rowptr[r]; e < rowptr[r + 1]; ++e) {
        const int64_t c = (int64_t)col[e] * K;
        double s = 0.0;
#pragma unroll
        for (int j = 0; j < K; ++j) s += l[j] * x[c + j];
        grad[e] = -s;
    }
}

}  // namespace uhip

using namespace uhip;

// ---- dispatch helpers (K in {1, 2, 4, 8, 16}) ----
#define UHIP_K_SWITCH(k, ...)                                         \
    switch (k) {                                                      \
        case 1: { constexpr int KK = 1; __VA_ARGS__; } break;         \
        case 2: { constexpr int KK = 2; __VA_ARGS__; } break;         \
        case 4: { constexpr int KK = 4; __VA_ARGS__; } break;         \
        case 8: { constexpr int KK = 8; __VA_ARGS__; } break;         \
        case 16: { constexpr int KK = 16; __VA_ARGS__; } break;       \
        default: return set_error(UHIP_ERR_INVALID, "K=%d not in {1,2,4,8,16}", k); \
    }

extern "C" {

int uhip_spmm_by_wave(const uhip_csr *A) {
    return A->spmm_kernel == 2 || (A->spmm_kernel != 1 && A->nnz >= 32LL * A->nrows);
}

int uhip_spmm(uhip_ctx ctx, const uhip_csr *A, int k, const void *X, int x_dtype, void *Y, int y_dtype, int op,
              const void *B, int b_dtype) {
    UHIP_REQUIRE(ctx && A && X && Y, "uhip_spmm: null argument");
    UHIP_REQUIRE(op >= 0 && op <= 2, "uhip_spmm: op %d", op);
    UHIP_REQUIRE(op != 2 || B, "uhip_spmm: residual needs B");
    // op 0: Y = A X; 1: Y += A X; 2: Y = B - A X. Accumulation in the matrix precision.
#define UHIP_SPMM_T(TA, TX, TY, TB)                                                                          \
    do {                                                                                                     \
        if (op == 0) {                                                                                       \
            UHIP_K_SWITCH(k, UHIP_TRY((launch_spmm<KK, TA, EpiKStore<TA, TY>, TA, TX>(                 \
                                 ctx, A, (const TX *)X, EpiKStore<TA, TY>{(TY *)Y}))));                  \
        } else if (op == 1) {                                                                                \
            UHIP_K_SWITCH(k, UHIP_TRY((launch_spmm<KK, TA, EpiKAdd<TA, TY>, TA, TX>(                   \
                                 ctx, A, (const TX *)X, EpiKAdd<TA, TY>{(TY *)Y}))));                    \
        } else {                                                                                             \
            UHIP_K_SWITCH(k, UHIP_TRY((launch_spmm<KK, TA, EpiKResidual<TA, TB, TY>, TA, TX>(          \
                                 ctx, A, (const TX *)X, EpiKResidual<TA, TB, TY>{(const TB *)B, (TY *)Y})))); \
        }                                                                                                    \
        return UHIP_OK;                                                                                      \
    } while (0)
    if (A->dtype == UHIP_F64) {
        if (x_dtype == UHIP_F64 && y_dtype == UHIP_F64) UHIP_SPMM_T(double, double, double, double);
        if (x_dtype == UHIP_F32 && y_dtype == UHIP_F32) UHIP_SPMM_T(double, float, float, double);
        if (x_dtype == UHIP_F32 && y_dtype == UHIP_F64) UHIP_SPMM_T(double, float, double, double);
        if (x_dtype == UHIP_F64 && y_dtype == UHIP_F32) UHIP_SPMM_T(double, double, float, double);
    } else {
        UHIP_REQUIRE(y_dtype == UHIP_F32, "uhip_spmm: FP32 matrix writes FP32");
        if (x_dtype == UHIP_F32) {
            if (op != 2 || b_dtype == UHIP_F32) UHIP_SPMM_T(float, float, float, float);
            UHIP_SPMM_T(float, float, float, double);
        }
    }
#undef UHIP_SPMM_T
    return set_error(UHIP_ERR_INVALID, "uhip_spmm: dtype combination");
}

int uhip_csr_autotune_spmm(uhip_ctx ctx, uhip_csr *A, int k, int reps, int32_t *choice, float *ms_out) {
    UHIP_REQUIRE(ctx && A && reps > 0, "uhip_csr_autotune_spmm: bad argument");
    UHIP_REQUIRE(k == 1 || k == 2 || k == 4 || k == 8 || k == 16, "uhip_csr_autotune_spmm: K=%d", k);
    const size_t vb = A->dtype == UHIP_F64 ? sizeof(double) : sizeof(float);
    void *x = nullptr, *y = nullptr;
    UHIP_CHECK_HIP(hipMalloc(&x, vb * (size_t)k * (size_t)std::max(A->ncols, 1)));
    UHIP_CHECK_HIP(hipMalloc(&y, vb * (size_t)k * (size_t)std::max(A->nrows, 1)));
    UHIP_CHECK_HIP(hipMemsetAsync(x, 0, vb * (size_t)k * (size_t)std::max(A->ncols, 1), ctx->stream));
    hipEvent_t e0, e1;
    UHIP_CHECK_HIP(hipEventCreate(&e0));
    UHIP_CHECK_HIP(hipEventCreate(&e1));
    const int32_t saved = A->spmm_kernel;
    float best = 1e30f;
    int32_t win = 1;
    int st = UHIP_OK;
    const int dt = A->dtype;
    for (int32_t cand = 1; cand <= 2 && st == UHIP_OK; ++cand) {
        A->spmm_kernel = cand;
        if ((st = uhip_spmm(ctx, A, k, x, dt, y, dt, 0, nullptr, 0)) != UHIP_OK) break;  // warm-up
        hipEventRecord(e0, ctx->stream);
        for (int r = 0; r < reps && st == UHIP_OK; ++r) st = uhip_spmm(ctx, A, k, x, dt, y, dt, 0, nullptr, 0);
        hipEventRecord(e1, ctx->stream);
        hipEventSynchronize(e1);
        float ms = 0.f;
        hipEventElapsedTime(&ms, e0, e1);
        ms /= (float)reps;
        if (ms < best) best = ms, win = cand;
    }
    hipEventDestroy(e0);
    hipEventDestroy(e1);
    hipStreamSynchronize(ctx->stream);
    hipFree(x);
    hipFree(y);
    if (st != UHIP_OK) {
        A->spmm_kernel = saved;
        return st;
    }
    A->spmm_kernel = win;
    if (choice) *choice = win;
    if (ms_out) *ms_out = best;
    return UHIP_OK;
}

int uhip_spmm_cheb_step(uhip_ctx ctx, const uhip_csr *A, int k, const void *pprev, int p_dtype, const void *rprev,
                        const void *xin, void *xout, int x_dtype, void *rout, void *pout, const int32_t *rowseg,
                        const double *coef, int last) {
    UHIP_REQUIRE(ctx && A && pprev && xout && rowseg && coef, "uhip_spmm_cheb_step: null argument");
    UHIP_REQUIRE(last || (rout && pout), "uhip_spmm_cheb_step: rout/pout needed");
#define UHIP_SPMM_CHEB(TA, TP, TX)                                                                              \
    do {                                                                                                        \
        UHIP_K_SWITCH(k,                                                                                      \
                          EpiKCheb<TA, TP, TX> e{(const TP *)pprev, (const TA *)rprev, (const TA *)xin,     \
                                                     (TX *)xout,         (TA *)rout,         (TA *)pout,         \
                                                     rowseg,             coef,               last, nullptr};     \
                          UHIP_TRY((launch_spmm<KK, TA, EpiKCheb<TA, TP, TX>, TA, TP>(ctx, A, (const TP *)pprev, \
                                                                                           e)));                \
                      );                                                                                      \
        return UHIP_OK;                                                                                         \
    } while (0)
    if (A->dtype == UHIP_F64) {
        UHIP_REQUIRE(p_dtype == UHIP_F64 && x_dtype == UHIP_F64, "uhip_spmm_cheb_step: FP64 level");
        UHIP_SPMM_CHEB(double, double, double);
    }
    if (p_dtype == UHIP_F32 && x_dtype == UHIP_F32) UHIP_SPMM_CHEB(float, float, float);
    if (p_dtype == UHIP_F64 && x_dtype == UHIP_F32) UHIP_SPMM_CHEB(float, double, float);
    if (p_dtype == UHIP_F32 && x_dtype == UHIP_F64) UHIP_SPMM_CHEB(float, float, double);
    if (p_dtype == UHIP_F64 && x_dtype == UHIP_F64) UHIP_SPMM_CHEB(float, double, double);
#undef UHIP_SPMM_CHEB
    return set_error(UHIP_ERR_INVALID, "uhip_spmm_cheb_step: dtypes");
}

int uhip_axpy_seg(uhip_ctx ctx, int32_t n, int k, const int32_t *rowseg, const double *coef, const void *p,
                  int p_dtype, const void *xin, void *out, int out_dtype, int level_dtype) {
    UHIP_REQUIRE(ctx && rowseg && coef && p && out, "uhip_axpy_seg: null argument");
    if (n == 0) return UHIP_OK;
    const int64_t m = (int64_t)n * k;
    dim3 g((unsigned)((m + 255) / 256)), b(256);
#define UHIP_AXS(TP, TX, TO, TA)                                                                              \
    UHIP_K_SWITCH(k, hipLaunchKernelGGL((k_axpy_seg<KK, TP, TX, TO, TA>), g, b, 0, ctx->stream, ctx->gate, n, rowseg, coef, \
                                         (const TP *)p, (const TX *)xin, (TO *)out))
    if (level_dtype == UHIP_F64) {
        UHIP_AXS(double, double, double, double);
    } else if (p_dtype == UHIP_F64 && out_dtype == UHIP_F32) {
        UHIP_AXS(double, float, float, float);
    } else if (p_dtype == UHIP_F32 && out_dtype == UHIP_F64) {
        UHIP_AXS(float, float, double, float);
    } else if (p_dtype == UHIP_F64 && out_dtype == UHIP_F64) {
        UHIP_AXS(double, float, double, float);
    } else {
        UHIP_AXS(float, float, float, float);
    }
#undef UHIP_AXS
    UHIP_CHECK_LAUNCH();
    return UHIP_OK;
}

static int finish_chunks(uhip_ctx ctx, int k, int32_t nseg, const int32_t *seg_c0, double *out, int take_sqrt,
                         int per_chunk) {
    UHIP_K_SWITCH(k, hipLaunchKernelGGL((k_segdot_finish<KK>), dim3(nseg), dim3(256), 0, ctx->stream, ctx->gate, seg_c0,
                                         ctx->partials, out, take_sqrt, per_chunk));
    UHIP_CHECK_LAUNCH();
    return UHIP_OK;
}

int uhip_segdot(uhip_ctx ctx, int k, int32_t nchunks, const int32_t *c_row0, const int32_t *c_row1, int32_t nseg,
                const int32_t *seg_c0, const void *x, const void *y, int dtype, double *out, int take_sqrt) {
    UHIP_REQUIRE(ctx && c_row0 && c_row1 && seg_c0 && x && y && out, "uhip_segdot: null argument");
    if (nchunks == 0) return UHIP_OK;
    UHIP_TRY(ensure_partials(ctx, (int64_t)nchunks * k));
    if (dtype == UHIP_F64) {
        UHIP_K_SWITCH(k, hipLaunchKernelGGL((k_segdot_chunk<KK, double, double>), dim3(nchunks), dim3(256), 0,
                                             ctx->stream, ctx->gate, c_row0, c_row1, (const double *)x, (const double *)y,
                                             ctx->partials));
    } else {
        UHIP_K_SWITCH(k, hipLaunchKernelGGL((k_segdot_chunk<KK, float, float>), dim3(nchunks), dim3(256), 0,
                                             ctx->stream, ctx->gate, c_row0, c_row1, (const float *)x, (const float *)y,
                                             ctx->partials));
    }
    UHIP_CHECK_LAUNCH();
    return finish_chunks(ctx, k, nseg, seg_c0, out, take_sqrt, 1);
}

int uhip_spmm_dot(uhip_ctx ctx, const uhip_csr *A, int k, const double *X, double *Y, int32_t nchunks,
                  const int32_t *c_row0, const int32_t *c_row1, int32_t nseg, const int32_t *seg_c0, double *out) {
    UHIP_REQUIRE(ctx && A && X && Y && c_row0 && c_row1 && seg_c0 && out && A->dtype == UHIP_F64,
                 "uhip_spmm_dot: bad argument");
    if (nchunks == 0) return UHIP_OK;
    UHIP_TRY(ensure_partials(ctx, (int64_t)nchunks * kDotGroups * k));
    using Epi = EpiKStoreDot<double, double, double>;
    UHIP_K_SWITCH(k, UHIP_EB_SWITCH(A, hipLaunchKernelGGL((k_spmm_csr_dot<KK, EB, double, Epi, double, double>),
                                                          dim3(nchunks * kDotGroups), dim3(256), 0, ctx->stream, ctx->gate,
                                                          c_row0, c_row1, A->rowptr, A->col, (const double *)A->val, X,
                                                          Epi{X, Y}, ctx->partials)));
    UHIP_CHECK_LAUNCH();
    return finish_chunks(ctx, k, nseg, seg_c0, out, 0, kDotGroups);
}

int uhip_spmm_cheb_last_dot(uhip_ctx ctx, const uhip_csr *A, int k, const void *pprev, const void *rprev,
                            const void *xin, void *xout, const int32_t *rowseg, const double *coef,
                            const double *with, int32_t nchunks, const int32_t *c_row0, const int32_t *c_row1,
                            int32_t nseg, const int32_t *seg_c0, double *out) {
    UHIP_REQUIRE(ctx && A && pprev && xout && rowseg && coef && with && c_row0 && c_row1 && seg_c0 && out,
                 "uhip_spmm_cheb_last_dot: null argument");
    if (nchunks == 0) return UHIP_OK;
    UHIP_TRY(ensure_partials(ctx, (int64_t)nchunks * kDotGroups * k));
#define UHIP_CHEB_DOT(T)                                                                                               \
    UHIP_K_SWITCH(k, UHIP_EB_SWITCH(A, hipLaunchKernelGGL(                                                             \
                         (k_spmm_csr_dot<KK, EB, T, EpiKCheb<T, T, T, true>, T, T>), dim3(nchunks * kDotGroups), dim3(256), \
                         0, ctx->stream, ctx->gate, c_row0, c_row1, A->rowptr, A->col, (const T *)A->val,              \
                         (const T *)pprev,                                                                             \
                         EpiKCheb<T, T, T, true>{(const T *)pprev, (const T *)rprev, (const T *)xin, (T *)xout,        \
                                                 nullptr, nullptr, rowseg, coef, 1, with},                             \
                         ctx->partials)))
    if (A->dtype == UHIP_F64) {
        UHIP_CHEB_DOT(double);
    } else {
        UHIP_CHEB_DOT(float);
    }
#undef UHIP_CHEB_DOT
    UHIP_CHECK_LAUNCH();
    return finish_chunks(ctx, k, nseg, seg_c0, out, 0, kDotGroups);
}

int uhip_bcg_alpha(uhip_ctx ctx, int32_t m, double *const *state_d, int32_t *flags, int32_t *pending) {
    UHIP_REQUIRE(ctx && state_d && flags && pending, "uhip_bcg_alpha: null argument");
    BCGState st{state_d[0], state_d[1], state_d[2], state_d[3], state_d[4], state_d[5], state_d[6], flags, nullptr};
    hipLaunchKernelGGL(k_bcg_alpha_pending, dim3((m + 255) / 256), dim3(256), 0, ctx->stream, ctx->gate, m, st, pending);
    UHIP_CHECK_LAUNCH();
    return UHIP_OK;
}

int uhip_bcg_residual(uhip_ctx ctx, int k, const int32_t *rowseg, const double *alpha, double *r, const double *Ap,
                      float *r32, int32_t nchunks, const int32_t *c_row0, const int32_t *c_row1, int32_t nseg,
                      const int32_t *seg_c0, double *norm) {
    UHIP_REQUIRE(ctx && rowseg && alpha && r && Ap && c_row0 && c_row1 && seg_c0 && norm, "uhip_bcg_residual: null argument");
    if (nchunks == 0) return UHIP_OK;
    UHIP_TRY(ensure_partials(ctx, (int64_t)nchunks * kDotGroups * k));
    UHIP_K_SWITCH(k, hipLaunchKernelGGL((k_bcg_residual<KK>), dim3(nchunks * kDotGroups), dim3(256), 0, ctx->stream, ctx->gate,
                                         c_row0, c_row1, rowseg, alpha, r, Ap, r32, ctx->partials));
    UHIP_CHECK_LAUNCH();
    return finish_chunks(ctx, k, nseg, seg_c0, norm, 1, kDotGroups);
}

int uhip_bcg_beta(uhip_ctx ctx, int32_t m, double *const *state_d, int32_t *flags) {
    UHIP_REQUIRE(ctx && state_d && flags, "uhip_bcg_beta: null argument");
    BCGState st{state_d[0], state_d[1], state_d[2], state_d[3], state_d[4], state_d[5], state_d[6], flags, nullptr};
    hipLaunchKernelGGL(k_bcg_beta, dim3((m + 255) / 256), dim3(256), 0, ctx->stream, ctx->gate, m, st);
    UHIP_CHECK_LAUNCH();
    return UHIP_OK;
}

int uhip_bcg_xpupdate(uhip_ctx ctx, int32_t n, int k, const int32_t *rowseg, const double *alpha, const double *beta,
                      double *x, double *p, const void *z, int z_dtype, const int32_t *pending,
                      const int32_t *active) {
    UHIP_REQUIRE(ctx && rowseg && alpha && beta && x && p && z && pending && active, "uhip_bcg_xpupdate: null argument");
    if (n == 0) return UHIP_OK;
    const int64_t threads = (int64_t)n * (k >= 2 ? k / 2 : 1);
    const dim3 g((unsigned)((threads + 255) / 256)), b(256);
    if (z_dtype == UHIP_F64) {
        UHIP_K_SWITCH(k, hipLaunchKernelGGL((k_bcg_xpupdate<KK, double>), g, b, 0, ctx->stream, pending, active, n, rowseg,
                                             alpha, beta, x, p, (const double *)z));
    } else {
        UHIP_K_SWITCH(k, hipLaunchKernelGGL((k_bcg_xpupdate<KK, float>), g, b, 0, ctx->stream, pending, active, n, rowseg,
                                             alpha, beta, x, p, (const float *)z));
    }
    UHIP_CHECK_LAUNCH();
    return UHIP_OK;
}

int uhip_bcg_step(uhip_ctx ctx, int stage, int32_t n, int k, int32_t m, const int32_t *rowseg, double *x, double *p,
                  double *r, const double *Ap, const double *z, double *const *state_d, int32_t *flags,
                  int32_t *conv_it, int32_t *iter, int32_t *active_count) {
    // state_d: rz, pap, alpha, beta, rznew, rr, atol
    UHIP_REQUIRE(ctx && state_d && flags && conv_it && iter && active_count, "uhip_bcg_step: null argument");
    BCGState st{state_d[0], state_d[1], state_d[2], state_d[3], state_d[4], state_d[5], state_d[6], flags, conv_it};
    const int64_t nk = (int64_t)n * k;
    dim3 gm((m + 255) / 256), gv((unsigned)((nk + 255) / 256)), b(256);
    switch (stage) {
        case 0:  // alpha and x, r update
            hipLaunchKernelGGL(k_bcg_alpha, gm, b, 0, ctx->stream, ctx->gate, m, st);
            UHIP_CHECK_LAUNCH();
            if (nk > 0) {
                UHIP_K_SWITCH(k, hipLaunchKernelGGL((k_bcg_update<KK>), gv, b, 0, ctx->stream, ctx->gate, n, rowseg, st.alpha, x,
                                                     (const double *)p, r, Ap));
                UHIP_CHECK_LAUNCH();
            }
            return UHIP_OK;
        case 1:  // convergence check (rr holds |r|)
            hipLaunchKernelGGL(k_bcg_check, dim3(1), b, 0, ctx->stream, ctx->gate, m, st, iter, active_count);
            UHIP_CHECK_LAUNCH();
            return UHIP_OK;
        case 2:  // beta and p update
            hipLaunchKernelGGL(k_bcg_beta, gm, b, 0, ctx->stream, ctx->gate, m, st);
            UHIP_CHECK_LAUNCH();
            if (nk > 0) {
                UHIP_K_SWITCH(k, hipLaunchKernelGGL((k_bcg_pupdate<KK>), gv, b, 0, ctx->stream, ctx->gate, n, rowseg, st.beta, p,
                                                     z));
                UHIP_CHECK_LAUNCH();
            }
            return UHIP_OK;
        default:
            return set_error(UHIP_ERR_INVALID, "uhip_bcg_step: stage %d", stage);
    }
}

int uhip_seg_scale(uhip_ctx ctx, int32_t n, const int32_t *rowseg, const double *norm, const int32_t *done,
                   const double *w, double *v) {
    UHIP_REQUIRE(ctx && rowseg && norm && w && v, "uhip_seg_scale: null argument");
    if (n == 0) return UHIP_OK;
    hipLaunchKernelGGL(k_seg_scale, dim3((n + 255) / 256), dim3(256), 0, ctx->stream, n, rowseg, norm, done, w, v);
    UHIP_CHECK_LAUNCH();
    return UHIP_OK;
}

int uhip_pattern_grad(uhip_ctx ctx, const uhip_csr *A, int k, const double *lambda, const double *x, double *grad) {
    UHIP_REQUIRE(ctx && A && lambda && x && grad, "uhip_pattern_grad: null argument");
    const int32_t n = A->nrows;
    if (n == 0) return UHIP_OK;
    UHIP_K_SWITCH(k, hipLaunchKernelGGL((k_pattern_grad<KK>), dim3((n + 255) / 256), dim3(256), 0, ctx->stream, n,
                                         A->rowptr, A->col, lambda, x, grad));
    UHIP_CHECK_LAUNCH();
    return UHIP_OK;
}

}  // extern "C"
