// Setup-time sparse products: transpose, C = A*B and the Galerkin triple
// product Ac = P^T A P. All pattern work is integer-exact and the value of
// each C_ij is summed in the order a row-wise (Gustavson) product visits it:
// over k in A's row order, so results are deterministic and equal to a
// sequential dense-accumulator loop.
//
// Rows of C are accumulated in small LDS hash tables (k_spgemm_hash), the
// rows with too many distinct columns, and products of long rows with few
// duplicates, by sorting all candidates (k_spgemm_rows). Galerkin product of a
// 96^3 7-point operator (885k rows): 12.0 ms with every row sorted, 0.94 ms; the
// first of a context, which takes its temporaries from the driver, 2.0 to 2.3 ms.
#include <hipcub/hipcub.hpp>

#include "uhip_common.hpp"

namespace uhip {

// Entries per column, and each entry's arrival number within its column.
__global__ __launch_bounds__(kBlock) void k_col_hist(int64_t nnz, const int32_t *__restrict__ col,
                                                     int32_t *__restrict__ cnt, int32_t *__restrict__ slot) {
    for (int64_t e = (int64_t)blockIdx.x * kBlock + threadIdx.x; e < nnz; e += (int64_t)gridDim.x * kBlock)
        slot[e] = atomicAdd(&cnt[col[e]], 1);
}

// Entry e of row r goes to row col[e] of the transpose, at its arrival number: rows come out complete
// but in any order, k_transpose_order puts them in order.
__global__ __launch_bounds__(kBlock) void k_transpose_scatter(int32_t n, const int32_t *__restrict__ rowptr,
                                                              const int32_t *__restrict__ col,
                                                              const int32_t *__restrict__ slot,
                                                              const int32_t *__restrict__ trp,
                                                              int2 *__restrict__ entry) {
    const int32_t r = blockIdx.x * kBlock + threadIdx.x;
    if (r >= n) return;
    for (int32_t e = rowptr[r]; e < rowptr[r + 1]; ++e) entry[trp[col[e]] + slot[e]] = int2{r, e};
}

// Rows of up to kOrderMax entries put in the order of their entry numbers in A (which is that of the
// rows of A, duplicates included) by counting the smaller ones, 32 lanes a row. A restriction's rows
// have 27 entries, one a lane; longer ones are read again for each 32 of their entries, which the limit
// keeps to 16 times. The (column, row) radix sort this replaces for short rows took 0.4 ms on the 3.0M
// entries of a 96^3 interpolation, this and the scatter 65 us.
constexpr int32_t kOrderMax = 512;
template <typename T>
__global__ __launch_bounds__(kBlock) void k_transpose_order(int32_t m, const int32_t *__restrict__ trp,
                                                            const int2 *__restrict__ entry,
                                                            const T *__restrict__ aval, int32_t *__restrict__ col,
                                                            T *__restrict__ val) {
    const int lane = threadIdx.x & 31;
    for (int64_t r = (blockIdx.x * (int64_t)kBlock + threadIdx.x) >> 5; r < m; r += (int64_t)gridDim.x * (kBlock / 32)) {
        const int32_t a = trp[r], len = trp[r + 1] - a;
        if (len <= 32) {
            const int2 c = lane < len ? entry[a + lane] : int2{0, INT32_MAX};
            int32_t rank = 0;
#pragma unroll
            for (int j = 0; j < 32; ++j) rank += __shfl(c.y, j, 32) < c.y ? 1 : 0;
            if (lane < len) {
                col[a + rank] = c.x;
                val[a + rank] = aval[c.y];
            }
            continue;
        }
        for (int32_t i = lane; i < len; i += 32) {
            const int2 c = entry[a + i];
            int32_t rank = 0;
            for (int32_t j = 0; j < len; ++j) rank += entry[a + j].y < c.y ? 1 : 0;
            col[a + rank] = c.x;
            val[a + rank] = aval[c.y];
        }
    }
}

// Workgroups for `items` with `per` a workgroup: kernels with several lanes an item take more items a workgroup where
// a launch would have 2^32 threads, which it may not (at 32 lanes a row: 2^27 rows).
static unsigned lanes_grid(int64_t items, int per) {
    return (unsigned)std::min<int64_t>((items + per - 1) / per, int64_t(1) << 22);
}

// *mx = the largest v of the launch (blocks of kBlock, all threads): one atomic where a workgroup raises the maximum
__device__ __forceinline__ void raise_max(int32_t v, int32_t *mx) {
    __shared__ int32_t red[kBlock / 64];
#pragma unroll
    for (int d = 32; d > 0; d >>= 1) v = max(v, __shfl_xor(v, d, 64));
    if ((threadIdx.x & 63) == 0) red[threadIdx.x >> 6] = v;
    __syncthreads();
    if (threadIdx.x == 0) {
#pragma unroll
        for (int i = 1; i < kBlock / 64; ++i) v = max(v, red[i]);
        if (v > __hip_atomic_load(mx, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT)) atomicMax(mx, v);
    }
    __syncthreads();
}

__global__ __launch_bounds__(kBlock) void k_max_len(int32_t m, const int32_t *__restrict__ cnt,
                                                    int32_t *__restrict__ mx) {
    int32_t v = 0;
    for (int64_t i = blockIdx.x * kBlock + threadIdx.x; i < m; i += gridDim.x * kBlock) v = max(v, cnt[i]);
    raise_max(v, mx);
}

template <typename T>
__global__ __launch_bounds__(kBlock) void k_transpose_keys(int32_t n, const int32_t *__restrict__ rowptr,
                                                           const int32_t *__restrict__ col,
                                                           const T *__restrict__ val,
                                                           uint64_t *__restrict__ keys, T *__restrict__ vals) {
    const int32_t r = blockIdx.x * kBlock + threadIdx.x;
    if (r >= n) return;
    for (int32_t e = rowptr[r]; e < rowptr[r + 1]; ++e) {
        keys[e] = ((uint64_t)(uint32_t)col[e] << 32) | (uint32_t)r;
        vals[e] = val[e];
    }
}

__global__ __launch_bounds__(kBlock) void k_keys_low(int64_t nnz, const uint64_t *__restrict__ keys,
                                                     int32_t *__restrict__ col) {
    for (int64_t e = (int64_t)blockIdx.x * kBlock + threadIdx.x; e < nnz; e += (int64_t)gridDim.x * kBlock)
        col[e] = (int32_t)(keys[e] & 0xffffffffu);
}

// The most candidate products (sum of |B_k| over k in A_i) of a row of A*B.
__global__ __launch_bounds__(kBlock) void k_row_ub(int32_t n, const int32_t *__restrict__ arp,
                                                   const int32_t *__restrict__ acol,
                                                   const int32_t *__restrict__ brp, int32_t *__restrict__ mx) {
    int64_t s = 0;
    const int32_t r = blockIdx.x * kBlock + threadIdx.x;
    if (r < n)
#pragma unroll 8
        for (int32_t e = arp[r]; e < arp[r + 1]; ++e) {
            const int32_t k = acol[e];
            s += brp[k + 1] - brp[k];
        }
    raise_max((int32_t)(s > 0x7fffffff ? 0x7fffffff : s), mx);
}

// The rows of the lanes with `take` to the end of a list: one atomic a wavefront (one a row is 10 ns a row, all on one
// word: 280 us for 28,000 rows).
__device__ __forceinline__ void append(bool take, int32_t row, int32_t *__restrict__ list, int32_t *__restrict__ n) {
    const uint64_t mask = __ballot(take);
    if (mask == 0) return;
    const int lane = threadIdx.x & 63, first = __builtin_ctzll(mask);
    int32_t at = 0;
    if (lane == first) at = atomicAdd(n, (int32_t)__popcll(mask));
    at = __shfl(at, first, 64) + (int32_t)__popcll(mask & ((1ull << lane) - 1));
    if (take) list[at] = row;
}

// Rows of C = A*B in LDS hash tables: G lanes own a row, the table holds T (column, sum) slots.
// The entries k of the A row are taken one after the other; in each step the lanes hold the entries of
// row B_k, whose columns are distinct, so no two lanes of a step meet in one sum and every C_ij adds
// its products over k in A's row order. What bounds it is latency (row pointer -> columns -> table),
// so the (column, value) pairs of 8 steps are loaded before the first is used, and G follows the
// length of B's rows: 8 rows of C a wavefront where they average up to 8 entries (an interpolation),
// 4 where they have up to 16 (A P), else 2. T = 64 holds a stencil hierarchy's rows (up to 27
// columns), T = 512 with a wavefront a row the longer ones; a table is filled to kHashRows<T> columns, beyond which the
// longest of a step's probe chains takes over (filled to 7/8, one row of 578 columns took 150 us).
// PASS 0 writes the number of distinct columns to cnt[i]; a row over the limit goes to `dense_list` if its columns
// come up again and again (1.5 candidates a column so far: a product of stencils), else to `sort_list`: sorting takes
// the same few steps for a row of few duplicates. (The table of T = 512 sends what it does not hold there as well.)
// PASS 1 writes sorted columns and values at crp[i], for the rows within the limit.
// Ragged rows of 8 on average, 2,000 x 2,000 / 60,000 x 60,000: every row sorted 306 / 871 us, tables filled to 7/8 and
// only checked after G entries of a row of A 1674 / 3296.
template <int T>
constexpr int32_t kHashRows = T == 32 ? 28 : (T == 64 ? 40 : 256);

template <int G, int T, int PASS, bool LIST>
__global__ __launch_bounds__(256) void k_spgemm_hash(int32_t n, const int32_t *__restrict__ list,
                                                     const int32_t *__restrict__ list_n,
                                                     const int32_t *__restrict__ arp,
                                                     const int32_t *__restrict__ acol,
                                                     const double *__restrict__ aval,
                                                     const int32_t *__restrict__ brp,
                                                     const int32_t *__restrict__ bcol,
                                                     const double *__restrict__ bval, int32_t *__restrict__ cnt,
                                                     int32_t *__restrict__ dense_list, int32_t *__restrict__ dense_n,
                                                     int32_t *__restrict__ sort_list, int32_t *__restrict__ sort_n,
                                                     const int32_t *__restrict__ crp, int32_t *__restrict__ ccol,
                                                     double *__restrict__ cval) {
    constexpr int R = 256 / G, U = 8, S = T / G;
    constexpr int kShift = T == 32 ? 27 : (T == 64 ? 26 : 23);
    static_assert(T == 32 || T == 64 || T == 512, "hash shift");
    __shared__ __align__(16) int32_t keys[R * T];
    __shared__ double sums[PASS == 1 ? R * T : 1];
    const int lane = threadIdx.x % G, g = threadIdx.x / G;
    volatile int32_t *kt = keys + g * T;
    double *vt = sums + (PASS == 1 ? g * T : 0);
    const uint64_t gmask = (G == 64 ? ~0ull : ((1ull << (G & 63)) - 1)) << ((threadIdx.x & 63) / G * G);
    const int32_t total_rows = LIST ? *list_n : n;
    // a wavefront's own tables: its LDS operations are in order, the fence keeps the compiler to it
    auto step_done = [] {
        __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
        __builtin_amdgcn_wave_barrier();
    };
    for (int64_t i0 = (int64_t)blockIdx.x * R; i0 < total_rows; i0 += (int64_t)gridDim.x * R) {
        const bool have = i0 + g < total_rows;
        const int32_t row = !have ? 0 : (LIST ? list[i0 + g] : (int32_t)(i0 + g));
        const int32_t a0 = have ? arp[row] : 0;
        int32_t a1 = have ? arp[row + 1] : 0, c0 = 0;
        if (PASS == 1) {
            c0 = have ? crp[row] : 0;
            if (have && crp[row + 1] - c0 > kHashRows<T>) a1 = a0;  // the next kernel's row
        }
#pragma unroll
        for (int s = 0; s < S; ++s) {
            kt[lane + s * G] = -1;
            if (PASS == 1) vt[lane + s * G] = -0.0;  // -0.0 + p == p for every p
        }
        step_done();
        // distinct columns and candidates so far (PASS 0; the same in all of the row's lanes)
        int32_t added = 0, seen = 0;
        for (int32_t e0 = a0; e0 < a1 && added <= kHashRows<T>; e0 += G) {
            const int32_t e = e0 + lane;
            int32_t b0 = 0, len = 0;
            double av = 0.0;
            if (e < a1) {
                const int32_t k = acol[e];
                if (PASS == 1) av = aval[e];
                b0 = brp[k];
                len = brp[k + 1] - b0;
            }
            const int m = min(G, a1 - e0);
            for (int j0 = 0; j0 < m && added <= kHashRows<T>; j0 += U) {
                int32_t bs[U], ln[U], cc[U];
                double vv[U];
#pragma unroll
                for (int u = 0; u < U; ++u) {
                    bs[u] = __shfl(b0, (j0 + u) & (G - 1), G);
                    ln[u] = __shfl(len, (j0 + u) & (G - 1), G);
                    if (j0 + u >= m) ln[u] = 0;
                    cc[u] = 0;
                    vv[u] = 0.0;
                    if (lane < ln[u]) {
                        cc[u] = bcol[bs[u] + lane];
                        if (PASS == 1) vv[u] = bval[bs[u] + lane];
                    }
                }
#pragma unroll
                for (int u = 0; u < U; ++u) {
                    const double a = PASS == 1 ? __shfl(av, (j0 + u) & (G - 1), G) : 0.0;
                    int32_t c = cc[u];
                    double v = vv[u];
                    for (int32_t q0 = 0; q0 < ln[u]; q0 += G) {
                        // a row over the limit is the next kernel's: a table that goes on filling up is probed from
                        // end to end by every entry (512 slots: 1.6 ms a row)
                        if (PASS == 0 && added > kHashRows<T>) break;
                        const int32_t q = q0 + lane;
                        bool fresh = false;
                        if (q < ln[u]) {
                            if (q0 > 0) {
                                c = bcol[bs[u] + q];
                                if (PASS == 1) v = bval[bs[u] + q];
                            }
                            uint32_t h = ((uint32_t)c * 2654435769u) >> kShift;
                            for (int probe = 0; probe < T; ++probe) {
                                const int32_t cur = kt[h];
                                if (cur == c) break;
                                if (cur == -1) {
                                    const int32_t was = atomicCAS((int32_t *)&kt[h], -1, c);
                                    fresh = was == -1;
                                    if (fresh || was == c) break;
                                }
                                h = (h + 1) & (T - 1);
                            }
                            if (PASS == 1) vt[h] += a * v;  // a PASS 1 row fits
                        }
                        if (PASS == 0) {
                            added += __popcll(__ballot(fresh) & gmask);
                            seen += min(G, ln[u] - q0);
                        }
                    }
                    step_done();
                }
            }
        }
        if (PASS == 0) {
            const bool over = have && lane == 0 && added > kHashRows<T>;
            const bool dense = over && !LIST && 2 * seen >= 3 * added;
            if (have && lane == 0 && !over) cnt[row] = added;
            if (!LIST) append(dense, row, dense_list, dense_n);
            append(over && !dense, row, sort_list, sort_n);
        } else {
            int32_t kk[S], mine = 0;
            double vv[S];
#pragma unroll
            for (int s = 0; s < S; ++s) {
                kk[s] = kt[lane + s * G];
                vv[s] = vt[lane + s * G];
                mine += kk[s] >= 0 ? 1 : 0;
            }
            int32_t incl = mine;
#pragma unroll
            for (int d = 1; d < G; d <<= 1) {
                const int32_t y = __shfl_up(incl, d, G);
                if (lane >= d) incl += y;
            }
            const int32_t count = __shfl(incl, G - 1, G);
            step_done();
            int32_t at = incl - mine;
#pragma unroll
            for (int s = 0; s < S; ++s)
                if (kk[s] >= 0) kt[at++] = kk[s];  // the row's columns, packed, and up to a multiple of four
            if (lane < 4) kt[count + lane] = INT32_MAX;  // (count + 3 < T)
            step_done();
            int32_t rank[S];
#pragma unroll
            for (int s = 0; s < S; ++s) rank[s] = 0;
            const int4 *packed = (const int4 *)(keys + g * T);
            for (int32_t j = 0; j < count; j += 4) {
                const int4 c = packed[j >> 2];
#pragma unroll
                for (int s = 0; s < S; ++s)
                    rank[s] += (c.x < kk[s] ? 1 : 0) + (c.y < kk[s] ? 1 : 0) + (c.z < kk[s] ? 1 : 0) + (c.w < kk[s] ? 1 : 0);
            }
#pragma unroll
            for (int s = 0; s < S; ++s)
                if (kk[s] >= 0) {
                    ccol[c0 + rank[s]] = kk[s];
                    cval[c0 + rank[s]] = vv[s];
                }
        }
        step_done();
    }
}

// How the rows of A*B look, from kSampled of them: out[0] += candidates, and of a row's first 128 or so, out[1] +=
// candidates, out[2] += distinct columns. A wavefront a row.
constexpr int kSampled = 128;
__global__ __launch_bounds__(256) void k_spgemm_sample(int32_t n, const int32_t *__restrict__ arp,
                                                       const int32_t *__restrict__ acol,
                                                       const int32_t *__restrict__ brp,
                                                       const int32_t *__restrict__ bcol, int32_t *__restrict__ out) {
    constexpr int T = 512, kSeen = 128;  // at most kSeen + 63 columns come into the table
    __shared__ int32_t tables[4 * T];
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    volatile int32_t *kt = tables + wave * T;
    const int32_t row = (int32_t)((int64_t)(blockIdx.x * 4 + wave) * n / kSampled);
    const int32_t a0 = arp[row], a1 = arp[row + 1];
    int32_t m = 0, b0 = 0, len = 0;  // the lane's entry of the row's first 64
    for (int32_t e = a0 + lane; e < a1; e += 64) {
        const int32_t b = brp[acol[e]], l = brp[acol[e] + 1] - b;
        m += l;
        if (e == a0 + lane) b0 = b, len = l;
    }
#pragma unroll
    for (int d = 32; d > 0; d >>= 1) m += __shfl_xor(m, d, 64);
    for (int i = lane; i < T; i += 64) kt[i] = -1;
    __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
    __builtin_amdgcn_wave_barrier();
    int32_t seen = 0, added = 0;
    constexpr int U = 8;  // rows of B loaded together; of each at most 64 entries count
    for (int j0 = 0; j0 < min(64, a1 - a0) && seen < kSeen; j0 += U) {
        int32_t c[U], l[U];
#pragma unroll
        for (int u = 0; u < U; ++u) {
            l[u] = min(64, __shfl(len, j0 + u, 64));
            c[u] = lane < l[u] ? bcol[__shfl(b0, j0 + u, 64) + lane] : -1;
        }
#pragma unroll
        for (int u = 0; u < U; ++u) {
            if (seen >= kSeen) break;
            bool fresh = false;
            uint32_t h = ((uint32_t)c[u] * 2654435769u) >> 23;
            for (int probe = 0; lane < l[u] && probe < T; ++probe) {
                const int32_t cur = kt[h];
                if (cur == c[u]) break;
                if (cur == -1) {
                    const int32_t was = atomicCAS((int32_t *)&kt[h], -1, c[u]);
                    fresh = was == -1;
                    if (fresh || was == c[u]) break;
                }
                h = (h + 1) & (T - 1);
            }
            added += __popcll(__ballot(fresh));
            seen += l[u];
        }
    }
    if (lane == 0) {
        atomicAdd(out, m);
        atomicAdd(out + 1, seen);
        atomicAdd(out + 2, added);
    }
}

// The rows of a list with lo < m <= CAP candidates (none has more than `most`), one per block iteration, by sorting their candidates: for rows with
// more distinct columns than the hash tables hold. PASS 0 writes the number of distinct
// columns to cnt[i]; PASS 1 writes sorted columns and values at crp[i].
// list NULL: all of rows 0 .. n - 1. Candidates get key (col << 32 | position) so equal columns stay in visiting
// order through the (unstable) bitonic sort. CAP, the most candidates, sets how many rows a CU has at work (16 bytes
// each), NT how fast one row's chain of steps is: a list's rows are taken in classes.
template <int NT, int CAP, int PASS>
__global__ __launch_bounds__(NT) void k_spgemm_rows(int32_t n, const int32_t *__restrict__ list,
                                                    const int32_t *__restrict__ list_n, int32_t lo, int32_t most,
                                                    const int32_t *__restrict__ arp,
                                                    const int32_t *__restrict__ acol,
                                                    const double *__restrict__ aval,
                                                    const int32_t *__restrict__ brp,
                                                    const int32_t *__restrict__ bcol,
                                                    const double *__restrict__ bval, int32_t *__restrict__ cnt,
                                                    const int32_t *__restrict__ crp, int32_t *__restrict__ ccol,
                                                    double *__restrict__ cval) {
    __shared__ uint64_t key[CAP];
    __shared__ double val[CAP];
    __shared__ int32_t off[NT + 1];
    __shared__ int32_t wsum[NT / 64 + 1];
    const int tid = threadIdx.x;
    if (list) n = *list_n;
    for (int32_t i = blockIdx.x; i < n; i += gridDim.x) {
        const int32_t row = list ? list[i] : i;
        const int32_t a0 = arp[row], a1 = arp[row + 1];
        if (lo >= 0 || most > CAP) {
            int32_t len = 0;  // (the sum fits: no row has more than 8192)
            for (int32_t t = a0 + tid; t < a1; t += NT) len += brp[acol[t] + 1] - brp[acol[t]];
#pragma unroll
            for (int d = 32; d > 0; d >>= 1) len += __shfl_xor(len, d, 64);
            if ((tid & 63) == 0) wsum[tid >> 6] = len;
            __syncthreads();
            len = 0;
            for (int w = 0; w < NT / 64; ++w) len += wsum[w];
            __syncthreads();
            if (len <= lo || len > CAP) continue;
        }
        int32_t m = 0;  // candidates so far
        for (int32_t c0 = a0; c0 < a1; c0 += NT) {
            const int32_t t = c0 + tid;
            int32_t k = 0, len = 0;
            double av = 0.0;
            if (t < a1) {
                k = acol[t];
                av = aval[t];
                len = brp[k + 1] - brp[k];
            }
            // block exclusive scan of len
            int32_t incl = len;
#pragma unroll
            for (int d = 1; d < 64; d <<= 1) {
                const int32_t y = __shfl_up(incl, d, 64);
                if ((tid & 63) >= d) incl += y;
            }
            if ((tid & 63) == 63) wsum[tid >> 6] = incl;
            __syncthreads();
            int32_t wbase = 0;
            for (int w = 0; w < (tid >> 6); ++w) wbase += wsum[w];
            const int32_t excl = wbase + incl - len;
            int32_t total = 0;
            for (int w = 0; w < NT / 64; ++w) total += wsum[w];
            if (t < a1) {
                const int32_t b0 = brp[k];
                for (int32_t q = 0; q < len; ++q) {
                    const int32_t p = m + excl + q;
                    key[p] = ((uint64_t)(uint32_t)bcol[b0 + q] << 32) | (uint32_t)p;
                    if (PASS == 1) val[p] = av * bval[b0 + q];
                }
            }
            m += total;
            __syncthreads();
        }
        // pad to a power of two and sort
        int32_t P = 1;
        while (P < m) P <<= 1;
        for (int32_t p = m + tid; p < P; p += NT) key[p] = ~0ull;
        __syncthreads();
        for (int32_t size = 2; size <= P; size <<= 1) {
            for (int32_t stride = size >> 1; stride > 0; stride >>= 1) {
                for (int32_t i = tid; i < P; i += NT) {
                    const int32_t j = i ^ stride;
                    if (j > i) {
                        const bool up = (i & size) == 0;
                        const uint64_t ki = key[i], kj = key[j];
                        if ((ki > kj) == up) {
                            key[i] = kj;
                            key[j] = ki;
                            if (PASS == 1) {
                                const double vi = val[i];
                                val[i] = val[j];
                                val[j] = vi;
                            }
                        }
                    }
                }
                __syncthreads();
            }
        }
        // run heads: chunk [tid*per, (tid+1)*per) per thread, then a block scan of head counts
        const int32_t per = (m + NT - 1) / NT;
        const int32_t s0 = tid * per, s1 = min(m, s0 + per);
        int32_t heads = 0;
        for (int32_t i = s0; i < s1; ++i)
            if (i == 0 || (key[i] >> 32) != (key[i - 1] >> 32)) ++heads;
        int32_t incl = heads;
#pragma unroll
        for (int d = 1; d < 64; d <<= 1) {
            const int32_t y = __shfl_up(incl, d, 64);
            if ((tid & 63) >= d) incl += y;
        }
        if ((tid & 63) == 63) wsum[tid >> 6] = incl;
        __syncthreads();
        int32_t wbase = 0;
        for (int w = 0; w < (tid >> 6); ++w) wbase += wsum[w];
        int32_t total = 0;
        for (int w = 0; w < NT / 64; ++w) total += wsum[w];
        if (PASS == 0) {
            if (tid == 0) cnt[row] = total;
        } else {
            int32_t rank = wbase + incl - heads;
            const int32_t base = crp[row];
            for (int32_t i = s0; i < s1; ++i) {
                if (i == 0 || (key[i] >> 32) != (key[i - 1] >> 32)) {
                    const uint64_t c = key[i] >> 32;
                    double s = val[i];
                    for (int32_t j = i + 1; j < m && (key[j] >> 32) == c; ++j) s += val[j];
                    ccol[base + rank] = (int32_t)c;
                    cval[base + rank] = s;
                    ++rank;
                }
            }
        }
        __syncthreads();
    }
}

// PASS 0 or 1 of C = A B: the hash kernel over all rows, then over the rows that its tables do not
// hold: list1 (T = 512), list2 (sorted). nlist: the lists' lengths. maxub: the most candidates of a row,
// maxcnt (PASS 1): the most columns of a row of C.
// by_hash: false: every row is sorted.
template <int PASS>
static int spgemm_pass(uhip_ctx ctx, const uhip_csr *A, const uhip_csr *B, const uhip_csr *C, int32_t maxub,
                       int32_t maxcnt, bool by_hash, int32_t *cnt, int32_t *list1, int32_t *list2, int32_t *nlist) {
    hipStream_t s = ctx->stream;
    const int32_t n = A->nrows;
    const double *av = (const double *)A->val, *bv = (const double *)B->val;
    double *cv = (double *)C->val;
    if (by_hash) {
#define UHIP_HASH(G, T, LIST, GRID, L, LN)                                                                         \
    hipLaunchKernelGGL((k_spgemm_hash<G, T, PASS, LIST>), dim3(GRID), dim3(256), 0, s, n, L, LN, A->rowptr, A->col, av, \
                       B->rowptr, B->col, bv, cnt, list1, nlist, list2, nlist + 1, C->rowptr, C->col, cv)
        // lanes a row by the mean length of B's rows, so that most of a row's entries go in one step
        const int64_t per = B->nnz / std::max(B->nrows, 1);
        // tables of 32 slots where every row fits and the mean row fills at most half of them: A P of
        // the 96^3 product (11 a row) 225 -> 192 us; its R (A P), 27 in each row, 155 -> 267 us
        if (PASS == 1 && maxcnt <= kHashRows<32> && C->nnz <= 16 * (int64_t)n && per <= 8) {
            UHIP_HASH(8, 32, false, lanes_grid(n, 32), nullptr, nullptr);
            UHIP_CHECK_LAUNCH();
            return UHIP_OK;
        }
        if (per <= 8) UHIP_HASH(8, 64, false, lanes_grid(n, 32), nullptr, nullptr);
        else if (per <= 16) UHIP_HASH(16, 64, false, lanes_grid(n, 16), nullptr, nullptr);
        else UHIP_HASH(32, 64, false, lanes_grid(n, 8), nullptr, nullptr);
        UHIP_CHECK_LAUNCH();
        if (maxub <= kHashRows<64> || (PASS == 1 && maxcnt <= kHashRows<64>)) return UHIP_OK;
        if (2 * maxub >= 3 * kHashRows<64>) {
            UHIP_HASH(64, 512, true, std::min(lanes_grid(n, 4), 2048u), list1, nlist);
            UHIP_CHECK_LAUNCH();
        }
#undef UHIP_HASH
    }
    // A row's chain of steps is shorter with four wavefronts, and a CU holds more rows with the smaller arrays: two
    // launches where no row has more than 1024 candidates (2,000 ragged rows of 8: 232 -> 136 us for both passes
    // against one wavefront and 1024 for all). Longer rows are the launch's tail anyway, one launch has one.
    int32_t *const list = by_hash ? list2 : nullptr;
#define UHIP_SORT(NT, CAP, LO)                                                                                      \
    hipLaunchKernelGGL((k_spgemm_rows<NT, CAP, PASS>), dim3(std::min(n, list ? (1 << 19) / NT : 1 << 16)), dim3(NT), 0, s, n, \
                       list, nlist + 1, LO, maxub, A->rowptr, A->col, av, B->rowptr, B->col, bv, cnt, C->rowptr, C->col, cv)
    if (maxub <= 1024) {
        UHIP_SORT(64, 256, -1);
        UHIP_CHECK_LAUNCH();
        if (maxub > 256) UHIP_SORT(256, 1024, 256);
    } else if (maxub <= 4096) UHIP_SORT(256, 4096, -1);
    else UHIP_SORT(256, 8192, -1);
#undef UHIP_SORT
    UHIP_CHECK_LAUNCH();
    return UHIP_OK;
}

// info[0], info[1]: the longest row of A and of B; info[2] = 1 when a row of B has columns that do not
// increase strictly.
__global__ __launch_bounds__(kBlock) void k_row_info(int32_t na, const int32_t *__restrict__ arp, int32_t nb,
                                                     const int32_t *__restrict__ brp,
                                                     const int32_t *__restrict__ bcol, int32_t *__restrict__ info) {
    int32_t la = 0, lb = 0;
    bool bad = false;
    const int32_t st = gridDim.x * kBlock;
    for (int64_t r = blockIdx.x * kBlock + threadIdx.x; r < max(na, nb); r += st) {
        if (r < na) la = max(la, arp[r + 1] - arp[r]);
        if (r < nb) {
            const int32_t b0 = brp[r], b1 = brp[r + 1];
            lb = max(lb, b1 - b0);
            // no early end: the loads then do not wait for each other
#pragma unroll 8
            for (int32_t e = b0 + 1; e < b1; ++e) bad = bad | (bcol[e] <= bcol[e - 1]);
        }
    }
    raise_max(la, info);
    raise_max(lb, info + 1);
    if (bad) info[2] = 1;
}

__global__ __launch_bounds__(kBlock) void k_to_dense(int32_t n, int32_t ncols, const int32_t *__restrict__ rowptr,
                                                     const int32_t *__restrict__ col,
                                                     const double *__restrict__ val, double *__restrict__ dense) {
    const int32_t r = blockIdx.x * kBlock + threadIdx.x;
    if (r >= n) return;
    for (int32_t e = rowptr[r]; e < rowptr[r + 1]; ++e) dense[(int64_t)r * ncols + col[e]] += val[e];
}

}  // namespace uhip

using namespace uhip;

extern "C" {

int uhip_csr_free(uhip_ctx ctx, uhip_csr *A) {
    if (!A) return UHIP_OK;
    if (ctx) UHIP_CHECK_HIP(hipStreamSynchronize(ctx->stream));
    if (A->rowptr) hipFree(A->rowptr);
    if (A->col) hipFree(A->col);
    if (A->val) hipFree(A->val);
    A->rowptr = nullptr;
    A->col = nullptr;
    A->val = nullptr;
    return uhip_csr_plan_destroy(ctx, A);
}

}  // extern "C"

// Arrays of a result: the caller's own allocations (freed by uhip_csr_free), or, for an intermediate of
// a product, blocks of the context's cache.
struct CsrBlocks {
    explicit CsrBlocks(uhip_ctx c) : ctx(c) {}
    ~CsrBlocks() {
        for (int i = 0; i < 3; ++i)
            if (ptr[i]) ctx->cache.put(ptr[i], held[i]);
    }
    uhip_ctx ctx;
    void *ptr[3] = {nullptr, nullptr, nullptr};
    size_t held[3] = {0, 0, 0};
};
static int csr_array(CsrBlocks *own, int which, size_t bytes, void **out) {
    if (!own) {
        UHIP_CHECK_HIP(hipMalloc(out, bytes));
        return UHIP_OK;
    }
    UHIP_TRY(own->ctx->cache.take(bytes, &own->ptr[which], &own->held[which]));
    *out = own->ptr[which];
    return UHIP_OK;
}

// own: NULL, or the holder of an intermediate's arrays. Work on the stream may be pending on return.
template <typename T>
static int transpose_typed(uhip_ctx ctx, const uhip_csr *A, uhip_csr *B, CsrBlocks *own = nullptr) {
    hipStream_t s = ctx->stream;
    const int64_t nnz = A->nnz;
    const int32_t n = A->nrows, m = A->ncols;
    memset(B, 0, sizeof(*B));
    B->nrows = m;
    B->ncols = n;
    B->nnz = nnz;
    B->dtype = A->dtype;
    UHIP_TRY(csr_array(own, 0, sizeof(int32_t) * ((size_t)m + 1), (void **)&B->rowptr));
    UHIP_TRY(csr_array(own, 1, sizeof(int32_t) * std::max<int64_t>(nnz, 1), (void **)&B->col));
    UHIP_TRY(csr_array(own, 2, sizeof(T) * std::max<int64_t>(nnz, 1), &B->val));
    size_t tb = 0;
    UHIP_CHECK_HIP(hipcub::DeviceScan::ExclusiveSum(nullptr, tb, (int32_t *)nullptr, B->rowptr, m + 1, s));
    Scratch w(ctx);
    const size_t o_cnt = w.add(sizeof(int32_t) * ((size_t)m + 2)), o_tmp = w.add(tb),
                 o_slot = w.add(sizeof(int32_t) * nnz), o_entry = w.add(sizeof(int2) * nnz);
    UHIP_TRY(w.allocate());
    int32_t *cnt = w.at<int32_t>(o_cnt), *slot = w.at<int32_t>(o_slot);
    UHIP_CHECK_HIP(hipMemsetAsync(cnt, 0, sizeof(int32_t) * ((size_t)m + 2), s));
    if (nnz > 0) {
        hipLaunchKernelGGL(k_col_hist, dim3(grid_for(nnz, 4, 1 << 16)), dim3(kBlock), 0, s, nnz, A->col, cnt, slot);
        UHIP_CHECK_LAUNCH();
        hipLaunchKernelGGL(k_max_len, dim3(grid_for(m, 4, 256)), dim3(kBlock), 0, s, m, cnt, cnt + m + 1);
        UHIP_CHECK_LAUNCH();
    }
    UHIP_CHECK_HIP(hipcub::DeviceScan::ExclusiveSum(w.at<void>(o_tmp), tb, cnt, B->rowptr, m + 1, s));
    if (nnz == 0) return UHIP_OK;
    int32_t longest = 0;
    UHIP_TRY(read_ints(ctx, cnt + m + 1, 1, &longest));
    if (longest <= kOrderMax) {
        hipLaunchKernelGGL(k_transpose_scatter, dim3((n + kBlock - 1) / kBlock), dim3(kBlock), 0, s, n, A->rowptr,
                           A->col, slot, B->rowptr, w.at<int2>(o_entry));
        UHIP_CHECK_LAUNCH();
        hipLaunchKernelGGL(k_transpose_order<T>, dim3(lanes_grid(m, 8)), dim3(kBlock), 0, s, m, B->rowptr,
                           w.at<int2>(o_entry), (const T *)A->val, B->col, (T *)B->val);
        UHIP_CHECK_LAUNCH();
        return UHIP_OK;
    }
    // a long column: all entries sorted by (column, row)
    int hi_bits = 1;
    while ((1ll << hi_bits) < (int64_t)m) ++hi_bits;
    const int end_bit = 32 + hi_bits;
    Scratch x(ctx);
    const size_t o_k0 = x.add(sizeof(uint64_t) * nnz), o_k1 = x.add(sizeof(uint64_t) * nnz),
                 o_v0 = x.add(sizeof(T) * nnz);
    UHIP_CHECK_HIP(hipcub::DeviceRadixSort::SortPairs(nullptr, tb, (uint64_t *)nullptr, (uint64_t *)nullptr,
                                                      (T *)nullptr, (T *)B->val, (int)nnz, 0, end_bit, s));
    const size_t o_sort = x.add(tb);
    UHIP_TRY(x.allocate());
    uint64_t *k0 = x.at<uint64_t>(o_k0), *k1 = x.at<uint64_t>(o_k1);
    T *v0 = x.at<T>(o_v0);
    hipLaunchKernelGGL(k_transpose_keys<T>, dim3((n + kBlock - 1) / kBlock), dim3(kBlock), 0, s, n, A->rowptr, A->col,
                       (const T *)A->val, k0, v0);
    UHIP_CHECK_LAUNCH();
    UHIP_CHECK_HIP(hipcub::DeviceRadixSort::SortPairs(x.at<void>(o_sort), tb, k0, k1, v0, (T *)B->val, (int)nnz, 0,
                                                      end_bit, s));
    hipLaunchKernelGGL(k_keys_low, dim3(grid_for(nnz, 4, 1 << 16)), dim3(kBlock), 0, s, nnz, k1, B->col);
    UHIP_CHECK_LAUNCH();
    return UHIP_OK;
}

// C = A B into hipMalloc'd arrays, or (own) blocks of the cache. Work may be pending on return.
static int spgemm_into(uhip_ctx ctx, const uhip_csr *A, const uhip_csr *B, uhip_csr *C, CsrBlocks *own) {
    hipStream_t s = ctx->stream;
    const int32_t n = A->nrows;
    memset(C, 0, sizeof(*C));
    C->nrows = n;
    C->ncols = B->ncols;
    C->dtype = UHIP_F64;
    UHIP_TRY(csr_array(own, 0, sizeof(int32_t) * ((size_t)n + 1), (void **)&C->rowptr));
    if (n == 0) {
        UHIP_CHECK_HIP(hipMemsetAsync(C->rowptr, 0, sizeof(int32_t), s));
        UHIP_TRY(csr_array(own, 1, sizeof(int32_t), (void **)&C->col));
        return csr_array(own, 2, sizeof(double), &C->val);
    }
    size_t tb = 0;
    UHIP_CHECK_HIP(hipcub::DeviceScan::ExclusiveSum(nullptr, tb, (int32_t *)nullptr, C->rowptr, n + 1, s));
    Scratch w(ctx);
    // ints: the lists' lengths (2), the longest row of A and of B, whether a row of B is not sorted, the
    // most candidates of a row, the sample (3), the entries of C and of its longest row
    const size_t o_ints = w.add(sizeof(int32_t) * 11), o_cnt = w.add(sizeof(int32_t) * ((size_t)n + 1)),
                 o_l1 = w.add(sizeof(int32_t) * n), o_l2 = w.add(sizeof(int32_t) * n), o_tmp = w.add(tb);
    UHIP_TRY(w.allocate());
    int32_t *ints = w.at<int32_t>(o_ints), *cnt = w.at<int32_t>(o_cnt);
    UHIP_CHECK_HIP(hipMemsetAsync(ints, 0, sizeof(int32_t) * 11, s));
    hipLaunchKernelGGL(k_row_info, dim3(grid_for(std::max(n, B->nrows), 1, 1024)), dim3(kBlock), 0, s, n,
                       A->rowptr, B->nrows, B->rowptr, B->col, ints + 2);
    UHIP_CHECK_LAUNCH();
    int32_t info[3];
    UHIP_TRY(read_ints(ctx, ints + 2, 3, info));
    // Columns of B's rows that increase strictly are what the hash kernel needs (a column twice in a row of B would
    // meet itself in one step); otherwise every row is sorted.
    bool by_hash = info[2] == 0;
    // the longest rows' product bounds a row's candidates; the exact count only where that is too many
    int32_t maxub = (int32_t)std::min<int64_t>((int64_t)info[0] * info[1], 0x7fffffff);
    if (maxub > 1024) {
        hipLaunchKernelGGL(k_row_ub, dim3((n + kBlock - 1) / kBlock), dim3(kBlock), 0, s, n, A->rowptr, A->col,
                           B->rowptr, ints + 5);
        UHIP_CHECK_LAUNCH();
        if (by_hash) {
            hipLaunchKernelGGL(k_spgemm_sample, dim3(kSampled / 4), dim3(256), 0, s, n, A->rowptr, A->col, B->rowptr, B->col,
                               ints + 6);
            UHIP_CHECK_LAUNCH();
        }
        int32_t look[4];
        UHIP_TRY(read_ints(ctx, ints + 5, 4, look));
        maxub = look[0];
        // Long rows of few duplicates: a table would be filled in vain before each is sorted. Sorting every row
        // / tables first: 2,000 ragged rows of 8 (56 candidates) 231 / 292 us, of 20 (377) 436 / 586; 60,000 of 8
        // 657 / 861, of 20 5946 / 5207; 200 rows of 720 candidates 239 / 368.
        if (look[1] > kSampled * kHashRows<64> && 2 * look[2] < 3 * look[3]) by_hash = false;
    }
    if (maxub > 8192) {
        if (!own) (void)hipFree(C->rowptr);
        C->rowptr = nullptr;
        return set_error(UHIP_ERR_UNSUPPORTED, "uhip_csr_spgemm: a row has %d candidate products (> 8192)", maxub);
    }
    UHIP_TRY(spgemm_pass<0>(ctx, A, B, C, maxub, 0, by_hash, cnt, w.at<int32_t>(o_l1), w.at<int32_t>(o_l2), ints));
    UHIP_CHECK_HIP(hipMemsetAsync(cnt + n, 0, sizeof(int32_t), s));
    UHIP_CHECK_HIP(hipcub::DeviceScan::ExclusiveSum(w.at<void>(o_tmp), tb, cnt, C->rowptr, n + 1, s));
    hipLaunchKernelGGL(k_max_len, dim3(grid_for(n, 4, 256)), dim3(kBlock), 0, s, n, cnt, ints + 10);
    UHIP_CHECK_LAUNCH();
    UHIP_CHECK_HIP(hipMemcpyAsync(ints + 9, C->rowptr + n, sizeof(int32_t), hipMemcpyDeviceToDevice, s));
    int32_t size[2];  // entries of C, the most of a row
    UHIP_TRY(read_ints(ctx, ints + 9, 2, size));
    const int32_t nnz = size[0];
    C->nnz = nnz;
    UHIP_TRY(csr_array(own, 1, sizeof(int32_t) * std::max<int64_t>(nnz, 1), (void **)&C->col));
    UHIP_TRY(csr_array(own, 2, sizeof(double) * std::max<int64_t>(nnz, 1), &C->val));
    return spgemm_pass<1>(ctx, A, B, C, maxub, size[1], by_hash, cnt, w.at<int32_t>(o_l1), w.at<int32_t>(o_l2), ints);
}

extern "C" {

int uhip_csr_transpose(uhip_ctx ctx, const uhip_csr *A, uhip_csr *B) {
    UHIP_REQUIRE(ctx && A && B, "uhip_csr_transpose: null argument");
    UHIP_REQUIRE(A->dtype == UHIP_F64 || A->dtype == UHIP_F32, "uhip_csr_transpose: dtype %d", A->dtype);
    UHIP_TRY(A->dtype == UHIP_F64 ? transpose_typed<double>(ctx, A, B) : transpose_typed<float>(ctx, A, B));
    UHIP_CHECK_HIP(hipStreamSynchronize(ctx->stream));
    return UHIP_OK;
}

int uhip_csr_spgemm(uhip_ctx ctx, const uhip_csr *A, const uhip_csr *B, uhip_csr *C) {
    UHIP_REQUIRE(ctx && A && B && C, "uhip_csr_spgemm: null argument");
    UHIP_REQUIRE(A->dtype == UHIP_F64 && B->dtype == UHIP_F64, "uhip_csr_spgemm: FP64 matrices only");
    UHIP_REQUIRE(A->ncols == B->nrows, "uhip_csr_spgemm: inner dimensions %d != %d", A->ncols, B->nrows);
    UHIP_TRY(spgemm_into(ctx, A, B, C, nullptr));
    UHIP_CHECK_HIP(hipStreamSynchronize(ctx->stream));
    return UHIP_OK;
}

int uhip_csr_ptap(uhip_ctx ctx, const uhip_csr *A, const uhip_csr *P, uhip_csr *Ac) {
    UHIP_REQUIRE(ctx && A && P && Ac, "uhip_csr_ptap: null argument");
    UHIP_REQUIRE(A->nrows == A->ncols && P->nrows == A->ncols, "uhip_csr_ptap: shapes A %dx%d P %dx%d", A->nrows,
                 A->ncols, P->nrows, P->ncols);
    UHIP_REQUIRE(A->dtype == UHIP_F64 && P->dtype == UHIP_F64, "uhip_csr_spgemm: FP64 matrices only");
    // P^T and A P are dropped here: they live in the context's cache
    uhip_csr R, AP;
    CsrBlocks r(ctx), ap(ctx);
    UHIP_TRY(transpose_typed<double>(ctx, P, &R, &r));
    UHIP_TRY(spgemm_into(ctx, A, P, &AP, &ap));
    UHIP_TRY(spgemm_into(ctx, &R, &AP, Ac, nullptr));
    UHIP_CHECK_HIP(hipStreamSynchronize(ctx->stream));
    return UHIP_OK;
}

int uhip_csr_to_dense(uhip_ctx ctx, const uhip_csr *A, double *dense) {
    UHIP_REQUIRE(ctx && A && dense, "uhip_csr_to_dense: null argument");
    UHIP_REQUIRE(A->dtype == UHIP_F64, "uhip_csr_to_dense: FP64 only");
    const int32_t n = A->nrows;
    UHIP_CHECK_HIP(hipMemsetAsync(dense, 0, sizeof(double) * (size_t)n * A->ncols, ctx->stream));
    if (n == 0) return UHIP_OK;
    hipLaunchKernelGGL(k_to_dense, dim3((n + kBlock - 1) / kBlock), dim3(kBlock), 0, ctx->stream, n, A->ncols,
                       A->rowptr, A->col, (const double *)A->val, dense);
    UHIP_CHECK_LAUNCH();
    return UHIP_OK;
}

}  // extern "C"
