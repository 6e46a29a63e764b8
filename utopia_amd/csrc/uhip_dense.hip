// Dense FP64 kernels for the coarsest multigrid level (4096 rows: factor and inverse 22.2 -> 4.4 ms with
// the forms below against one launch per 64-column step of each solve): blocked Cholesky
// (A = L L^T) whose GEMM-shaped trailing updates run on the FP64 matrix cores
// (v_mfma_f64_16x16x4f64), the explicit inverse A^-1 = L^-T L^-1, and the GEMV
// that applies it once per V-cycle.
#include "uhip_common.hpp"

namespace uhip {

constexpr int kNB = 64;  // panel width

typedef double v4d __attribute__((ext_vector_type(4)));

typedef double v2d __attribute__((ext_vector_type(2), aligned(8)));

// Operand lanes of v_mfma_f64_16x16x4f64: lane l supplies A[l%16][l/16] and B[l/16][l%16]
// (k = l/16); item r of lane l of the result is D[4*r + l/16][l%16].

// One triangular matrix product per block (blockIdx.z) on the matrix cores: a 64x64 tile of
// C = alpha A B^T (kLowerC: C += alpha A B^T) per workgroup, 4 waves with a 32x32 quarter (2x2 MFMA tiles) each.
//   KC: operand stored with k contiguous (element (i,k) at i*ld + k), else with i contiguous
//       (k*ld + i); either way a chunk of 32 k is loaded in 16-byte pairs, kept in registers while
//       the previous chunk is multiplied, and staged in LDS at a stride free of bank conflicts for
//       the MFMA reads (34 doubles along k, 80 along i).
//   TRI: which tiles are computed, and which k of a tile are zero for good and left out
// Measured at n = 4096: A^-1 = Y^T Y 782 us (22.9 GFLOP, 29 TFLOP/s; about 70 is the matrix cores' rate),
// the inverse's 12 products 814 us, a trailing update of the factor 18.5 us in the mean (C's values read
// before the products: 23.6 us where each was read as it was replaced).
enum class Tri {
    kNone,     // all k
    kLowerC,   // C symmetric, lower tiles only; all k (trailing update)
    kBLower,   // B(j,k) = Y[k][j], Y lower triangular: k >= tile's first j
    kALower,   // A lower triangular: k <= tile's last i
    kGram,     // A = B = Y^T, Y lower triangular: k >= tile's first i (i >= j); lower tiles, mirrored
};

constexpr int kBK = 32;

struct GemmBlocks {
    // block z's operands: base + z * step; its M, N, K shrink where the matrix ends
    const double *A, *B;
    double *C;
    int64_t lda, ldb, ldc;
    int64_t stepA, stepB, stepC;
    int M, N, K;
    int n, row0, rowstep;  // rows of C: row0 + z * rowstep + [0, M) below n
    double alpha;
};

template <bool AK, bool BK_, Tri TRI>
__global__ __launch_bounds__(256) void k_gemm_f64(GemmBlocks g) {
    constexpr int SA = AK ? kBK + 2 : 80, SB = BK_ ? kBK + 2 : 80;
    __shared__ __align__(16) double As[AK ? 64 * SA : kBK * SA];
    __shared__ __align__(16) double Bs[BK_ ? 64 * SB : kBK * SB];
    const int z = blockIdx.z;
    const int ti = blockIdx.y * 64, tj = blockIdx.x * 64;
    if ((TRI == Tri::kLowerC || TRI == Tri::kGram) && tj > ti) return;
    const int M = min(g.M, g.n - (g.row0 + z * g.rowstep));
    if (ti >= M) return;
    const int N = (TRI == Tri::kLowerC || TRI == Tri::kGram) ? M : g.N;
    // rows of the blocks on the diagonal end with the matrix too
    const int K = (TRI == Tri::kALower || TRI == Tri::kGram) ? M : g.K;
    const double *A = g.A + z * g.stepA, *B = g.B + z * g.stepB;
    double *C = g.C + z * g.stepC;
    int kb = 0, ke = K;
    if (TRI == Tri::kBLower) kb = tj;
    if (TRI == Tri::kALower) ke = min(K, ti + 64);
    if (TRI == Tri::kGram) kb = ti;
    const int tid = threadIdx.x, wave = tid >> 6, lane = tid & 63;
    const int wi = (wave >> 1) * 32, wj = (wave & 1) * 32;
    v4d acc[2][2];
#pragma unroll
    for (int a = 0; a < 2; ++a)
#pragma unroll
        for (int b = 0; b < 2; ++b) acc[a][b] = v4d{0.0, 0.0, 0.0, 0.0};
    v2d ra[4], rb[4];
    // C's values, where they are needed, come with the first loads (item r of tile (a, b))
    auto c_at = [&](int a, int b, int r, int &gi, int &gj) {
        gi = ti + wi + a * 16 + 4 * r + (lane >> 4);
        gj = tj + wj + b * 16 + (lane & 15);
        return gi < M && gj < N && !((TRI == Tri::kLowerC || TRI == Tri::kGram) && gj > gi);
    };
    double cv[2][2][4];
    if (TRI == Tri::kLowerC) {
#pragma unroll
        for (int a = 0; a < 2; ++a)
#pragma unroll
            for (int b = 0; b < 2; ++b)
#pragma unroll
                for (int r = 0; r < 4; ++r) {
                    int gi, gj;
                    (void)c_at(a, b, r, gi, gj);
                    cv[a][b][r] = C[(int64_t)min(gi, M - 1) * g.ldc + min(gj, N - 1)];
                }
    }
    // thread's pair p of a chunk: (row, k) for a k-contiguous operand, (k, row) otherwise. A chunk
    // inside the operands is loaded without a test.
    const bool inner = ti + 64 <= M && tj + 64 <= N;
    auto fetch = [&](const double *X, int64_t ld, int t0, int lim, bool kc, int k0, v2d (&r)[4]) {
        if (inner && k0 + kBK <= ke) {
            const double *q = kc ? X + (int64_t)(t0 + (tid >> 4)) * ld + k0 + 2 * (tid & 15)
                                 : X + (int64_t)(k0 + (tid >> 5)) * ld + t0 + 2 * (tid & 31);
            const int64_t step = (kc ? 16 : 8) * ld;
#pragma unroll
            for (int p = 0; p < 4; ++p) r[p] = *(const v2d *)(q + p * step);
            return;
        }
#pragma unroll
        for (int p = 0; p < 4; ++p) {
            const int e = tid + 256 * p;
            const int row = t0 + (kc ? e >> 4 : 2 * (e & 31));
            const int k = k0 + (kc ? 2 * (e & 15) : e >> 5);
            const bool in0 = row < lim && k < ke;
            const bool in1 = kc ? (row < lim && k + 1 < ke) : (row + 1 < lim && k < ke);
            const double *q = kc ? X + (int64_t)row * ld + k : X + (int64_t)k * ld + row;
            v2d v = v2d{0.0, 0.0};
            if (in1) v = *(const v2d *)q;
            else if (in0) v.x = *q;
            r[p] = v;
        }
    };
    auto stage = [&](double *S, int stride, bool kc, const v2d (&r)[4]) {
#pragma unroll
        for (int p = 0; p < 4; ++p) {
            const int e = tid + 256 * p;
            double *q = kc ? S + (e >> 4) * stride + 2 * (e & 15) : S + (e >> 5) * stride + 2 * (e & 31);
            q[0] = r[p].x;
            q[1] = r[p].y;
        }
    };
    if (kb < ke) {
        fetch(A, g.lda, ti, M, AK, kb, ra);
        fetch(B, g.ldb, tj, N, BK_, kb, rb);
    }
    for (int k0 = kb; k0 < ke; k0 += kBK) {
        __syncthreads();
        stage(As, SA, AK, ra);
        stage(Bs, SB, BK_, rb);
        __syncthreads();
        if (k0 + kBK < ke) {
            fetch(A, g.lda, ti, M, AK, k0 + kBK, ra);
            fetch(B, g.ldb, tj, N, BK_, k0 + kBK, rb);
        }
#pragma unroll
        for (int ks = 0; ks < kBK; ks += 4) {
            const int kl = ks + (lane >> 4);
            double av[2], bv[2];
#pragma unroll
            for (int a = 0; a < 2; ++a) {
                const int i = wi + a * 16 + (lane & 15), j = wj + a * 16 + (lane & 15);
                av[a] = AK ? As[i * SA + kl] : As[kl * SA + i];
                bv[a] = BK_ ? Bs[j * SB + kl] : Bs[kl * SB + j];
            }
#pragma unroll
            for (int a = 0; a < 2; ++a)
#pragma unroll
                for (int b = 0; b < 2; ++b)
                    acc[a][b] = __builtin_amdgcn_mfma_f64_16x16x4f64(av[a], bv[b], acc[a][b], 0, 0, 0);
        }
    }
#pragma unroll
    for (int a = 0; a < 2; ++a)
#pragma unroll
        for (int b = 0; b < 2; ++b)
#pragma unroll
            for (int r = 0; r < 4; ++r) {
                int gi, gj;
                if (c_at(a, b, r, gi, gj)) {
                    const double v = (TRI == Tri::kLowerC ? cv[a][b][r] : 0.0) + g.alpha * acc[a][b][r];
                    C[(int64_t)gi * g.ldc + gj] = v;
                    if (TRI == Tri::kGram) C[(int64_t)gj * g.ldc + gi] = v;
                }
            }
}

__device__ __forceinline__ double lane_value(double v, int src) {
    return __hiloint2double(__builtin_amdgcn_readlane(__double2hiint(v), src),
                            __builtin_amdgcn_readlane(__double2loint(v), src));
}

constexpr int kLS = kNB + 2;  // LDS stride of a 64-column block: MFMA reads free of bank conflicts

// The lower triangle of the nb x nb block at (k, k) into T, continued by the identity: 16 values a
// thread, all loaded (at clamped places) before the first is stored.
__device__ __forceinline__ void load_lower(const double *A, int64_t lda, int k, int nb, double *T, int tid) {
    const int c = tid & 63, i0 = tid >> 6;
    const double *q = A + (int64_t)k * lda + k + min(c, nb - 1);
    double v[16];
#pragma unroll
    for (int p = 0; p < 16; ++p) v[p] = q[min(i0 + 4 * p, nb - 1) * lda];
#pragma unroll
    for (int p = 0; p < 16; ++p) {
        const int i = i0 + 4 * p;
        T[i * kLS + c] = (i < nb && c <= i) ? v[p] : (i == c ? 1.0 : 0.0);
    }
}

// The inverse of the 16x16 lower triangular block at (o, o) of T into V (row stride vs), a column per
// lane (lanes 0 .. 15); rd: the reciprocals of the diagonal.
__device__ __forceinline__ void invert16(const double *T, int o, const double *rd, double *V, int vs, int lane) {
    if (lane >= 16) return;
    double v[16];
#pragma unroll
    for (int i = 0; i < 16; ++i) v[i] = i == lane ? 1.0 : 0.0;
#pragma unroll
    for (int i = 0; i < 16; ++i) {
        v[i] = v[i] * rd[o + i];
#pragma unroll
        for (int q = i + 1; q < 16; ++q) v[q] = v[q] - T[(o + q) * kLS + o + i] * v[i];
    }
#pragma unroll
    for (int i = 0; i < 16; ++i) V[i * vs + lane] = v[i];
}

// One step of the blocked Cholesky, columns k .. k+63: the diagonal block's factor (every workgroup
// computes it for itself: cheaper than a launch of its own before the panel's), then 64 rows of the
// panel L(i, k:k+64) = A(i, k:k+64) Lkk^-T per workgroup. Both go by 16 columns: the first wave
// factors 16 columns of the 64-row block with a row per lane in registers (pivots and multipliers
// move by readlane), the matrix cores update the rest; the panel rows are multiplied by the inverses
// of the four 16x16 diagonal blocks. A serial chain of 64 pivots bounds it. n = 4096: 24.6 us a step
// (one launch with a thread per entry for the block, 85 us, and one with a row per thread below, 51 us).
// Other workgroups still read the diagonal block of A, so its factor goes to Dk (64 x 64) and
// k_put_diag puts all of them in place at the end.
__global__ __launch_bounds__(256) void k_cholesky_panel(int n, double *__restrict__ A, int64_t lda, int k,
                                                        double *__restrict__ Dk, int *__restrict__ info) {
    __shared__ __align__(16) double T[kNB * kLS];    // the diagonal block, then its factor
    __shared__ __align__(16) double V[kNB * 18];     // inverses of its 16x16 diagonal blocks
    __shared__ __align__(16) double X[4][16 * kLS];  // a wave's 16 rows of the panel
    __shared__ double rd[kNB];                       // 1 / diagonal
    const int nb = min(kNB, n - k);
    const int tid = threadIdx.x, wave = tid >> 6, lane = tid & 63;
    const int l16 = lane & 15, l4 = lane >> 4;
    load_lower(A, lda, k, nb, T, tid);
    // the wave's panel rows, loaded behind the factorisation (item r of tile b: row 4 r + l4, column 16 b + l16)
    const int row0 = k + nb + (int)blockIdx.x * 64 + wave * 16;
    v4d x[4];
#pragma unroll
    for (int b = 0; b < 4; ++b)
#pragma unroll
        for (int r = 0; r < 4; ++r) {
            const int i = row0 + 4 * r + l4;
            // rows past the end compute nothing that is kept; below n the block above is a full one
            x[b][r] = A[(int64_t)min(i, n - 1) * lda + min(k + 16 * b + l16, n - 1)];
        }
    __syncthreads();
    for (int kb = 0; kb < 4; ++kb) {
        const int c0 = 16 * kb;
        if (wave == 0) {
            double r[16];
#pragma unroll
            for (int c = 0; c < 16; ++c) r[c] = T[lane * kLS + c0 + c];
#pragma unroll
            for (int j = 0; j < 16; ++j) {
                const double d = lane_value(r[j], c0 + j);
                const bool ok = d > 0.0;
                if (!ok && blockIdx.x == 0 && lane == 0 && c0 + j < nb && *info == 0) *info = k + c0 + j + 1;
                // 1/sqrt(d) once a column: multipliers by a product; sqrt(d) corrected by one Newton step
                const double y = ok ? rsqrt(d) : 1.0;
                double s = d * y;
                s = ok ? fma(0.5 * y, fma(-s, s, d), s) : 1.0;
                const double l = r[j] * y;
                r[j] = lane == c0 + j ? s : l;
                if (lane == 0) rd[c0 + j] = y;
#pragma unroll
                for (int c = j + 1; c < 16; ++c) r[c] = r[c] - l * lane_value(l, c0 + c);
            }
#pragma unroll
            for (int c = 0; c < 16; ++c)
                if (lane >= c0) T[lane * kLS + c0 + c] = c0 + c <= lane ? r[c] : 0.0;
        }
        __syncthreads();
        // T(i, j) -= L(i, c0:c0+16) L(j, c0:c0+16)^T on the 16x16 tiles below
        int t = 0;
        for (int bi = kb + 1; bi < 4; ++bi)
            for (int bj = kb + 1; bj <= bi; ++bj, ++t) {
                if ((t & 3) != wave) continue;
                v4d acc = v4d{0.0, 0.0, 0.0, 0.0};
#pragma unroll
                for (int ks = 0; ks < 16; ks += 4)
                    acc = __builtin_amdgcn_mfma_f64_16x16x4f64(T[(16 * bi + l16) * kLS + c0 + ks + l4],
                                                               T[(16 * bj + l16) * kLS + c0 + ks + l4], acc, 0, 0, 0);
#pragma unroll
                for (int r = 0; r < 4; ++r) T[(16 * bi + 4 * r + l4) * kLS + 16 * bj + l16] -= acc[r];
            }
        __syncthreads();
    }
    if (blockIdx.x == 0)
        for (int e = tid; e < kNB * kNB; e += 256) {
            const double v = T[(e >> 6) * kLS + (e & 63)];
            // the root of an infinite pivot comes out as inf * 0 (and only that); its row is held at zero
            Dk[e] = (e >> 6) == (e & 63) && v != v ? HUGE_VAL : v;
        }
    if (k + nb >= n) return;
    invert16(T, 16 * wave, rd, V + 16 * wave * 18, 18, lane);
    __syncthreads();
    // X_b = (A_b - sum_{j < b} X_j L_bj^T) V_b^T
    double *xs = X[wave];
#pragma unroll
    for (int b = 0; b < 4; ++b) {
        v4d acc = v4d{0.0, 0.0, 0.0, 0.0};
#pragma unroll
        for (int ks = 0; ks < 16 * b; ks += 4)
            acc = __builtin_amdgcn_mfma_f64_16x16x4f64(xs[l16 * kLS + ks + l4], T[(16 * b + l16) * kLS + ks + l4], acc,
                                                       0, 0, 0);
        // the tile as an A operand: through LDS (this wave's rows only)
#pragma unroll
        for (int r = 0; r < 4; ++r) xs[(4 * r + l4) * kLS + 16 * b + l16] = x[b][r] - acc[r];
        __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
        __builtin_amdgcn_wave_barrier();
        v4d y = v4d{0.0, 0.0, 0.0, 0.0};
#pragma unroll
        for (int ks = 0; ks < 16; ks += 4)
            y = __builtin_amdgcn_mfma_f64_16x16x4f64(xs[l16 * kLS + 16 * b + ks + l4], V[(16 * b + l16) * 18 + ks + l4],
                                                     y, 0, 0, 0);
        __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
        __builtin_amdgcn_wave_barrier();
#pragma unroll
        for (int r = 0; r < 4; ++r) {
            xs[(4 * r + l4) * kLS + 16 * b + l16] = y[r];
            const int i = row0 + 4 * r + l4;
            if (i < n) A[(int64_t)i * lda + k + 16 * b + l16] = y[r];
        }
        __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
        __builtin_amdgcn_wave_barrier();
    }
}

// The factored diagonal blocks to their places in A.
__global__ __launch_bounds__(256) void k_put_diag(int n, double *__restrict__ A, int64_t lda,
                                                  const double *__restrict__ D) {
    const int k = (int)blockIdx.x * kNB, nb = min(kNB, n - k);
    for (int e = threadIdx.x; e < kNB * kNB; e += 256) {
        const int i = e >> 6, c = e & 63;
        if (i < nb && c < nb) A[(int64_t)(k + i) * lda + k + c] = D[(int64_t)blockIdx.x * kNB * kNB + e];
    }
}

// Y = L^-1 on the 64x64 diagonal blocks (zeros above the diagonal): the 16x16 diagonal inverses, a wave
// each, then two doubling steps (16, 32) on the matrix cores, all in LDS. n = 4096: 8 us (a column
// per thread by substitution: 303 us).
__global__ __launch_bounds__(256) void k_tri_inverse_diag(int n, const double *__restrict__ L, int64_t lda,
                                                          double *__restrict__ Y, int64_t ldy) {
    __shared__ __align__(16) double T[kNB * kLS], V[kNB * kLS], W[32 * kLS];
    __shared__ double rd[kNB];
    const int k = (int)blockIdx.x * kNB, nb = min(kNB, n - k);
    const int tid = threadIdx.x, wave = tid >> 6, lane = tid & 63, l16 = lane & 15, l4 = lane >> 4;
    load_lower(L, lda, k, nb, T, tid);
    for (int e = tid; e < kNB * kLS; e += 256) V[e] = 0.0;
    __syncthreads();
    if (tid < kNB) rd[tid] = 1.0 / T[tid * kLS + tid];
    __syncthreads();
    invert16(T, 16 * wave, rd, V + 16 * wave * kLS + 16 * wave, kLS, lane);
    __syncthreads();
    // 16x16 tile of A B from LDS rows (A: rows ra.., B: rows rb.. of stride kLS, K deep)
    auto tile = [&](const double *A, const double *B, int K) {
        v4d acc = v4d{0.0, 0.0, 0.0, 0.0};
        for (int ks = 0; ks < K; ks += 4)
            acc = __builtin_amdgcn_mfma_f64_16x16x4f64(A[l16 * kLS + ks + l4], B[(ks + l4) * kLS + l16], acc, 0, 0, 0);
        return acc;
    };
    auto put = [&](double *C, const v4d &v, double f) {
#pragma unroll
        for (int r = 0; r < 4; ++r) C[(4 * r + l4) * kLS + l16] = f * v[r];
    };
#pragma unroll
    for (int s = 16; s < kNB; s *= 2) {
        // W = L21 Y11 of every pair, tiles taken in turn; then Y21 = -Y22 W
        const int side = s / 16, tiles = side * side * (kNB / (2 * s));
        for (int t = wave; t < tiles; t += 4) {
            const int p = t / (side * side), i = t / side % side, j = t % side, o = 2 * s * p;
            put(W + (s * p + 16 * i) * kLS + 16 * j, tile(T + (o + s + 16 * i) * kLS + o, V + o * kLS + o + 16 * j, s),
                1.0);
        }
        __syncthreads();
        for (int t = wave; t < tiles; t += 4) {
            const int p = t / (side * side), i = t / side % side, j = t % side, o = 2 * s * p;
            put(V + (o + s + 16 * i) * kLS + o + 16 * j,
                tile(V + (o + s + 16 * i) * kLS + o + s, W + s * p * kLS + 16 * j, s), -1.0);
        }
        __syncthreads();
    }
    for (int e = tid; e < kNB * kNB; e += 256) {
        const int i = e >> 6, c = e & 63;
        if (i < nb && c < nb) Y[(int64_t)(k + i) * ldy + k + c] = V[i * kLS + c];
    }
}

// y = M x, one wavefront per row. Lane l keeps eight chains, chain u summing columns
// l + 64 u + 512 j in order; the chains are combined in a fixed tree and the lanes by the
// butterfly, so the result is the same on every run. M is streamed (non-temporal loads). With
// an FP32 x the main loop issues two steps' loads (sixteen per lane) before adding them to the
// chains in the same order as one step at a time; an FP64 x keeps one step's eight. Measured
// with the 4096-row coarse inverse of a 256^3 MG-PCG hierarchy: FP32 x 30.5 -> 23.8 us per
// product; sixteen loads with an FP64 x took 35.7 us against 29.8 (the streamed M alone: FP64
// MG-PCG -2 ms).
template <typename TX, typename TY, typename TM = double>
__global__ __launch_bounds__(256) void k_gemv(int n, const TM *__restrict__ M, const TX *__restrict__ x,
                                              TY *__restrict__ y) {
    const int row = blockIdx.x * 4 + (threadIdx.x >> 6);
    const int lane = threadIdx.x & 63;
    if (row >= n) return;
    const TM *m = M + (int64_t)row * n;
    double a[8] = {0, 0, 0, 0, 0, 0, 0, 0};
    int c = lane;
    if constexpr (sizeof(TX) == 4) {
        for (; c + 15 * 64 < n; c += 16 * 64) {
            double mv[16], xv[16];
#pragma unroll
            for (int u = 0; u < 16; ++u) {
                mv[u] = (double)__builtin_nontemporal_load(m + c + u * 64);
                xv[u] = (double)x[c + u * 64];
            }
#pragma unroll
            for (int u = 0; u < 8; ++u) a[u] += mv[u] * xv[u];
#pragma unroll
            for (int u = 0; u < 8; ++u) a[u] += mv[8 + u] * xv[8 + u];
        }
    }
    for (; c + 7 * 64 < n; c += 8 * 64) {
        double mv[8], xv[8];
#pragma unroll
        for (int u = 0; u < 8; ++u) {
            mv[u] = (double)__builtin_nontemporal_load(m + c + u * 64);
            xv[u] = (double)x[c + u * 64];
        }
#pragma unroll
        for (int u = 0; u < 8; ++u) a[u] += mv[u] * xv[u];
    }
    for (int u = 0; c < n; c += 64, ++u) a[u] += (double)m[c] * (double)x[c];
    double s = ((a[0] + a[1]) + (a[2] + a[3])) + ((a[4] + a[5]) + (a[6] + a[7]));
    s = wave_sum(s);
    if (lane == 0) y[row] = (TY)s;
}

template <bool AK, bool BK_, Tri TRI>
static int gemm(uhip_ctx ctx, const GemmBlocks &g, int blocks) {
    if (g.M <= 0 || g.N <= 0 || blocks <= 0) return UHIP_OK;
    hipLaunchKernelGGL((k_gemm_f64<AK, BK_, TRI>), dim3((g.N + 63) / 64, (g.M + 63) / 64, blocks), dim3(256), 0,
                       ctx->stream, g);
    UHIP_CHECK_LAUNCH();
    return UHIP_OK;
}

}  // namespace uhip

using namespace uhip;

extern "C" {

int uhip_dense_cholesky(uhip_ctx ctx, int32_t n, double *A, int32_t lda, int *info_h) {
    UHIP_REQUIRE(ctx && A && info_h && n >= 0 && lda >= n, "uhip_dense_cholesky: bad argument");
    int *info = (int *)ctx->counters;
    UHIP_CHECK_HIP(hipMemsetAsync(info, 0, sizeof(int), ctx->stream));
    const int nblk = (n + kNB - 1) / kNB;
    Scratch w(ctx);
    const size_t o_d = w.add(sizeof(double) * kNB * kNB * (size_t)std::max(nblk, 1));
    UHIP_TRY(w.allocate());
    double *D = w.at<double>(o_d);
    for (int b = 0; b < nblk; ++b) {
        const int k = b * kNB, rest = n - k - kNB;
        hipLaunchKernelGGL(k_cholesky_panel, dim3(std::max(1, (rest + 63) / 64)), dim3(256), 0, ctx->stream, n, A,
                           (int64_t)lda, k, D + (size_t)b * kNB * kNB, info);
        UHIP_CHECK_LAUNCH();
        if (rest > 0) {
            // A22 -= L21 L21^T (lower triangle)
            const double *L21 = A + (int64_t)(k + kNB) * lda + k;
            const GemmBlocks g{L21, L21, A + (int64_t)(k + kNB) * lda + k + kNB, lda, lda, lda, 0, 0, 0,
                               rest, rest, kNB, n, k + kNB, 0, -1.0};
            UHIP_TRY((gemm<true, true, Tri::kLowerC>(ctx, g, 1)));
        }
    }
    if (nblk > 0) {
        hipLaunchKernelGGL(k_put_diag, dim3(nblk), dim3(256), 0, ctx->stream, n, A, (int64_t)lda, D);
        UHIP_CHECK_LAUNCH();
    }
    int32_t i32 = 0;
    UHIP_TRY(read_ints(ctx, info, 1, &i32));
    *info_h = i32;
    return UHIP_OK;
}

// Y = L^-1 by doubling: the 64x64 diagonal blocks first, all at once; then, for s = 64, 128, ..., every
// pair of neighbouring s x s diagonal inverses gets the block between them, Y21 = -Y22 (L21 Y11). 2 log2(n/64)
// launches in place of a chain of 2 n/64, and every product at least s deep. A^-1 = Y^T Y follows
// (one triangle, mirrored). The products leave out the zero halves of Y. Ainv is written by the last product
// only, which reads Y alone: it may be L's memory.
int uhip_dense_cholesky_inverse(uhip_ctx ctx, int32_t n, const double *L, int32_t lda, double *Ainv) {
    UHIP_REQUIRE(ctx && L && Ainv && n >= 0 && lda >= n, "uhip_dense_cholesky_inverse: bad argument");
    if (n == 0) return UHIP_OK;
    Scratch w(ctx);
    const size_t o_y = w.add(sizeof(double) * (size_t)n * n);
    const auto pairs_of = [n](int64_t s) { return (n - s + 2 * s - 1) / (2 * s); };
    int64_t t_size = 0;  // L21 Y11 of all pairs, s columns each; the last pair's rows end with the matrix
    for (int64_t s = kNB; s < n; s *= 2) {
        const int64_t before = pairs_of(s) - 1;
        t_size = std::max(t_size, before * s * s + std::min(s, n - s - before * 2 * s) * s);
    }
    const size_t o_t = w.add(sizeof(double) * (size_t)t_size);
    UHIP_TRY(w.allocate());
    double *Y = w.at<double>(o_y), *T = w.at<double>(o_t);
    hipLaunchKernelGGL(k_tri_inverse_diag, dim3((n + kNB - 1) / kNB), dim3(256), 0, ctx->stream, n, L, (int64_t)lda, Y,
                       (int64_t)n);
    UHIP_CHECK_LAUNCH();
    for (int64_t s = kNB; s < n; s *= 2) {
        const int si = (int)s, pairs = (int)pairs_of(s);
        const GemmBlocks t{L + s * lda, Y, T, lda, n, s, 2 * s * lda + 2 * s, 2 * s * n + 2 * s, s * s,
                           si, si, si, n, si, 2 * si, 1.0};
        UHIP_TRY((gemm<true, false, Tri::kBLower>(ctx, t, pairs)));
        const GemmBlocks y{Y + s * n + s, T, Y + s * n, n, s, n, 2 * s * n + 2 * s, s * s,
                           2 * s * n + 2 * s, si, si, si, n, si, 2 * si, -1.0};
        UHIP_TRY((gemm<true, false, Tri::kALower>(ctx, y, pairs)));
    }
    // A^-1 = Y^T Y:  Ainv(i,j) = sum_k Y(k,i) Y(k,j)
    const GemmBlocks a{Y, Y, Ainv, n, n, n, 0, 0, 0, n, n, n, n, 0, 0, 1.0};
    UHIP_TRY((gemm<false, false, Tri::kGram>(ctx, a, 1)));
    UHIP_CHECK_HIP(hipStreamSynchronize(ctx->stream));
    return UHIP_OK;
}

int uhip_dense_gemv(uhip_ctx ctx, int32_t n, const double *M, const void *x, int x_dtype, void *y, int y_dtype) {
    UHIP_REQUIRE(ctx && M && x && y && n >= 0, "uhip_dense_gemv: bad argument");
    if (n == 0) return UHIP_OK;
    dim3 g((n + 3) / 4), b(256);
    hipStream_t s = ctx->stream;
    if (x_dtype == UHIP_F64 && y_dtype == UHIP_F64)
        hipLaunchKernelGGL((k_gemv<double, double>), g, b, 0, s, n, M, (const double *)x, (double *)y);
    else if (x_dtype == UHIP_F32 && y_dtype == UHIP_F32)
        hipLaunchKernelGGL((k_gemv<float, float>), g, b, 0, s, n, M, (const float *)x, (float *)y);
    else if (x_dtype == UHIP_F32 && y_dtype == UHIP_F64)
        hipLaunchKernelGGL((k_gemv<float, double>), g, b, 0, s, n, M, (const float *)x, (double *)y);
    else
        hipLaunchKernelGGL((k_gemv<double, float>), g, b, 0, s, n, M, (const double *)x, (float *)y);
    UHIP_CHECK_LAUNCH();
    return UHIP_OK;
}

}  // extern "C"
