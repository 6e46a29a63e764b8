// Fused vector kernels of the Krylov and smoother loops. Step lengths are read
// from device scalars so a CG iteration needs one host read-back (the residual
// norm) instead of one per dot product.
#include <algorithm>

#include "uhip_common.hpp"
#include "uhip_spmv.hpp"

namespace uhip {

// out = xin + a * p   (xin may be null = 0), with dtype conversion. a == 0 adds nothing
// (VecAXPY with alpha 0 is a no-op), so the call is an exact copy / cast of xin.
template <typename TP, typename TX, typename TO, typename TAcc>
__global__ __launch_bounds__(kBlock) void k_axpy_cast(int64_t n, TAcc a, const TP *__restrict__ p,
                                                      const TX *__restrict__ xin, TO *__restrict__ out) {
    for (int64_t i = (int64_t)blockIdx.x * kBlock + threadIdx.x; i < n; i += (int64_t)gridDim.x * kBlock) {
        TAcc v = xin ? (TAcc)xin[i] : TAcc(0);
        if (a != TAcc(0)) v = v + a * (TAcc)p[i];
        out[i] = (TO)v;
    }
}

// alpha = s[i_num]/s[i_den]; x += alpha*p; rn = r - alpha*Ap; partial |rn|^2.
// Block 0 stores alpha to s[i_alpha].
__global__ __launch_bounds__(kBlock) void k_cg_update(int64_t n, double *__restrict__ x,
                                                      const double *__restrict__ p, const double *__restrict__ r,
                                                      const double *__restrict__ Ap, double *__restrict__ rn,
                                                      double *__restrict__ s, int i_num, int i_den, int i_alpha,
                                                      double *__restrict__ partials) {
    const double alpha = s[i_num] / s[i_den];
    if (!isfinite(alpha)) {  // CG stops before touching x (utopia_ConjugateGradient_impl.hpp:241-244)
        if (blockIdx.x == 0 && threadIdx.x == 0) s[i_alpha] = alpha;
        return;
    }
    double acc = 0.0;
    for (int64_t i = (int64_t)blockIdx.x * kBlock + threadIdx.x; i < n; i += (int64_t)gridDim.x * kBlock) {
        x[i] = x[i] + alpha * p[i];
        const double v = r[i] - alpha * Ap[i];
        rn[i] = v;
        acc += v * v;
    }
    acc = block_sum<kBlock>(acc);
    if (threadIdx.x == 0) {
        partials[blockIdx.x] = acc;
        if (blockIdx.x == 0) s[i_alpha] = alpha;
    }
}

// beta = s[i_num]/s[i_den]; p = z + beta*p; afterwards s[i_den] = s[i_num] (the
// next iteration's dot(z, r) is this iteration's dot(z_new, r_new)).
__global__ __launch_bounds__(kBlock) void k_cg_pupdate(int64_t n, double *__restrict__ p, const double *__restrict__ z,
                                                       const double *__restrict__ s, int i_num, int i_den) {
    const double beta = s[i_num] / s[i_den];
    for (int64_t i = (int64_t)blockIdx.x * kBlock + threadIdx.x; i < n; i += (int64_t)gridDim.x * kBlock)
        p[i] = z[i] + beta * p[i];
}

// alpha = s[i_num]/den, den the sum of den_n partial sums (or one finished); rn = r - alpha*Ap (and
// rn32 = (float)rn when given); partial |rn|^2. x is left to k_cg_xpupdate. Block 0 stores alpha.
__global__ __launch_bounds__(kBlock) void k_cg_residual(int64_t n, const double *__restrict__ r,
                                                        const double *__restrict__ Ap, double *__restrict__ rn,
                                                        float *__restrict__ rn32, double *__restrict__ s, int i_num,
                                                        const double *__restrict__ den, int den_n, int i_alpha,
                                                        double *__restrict__ partials) {
    double d[1];
    sum_partials<kBlock, 1>(den, 0, den_n, d);
    const double alpha = s[i_num] / d[0];
    if (!isfinite(alpha)) {
        if (blockIdx.x == 0 && threadIdx.x == 0) s[i_alpha] = alpha;
        return;
    }
    // four grid-strided entries per step, their loads issued together (the grid is capped at
    // kMaxRedBlocks, so each thread covers many entries)
    double acc = 0.0;
    const int64_t st = (int64_t)gridDim.x * kBlock;
    int64_t i = (int64_t)blockIdx.x * kBlock + threadIdx.x;
    for (; i + 3 * st < n; i += 4 * st) {
        double rv[4], av[4];
#pragma unroll
        for (int u = 0; u < 4; ++u) {
            rv[u] = __builtin_nontemporal_load(r + i + u * st);
            av[u] = __builtin_nontemporal_load(Ap + i + u * st);
        }
#pragma unroll
        for (int u = 0; u < 4; ++u) {
            const double v = rv[u] - alpha * av[u];
            __builtin_nontemporal_store(v, rn + i + u * st);
            // the FP32 copy is the preconditioner's next input: a cached store keeps it in the MALL
            if (rn32) rn32[i + u * st] = (float)v;
            acc += v * v;
        }
    }
    for (; i < n; i += st) {
        const double v = r[i] - alpha * Ap[i];
        __builtin_nontemporal_store(v, rn + i);
        if (rn32) rn32[i] = (float)v;
        acc += v * v;
    }
    acc = block_sum<kBlock>(acc);
    if (threadIdx.x == 0) {
        partials[blockIdx.x] = acc;
        if (blockIdx.x == 0) s[i_alpha] = alpha;
    }
}

// What a CG iteration tells the host: alpha (value[0]) and |r| (value[1]) of iteration seq.
__device__ __forceinline__ void report_iteration(RunStatus *status, long long seq, double alpha, double rr) {
    status->value[0] = alpha;
    status->value[1] = sqrt(rr);
    __hip_atomic_store(&status->steps, seq, __ATOMIC_RELEASE, __HIP_MEMORY_SCOPE_SYSTEM);
}

__global__ __launch_bounds__(kBlock) void k_cg_report(const double *__restrict__ s, int i_alpha,
                                                      const double *__restrict__ rr, int rr_n, long long seq,
                                                      RunStatus *__restrict__ status) {
    double t[1];
    sum_partials<kBlock, 1>(rr, 0, rr_n, t);
    if (threadIdx.x == 0) report_iteration(status, seq, s[i_alpha], t[0]);
}

// x += s[i_alpha]*p, then (z given) p = z + beta*p with beta = num/s[i_den], num the sum of num_n partial sums
// (or one finished): the x update of iteration k uses p_k before it is replaced by p_{k+1}.
// REPORT: block 0 keeps num as s[i_num] and tells the host of iteration seq (|r| from rr_n partial sums).
template <typename TZ, bool REPORT>
__global__ __launch_bounds__(kBlock) void k_cg_xpupdate(int64_t n, double *__restrict__ x, double *__restrict__ p,
                                                        const TZ *__restrict__ z, double *__restrict__ s,
                                                        int i_alpha, int i_num, int i_den,
                                                        const double *__restrict__ num, int num_n,
                                                        const double *__restrict__ rr, int rr_n, long long seq,
                                                        RunStatus *__restrict__ status) {
    const double alpha = s[i_alpha];
    if (REPORT && blockIdx.x == 0) {
        double t[1];
        sum_partials<kBlock, 1>(rr, 0, rr_n, t);
        if (threadIdx.x == 0) report_iteration(status, seq, alpha, t[0]);
    }
    if (!isfinite(alpha)) return;  // the CG stops before touching x
    double beta = 0.0;
    if (z) {
        double t[1];
        sum_partials<kBlock, 1>(num, 0, num_n, t);
        beta = t[0] / s[i_den];
        // a finished num is s[i_num] itself, which the other workgroups read: nothing to store
        if (REPORT && num != s + i_num && blockIdx.x == 0 && threadIdx.x == 0) s[i_num] = t[0];
    }
    // x streams (loaded and stored non-temporally: it is next read by the next iteration's update,
    // so caching it only evicts the next product's operands); p and z go through the caches (z was
    // just written by the preconditioner, p is read next by A p). Measured at 256^3 against
    // cached x loads: MG-PCG mixed -1.4 to -1.8 ms, FP64 -2 to -3 ms; loading p and z
    // non-temporally as well gave back 1.2 - 1.5 ms of it.
    for (int64_t i = (int64_t)blockIdx.x * kBlock + threadIdx.x; i < n; i += (int64_t)gridDim.x * kBlock) {
        const double pi = p[i];
        __builtin_nontemporal_store(__builtin_nontemporal_load(x + i) + alpha * pi, x + i);
        if (z) p[i] = (double)z[i] + beta * pi;
    }
}

// CG preconditioned by the inverse diagonal (InvDiagPreconditioner), an iteration in three launches:
// A p with p.Ap, the two kernels below; in two on small diagonal plans, where the update joins the next product
// (k_jcg_product_dia). Each adds its producer's partial sums itself and the host does
// not wait for an iteration: block 0 reports alpha's validity and |r| to pinned memory, and the
// iterations that the host has already sent past the end do nothing. 2D Poisson, 256 x 256 (749
// iterations): 35.5 -> 12.9 us an iteration in three launches, 10.2 in two, of 4 to 5.5 us each (latency: their partial
// sums, one block sum, one pass over vectors that the caches hold).
// The scalars that iterations hand on: rz[j & 1] of iteration j, alpha; the loop's end: the last
// iteration that counts (kernels of later ones return).
struct JcgScalars {
    double rz[2];
    double alpha;
    long long last;
};

// Iteration j: alpha = rz / p.Ap; r -= alpha Ap; partial sums of r.r and r.z with z = d r (kept when given).
__global__ __launch_bounds__(kBlock) void k_jcg_residual(int64_t n, long long j, double *__restrict__ r,
                                                         const double *__restrict__ Ap, const double *__restrict__ d,
                                                         const double *__restrict__ pap, int pap_n,
                                                         JcgScalars *__restrict__ s, double *__restrict__ parts,
                                                         int64_t stride, RunStatus *__restrict__ status,
                                                         double *__restrict__ z) {
    constexpr int U = 4;
    const int64_t st = (int64_t)gridDim.x * kBlock, i0 = (int64_t)blockIdx.x * kBlock + threadIdx.x;
    double rv[U], av[U], dv[U];
    auto load = [&](int64_t i) {
#pragma unroll
        for (int u = 0; u < U; ++u) {
            const int64_t k = i + u * st < n ? i + u * st : n - 1;
            rv[u] = r[k];
            av[u] = Ap[k];
            dv[u] = d[k];
        }
    };
    load(i0);  // behind the sum of the partial sums
    if (s->last < j) return;
    double den[1];
    sum_partials<kBlock, 1>(pap, 0, pap_n, den);
    const double alpha = s->rz[j & 1] / den[0];
    const bool first = blockIdx.x == 0 && threadIdx.x == 0;
    if (!isfinite(alpha)) {  // stops before touching x (utopia_ConjugateGradient_impl.hpp:241-244)
        if (first) {
            s->last = j - 1;
            status->done = 2;
            __threadfence_system();
        }
        return;
    }
    double dots[2] = {0.0, 0.0};
    for (int64_t i = i0; i < n; i += U * st) {
        if (i != i0) load(i);
#pragma unroll
        for (int u = 0; u < U; ++u)
            if (i + u * st < n) {
                const double v = rv[u] - alpha * av[u];
                r[i + u * st] = v;
                if (z) z[i + u * st] = dv[u] * v;
                dots[0] += v * v;
                dots[1] += (dv[u] * v) * v;
            }
    }
    block_totals<kBlock, 2>(dots);
    if (threadIdx.x == 0) {
        parts[blockIdx.x] = dots[0];
        parts[stride + blockIdx.x] = dots[1];
        if (blockIdx.x == 0) s->alpha = alpha;
    }
}

// Iteration j: x += alpha p; p = d r + (r.z / rz) p. Block 0 hands r.z on and reports |r|; with |r| <= atol
// iteration j is the last.
__global__ __launch_bounds__(kBlock) void k_jcg_update(int64_t n, long long j, double *__restrict__ x,
                                                       double *__restrict__ p, const double *__restrict__ r,
                                                       const double *__restrict__ d, const double *__restrict__ sums,
                                                       int sums_n, int64_t stride, double atol,
                                                       JcgScalars *__restrict__ s, RunStatus *__restrict__ status) {
    constexpr int U = 4;
    const int64_t st = (int64_t)gridDim.x * kBlock, i0 = (int64_t)blockIdx.x * kBlock + threadIdx.x;
    double xv[U], pv[U], rv[U], dv[U];
    auto load = [&](int64_t i) {
#pragma unroll
        for (int u = 0; u < U; ++u) {
            const int64_t k = i + u * st < n ? i + u * st : n - 1;
            xv[u] = x[k];
            pv[u] = p[k];
            rv[u] = r[k];
            dv[u] = d[k];
        }
    };
    load(i0);
    if (s->last < j) return;
    double dots[2];  // r.r, r.z
    sum_partials<kBlock, 2>(sums, stride, sums_n, dots);
    const double alpha = s->alpha, beta = dots[1] / s->rz[j & 1];
    if (blockIdx.x == 0 && threadIdx.x == 0) {
        const double norm = sqrt(dots[0]);
        s->rz[(j + 1) & 1] = dots[1];
        status->value[0] = norm;
        if (norm <= atol) {
            s->last = j;
            status->done = 1;
        }
        __hip_atomic_store(&status->steps, j + 1, __ATOMIC_RELEASE, __HIP_MEMORY_SCOPE_SYSTEM);
    }
    for (int64_t i = i0; i < n; i += U * st) {
        if (i != i0) load(i);
#pragma unroll
        for (int u = 0; u < U; ++u)
            if (i + u * st < n) {
                x[i + u * st] = xv[u] + alpha * pv[u];
                p[i + u * st] = dv[u] * rv[u] + beta * pv[u];
            }
    }
}

// The end of iteration j - 1 (as k_jcg_update) and the product of iteration j in one launch, on a DIA plan: p = z + beta
// p_old is formed again at each entry's column (the same operations, so the same bits), from z and p_old that no
// kernel is writing, and stored to the other of two buffers. One row a thread and the rows' loads issued before the
// partial sums are added, as in k_spmv_dia on few rows.
template <typename TM, bool SYM>
__global__ __launch_bounds__(kBlock) void k_jcg_product_dia(int32_t n, int32_t ndiag, const int32_t *__restrict__ off,
                                                            const double *__restrict__ val, const TM *__restrict__ mask,
                                                            long long j, double *__restrict__ x,
                                                            const double *__restrict__ z, const double *__restrict__ p,
                                                            double *__restrict__ pn, double *__restrict__ Ap,
                                                            const double *__restrict__ sums, int sums_n, int64_t stride,
                                                            double atol, JcgScalars *__restrict__ s,
                                                            double *__restrict__ parts,
                                                            RunStatus *__restrict__ status) {
    constexpr int G = sizeof(TM) == 1 ? 8 : 16;  // diagonals whose loads are in flight together
    const int b = xcd_remap(blockIdx.x, gridDim.x);
    const int32_t row = b * kBlock + (int32_t)threadIdx.x, rc = min(row, n - 1), k = ndiag >> 1;
    const int64_t ld = dia_ld(n);
    const uint32_t m = (uint32_t)mask[rc];
    const double xo = x[rc], zo = z[rc], po = p[rc];
    double vv[G], zv[G], pv[G];
    auto load = [&](int d) {
#pragma unroll
        for (int u = 0; u < G; ++u)
            if (d + u < ndiag) {
                const int32_t o = off[d + u], c = min(max(rc + o, 0), n - 1);
                if constexpr (SYM)
                    vv[u] = val[(int64_t)(d + u < k ? k - d - u : d + u - k) * ld + min(max(rc + (d + u < k ? o : 0), 0), (int32_t)ld - 1)];
                else
                    vv[u] = val[(int64_t)(d + u) * ld + rc];
                zv[u] = z[c];
                pv[u] = p[c];
            }
    };
    load(0);
    if (s->last < j - 1) return;
    double dots[2];  // r.r, r.z of iteration j - 1
    sum_partials<kBlock, 2>(sums, stride, sums_n, dots);
    const double alpha = s->alpha, beta = dots[1] / s->rz[(j - 1) & 1], norm = sqrt(dots[0]);
    if (blockIdx.x == 0 && threadIdx.x == 0) {
        s->rz[j & 1] = dots[1];
        status->value[0] = norm;
        if (norm <= atol) {
            s->last = j - 1;
            status->done = 1;
        }
        __hip_atomic_store(&status->steps, j, __ATOMIC_RELEASE, __HIP_MEMORY_SCOPE_SYSTEM);
    }
    const double pi = zo + beta * po;
    if (row < n) {
        x[row] = xo + alpha * po;
        pn[row] = pi;
    }
    if (norm <= atol) return;
    double acc = 0.0;
    for (int d = 0; d < ndiag; d += G) {
        if (d > 0) load(d);
#pragma unroll
        for (int u = 0; u < G; ++u)
            if (d + u < ndiag) {
                const double t = vv[u] * (zv[u] + beta * pv[u]);
                acc = ((m >> (d + u)) & 1u) ? acc + t : acc;
            }
    }
    if (row < n) Ap[row] = acc;
    const double t = block_sum<kBlock>(row < n ? pi * acc : 0.0);
    if (threadIdx.x == 0) parts[b] = t;
}

__global__ void k_jcg_begin(JcgScalars *__restrict__ s, const double *__restrict__ rz) {
    s->rz[0] = *rz;
    s->last = 0x7fffffffffffffffll;
}

__global__ void k_scalar_copy(double *s, int dst, int src) { s[dst] = s[src]; }

}  // namespace uhip

using namespace uhip;

extern "C" {

int uhip_vec_axpy_cast(uhip_ctx ctx, int64_t n, double a, const void *p, int p_dtype, const void *xin, int x_dtype,
                       void *out, int out_dtype) {
    UHIP_REQUIRE(ctx && p && out, "uhip_vec_axpy_cast: null argument");
    if (n <= 0) return UHIP_OK;
    dim3 g(grid_for(n, 1, 1 << 16)), b(kBlock);
    hipStream_t s = ctx->stream;
    // working precision: float only if every operand is float
    const bool f32 = p_dtype == UHIP_F32 && (xin == nullptr || x_dtype == UHIP_F32) && out_dtype == UHIP_F32;
#define UHIP_AC(TP, TX, TO, TA)                                                                     \
    hipLaunchKernelGGL((k_axpy_cast<TP, TX, TO, TA>), g, b, 0, s, n, (TA)a, (const TP *)p, (const TX *)xin, \
                       (TO *)out)
    if (f32) {
        UHIP_AC(float, float, float, float);
    } else if (p_dtype == UHIP_F64 && x_dtype != UHIP_F32 && out_dtype == UHIP_F64) {
        UHIP_AC(double, double, double, double);
    } else if (p_dtype == UHIP_F32 && out_dtype == UHIP_F64) {
        if (xin && x_dtype == UHIP_F64) UHIP_AC(float, double, double, double);
        else UHIP_AC(float, float, double, float);
    } else if (p_dtype == UHIP_F64 && out_dtype == UHIP_F32) {
        if (xin && x_dtype == UHIP_F64) UHIP_AC(double, double, float, double);
        else UHIP_AC(double, float, float, float);
    } else {
        UHIP_AC(double, float, double, double);
    }
#undef UHIP_AC
    UHIP_CHECK_LAUNCH();
    return UHIP_OK;
}

int uhip_cg_update_f64(uhip_ctx ctx, int64_t n, double *x, const double *p, const double *r, const double *Ap,
                       double *r_new, double *scalars, int i_num, int i_den, int i_alpha, int i_rnorm) {
    UHIP_REQUIRE(ctx && x && p && r && Ap && r_new && scalars, "uhip_cg_update_f64: null argument");
    const int g = grid_for(n, 4, kMaxRedBlocks);
    UHIP_TRY(ensure_partials(ctx, g));
    hipLaunchKernelGGL(k_cg_update, dim3(g), dim3(kBlock), 0, ctx->stream, n, x, p, r, Ap, r_new, scalars, i_num,
                       i_den, i_alpha, ctx->partials);
    UHIP_CHECK_LAUNCH();
    return finish_sums(ctx, 1, g, ctx->max_partials, scalars + i_rnorm, 1u);
}

int uhip_cg_pupdate_f64(uhip_ctx ctx, int64_t n, double *p, const double *z, double *scalars, int i_num, int i_den) {
    UHIP_REQUIRE(ctx && p && z && scalars, "uhip_cg_pupdate_f64: null argument");
    UHIP_TRY(finish_left(ctx));
    if (n > 0) {
        hipLaunchKernelGGL(k_cg_pupdate, dim3(grid_for(n, 4, 1 << 16)), dim3(kBlock), 0, ctx->stream, n, p, z,
                           scalars, i_num, i_den);
        UHIP_CHECK_LAUNCH();
    }
    hipLaunchKernelGGL(k_scalar_copy, dim3(1), dim3(1), 0, ctx->stream, scalars, i_den, i_num);
    UHIP_CHECK_LAUNCH();
    return UHIP_OK;
}

int uhip_cg_residual_f64(uhip_ctx ctx, int64_t n, const double *r, const double *Ap, double *r_new, float *r_new32,
                         double *scalars, int i_num, int i_den, int i_alpha, int i_rnorm) {
    UHIP_REQUIRE(ctx && r && Ap && r_new && scalars, "uhip_cg_residual_f64: null argument");
    const int g = grid_for(n, 4, kMaxRedBlocks);
    UHIP_TRY(ensure_partials(ctx, g));
    hipLaunchKernelGGL(k_cg_residual, dim3(g), dim3(kBlock), 0, ctx->stream, n, r, Ap, r_new, r_new32, scalars, i_num,
                       scalars + i_den, 1, i_alpha, ctx->partials);
    UHIP_CHECK_LAUNCH();
    return finish_sums(ctx, 1, g, ctx->max_partials, scalars + i_rnorm, 1u);
}

int uhip_cg_xpupdate_f64(uhip_ctx ctx, int64_t n, double *x, double *p, const double *z, double *scalars, int i_alpha,
                         int i_num, int i_den) {
    UHIP_REQUIRE(ctx && x && p && scalars, "uhip_cg_xpupdate_f64: null argument");
    UHIP_TRY(finish_left(ctx));
    if (n > 0) {
        hipLaunchKernelGGL((k_cg_xpupdate<double, false>), dim3(grid_for(n, 4, 1 << 16)), dim3(kBlock), 0, ctx->stream, n,
                           x, p, z, scalars, i_alpha, i_num, i_den, scalars + i_num, 1, nullptr, 0, 0ll, nullptr);
        UHIP_CHECK_LAUNCH();
    }
    if (z) {
        hipLaunchKernelGGL(k_scalar_copy, dim3(1), dim3(1), 0, ctx->stream, scalars, i_den, i_num);
        UHIP_CHECK_LAUNCH();
    }
    return UHIP_OK;
}

int uhip_cg_xpupdate2(uhip_ctx ctx, int64_t n, double *x, double *p, const void *z, int z_dtype, double *scalars,
                      int i_alpha, int i_num, int i_den) {
    UHIP_REQUIRE(ctx && x && p && z && scalars, "uhip_cg_xpupdate2: null argument");
    UHIP_REQUIRE(z_dtype == UHIP_F64 || z_dtype == UHIP_F32, "uhip_cg_xpupdate2: z dtype");
    UHIP_TRY(finish_left(ctx));
    if (n <= 0) return UHIP_OK;
    const dim3 g(grid_for(n, 4, 1 << 16)), b(kBlock);
    if (z_dtype == UHIP_F64)
        hipLaunchKernelGGL((k_cg_xpupdate<double, false>), g, b, 0, ctx->stream, n, x, p, (const double *)z, scalars, i_alpha,
                           i_num, i_den, scalars + i_num, 1, nullptr, 0, 0ll, nullptr);
    else
        hipLaunchKernelGGL((k_cg_xpupdate<float, false>), g, b, 0, ctx->stream, n, x, p, (const float *)z, scalars, i_alpha,
                           i_num, i_den, scalars + i_num, 1, nullptr, 0, 0ll, nullptr);
    UHIP_CHECK_LAUNCH();
    return UHIP_OK;
}

// the partial sums of the dot wanted at `finished` where it was left as such, or its finished value
static int take_sum(uhip_ctx ctx, double *finished, const double **parts, int *count) {
    *parts = finished;
    *count = 1;
    if (ctx->left == 0 || ctx->left_for != finished) return finish_left(ctx);
    *parts = ctx->partials;
    *count = ctx->left;
    ctx->left = 0;
    return UHIP_OK;
}

int64_t uhip_cg_residual_parts(int64_t n) { return grid_for(n, 4, kMaxRedBlocks); }

int uhip_cg_begin(uhip_ctx ctx) {
    UHIP_REQUIRE(ctx, "uhip_cg_begin: null context");
    UHIP_CHECK_HIP(hipStreamSynchronize(ctx->stream));  // no kernel of an earlier loop still reports
    memset(run_record(ctx), 0, sizeof(RunStatus));
    return UHIP_OK;
}

int uhip_cg_residual2_f64(uhip_ctx ctx, int64_t n, const double *r, const double *Ap, double *r_new, float *r_new32,
                          double *scalars, int i_num, int i_den, int i_alpha, double *rr_parts) {
    UHIP_REQUIRE(ctx && r && Ap && r_new && scalars && rr_parts, "uhip_cg_residual2_f64: null argument");
    const double *den = nullptr;
    int den_n = 0;
    UHIP_TRY(take_sum(ctx, scalars + i_den, &den, &den_n));
    hipLaunchKernelGGL(k_cg_residual, dim3((unsigned)uhip_cg_residual_parts(n)), dim3(kBlock), 0, ctx->stream, n, r, Ap,
                       r_new, r_new32, scalars, i_num, den, den_n, i_alpha, rr_parts);
    UHIP_CHECK_LAUNCH();
    return UHIP_OK;
}

int uhip_cg_report(uhip_ctx ctx, int64_t n, const double *scalars, int i_alpha, const double *rr_parts, int64_t seq) {
    UHIP_REQUIRE(ctx && scalars && rr_parts, "uhip_cg_report: null argument");
    hipLaunchKernelGGL(k_cg_report, dim3(1), dim3(kBlock), 0, ctx->stream, scalars, i_alpha, rr_parts,
                       (int)uhip_cg_residual_parts(n), (long long)seq, run_record(ctx));
    UHIP_CHECK_LAUNCH();
    return UHIP_OK;
}

int uhip_cg_xpupdate3(uhip_ctx ctx, int64_t n, double *x, double *p, const void *z, int z_dtype, double *scalars,
                      int i_alpha, int i_num, int i_den, const double *rr_parts, int64_t seq) {
    UHIP_REQUIRE(ctx && x && p && z && scalars && rr_parts, "uhip_cg_xpupdate3: null argument");
    UHIP_REQUIRE(z_dtype == UHIP_F64 || z_dtype == UHIP_F32, "uhip_cg_xpupdate3: z dtype");
    const double *num = nullptr;
    int num_n = 0;
    UHIP_TRY(take_sum(ctx, scalars + i_num, &num, &num_n));
    const dim3 g(grid_for(n, 4, 1 << 16)), b(kBlock);
    const int rr_n = (int)uhip_cg_residual_parts(n);
    if (z_dtype == UHIP_F64)
        hipLaunchKernelGGL((k_cg_xpupdate<double, true>), g, b, 0, ctx->stream, n, x, p, (const double *)z, scalars, i_alpha,
                           i_num, i_den, num, num_n, rr_parts, rr_n, (long long)seq, run_record(ctx));
    else
        hipLaunchKernelGGL((k_cg_xpupdate<float, true>), g, b, 0, ctx->stream, n, x, p, (const float *)z, scalars, i_alpha,
                           i_num, i_den, num, num_n, rr_parts, rr_n, (long long)seq, run_record(ctx));
    UHIP_CHECK_LAUNCH();
    return UHIP_OK;
}

int uhip_cg_wait(uhip_ctx ctx, int64_t seq, double *alpha, double *r_norm) {
    UHIP_REQUIRE(ctx && alpha && r_norm, "uhip_cg_wait: null argument");
    UHIP_TRY(run_wait(ctx, (long long)seq));
    volatile RunStatus *st = run_record(ctx);
    *alpha = st->value[0];
    *r_norm = st->value[1];
    return UHIP_OK;
}

int uhip_cg_jacobi_f64(uhip_ctx ctx, const uhip_csr *A, const double *dinv, double *x, double *r, double *p, double *Ap,
                       const double *rz_d, double atol, int64_t max_steps, int64_t *steps, double *r_norm,
                       int *reason) {
    UHIP_REQUIRE(ctx && A && dinv && x && r && p && Ap && rz_d && steps && r_norm && reason,
                 "uhip_cg_jacobi_f64: null argument");
    UHIP_REQUIRE(A->nrows == A->ncols && A->dtype == UHIP_F64, "uhip_cg_jacobi_f64: square FP64 matrix");
    const int64_t n = A->nrows;
    *steps = 0;
    *reason = n == 0 ? 2 : 0;  // nothing to iterate on: alpha = 0 / 0
    if (n == 0 || max_steps <= 0) return UHIP_OK;
    hipStream_t st = ctx->stream;
    // one entry a thread up to 1024 workgroups: more of the chip on short vectors
    const int g = grid_for(n, 1, kMaxRedBlocks);
    const int64_t np = spmv_parts(A);
    // Few rows on a DIA plan that the general DIA kernel takes: the launches are what takes the time, so the update goes
    // with the next product, at two more loads an entry. An iteration in three launches / in two: 5 diagonals
    // 4096 rows 11.1 / 9.2 us, 65,536 11.8 / 9.5, 160,000 15.9 / 13.0, 524,176 22.6 / 21.9; 9 diagonals 65,536 12.5 / 10.3,
    // 490,000 25.1 / 26.2; 27 diagonals 2744 13.4 / 12.1, 91,125 17.0 / 15.1, 238,328 27.9 / 26.7.
    const bool two = max_steps > 1 && A->format == UHIP_FMT_DIA && !A->dia_w27 && A->dia_sym != 2 && !A->dia_delta &&
                     n <= 1 << 18;
    const int gp = (int)((n + kBlock - 1) / kBlock);
    Scratch w(ctx);
    const size_t o_pap = w.add(sizeof(double) * (size_t)std::max<int64_t>(np, two ? gp : 1)),
                 o_dots = w.add(sizeof(double) * 2 * g), o_s = w.add(sizeof(JcgScalars)), o_sum = w.add(sizeof(double)),
                 o_p = w.add(two ? sizeof(double) * (size_t)n : 0), o_z = w.add(two ? sizeof(double) * (size_t)n : 0);
    UHIP_TRY(w.allocate());
    double *pap = w.at<double>(o_pap), *dots = w.at<double>(o_dots);
    double *buf[2] = {p, two ? w.at<double>(o_p) : p}, *z = two ? w.at<double>(o_z) : nullptr;  // p_j in buf[j & 1]
    JcgScalars *s = w.at<JcgScalars>(o_s);
    const bool many = np > kConsumerSums;
    RunScope scope(ctx);
    UHIP_TRY(scope.status());
    RunStatus *status = run_record(ctx);
    UHIP_CHECK_HIP(hipStreamSynchronize(st));  // no kernel of an earlier loop still reports
    memset(status, 0, sizeof(*status));
    hipLaunchKernelGGL(k_jcg_begin, dim3(1), dim3(1), 0, st, s, rz_d);
    UHIP_CHECK_LAUNCH();
    // the host stays kAhead iterations ahead: enough to hide the launches, few to run empty at the end
    constexpr int64_t kAhead = 6;
    volatile RunStatus *seen = status;
    int64_t j = 0;
    for (; j < max_steps && !seen->done; ++j) {
        int count = gp;
        if (!two || j == 0) {
            UHIP_TRY(spmv_dots_into(ctx, A, p, Ap, nullptr, pap, np, &count));
        } else {
#define UHIP_JCG(TM, SYM)                                                                                              \
    hipLaunchKernelGGL((k_jcg_product_dia<TM, SYM>), dim3(gp), dim3(kBlock), 0, st, A->nrows, A->ndiag, A->dia_off,    \
                       (const double *)A->dia_val, (const TM *)A->dia_mask, (long long)j, x, z, buf[(j - 1) & 1],      \
                       buf[j & 1], Ap, dots, g, (int64_t)g, atol, s, pap, status)
            if (A->ndiag <= 8) {
                if (A->dia_sym) UHIP_JCG(uint8_t, true);
                else UHIP_JCG(uint8_t, false);
            } else if (A->ndiag <= 16) {
                if (A->dia_sym) UHIP_JCG(uint16_t, true);
                else UHIP_JCG(uint16_t, false);
            } else {
                if (A->dia_sym) UHIP_JCG(uint32_t, true);
                else UHIP_JCG(uint32_t, false);
            }
#undef UHIP_JCG
            UHIP_CHECK_LAUNCH();
        }
        if (many) UHIP_TRY(finish_sums_from(ctx, pap, 1, count, np, w.at<double>(o_sum)));
        hipLaunchKernelGGL(k_jcg_residual, dim3(g), dim3(kBlock), 0, st, n, (long long)j, r, Ap, dinv,
                           many ? w.at<double>(o_sum) : pap, many ? 1 : count, s, dots, (int64_t)g, status, z);
        UHIP_CHECK_LAUNCH();
        if (!two || j + 1 == max_steps) {
            hipLaunchKernelGGL(k_jcg_update, dim3(g), dim3(kBlock), 0, st, n, (long long)j, x, buf[two ? j & 1 : 0], r, dinv, dots, g,
                               (int64_t)g, atol, s, status);
            UHIP_CHECK_LAUNCH();
        }
        if (j >= kAhead) UHIP_TRY(run_wait(ctx, j + 1 - kAhead));
    }
    UHIP_CHECK_HIP(hipStreamSynchronize(st));
    // the caller's p: written by the last update in place, else by the product after the last iteration
    if (two && ((seen->steps == max_steps ? max_steps - 1 : seen->steps) & 1)) {
        UHIP_CHECK_HIP(hipMemcpyAsync(p, buf[1], sizeof(double) * (size_t)n, hipMemcpyDeviceToDevice, st));
        UHIP_CHECK_HIP(hipStreamSynchronize(st));
    }
    *steps = seen->steps;
    *reason = seen->done;
    *r_norm = seen->value[0];
    return UHIP_OK;
}

}  // extern "C"
