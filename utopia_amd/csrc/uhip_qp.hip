// Box-constrained QP kernels: projection onto [lb, ub], the element-wise MPRGP
// operators (free gradient fi, chopped gradient beta, feasible step length), and
// the multicolour projected Gauss-Seidel sweep with its graph colouring.
#include <hipcub/hipcub.hpp>

#include <algorithm>
#include <cfloat>
#include <vector>

#include "uhip_common.hpp"

namespace uhip {

// VariableBoundSolverInterface::project (utopia_VariableBoundSolverInterface.hpp:107-155)
__device__ __forceinline__ double clamp_box(double x, double l, double u) { return (l >= x) ? l : ((u <= x) ? u : x); }

// ProjectedConjugateGradient::apply, element loop (utopia_ProjectedConjugateGradient.hpp:71-97).
// The active test reads z (the reference's x_view is a view of zk): elem = z_i,
// val = (|elem - ub_i| <= eps or |elem - lb_i| <= eps) ? max(u_i, 0) : u_i,
// z_i = (val == 0) ? max(p_i, 0) : p_i, w_i = val.
__global__ __launch_bounds__(kBlock) void k_pcg_wz(int64_t n, const double *__restrict__ u,
                                                   const double *__restrict__ lb, const double *__restrict__ ub,
                                                   const double *__restrict__ p, double *__restrict__ z,
                                                   double *__restrict__ w) {
    const double eps = DBL_EPSILON;
    for (int64_t i = (int64_t)blockIdx.x * kBlock + threadIdx.x; i < n; i += (int64_t)gridDim.x * kBlock) {
        const double elem = z[i];
        const double ui = u[i];
        const double val = (fabs(elem - ub[i]) <= eps || fabs(elem - lb[i]) <= eps) ? fmax(ui, 0.0) : ui;
        z[i] = (val == 0.0) ? fmax(p[i], 0.0) : p[i];
        w[i] = val;
    }
}

// ProjectedGradient::solve direction (utopia_ProjectedGradient.hpp:157-170):
// p_i = 0 where x_i is within 10 eps of a bound, else u_i.
__global__ __launch_bounds__(kBlock) void k_pg_dir(int64_t n, const double *__restrict__ x,
                                                   const double *__restrict__ u, const double *__restrict__ lb,
                                                   const double *__restrict__ ub, double *__restrict__ p) {
    const double tol = 10.0 * DBL_EPSILON;
    for (int64_t i = (int64_t)blockIdx.x * kBlock + threadIdx.x; i < n; i += (int64_t)gridDim.x * kBlock) {
        const double xi = x[i];
        p[i] = (fabs(xi - ub[i]) <= tol || fabs(xi - lb[i]) <= tol) ? 0.0 : u[i];
    }
}

// (a bound NULL: none on that side)
__global__ __launch_bounds__(kBlock) void k_project(int64_t n, const double *__restrict__ x,
                                                    const double *__restrict__ lb, const double *__restrict__ ub,
                                                    double *__restrict__ out) {
    for (int64_t i = (int64_t)blockIdx.x * kBlock + threadIdx.x; i < n; i += (int64_t)gridDim.x * kBlock)
        out[i] = clamp_box(x[i], lb ? lb[i] : -DBL_MAX, ub ? ub[i] : DBL_MAX);
}

// fi, beta, gp = fi + beta, and the three dots beta.beta, fi.fi, gp.gp (utopia_MPRGP.hpp:238-245)
__global__ __launch_bounds__(kBlock) void k_mprgp_state(int64_t n, const double *__restrict__ x,
                                                        const double *__restrict__ g, const double *__restrict__ lb,
                                                        const double *__restrict__ ub, double *__restrict__ fi,
                                                        double *__restrict__ beta, double *__restrict__ gp,
                                                        double *__restrict__ partials, int64_t stride) {
    double s0 = 0, s1 = 0, s2 = 0;
    for (int64_t i = (int64_t)blockIdx.x * kBlock + threadIdx.x; i < n; i += (int64_t)gridDim.x * kBlock) {
        const double xi = x[i], gi = g[i], li = lb ? lb[i] : -DBL_MAX, ui = ub ? ub[i] : DBL_MAX;
        const double f = free_grad(xi, gi, li, ui), b = chopped_grad(xi, gi, li, ui);
        const double q = f + b;
        if (fi) fi[i] = f;
        if (beta) beta[i] = b;
        if (gp) gp[i] = q;
        s0 += b * b;
        s1 += f * f;
        s2 += q * q;
    }
    s0 = block_sum<kBlock>(s0);
    s1 = block_sum<kBlock>(s1);
    s2 = block_sum<kBlock>(s2);
    if (threadIdx.x == 0) {
        partials[blockIdx.x] = s0;
        partials[stride + blockIdx.x] = s1;
        partials[2 * stride + blockIdx.x] = s2;
    }
}

__global__ __launch_bounds__(kBlock) void k_free_grad(int64_t n, const double *__restrict__ x,
                                                      const double *__restrict__ g, const double *__restrict__ lb,
                                                      const double *__restrict__ ub, double *__restrict__ fi) {
    for (int64_t i = (int64_t)blockIdx.x * kBlock + threadIdx.x; i < n; i += (int64_t)gridDim.x * kBlock)
        fi[i] = free_grad(x[i], g[i], lb[i], ub[i]);
}

// MPRGP::get_alpha_f (utopia_MPRGP.hpp:289-322): min over (x-l)/p for p > 0 and (x-u)/p for p < 0 (1e15 otherwise)
__global__ __launch_bounds__(kBlock) void k_alpha_f(int64_t n, const double *__restrict__ x,
                                                    const double *__restrict__ p, const double *__restrict__ lb,
                                                    const double *__restrict__ ub, double *__restrict__ partials) {
    double m = INFINITY;
    for (int64_t i = (int64_t)blockIdx.x * kBlock + threadIdx.x; i < n; i += (int64_t)gridDim.x * kBlock) {
        const double pi = p[i], xi = x[i];
        const double h1 = (pi > 0) ? ((xi - lb[i]) / pi) : 1e15;
        const double h2 = (pi < 0) ? ((xi - ub[i]) / pi) : 1e15;
        m = fmin(m, fmin(h1, h2));
    }
    __shared__ double red[kBlock];
    red[threadIdx.x] = m;
    __syncthreads();
    for (int s = kBlock / 2; s > 0; s >>= 1) {
        if (threadIdx.x < s) red[threadIdx.x] = fmin(red[threadIdx.x], red[threadIdx.x + s]);
        __syncthreads();
    }
    if (threadIdx.x == 0) partials[blockIdx.x] = red[0];
}

__global__ __launch_bounds__(kBlock) void k_min_finish(const double *__restrict__ partials, int64_t np,
                                                       double *__restrict__ out) {
    double m = INFINITY;
    for (int64_t b = threadIdx.x; b < np; b += kBlock) m = fmin(m, partials[b]);
    __shared__ double red[kBlock];
    red[threadIdx.x] = m;
    __syncthreads();
    for (int s = kBlock / 2; s > 0; s >>= 1) {
        if (threadIdx.x < s) red[threadIdx.x] = fmin(red[threadIdx.x], red[threadIdx.x + s]);
        __syncthreads();
    }
    if (threadIdx.x == 0) out[0] = red[0];
}

// CG step of MPRGP (utopia_MPRGP.hpp:167-182): x -= a p; g -= a Ap; fi = get_fi(x, g);
// partial fi.Ap. a = s[ia].
__global__ __launch_bounds__(kBlock) void k_mprgp_cg_step(int64_t n, double *__restrict__ x,
                                                          double *__restrict__ g, const double *__restrict__ p,
                                                          const double *__restrict__ Ap, const double *__restrict__ lb,
                                                          const double *__restrict__ ub, double *__restrict__ fi,
                                                          double a, double *__restrict__ partials) {
    double acc = 0.0;
    for (int64_t i = (int64_t)blockIdx.x * kBlock + threadIdx.x; i < n; i += (int64_t)gridDim.x * kBlock) {
        const double xi = x[i] - a * p[i];
        const double gi = g[i] - a * Ap[i];
        x[i] = xi;
        g[i] = gi;
        const double f = free_grad(xi, gi, lb[i], ub[i]);
        fi[i] = f;
        acc += f * Ap[i];
    }
    acc = block_sum<kBlock>(acc);
    if (threadIdx.x == 0) partials[blockIdx.x] = acc;
}

// CG step fused with the state that follows it (utopia_MPRGP.hpp:168-183 and the
// get_fi / chopped-gradient pass at the end of the iteration): x -= a p, g -= a Ap,
// then fi, beta, gp = fi + beta from the new x, g, and the dots beta.beta, fi.fi,
// gp.gp, fi.Ap. The grid and each thread's entries are those of k_mprgp_cg_step and
// k_mprgp_state, so the four sums are bit-identical to the two kernels'.
__global__ __launch_bounds__(kBlock) void k_mprgp_cg_step_state(int64_t n, double *__restrict__ x,
                                                                double *__restrict__ g, const double *__restrict__ p,
                                                                const double *__restrict__ Ap,
                                                                const double *__restrict__ lb,
                                                                const double *__restrict__ ub, double *__restrict__ fi,
                                                                double *__restrict__ beta, double *__restrict__ gp,
                                                                double a, double *__restrict__ partials,
                                                                int64_t stride) {
    double s0 = 0, s1 = 0, s2 = 0, s3 = 0;
    for (int64_t i = (int64_t)blockIdx.x * kBlock + threadIdx.x; i < n; i += (int64_t)gridDim.x * kBlock) {
        const double api = Ap[i];
        const double xi = x[i] - a * p[i];
        const double gi = g[i] - a * api;
        x[i] = xi;
        g[i] = gi;
        const double li = lb[i], ui = ub[i];
        const double f = free_grad(xi, gi, li, ui), b = chopped_grad(xi, gi, li, ui);
        const double q = f + b;
        fi[i] = f;
        beta[i] = b;
        gp[i] = q;
        s0 += b * b;
        s1 += f * f;
        s2 += q * q;
        s3 += f * api;
    }
    s0 = block_sum<kBlock>(s0);
    s1 = block_sum<kBlock>(s1);
    s2 = block_sum<kBlock>(s2);
    s3 = block_sum<kBlock>(s3);
    if (threadIdx.x == 0) {
        partials[blockIdx.x] = s0;
        partials[stride + blockIdx.x] = s1;
        partials[2 * stride + blockIdx.x] = s2;
        partials[3 * stride + blockIdx.x] = s3;
    }
}

// p = fi - (s[inum]/s[iden]) p
__global__ __launch_bounds__(kBlock) void k_mprgp_pupdate(int64_t n, double *__restrict__ p,
                                                          const double *__restrict__ fi, const double *__restrict__ s,
                                                          int inum, int iden) {
    const double beta_sc = s[inum] / s[iden];
    for (int64_t i = (int64_t)blockIdx.x * kBlock + threadIdx.x; i < n; i += (int64_t)gridDim.x * kBlock)
        p[i] = fi[i] - beta_sc * p[i];
}

// Expansion step (utopia_MPRGP.hpp:184-198): x -= af p; g -= af Ap; fi = get_fi(x, g);
// x = P(x - abar fi).
__global__ __launch_bounds__(kBlock) void k_mprgp_expand(int64_t n, double *__restrict__ x,
                                                         const double *__restrict__ g, const double *__restrict__ p,
                                                         const double *__restrict__ Ap, const double *__restrict__ lb,
                                                         const double *__restrict__ ub, double af, double abar) {
    for (int64_t i = (int64_t)blockIdx.x * kBlock + threadIdx.x; i < n; i += (int64_t)gridDim.x * kBlock) {
        const double li = lb[i], ui = ub[i];
        const double xi = x[i] - af * p[i];
        const double gi = g[i] - af * Ap[i];
        const double f = free_grad(xi, gi, li, ui);
        x[i] = clamp_box(xi - (abar * f), li, ui);
    }
}

// Proportioning step (utopia_MPRGP.hpp:223-235): x -= a beta; g -= a Abeta; p = get_fi(x, g)
__global__ __launch_bounds__(kBlock) void k_mprgp_prop(int64_t n, double *__restrict__ x, double *__restrict__ g,
                                                       const double *__restrict__ beta,
                                                       const double *__restrict__ Abeta,
                                                       const double *__restrict__ lb, const double *__restrict__ ub,
                                                       double *__restrict__ p, double a) {
    for (int64_t i = (int64_t)blockIdx.x * kBlock + threadIdx.x; i < n; i += (int64_t)gridDim.x * kBlock) {
        const double xi = x[i] - a * beta[i];
        const double gi = g[i] - a * Abeta[i];
        x[i] = xi;
        g[i] = gi;
        p[i] = free_grad(xi, gi, lb[i], ub[i]);
    }
}

// ---- MPRGP iterations that decide on the device (utopia_MPRGP.hpp:119-257) ----
// Iteration j: A p with p.Ap and g.p; k_mprgp_step chooses the step and takes it; an expansion step's
// g = A x - b (a launch that returns at once in the other steps); k_mprgp_direction forms the next
// direction. A proportioning step finds beta in p. The free and chopped gradients are functions of x, g
// and the bounds and are formed where they are used, never stored; each kernel adds its producer's partial
// sums itself; the host follows through pinned memory, some iterations behind.
// 1024 x 1024, 9-point, lower bounds: 79 -> 47 us an iteration (product 14.5, step 14.0, direction 9.3,
// gradient 14 in the fifth of the iterations that expand, else 5 for the empty launch). The vectors and the operator
// (150 MB) stay in the 256 MB MALL, which gives about 4.5 TB/s here, so the bytes are what is left; a bound
// that is absent is not read (51 -> 47 us).
constexpr int kMprgpGroups = 512;

__device__ __forceinline__ double block_min(double v) {
    __shared__ double red[kBlock / 64];
#pragma unroll
    for (int d = 32; d > 0; d >>= 1) v = fmin(v, __shfl_xor(v, d, 64));
    if ((threadIdx.x & 63) == 0) red[threadIdx.x >> 6] = v;
    __syncthreads();
    double m = red[0];
#pragma unroll
    for (int i = 1; i < kBlock / 64; ++i) m = fmin(m, red[i]);
    __syncthreads();
    return m;
}

// lb or ub NULL: no bound on that side (the value that fills a missing bound, not read from memory).
// sums: the state's partial sums (beta.beta, fi.fi, gp.gp, fi.Ap) of CG and proportioning steps
__global__ __launch_bounds__(kBlock) void k_mprgp_step(int64_t n, long long j, double *__restrict__ x,
                                                       double *__restrict__ g, const double *__restrict__ p,
                                                       const double *__restrict__ Ap, const double *__restrict__ lb,
                                                       const double *__restrict__ ub, double alpha_bar,
                                                       const double *__restrict__ dots, int dots_n, int64_t dots_st,
                                                       const double *__restrict__ mins, MprgpScalars *__restrict__ s,
                                                       double *__restrict__ sums, RunStatus *__restrict__ status) {
    constexpr int U = 4;
    const int64_t st = (int64_t)gridDim.x * kBlock, i0 = (int64_t)blockIdx.x * kBlock + threadIdx.x;
    double xv[U], gv[U], pv[U], av[U], lv[U], uv[U];
    auto load = [&](int64_t i) {
#pragma unroll
        for (int u = 0; u < U; ++u) {
            const int64_t k = i + u * st < n ? i + u * st : n - 1;
            xv[u] = x[k];
            gv[u] = g[k];
            pv[u] = p[k];
            av[u] = Ap[k];
            lv[u] = lb ? lb[k] : -DBL_MAX;
            uv[u] = ub ? ub[k] : DBL_MAX;
        }
    };
    load(i0);
    if (s->last < j) return;
    const bool prop = s->prop[j & 1] != 0;
    double pr[2], alpha_f = INFINITY;  // p.Ap, g.p
    add_partials<kBlock, 2>(dots, dots_st, dots_n, pr);
    for (int i = threadIdx.x; i < (int)gridDim.x; i += kBlock) alpha_f = fmin(alpha_f, mins[i]);
    block_totals<kBlock, 2>(pr);
    alpha_f = block_min(alpha_f);
    const double pap = pr[0], gp = pr[1];
    const bool first = blockIdx.x == 0 && threadIdx.x == 0;
    if (pap <= 0.0) {  // negative curvature
        if (first) {
            s->last = j - 1;
            status->done = 2;
            __threadfence_system();
        }
        return;
    }
    const double alpha = gp / pap;
    const int kind = prop ? 2 : (alpha <= alpha_f ? 0 : 1);
    if (first) {
        s->kind = kind;
        s->pap = pap;
    }
    double t[4] = {0, 0, 0, 0};
    for (int64_t i = i0; i < n; i += U * st) {
        if (i != i0) load(i);
#pragma unroll
        for (int u = 0; u < U; ++u) {
            if (i + u * st >= n) continue;
            if (kind == 1) {  // x = P(x - af p - abar fi(x - af p, g - af Ap))
                const double xi = xv[u] - alpha_f * pv[u];
                const double gi = gv[u] - alpha_f * av[u];
                x[i + u * st] = clamp_box(xi - (alpha_bar * free_grad(xi, gi, lv[u], uv[u])), lv[u], uv[u]);
            } else {
                const double xi = xv[u] - alpha * pv[u];
                const double gi = gv[u] - alpha * av[u];
                x[i + u * st] = xi;
                g[i + u * st] = gi;
                const double f = free_grad(xi, gi, lv[u], uv[u]), b = chopped_grad(xi, gi, lv[u], uv[u]), q = f + b;
                t[0] += b * b;
                t[1] += f * f;
                t[2] += q * q;
                t[3] += f * av[u];
            }
        }
    }
    if (kind == 1) return;
    block_totals<kBlock, 4>(t);
    if (threadIdx.x < 4) sums[threadIdx.x * gridDim.x + blockIdx.x] = t[threadIdx.x];
}

// p = fi - (fi.Ap / p.Ap) p after a CG step, fi after the others; beta where the next step is a
// proportioning one (beta.beta > fi.fi). Partial minima of get_alpha_f for the new p. Block 0 reports the
// projected gradient's norm and ends the loop. j < 0: the loop's start (the state of the first iterate).
__global__ __launch_bounds__(kBlock) void k_mprgp_direction(int64_t n, long long j, const double *__restrict__ x,
                                                            const double *__restrict__ g, double *__restrict__ p,
                                                            const double *__restrict__ lb,
                                                            const double *__restrict__ ub,
                                                            const double *__restrict__ sums,
                                                            const double *__restrict__ grad_sums, int grad_n,
                                                            int64_t grad_st, double atol, double rtol,
                                                            MprgpScalars *__restrict__ s, double *__restrict__ mins,
                                                            RunStatus *__restrict__ status) {
    constexpr int U = 4;
    const int64_t st = (int64_t)gridDim.x * kBlock, i0 = (int64_t)blockIdx.x * kBlock + threadIdx.x;
    double xv[U], gv[U], pv[U], lv[U], uv[U];
    auto load = [&](int64_t i) {
#pragma unroll
        for (int u = 0; u < U; ++u) {
            const int64_t k = i + u * st < n ? i + u * st : n - 1;
            xv[u] = x[k];
            gv[u] = g[k];
            pv[u] = p[k];
            lv[u] = lb ? lb[k] : -DBL_MAX;
            uv[u] = ub ? ub[k] : DBL_MAX;
        }
    };
    load(i0);
    if (s->last < j) return;
    const int kind = j < 0 ? 2 : s->kind;
    const double *q = kind == 1 ? grad_sums : sums;
    const int qn = kind == 1 ? grad_n : (int)gridDim.x;
    const int64_t qst = kind == 1 ? grad_st : (int64_t)gridDim.x;
    double t[4];  // beta.beta, fi.fi, gp.gp, and (CG steps) fi.Ap
    if (kind == 0) {
        sum_partials<kBlock, 4>(q, qst, qn, t);
    } else {
        double t3[3];
        sum_partials<kBlock, 3>(q, qst, qn, t3);
        t[0] = t3[0], t[1] = t3[1], t[2] = t3[2], t[3] = 0.0;
    }
    const bool prop = !(t[0] <= t[1]);
    const double scale = kind == 0 ? t[3] / s->pap : 0.0;
    if (blockIdx.x == 0 && threadIdx.x == 0) {
        s->prop[(j + 1) & 1] = prop ? 1 : 0;
        if (j >= 0) {
            const double norm = sqrt(t[2]);
            if (j == 0) s->gnorm0 = norm;
            const double norm0 = j == 0 ? norm : s->gnorm0;
            status->value[0] = norm;
            status->value[1] = norm0;
            if (norm <= atol || norm / norm0 <= rtol) {
                s->last = j;
                status->done = 1;
            }
            __hip_atomic_store(&status->steps, j + 1, __ATOMIC_RELEASE, __HIP_MEMORY_SCOPE_SYSTEM);
        }
    }
    double m = INFINITY;
    for (int64_t i = i0; i < n; i += U * st) {
        if (i != i0) load(i);
#pragma unroll
        for (int u = 0; u < U; ++u) {
            if (i + u * st >= n) continue;
            const double f = free_grad(xv[u], gv[u], lv[u], uv[u]);
            double d = kind == 0 ? f - scale * pv[u] : f;
            if (prop) d = chopped_grad(xv[u], gv[u], lv[u], uv[u]);
            p[i + u * st] = d;
            const double h1 = (d > 0) ? ((xv[u] - lv[u]) / d) : 1e15;
            const double h2 = (d < 0) ? ((xv[u] - uv[u]) / d) : 1e15;
            m = fmin(m, fmin(h1, h2));
        }
    }
    m = block_min(m);
    if (threadIdx.x == 0) mins[blockIdx.x] = m;
}

__global__ void k_mprgp_begin(MprgpScalars *__restrict__ s) {
    *s = MprgpScalars{0.0, 0.0, 0x7fffffffffffffffll, 2, {0, 0}};
}

// the loop's device memory: scalars, partial sums of the products, of the state, minima
struct MprgpWork {
    MprgpScalars *s;
    double *dots, *grad, *sums, *mins, *total;
    int64_t parts;
    int groups;
    size_t bytes;
};
static MprgpWork mprgp_work(const uhip_csr *A, void *base) {
    MprgpWork w;
    w.parts = std::max<int64_t>(spmv_parts(A), 1);
    w.groups = grid_for(A->nrows, 1, kMprgpGroups);
    char *q = (char *)base;
    w.s = (MprgpScalars *)q;
    double *d = (double *)(q + 256);
    w.dots = d;
    w.grad = w.dots + 2 * w.parts;
    w.sums = w.grad + 3 * w.parts;
    w.mins = w.sums + 4 * (int64_t)w.groups;
    w.total = w.mins + w.groups;  // finished sums: 2 of the product, 3 of the gradient
    w.bytes = 256 + sizeof(double) * (size_t)(5 * w.parts + 5 * (int64_t)w.groups + 8);
    return w;
}

// ActiveSet::determine (solvers/nonlinear/constrained/utopia_ActiveSet.hpp:41-79):
// ind_i = (x_i <= l_i + tol or x_i >= u_i - tol); partial count of changed entries.
__global__ __launch_bounds__(kBlock) void k_active_set(int64_t n, const double *__restrict__ x,
                                                       const double *__restrict__ lb, const double *__restrict__ ub,
                                                       double tol, double *__restrict__ ind,
                                                       double *__restrict__ partials) {
    double changed = 0.0;
    for (int64_t i = (int64_t)blockIdx.x * kBlock + threadIdx.x; i < n; i += (int64_t)gridDim.x * kBlock) {
        const double xi = x[i];
        const double v = (xi <= lb[i] + tol || xi >= ub[i] - tol) ? 1.0 : 0.0;
        changed += (v != ind[i]) ? 1.0 : 0.0;
        ind[i] = v;
    }
    changed = block_sum<kBlock>(changed);
    if (threadIdx.x == 0) partials[blockIdx.x] = changed;
}

// IPTruncatedTransfer::truncate_interpolation (transfer/utopia_IPTruncatedTransfer.hpp:203-223):
// the values of rows i with ind_i == 1 become zero (pattern kept).
__global__ __launch_bounds__(kBlock) void k_zero_rows(int32_t n, const int32_t *__restrict__ rowptr,
                                                      const double *__restrict__ ind, double *__restrict__ val) {
    const int32_t r = blockIdx.x * kBlock + threadIdx.x;
    if (r >= n || ind[r] != 1.0) return;
    for (int32_t e = rowptr[r]; e < rowptr[r + 1]; ++e) val[e] = 0.0;
}

// ---- multicolour projected Gauss-Seidel ----

__device__ __forceinline__ uint64_t mix64(uint64_t z) {
    z += 0x9E3779B97F4A7C15ull;
    z = (z ^ (z >> 30)) * 0xBF58476D1CE4E5B9ull;
    z = (z ^ (z >> 27)) * 0x94D049BB133111EBull;
    return z ^ (z >> 31);
}

// Jones-Plassmann round: an uncoloured row whose (hash, index) beats every
// uncoloured neighbour takes the smallest colour none of its coloured
// neighbours has. Rows chosen in one round are never adjacent, so they cannot
// conflict. Needs a structurally symmetric pattern.
__global__ __launch_bounds__(kBlock) void k_jp_round(int32_t n, const int32_t *__restrict__ rowptr,
                                                     const int32_t *__restrict__ col, int32_t *__restrict__ color,
                                                     uint64_t seed, unsigned int *__restrict__ remaining) {
    const int32_t i = blockIdx.x * kBlock + threadIdx.x;
    if (i >= n || color[i] >= 0) return;
    const uint64_t hi = mix64((uint64_t)i ^ seed);
    bool best = true;
    for (int32_t e = rowptr[i]; e < rowptr[i + 1]; ++e) {
        const int32_t j = col[e];
        if (j == i) continue;
        if (color[j] >= 0) continue;  // coloured in an earlier round
        const uint64_t hj = mix64((uint64_t)j ^ seed);
        if (hj > hi || (hj == hi && j > i)) {
            best = false;
            break;
        }
    }
    if (!best) {
        *remaining = 1u;  // every such row writes the same value: 30 -> 8 us a round against a counter
        return;
    }
    // smallest colour not used by a coloured neighbour (neighbours chosen in
    // this round are marked pending, <= -2, and are never adjacent to i)
    int32_t c = 0;
    for (;;) {
        bool used = false;
        for (int32_t e = rowptr[i]; e < rowptr[i + 1] && !used; ++e) used = (col[e] != i) && (color[col[e]] == c);
        if (!used) break;
        ++c;
    }
    color[i] = -2 - c;  // pending until k_jp_commit, after every row of the round has decided
}

__global__ __launch_bounds__(kBlock) void k_jp_commit(int32_t n, int32_t *__restrict__ color) {
    const int32_t i = blockIdx.x * kBlock + threadIdx.x;
    if (i < n && color[i] <= -2) color[i] = -2 - color[i];
}

// One colour of the projected sweep (ProjectedScalarGaussSeidelSweep::apply,
// utopia_ProjectedGaussSeidelSweep.hpp:191-235), bounds relative to x:
// lbl = lb - x, ubl = ub - x (ProjectedGaussSeidel::step, utopia_petsc_ProjectedGaussSeidel.cpp:384-385).
__global__ __launch_bounds__(kBlock) void k_pgs_color(int32_t cnt, const int32_t *__restrict__ rows,
                                                      const int32_t *__restrict__ rowptr,
                                                      const int32_t *__restrict__ col, const double *__restrict__ val,
                                                      const double *__restrict__ dinv, const double *__restrict__ r,
                                                      const double *__restrict__ x, const double *__restrict__ lb,
                                                      const double *__restrict__ ub, double *__restrict__ c,
                                                      int constrained) {
    const int32_t t = blockIdx.x * kBlock + threadIdx.x;
    if (t >= cnt) return;
    const int32_t i = rows[t];
    double v = r[i];
    const double d = dinv[i];
    if (constrained) {
        const double lbl = lb[i] - x[i], ubl = ub[i] - x[i];
        if (d <= 0.0) {
            c[i] = (v == 0.0) ? 0.0 : ((v > 0.0) ? lbl : ubl);
            return;
        }
        for (int32_t e = rowptr[i]; e < rowptr[i + 1]; ++e) {
            const int32_t j = col[e];
            const double a = val[e];
            if (j != i && a != 0.0) v -= a * c[j];
        }
        c[i] = fmax(lbl, fmin(d * v, ubl));
    } else {
        for (int32_t e = rowptr[i]; e < rowptr[i + 1]; ++e) {
            const int32_t j = col[e];
            const double a = val[e];
            if (j != i && a != 0.0) v -= a * c[j];
        }
        c[i] = d * v;
    }
}

// The same colour from the colours' own layout (ColorPlan): slices of 64 rows of one colour, entries
// column-major within a slice, so a wavefront's matrix loads are contiguous and need no row pointer;
// they go out before anything is gathered. A launch is one chain of three loads (slice offset, columns,
// c) against k_pgs_color's five, and one wavefront a workgroup spreads the few thousand rows of a colour
// over all CUs. FINAL (the row's last visit in the sweep): x_i += c_i as well.
// Padding entries point at the row itself. 500 x 300, 9-point, 8 colours: 8.9 -> 4.45 us a colour, a symmetric
// projected sweep 163 -> 87 us (15 of its 16 colour launches, no separate clearing, update and copy of x).
template <bool CONSTRAINED, bool FINAL>
__global__ __launch_bounds__(64) void k_color_slices(int32_t s0, const int32_t *__restrict__ slice_off,
                                                     const int32_t *__restrict__ slot_row,
                                                     const int32_t *__restrict__ col, const double *__restrict__ val,
                                                     const double *__restrict__ dinv, const double *__restrict__ r,
                                                     double *__restrict__ x, const double *__restrict__ lb,
                                                     const double *__restrict__ ub, double *c) {
    constexpr int U = 16;
    const int32_t s = s0 + (int32_t)blockIdx.x, lane = threadIdx.x;
    const int32_t row = slot_row[64 * (int64_t)s + lane];
    const int32_t o = slice_off[s], w = (slice_off[s + 1] - o) >> 6;
    const int32_t i = max(row, 0);
    double v = r[i];
    const double d = dinv[i], xi = (CONSTRAINED || FINAL) ? x[i] : 0.0;
    const double l = CONSTRAINED ? (lb ? lb[i] : -DBL_MAX) : 0.0, u = CONSTRAINED ? (ub ? ub[i] : DBL_MAX) : 0.0;
    const double r0 = v;
    for (int32_t j0 = 0; j0 < w; j0 += U) {
        int32_t cj[U];
        double a[U], cv[U];
#pragma unroll
        for (int k = 0; k < U; ++k)
            if (j0 + k < w) {
                cj[k] = col[o + 64 * (j0 + k) + lane];
                a[k] = val[o + 64 * (j0 + k) + lane];
            }
#pragma unroll
        for (int k = 0; k < U; ++k)
            if (j0 + k < w) cv[k] = c[cj[k]];
#pragma unroll
        for (int k = 0; k < U; ++k)
            if (j0 + k < w && cj[k] != i && a[k] != 0.0) v -= a[k] * cv[k];
    }
    if (row < 0) return;
    double t = d * v;
    if (CONSTRAINED) {
        const double lbl = l - xi, ubl = u - xi;
        t = fmax(lbl, fmin(t, ubl));
        if (d <= 0.0) t = (r0 == 0.0) ? 0.0 : ((r0 > 0.0) ? lbl : ubl);
    }
    c[i] = t;
    if (FINAL) x[i] = xi + 1.0 * t;
}

// rows: the matrix's rows grouped by colour; first_slot / first_row: per colour, its first slot (a multiple
// of 64) and its first place in rows.
__global__ __launch_bounds__(64) void k_color_slots(int32_t nslices, int32_t ncolors,
                                                    const int32_t *__restrict__ first_slot,
                                                    const int32_t *__restrict__ first_row,
                                                    const int32_t *__restrict__ rows, const int32_t *__restrict__ rowptr,
                                                    int32_t *__restrict__ slot_row, int64_t *__restrict__ width) {
    const int32_t s = blockIdx.x, lane = threadIdx.x;
    if (s == nslices) {
        if (lane == 0) width[s] = 0;
        return;
    }
    int32_t k = 0;
    while (k + 1 < ncolors && first_slot[k + 1] <= 64 * s) ++k;
    const int32_t at = first_row[k] + 64 * s - first_slot[k] + lane;
    const int32_t row = at < first_row[k + 1] ? rows[at] : -1;
    slot_row[64 * (int64_t)s + lane] = row;
    int32_t w = row >= 0 ? rowptr[row + 1] - rowptr[row] : 0;
#pragma unroll
    for (int d = 32; d > 0; d >>= 1) w = max(w, __shfl_xor(w, d, 64));
    if (lane == 0) width[s] = 64 * (int64_t)w;
}

// the slices' offsets, known to fit
__global__ __launch_bounds__(kBlock) void k_color_offsets(int32_t n, const int64_t *__restrict__ wide,
                                                          int32_t *__restrict__ off) {
    const int32_t i = blockIdx.x * kBlock + threadIdx.x;
    if (i < n) off[i] = (int32_t)wide[i];
}

__global__ __launch_bounds__(64) void k_color_fill(const int32_t *__restrict__ slice_off,
                                                   const int32_t *__restrict__ slot_row,
                                                   const int32_t *__restrict__ rowptr, const int32_t *__restrict__ col,
                                                   const double *__restrict__ val, int32_t *__restrict__ scol,
                                                   double *__restrict__ sval) {
    const int32_t s = blockIdx.x, lane = threadIdx.x;
    const int32_t row = slot_row[64 * (int64_t)s + lane], o = slice_off[s], w = (slice_off[s + 1] - o) >> 6;
    const int32_t e0 = row >= 0 ? rowptr[row] : 0, len = row >= 0 ? rowptr[row + 1] - e0 : 0;
    for (int32_t j = 0; j < w; ++j) {
        scol[o + 64 * j + lane] = j < len ? col[e0 + j] : max(row, 0);
        sval[o + 64 * j + lane] = j < len ? val[e0 + j] : 0.0;
    }
}

__global__ __launch_bounds__(kBlock) void k_max_color(int32_t n, const int32_t *__restrict__ color,
                                                      int32_t *__restrict__ mx) {
    int32_t v = 0;
    for (int64_t i = blockIdx.x * kBlock + threadIdx.x; i < n; i += gridDim.x * kBlock) v = max(v, color[i]);
#pragma unroll
    for (int d = 32; d > 0; d >>= 1) v = max(v, __shfl_xor(v, d, 64));
    if ((threadIdx.x & 63) == 0) atomicMax(mx, v);
}

__global__ __launch_bounds__(kBlock) void k_iota(int32_t n, int32_t *__restrict__ x) {
    const int32_t i = blockIdx.x * kBlock + threadIdx.x;
    if (i < n) x[i] = i;
}

// off[k] = the first place of a key >= k in the sorted keys, off[ncolors] = n
__global__ __launch_bounds__(kBlock) void k_group_offsets(int32_t n, int32_t ncolors, const int32_t *__restrict__ keys,
                                                          int32_t *__restrict__ off) {
    const int32_t i = blockIdx.x * kBlock + threadIdx.x;
    if (i >= n) return;
    const int32_t k0 = i > 0 ? keys[i - 1] : -1, k1 = keys[i];
    for (int32_t k = k0 + 1; k <= k1; ++k) off[k] = i;
    if (i == n - 1)
        for (int32_t k = k1 + 1; k <= ncolors; ++k) off[k] = n;
}

// d_inv_i = 1/a_ii where |a_ii| > 0, else 0 (init_from_local_matrix, :95-104)
__global__ __launch_bounds__(kBlock) void k_pgs_dinv(int32_t n, const int32_t *__restrict__ rowptr,
                                                     const int32_t *__restrict__ col, const double *__restrict__ val,
                                                     double *__restrict__ dinv) {
    const int32_t i = blockIdx.x * kBlock + threadIdx.x;
    if (i >= n) return;
    double d = 0.0;
    for (int32_t e = rowptr[i]; e < rowptr[i + 1]; ++e)
        if (col[e] == i) d = (fabs(val[e]) > 0.0) ? (1 / val[e]) : 0.0;
    dinv[i] = d;
}

}  // namespace uhip

using namespace uhip;

// Slots that a colour plan may have for its entries: a slice is as wide as its longest row. The copy is faster than the
// rows themselves at any padding (a projected symmetric sweep, 150,000 rows of 9 on average, from the copy / colour by
// colour: padding 1.8 102 / 223 us, 2.4 142 / 344, 3.8 419 / 1065, 6.7 5883 / 12993; one row of 2000 among rows of 9
// 499 / 1155), so the line is what it may take of memory: four times the entries (12 bytes a slot against a matrix'
// own 12 bytes an entry), and 12 MB for matrices so small that their colours leave most slices unfilled.
constexpr int64_t kColorPadding = 4, kColorSmall = 1 << 20;

struct uhip_color_plan_s {
    int32_t n = 0, ncolors = 0;
    int64_t nnz = 0;
    std::vector<int32_t> first_slice;  // ncolors + 1
    int32_t *slice_off = nullptr, *slot_row = nullptr, *col = nullptr;
    double *val = nullptr;
};

extern "C" {

int uhip_color_plan_destroy(uhip_ctx ctx, uhip_color_plan plan) {
    if (!plan) return UHIP_OK;
    if (ctx) UHIP_CHECK_HIP(hipStreamSynchronize(ctx->stream));
    for (void *q : {(void *)plan->slot_row, (void *)plan->val})  // the other arrays lie in these
        if (q) (void)hipFree(q);
    delete plan;
    return UHIP_OK;
}

int uhip_color_plan_create(uhip_ctx ctx, const uhip_csr *A, int32_t ncolors, const int32_t *rows,
                           const int32_t *offsets_h, uhip_color_plan *out) {
    UHIP_REQUIRE(ctx && A && rows && offsets_h && out && ncolors >= 0, "uhip_color_plan_create: bad argument");
    UHIP_REQUIRE(A->dtype == UHIP_F64 && A->nrows == A->ncols, "uhip_color_plan_create: square FP64 matrix");
    UHIP_REQUIRE(ncolors == 0 || offsets_h[ncolors] == A->nrows, "uhip_color_plan_create: the groups hold %d of %d rows",
                 ncolors ? offsets_h[ncolors] : 0, A->nrows);
    *out = nullptr;
    hipStream_t st = ctx->stream;
    auto *p = new uhip_color_plan_s();
    struct Guard {
        uhip_ctx ctx;
        uhip_color_plan_s *p;
        ~Guard() { (void)uhip_color_plan_destroy(ctx, p); }
    } guard{ctx, p};
    p->n = A->nrows;
    p->nnz = A->nnz;
    p->ncolors = ncolors;
    p->first_slice.assign((size_t)ncolors + 1, 0);
    std::vector<int32_t> host((size_t)2 * ncolors + 2, 0);  // first_slot, first_row
    for (int32_t k = 0; k < ncolors; ++k) {
        p->first_slice[(size_t)k + 1] = p->first_slice[(size_t)k] + (offsets_h[k + 1] - offsets_h[k] + 63) / 64;
        host[(size_t)k + 1] = 64 * p->first_slice[(size_t)k + 1];
    }
    const int32_t ns = p->first_slice[(size_t)ncolors];
    if (ns > 0) {
        for (int32_t k = 0; k <= ncolors; ++k) host[(size_t)ncolors + 1 + k] = offsets_h[k];
        size_t tb = 0;
        // slice offsets and rows in one allocation, values and columns in another
        UHIP_CHECK_HIP(hipMalloc(&p->slot_row, sizeof(int32_t) * (65 * (size_t)ns + 1)));
        p->slice_off = p->slot_row + 64 * (size_t)ns;
        UHIP_CHECK_HIP(hipcub::DeviceScan::ExclusiveSum(nullptr, tb, (int64_t *)nullptr, (int64_t *)nullptr, ns + 1, st));
        Scratch w(ctx);
        const size_t o_h = w.add(sizeof(int32_t) * host.size()), o_w = w.add(sizeof(int64_t) * ((size_t)ns + 1)),
                     o_o = w.add(sizeof(int64_t) * ((size_t)ns + 1)), o_t = w.add(tb);
        UHIP_TRY(w.allocate());
        UHIP_CHECK_HIP(hipMemcpyAsync(w.at<void>(o_h), host.data(), sizeof(int32_t) * host.size(), hipMemcpyHostToDevice, st));
        hipLaunchKernelGGL(k_color_slots, dim3(ns + 1), dim3(64), 0, st, ns, ncolors, w.at<int32_t>(o_h),
                           w.at<int32_t>(o_h) + ncolors + 1, rows, A->rowptr, p->slot_row, w.at<int64_t>(o_w));
        UHIP_CHECK_LAUNCH();
        UHIP_CHECK_HIP(hipcub::DeviceScan::ExclusiveSum(w.at<void>(o_t), tb, w.at<int64_t>(o_w), w.at<int64_t>(o_o),
                                                        ns + 1, st));
        int64_t total = 0;
        UHIP_TRY(read_ints(ctx, (const int32_t *)(w.at<int64_t>(o_o) + ns), 2, (int32_t *)&total));
        if (total > kColorPadding * A->nnz + kColorSmall || total > INT32_MAX)
            return set_error(UHIP_ERR_UNSUPPORTED, "uhip_color_plan_create: %lld slots for %lld entries", (long long)total,
                             (long long)A->nnz);
        hipLaunchKernelGGL(k_color_offsets, dim3(ns / kBlock + 1), dim3(kBlock), 0, st, ns + 1, w.at<int64_t>(o_o),
                           p->slice_off);
        UHIP_CHECK_LAUNCH();
        UHIP_CHECK_HIP(hipMalloc(&p->val, (sizeof(double) + sizeof(int32_t)) * (size_t)std::max<int64_t>(total, 1)));
        p->col = (int32_t *)(p->val + total);
        hipLaunchKernelGGL(k_color_fill, dim3(ns), dim3(64), 0, st, p->slice_off, p->slot_row, A->rowptr, A->col,
                           (const double *)A->val, p->col, p->val);
        UHIP_CHECK_LAUNCH();
        UHIP_CHECK_HIP(hipStreamSynchronize(st));
    }
    guard.p = nullptr;
    *out = p;
    return UHIP_OK;
}

int uhip_color_plan_refresh(uhip_ctx ctx, uhip_color_plan plan, const uhip_csr *A) {
    UHIP_REQUIRE(ctx && plan && A && A->dtype == UHIP_F64, "uhip_color_plan_refresh: bad argument");
    UHIP_REQUIRE(A->nrows == plan->n && A->ncols == plan->n && A->nnz == plan->nnz,
                 "uhip_color_plan_refresh: not the plan's pattern");
    const int32_t ns = plan->first_slice.back();
    if (ns == 0) return UHIP_OK;
    hipLaunchKernelGGL(k_color_fill, dim3(ns), dim3(64), 0, ctx->stream, plan->slice_off, plan->slot_row, A->rowptr, A->col,
                       (const double *)A->val, plan->col, plan->val);
    UHIP_CHECK_LAUNCH();
    return UHIP_OK;
}

int uhip_color_plan_sweep(uhip_ctx ctx, uhip_color_plan plan, const double *dinv, const double *r, double *x,
                          const double *lb, const double *ub, double *c, int constrained, int symmetric, int add) {
    UHIP_REQUIRE(ctx && plan && dinv && r && c, "uhip_color_plan_sweep: null argument");
    UHIP_REQUIRE(x || !(constrained || add), "uhip_color_plan_sweep: x needed");
    const int32_t nc = plan->ncolors;
    // forward over the colours, then backward. The backward pass would begin with the colour that the
    // forward pass ended with: none of its rows' neighbours has changed in between, so its second visit
    // would compute the same values and is left out.
    for (int pass = 0; pass < (symmetric ? 2 : 1); ++pass)
        for (int32_t t = pass; t < nc; ++t) {
            const int32_t k = pass == 0 ? t : nc - 1 - t;
            const int32_t s0 = plan->first_slice[(size_t)k], ns = plan->first_slice[(size_t)k + 1] - s0;
            if (ns == 0) continue;
            const bool final_visit = add && (!symmetric || pass == 1 || t == nc - 1);
#define UHIP_COLOR(CON, FIN)                                                                                        \
    hipLaunchKernelGGL((k_color_slices<CON, FIN>), dim3(ns), dim3(64), 0, ctx->stream, s0, plan->slice_off,         \
                       plan->slot_row, plan->col, plan->val, dinv, r, x, lb, ub, c)
            if (constrained && final_visit) UHIP_COLOR(true, true);
            else if (constrained) UHIP_COLOR(true, false);
            else if (final_visit) UHIP_COLOR(false, true);
            else UHIP_COLOR(false, false);
#undef UHIP_COLOR
            UHIP_CHECK_LAUNCH();
        }
    return UHIP_OK;
}

int uhip_active_set_f64(uhip_ctx ctx, int64_t n, const double *x, const double *lb, const double *ub, double tol,
                        double *indicator, double *changed_d) {
    UHIP_REQUIRE(ctx && x && lb && ub && indicator && changed_d, "uhip_active_set_f64: null argument");
    const int g = grid_for(n, 4, kMaxRedBlocks);
    UHIP_TRY(ensure_partials(ctx, g));
    hipLaunchKernelGGL(k_active_set, dim3(g), dim3(kBlock), 0, ctx->stream, n, x, lb, ub, tol, indicator,
                       ctx->partials);
    UHIP_CHECK_LAUNCH();
    return finish_sums(ctx, 1, g, ctx->max_partials, changed_d, 0u);
}

int uhip_csr_zero_rows(uhip_ctx ctx, uhip_csr *A, const double *indicator) {
    UHIP_REQUIRE(ctx && A && indicator && A->dtype == UHIP_F64, "uhip_csr_zero_rows: bad argument");
    if (A->nrows == 0) return UHIP_OK;
    hipLaunchKernelGGL(k_zero_rows, dim3((A->nrows + kBlock - 1) / kBlock), dim3(kBlock), 0, ctx->stream, A->nrows,
                       A->rowptr, indicator, (double *)A->val);
    UHIP_CHECK_LAUNCH();
    return UHIP_OK;
}

int uhip_pcg_wz_f64(uhip_ctx ctx, int64_t n, const double *u, const double *lb, const double *ub, const double *p,
                    double *z, double *w) {
    UHIP_REQUIRE(ctx && u && lb && ub && p && z && w, "uhip_pcg_wz_f64: null argument");
    if (n <= 0) return UHIP_OK;
    hipLaunchKernelGGL(k_pcg_wz, dim3(grid_for(n, 4, 1 << 16)), dim3(kBlock), 0, ctx->stream, n, u, lb, ub, p, z, w);
    UHIP_CHECK_LAUNCH();
    return UHIP_OK;
}

int uhip_pg_direction_f64(uhip_ctx ctx, int64_t n, const double *x, const double *u, const double *lb,
                          const double *ub, double *p) {
    UHIP_REQUIRE(ctx && x && u && lb && ub && p, "uhip_pg_direction_f64: null argument");
    if (n <= 0) return UHIP_OK;
    hipLaunchKernelGGL(k_pg_dir, dim3(grid_for(n, 4, 1 << 16)), dim3(kBlock), 0, ctx->stream, n, x, u, lb, ub, p);
    UHIP_CHECK_LAUNCH();
    return UHIP_OK;
}

int uhip_box_project_f64(uhip_ctx ctx, int64_t n, const double *x, const double *lb, const double *ub, double *out) {
    UHIP_REQUIRE(ctx && x && lb && ub && out, "uhip_box_project_f64: null argument");
    if (n <= 0) return UHIP_OK;
    hipLaunchKernelGGL(k_project, dim3(grid_for(n, 4, 1 << 16)), dim3(kBlock), 0, ctx->stream, n, x, lb, ub, out);
    UHIP_CHECK_LAUNCH();
    return UHIP_OK;
}

int uhip_mprgp_state_f64(uhip_ctx ctx, int64_t n, const double *x, const double *g, const double *lb, const double *ub,
                         double *fi, double *beta, double *gp, double *dots_d) {
    UHIP_REQUIRE(ctx && x && g && lb && ub && dots_d, "uhip_mprgp_state_f64: null argument");
    const int gr = grid_for(n, 4, kMaxRedBlocks);
    UHIP_TRY(ensure_partials(ctx, gr));
    hipLaunchKernelGGL(k_mprgp_state, dim3(gr), dim3(kBlock), 0, ctx->stream, n, x, g, lb, ub, fi, beta, gp,
                       ctx->partials, ctx->max_partials);
    UHIP_CHECK_LAUNCH();
    return finish_sums(ctx, 3, gr, ctx->max_partials, dots_d, 0u);
}

int uhip_mprgp_free_grad_f64(uhip_ctx ctx, int64_t n, const double *x, const double *g, const double *lb,
                             const double *ub, double *fi) {
    UHIP_REQUIRE(ctx && x && g && lb && ub && fi, "uhip_mprgp_free_grad_f64: null argument");
    if (n <= 0) return UHIP_OK;
    hipLaunchKernelGGL(k_free_grad, dim3(grid_for(n, 4, 1 << 16)), dim3(kBlock), 0, ctx->stream, n, x, g, lb, ub, fi);
    UHIP_CHECK_LAUNCH();
    return UHIP_OK;
}

int64_t uhip_mprgp_work_bytes(const uhip_csr *A) { return A ? (int64_t)mprgp_work(A, nullptr).bytes : 0; }

int uhip_mprgp_begin_f64(uhip_ctx ctx, const uhip_csr *A, const double *b, const double *lb, const double *ub,
                         double *x, double *g, double *p, void *work) {
    UHIP_REQUIRE(ctx && A && b && x && g && p && work, "uhip_mprgp_begin_f64: null argument");
    UHIP_REQUIRE(A->nrows == A->ncols && A->dtype == UHIP_F64, "uhip_mprgp_begin_f64: square FP64 matrix");
    const int64_t n = A->nrows;
    if (n == 0) return UHIP_OK;
    const MprgpWork w = mprgp_work(A, work);
    hipStream_t st = ctx->stream;
    const dim3 blk(kBlock);
    hipLaunchKernelGGL(k_mprgp_begin, dim3(1), dim3(1), 0, st, w.s);
    UHIP_CHECK_LAUNCH();
    hipLaunchKernelGGL(k_project, dim3(grid_for(n, 4, 1 << 16)), blk, 0, st, n, x, lb, ub, x);
    UHIP_CHECK_LAUNCH();
    UHIP_TRY(uhip_spmv_axpbz(ctx, A, 1.0, x, -1.0, b, g));
    hipLaunchKernelGGL(k_mprgp_state, dim3(w.groups), dim3(kBlock), 0, st, n, x, g, lb, ub, nullptr, nullptr, nullptr,
                       w.sums, (int64_t)w.groups);
    UHIP_CHECK_LAUNCH();
    hipLaunchKernelGGL(k_mprgp_direction, dim3(w.groups), dim3(kBlock), 0, st, n, -1ll, x, g, p, lb, ub, w.sums, w.grad, 1,
                       w.parts, 0.0, 0.0, w.s, w.mins, run_record(ctx));
    UHIP_CHECK_LAUNCH();
    return UHIP_OK;
}

int uhip_mprgp_run_f64(uhip_ctx ctx, const uhip_csr *A, const double *b, const double *lb, const double *ub, double *x,
                       double *g, double *p, double *Ap, void *work, double alpha_bar, double atol, double rtol,
                       int64_t first, int64_t max_steps, int64_t *steps, double *norm, double *norm0, int *reason) {
    UHIP_REQUIRE(ctx && A && b && x && g && p && Ap && work && steps && norm && norm0 && reason,
                 "uhip_mprgp_run_f64: null argument");
    UHIP_REQUIRE(A->nrows == A->ncols && A->dtype == UHIP_F64 && first >= 0, "uhip_mprgp_run_f64: square FP64 matrix");
    const int64_t n = A->nrows;
    *steps = 0;
    *reason = n == 0 ? 2 : 0;  // nothing to iterate on: p.Ap = 0
    if (n == 0 || max_steps <= 0) return UHIP_OK;
    const MprgpWork w = mprgp_work(A, work);
    hipStream_t st = ctx->stream;
    RunScope scope(ctx);
    UHIP_TRY(scope.status());
    RunStatus *status = run_record(ctx);
    UHIP_CHECK_HIP(hipStreamSynchronize(st));  // no kernel of an earlier loop still reports
    memset(status, 0, sizeof(*status));
    status->steps = first;
    constexpr int64_t kAhead = 4;  // iterations that the host is ahead; those past the end return at once
    volatile RunStatus *seen = status;
    const bool many = w.parts > kConsumerSums;
    const dim3 grid(w.groups), blk(kBlock);
    for (int64_t j = first; j < first + max_steps && !seen->done; ++j) {
        UHIP_TRY(mprgp_product(ctx, A, p, Ap, g, w.dots, w.parts));
        if (many) UHIP_TRY(finish_sums_from(ctx, w.dots, 2, w.parts, w.parts, w.total));
        hipLaunchKernelGGL(k_mprgp_step, grid, blk, 0, st, n, (long long)j, x, g, p, Ap, lb, ub, alpha_bar,
                           many ? w.total : w.dots, many ? 1 : (int)w.parts, many ? (int64_t)1 : w.parts, w.mins, w.s,
                           w.sums, status);
        UHIP_CHECK_LAUNCH();
        UHIP_TRY(mprgp_gradient(ctx, A, x, g, b, lb, ub, w.s, (long long)j, w.grad, w.parts));
        if (many) UHIP_TRY(finish_sums_from(ctx, w.grad, 3, w.parts, w.parts, w.total + 2));
        hipLaunchKernelGGL(k_mprgp_direction, grid, blk, 0, st, n, (long long)j, x, g, p, lb, ub, w.sums,
                           many ? w.total + 2 : w.grad, many ? 1 : (int)w.parts, many ? (int64_t)1 : w.parts, atol, rtol,
                           w.s, w.mins, status);
        UHIP_CHECK_LAUNCH();
        if (j - first >= kAhead) UHIP_TRY(run_wait(ctx, j + 1 - kAhead));
    }
    UHIP_CHECK_HIP(hipStreamSynchronize(st));
    *steps = seen->steps - first;
    *reason = seen->done;
    *norm = seen->value[0];
    *norm0 = seen->value[1];
    return UHIP_OK;
}

int uhip_mprgp_alpha_f_f64(uhip_ctx ctx, int64_t n, const double *x, const double *p, const double *lb,
                           const double *ub, double *result_d) {
    UHIP_REQUIRE(ctx && x && p && lb && ub && result_d, "uhip_mprgp_alpha_f_f64: null argument");
    const int gr = grid_for(n, 4, kMaxRedBlocks);
    UHIP_TRY(ensure_partials(ctx, gr));
    hipLaunchKernelGGL(k_alpha_f, dim3(gr), dim3(kBlock), 0, ctx->stream, n, x, p, lb, ub, ctx->partials);
    UHIP_CHECK_LAUNCH();
    hipLaunchKernelGGL(k_min_finish, dim3(1), dim3(kBlock), 0, ctx->stream, ctx->partials, (int64_t)gr, result_d);
    UHIP_CHECK_LAUNCH();
    return UHIP_OK;
}

int uhip_mprgp_cg_step_f64(uhip_ctx ctx, int64_t n, double *x, double *g, const double *p, const double *Ap,
                           const double *lb, const double *ub, double *fi, double alpha, double *scalars,
                           int i_fiAp) {
    UHIP_REQUIRE(ctx && x && g && p && Ap && lb && ub && fi && scalars, "uhip_mprgp_cg_step_f64: null argument");
    const int gr = grid_for(n, 4, kMaxRedBlocks);
    UHIP_TRY(ensure_partials(ctx, gr));
    hipLaunchKernelGGL(k_mprgp_cg_step, dim3(gr), dim3(kBlock), 0, ctx->stream, n, x, g, p, Ap, lb, ub, fi, alpha,
                       ctx->partials);
    UHIP_CHECK_LAUNCH();
    return finish_sums(ctx, 1, gr, ctx->max_partials, scalars + i_fiAp, 0u);
}

int uhip_mprgp_cg_step_state_f64(uhip_ctx ctx, int64_t n, double *x, double *g, const double *p, const double *Ap,
                                 const double *lb, const double *ub, double *fi, double *beta, double *gp,
                                 double alpha, double *dots_d) {
    UHIP_REQUIRE(ctx && x && g && p && Ap && lb && ub && fi && beta && gp && dots_d,
                 "uhip_mprgp_cg_step_state_f64: null argument");
    const int gr = grid_for(n, 4, kMaxRedBlocks);
    UHIP_TRY(ensure_partials(ctx, gr));
    hipLaunchKernelGGL(k_mprgp_cg_step_state, dim3(gr), dim3(kBlock), 0, ctx->stream, n, x, g, p, Ap, lb, ub, fi, beta,
                       gp, alpha, ctx->partials, ctx->max_partials);
    UHIP_CHECK_LAUNCH();
    return finish_sums(ctx, 4, gr, ctx->max_partials, dots_d, 0u);
}

int uhip_mprgp_pupdate_f64(uhip_ctx ctx, int64_t n, double *p, const double *fi, const double *scalars, int i_num,
                           int i_den) {
    UHIP_REQUIRE(ctx && p && fi && scalars, "uhip_mprgp_pupdate_f64: null argument");
    UHIP_TRY(finish_left(ctx));
    if (n <= 0) return UHIP_OK;
    hipLaunchKernelGGL(k_mprgp_pupdate, dim3(grid_for(n, 4, 1 << 16)), dim3(kBlock), 0, ctx->stream, n, p, fi, scalars,
                       i_num, i_den);
    UHIP_CHECK_LAUNCH();
    return UHIP_OK;
}

int uhip_mprgp_expand_f64(uhip_ctx ctx, int64_t n, double *x, const double *g, const double *p, const double *Ap,
                          const double *lb, const double *ub, double alpha_f, double alpha_bar) {
    UHIP_REQUIRE(ctx && x && g && p && Ap && lb && ub, "uhip_mprgp_expand_f64: null argument");
    if (n <= 0) return UHIP_OK;
    hipLaunchKernelGGL(k_mprgp_expand, dim3(grid_for(n, 4, 1 << 16)), dim3(kBlock), 0, ctx->stream, n, x, g, p, Ap, lb,
                       ub, alpha_f, alpha_bar);
    UHIP_CHECK_LAUNCH();
    return UHIP_OK;
}

int uhip_mprgp_proportion_f64(uhip_ctx ctx, int64_t n, double *x, double *g, const double *beta, const double *Abeta,
                              const double *lb, const double *ub, double *p, double alpha) {
    UHIP_REQUIRE(ctx && x && g && beta && Abeta && lb && ub && p, "uhip_mprgp_proportion_f64: null argument");
    if (n <= 0) return UHIP_OK;
    hipLaunchKernelGGL(k_mprgp_prop, dim3(grid_for(n, 4, 1 << 16)), dim3(kBlock), 0, ctx->stream, n, x, g, beta, Abeta,
                       lb, ub, p, alpha);
    UHIP_CHECK_LAUNCH();
    return UHIP_OK;
}

int uhip_graph_color(uhip_ctx ctx, const uhip_csr *A, uint64_t seed, int32_t *color, int32_t *ncolors) {
    UHIP_REQUIRE(ctx && A && color && ncolors, "uhip_graph_color: null argument");
    UHIP_REQUIRE(A->nrows == A->ncols, "uhip_graph_color: square pattern required");
    const int32_t n = A->nrows;
    *ncolors = 0;
    if (n == 0) return UHIP_OK;
    UHIP_CHECK_HIP(hipMemsetAsync(color, 0xff, sizeof(int32_t) * (size_t)n, ctx->stream));  // -1
    unsigned int *rem = ctx->counters + 1;
    dim3 g((n + kBlock - 1) / kBlock);
    // every round colours at least the uncoloured row of largest (hash, index); the host looks after each
    // fourth (a 9-point grid takes about 20 rounds; a round with nothing left changes nothing)
    for (int32_t round = 0; round < n; round += 4) {
        for (int k = 0; k < 4; ++k) {
            if (k == 3) UHIP_CHECK_HIP(hipMemsetAsync(rem, 0, sizeof(unsigned int), ctx->stream));
            hipLaunchKernelGGL(k_jp_round, g, dim3(kBlock), 0, ctx->stream, n, A->rowptr, A->col, color, seed, rem);
            UHIP_CHECK_LAUNCH();
            hipLaunchKernelGGL(k_jp_commit, g, dim3(kBlock), 0, ctx->stream, n, color);
            UHIP_CHECK_LAUNCH();
        }
        int32_t left = 0;
        UHIP_TRY(read_ints(ctx, (const int32_t *)rem, 1, &left));
        if (left == 0) {
            UHIP_CHECK_HIP(hipMemsetAsync(rem, 0, sizeof(unsigned int), ctx->stream));
            hipLaunchKernelGGL(k_max_color, dim3(grid_for(n, 4, 256)), dim3(kBlock), 0, ctx->stream, n, color,
                               (int32_t *)rem);
            UHIP_CHECK_LAUNCH();
            int32_t m = 0;
            UHIP_TRY(read_ints(ctx, (const int32_t *)rem, 1, &m));
            *ncolors = m + 1;
            return UHIP_OK;
        }
    }
    return set_error(UHIP_ERR_NUMERIC, "uhip_graph_color: did not terminate");
}

int uhip_pgs_dinv(uhip_ctx ctx, const uhip_csr *A, double *dinv) {
    UHIP_REQUIRE(ctx && A && dinv && A->dtype == UHIP_F64, "uhip_pgs_dinv: bad argument");
    const int32_t n = A->nrows;
    if (n == 0) return UHIP_OK;
    hipLaunchKernelGGL(k_pgs_dinv, dim3((n + kBlock - 1) / kBlock), dim3(kBlock), 0, ctx->stream, n, A->rowptr, A->col,
                       (const double *)A->val, dinv);
    UHIP_CHECK_LAUNCH();
    return UHIP_OK;
}

int uhip_pgs_color_sweep(uhip_ctx ctx, const uhip_csr *A, int32_t cnt, const int32_t *rows, const double *dinv,
                         const double *r, const double *x, const double *lb, const double *ub, double *c,
                         int constrained) {
    UHIP_REQUIRE(ctx && A && rows && dinv && r && c && A->dtype == UHIP_F64, "uhip_pgs_color_sweep: bad argument");
    UHIP_REQUIRE(!constrained || (x && lb && ub), "uhip_pgs_color_sweep: bounds needed");
    if (cnt <= 0) return UHIP_OK;
    hipLaunchKernelGGL(k_pgs_color, dim3((cnt + kBlock - 1) / kBlock), dim3(kBlock), 0, ctx->stream, cnt, rows,
                       A->rowptr, A->col, (const double *)A->val, dinv, r, x, lb, ub, c, constrained);
    UHIP_CHECK_LAUNCH();
    return UHIP_OK;
}

// rows grouped by colour (stable), offsets[k] .. offsets[k+1]
int uhip_color_groups(uhip_ctx ctx, int32_t n, const int32_t *color, int32_t ncolors, int32_t *rows,
                      int32_t *offsets_h) {
    UHIP_REQUIRE(ctx && color && rows && offsets_h && ncolors >= 0, "uhip_color_groups: bad argument");
    if (n == 0) {
        offsets_h[0] = 0;
        return UHIP_OK;
    }
    hipStream_t st = ctx->stream;
    size_t tb = 0;
    int bits = 1;
    while ((1 << bits) <= ncolors) ++bits;
    UHIP_CHECK_HIP(hipcub::DeviceRadixSort::SortPairs(nullptr, tb, color, (int32_t *)nullptr, (int32_t *)nullptr, rows, n, 0,
                                                      bits, st));
    Scratch w(ctx);
    const size_t o_k = w.add(sizeof(int32_t) * n), o_i = w.add(sizeof(int32_t) * n),
                 o_o = w.add(sizeof(int32_t) * ((size_t)ncolors + 1)), o_t = w.add(tb);
    UHIP_TRY(w.allocate());
    const dim3 g((n + kBlock - 1) / kBlock), blk(kBlock);
    hipLaunchKernelGGL(k_iota, g, blk, 0, st, n, w.at<int32_t>(o_i));
    UHIP_CHECK_LAUNCH();
    UHIP_CHECK_HIP(hipcub::DeviceRadixSort::SortPairs(w.at<void>(o_t), tb, color, w.at<int32_t>(o_k), w.at<int32_t>(o_i), rows,
                                                      n, 0, bits, st));
    hipLaunchKernelGGL(k_group_offsets, g, blk, 0, st, n, ncolors, w.at<int32_t>(o_k), w.at<int32_t>(o_o));
    UHIP_CHECK_LAUNCH();
    UHIP_CHECK_HIP(hipMemcpyAsync(offsets_h, w.at<void>(o_o), sizeof(int32_t) * ((size_t)ncolors + 1),
                                  hipMemcpyDeviceToHost, st));
    UHIP_CHECK_HIP(hipStreamSynchronize(st));
    return UHIP_OK;
}

}  // extern "C"
