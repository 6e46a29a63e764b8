// Solvers of the host layer on an operator that changes between update and apply (new plan, new values in
// place), run by tests/test_gpu_cpp_surface.py with the name of one check. Exit status 0 = pass.
#include <cfloat>
#include <cmath>
#include <cstdio>
#include <cstring>
#include <string>
#include <vector>

#include "utopia_hip_multigrid.hpp"
#include "utopia_hip_qp.hpp"

using namespace utopia;
using namespace utopia::hip;

static int fails = 0;
#define CHECK(c)                                              \
    do {                                                      \
        if (!(c)) {                                           \
            std::printf("FAIL %s (line %d)\n", #c, __LINE__); \
            ++fails;                                          \
        }                                                     \
    } while (0)

static std::shared_ptr<HipCrsMatrix> poisson(const HipContextPtr &ctx, int nx, int ny) {
    const int32_t n = nx * ny;
    std::vector<int32_t> rp((size_t)n + 1), col((size_t)uhip_gen_nnz(0, nx, ny, 1));
    std::vector<double> val(col.size());
    uhip_gen_stencil(0, nx, ny, 1, 0, 0.0, rp.data(), col.data(), val.data());
    auto A = std::make_shared<HipCrsMatrix>();
    A->from_host(ctx, n, n, rp.data(), col.data(), val.data());
    return A;
}

static HipVector uniform(const HipContextPtr &ctx, int seed, int64_t n, double lo, double hi) {
    std::vector<double> h((size_t)n);
    uhip_gen_uniform(seed, n, lo, hi, h.data());
    HipVector v(ctx, n);
    v.upload(h.data());
    return v;
}

static bool same(const HipVector &a, const HipVector &b) {
    const std::vector<double> x = a.to_host(), y = b.to_host();
    return x.size() == y.size() && std::memcmp(x.data(), y.data(), sizeof(double) * x.size()) == 0;
}

// MPRGP set up with one plan, run with another that has more partial sums
static void mprgp_replanned(const HipContextPtr &ctx) {
    const auto A = poisson(ctx, 120, 100);
    const HipVector b = uniform(ctx, 3, A->rows(), -1, 1);
    BoxConstraints box;
    box.lower = std::make_shared<HipVector>(ctx, A->rows(), -2.0);
    auto solver = [&] {
        MPRGP s;
        s.atol(1e-8);
        s.max_it(200);
        s.set_box_constraints(box);
        return s;
    };
    MPRGP s = solver(), fresh = solver();
    s.update(A);
    const int64_t before = uhip_mprgp_work_bytes(&A->raw());
    hip_check(uhip_csr_plan_format(ctx->get(), &A->raw(), UHIP_FMT_ROWBLOCK, 1024), "plan");
    CHECK(uhip_mprgp_work_bytes(&A->raw()) > before);
    fresh.update(A);
    HipVector x(ctx, A->rows(), 0.0), y(ctx, A->rows(), 0.0);
    s.apply(b, x);
    fresh.apply(b, y);
    CHECK(same(x, y));
    CHECK(s.solution_status().iterates == fresh.solution_status().iterates);
}

// Gauss-Seidel solvers on values that have changed in place since update: what a solver whose colours were made
// anew on the changed operator does with the first one's diagonal
static void sweep_values(const HipContextPtr &ctx, int32_t block_nnz) {
    const auto A = poisson(ctx, 60, 50);
    A->plan(block_nnz);  // 0: a layout that copies the values; else row blocks on the matrix' own
    const int64_t n = A->rows();
    const HipVector b = uniform(ctx, 3, n, -1, 1);
    BoxConstraints box;
    box.lower = std::make_shared<HipVector>(ctx, n, -0.05);
    ProjectedGaussSeidel pgs;
    pgs.set_box_constraints(box);
    pgs.update(A);
    GaussSeidel gs;
    gs.sweeps(3);
    gs.update(A);
    // off-diagonal values only, so that d_inv, which update makes, stays that of the operator
    auto change = [&](double f) {
        if (block_nnz == 0) {
            A->transform_values([f](double v) { return v < 0 ? f * v : v; });
            return;
        }
        std::vector<int32_t> rp, col;
        std::vector<double> val;
        const HipCrsMatrix &M = *A;
        M.to_host(rp, col, val);
        for (double &v : val) v = v < 0 ? f * v : v;
        hip_check(uhip_memcpy_htod(ctx->get(), M.raw().val, val.data(), sizeof(double) * val.size()), "values");
    };
    for (const double f : {0.5, 1.5}) {
        change(f);
        ProjectedGaussSeidel pgs_fresh;
        pgs_fresh.set_box_constraints(box);
        pgs_fresh.update(A);
        GaussSeidel gs_fresh;
        gs_fresh.sweeps(3);
        gs_fresh.update(A);
        HipVector x(ctx, n, 0.0), y(ctx, n, 0.0);
        pgs.smooth(b, x, 2);
        pgs_fresh.smooth(b, y, 2);
        CHECK(same(x, y));
        pgs.max_it(5);
        pgs_fresh.max_it(5);
        pgs.apply(b, x);
        pgs_fresh.apply(b, y);
        CHECK(same(x, y));
        x.set(0.0);
        y.set(0.0);
        gs.apply(b, x);
        gs_fresh.apply(b, y);
        CHECK(same(x, y));
    }
}

// A multigrid smoothed by Gauss-Seidel keeps its hierarchy when the fine operator changes: the fine level smooths
// and forms residuals with the new values
static void multigrid_values(const HipContextPtr &ctx) {
    const int nx = 33, ny = 33, cx = 17, cy = 17;
    const auto A = poisson(ctx, nx, ny);
    std::vector<int32_t> rp{0}, col;
    std::vector<double> val;
    for (int j = 0; j < ny; ++j)
        for (int i = 0; i < nx; ++i) {  // bilinear interpolation
            for (int dj = 0; dj <= j % 2; ++dj)
                for (int di = 0; di <= i % 2; ++di) {
                    col.push_back((j / 2 + dj) * cx + i / 2 + di);
                    val.push_back((j % 2 ? 0.5 : 1.0) * (i % 2 ? 0.5 : 1.0));
                }
            rp.push_back((int32_t)col.size());
        }
    auto P = std::make_shared<HipCrsMatrix>();
    P->from_host(ctx, nx * ny, cx * cy, rp.data(), col.data(), val.data());
    const HipVector b = uniform(ctx, 3, A->rows(), -1, 1);
    auto one_cycle = [&](Multigrid &mg) {
        HipVector x(ctx, A->rows(), 0.0);
        mg.max_it(1);
        mg.apply(b, x);
        return x;
    };
    auto hierarchy = [&] {
        auto mg = std::make_shared<Multigrid>(std::make_shared<GaussSeidel>(), std::make_shared<Factorization>());
        mg->set_transfer_operators({P});
        mg->must_generate_masks(false);
        mg->update(A);
        return mg;
    };
    const auto mg = hierarchy(), kept = hierarchy();
    const HipVector before = one_cycle(*mg);
    CHECK(same(before, one_cycle(*kept)));
    A->transform_values([](double v) { return v < 0 ? 0.5 * v : v; });
    // by hand: the cycle on the changed operator with the old coarse operator and the (unchanged) diagonal
    GaussSeidel gs;
    gs.sweeps(3);
    gs.update(A);
    HipVector x(ctx, A->rows(), 0.0), r(ctx, A->rows(), 0.0), rc, cc(ctx, P->cols(), 0.0), cf;
    gs.apply(b, x);
    A->residual(x, b, r);
    P->transpose_multiply(r, rc);
    Factorization coarse;
    coarse.factorize(kept->level_operator(0));
    coarse.apply(rc, cc);
    P->multiply(cc, cf);
    x.axpy(1.0, cf);
    gs.apply(b, x);
    const HipVector after = one_cycle(*mg);
    HipVector d(after);
    d.axpy(-1.0, x);
    CHECK(!same(before, after));
    CHECK(d.norm2() <= 1e-13 * x.norm2());
}

// The bounds that a solver has after a solve: the missing one filled, and a change of it seen by the next solve
template <class Solver>
static void bounds_after_solve(const HipContextPtr &ctx, Solver &s) {
    const auto A = poisson(ctx, 40, 30);
    const int64_t n = A->rows();
    const HipVector b = uniform(ctx, 3, n, 0, 1);
    BoxConstraints box;
    box.lower = std::make_shared<HipVector>(ctx, n, -1.0);
    s.set_box_constraints(box);
    s.max_it(300);
    s.update(A);
    CHECK(!s.get_box_constraints().upper);
    HipVector x(ctx, n, 0.0);
    s.apply(b, x);
    CHECK(x.max() > 0.5);
    const BoxConstraints &after = s.get_box_constraints();
    CHECK(after.lower == box.lower && after.upper && after.upper->size() == n);
    if (!after.upper) return;
    CHECK(after.upper->min() == DBL_MAX && after.upper->max() == DBL_MAX);
    after.upper->set(0.25);
    x.set(0.0);
    s.apply(b, x);
    CHECK(x.max() <= 0.25 && x.max() > 0.2);
    box.upper = std::make_shared<HipVector>(ctx, n, 0.5);  // new bounds are taken as they are
    box.lower = nullptr;
    s.set_box_constraints(box);
    CHECK(!s.get_box_constraints().lower && s.get_box_constraints().upper == box.upper);
}

// MPRGP without bounds as the preconditioner of a CG on the same context: a loop inside a loop's iteration
static void loop_in_loop(const HipContextPtr &ctx) {
    const auto A = poisson(ctx, 60, 50);
    const HipVector b = uniform(ctx, 3, A->rows(), -1, 1);
    const double atol = 1e-8 * b.norm2();
    for (const double inner_rtol : {1e-10, 1e-2}) {
        auto inner = std::make_shared<MPRGP>();
        inner->atol(0);
        inner->rtol(inner_rtol);
        inner->max_it(2000);
        ConjugateGradient<HipCrsMatrix, HipVector> cg;
        cg.set_preconditioner(inner);
        cg.atol(atol);
        cg.rtol(0);
        cg.stol(0);
        cg.max_it(50);
        cg.update(A);
        HipVector x(ctx, A->rows(), 0.0), r;
        CHECK(cg.apply(b, x));
        r = HipVector(ctx, A->rows(), 0.0);
        A->residual(x, b, r);
        const double true_norm = r.norm2(), norm = cg.solution_status().gradient_norm;
        std::printf("inner rtol %g: %lld iterations, |b - A x| %.3e, reported %.3e, atol %.3e\n", inner_rtol,
                    (long long)cg.solution_status().iterates, true_norm, norm, atol);
        CHECK(norm <= atol && std::fabs(true_norm - norm) <= 1e-3 * atol);
    }
}

int main(int argc, char **argv) {
    const std::string name = argc > 1 ? argv[1] : "";
    auto ctx = std::make_shared<HipContext>(0);
    if (name == "mprgp_replanned") mprgp_replanned(ctx);
    else if (name == "sweep_values") sweep_values(ctx, 0);
    else if (name == "sweep_values_row_blocks") sweep_values(ctx, 2048);
    else if (name == "multigrid_values") multigrid_values(ctx);
    else if (name == "bounds_mprgp") {
        MPRGP s;
        bounds_after_solve(ctx, s);
    } else if (name == "bounds_pgs") {
        ProjectedGaussSeidel s;
        bounds_after_solve(ctx, s);
    } else if (name == "loop_in_loop") loop_in_loop(ctx);
    else CHECK(!"a check of this name");
    std::printf(fails ? "FAILED (%d)\n" : "OK\n", fails);
    return fails ? 1 : 0;
}
