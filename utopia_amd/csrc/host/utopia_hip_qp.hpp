// Box-constrained QP solvers over the HIP backend:
//   BoxConstraints        solvers/nonlinear/constrained/utopia_BoxConstraints.hpp:19-345
//   MPRGP                 solvers/nonlinear/constrained/quadratic_programming/utopia_MPRGP.hpp:14-421
//   ProjectedGaussSeidel  backend/petsc/solvers/nonlinear/constrained/quadratic_programming/
//                         utopia_petsc_ProjectedGaussSeidel.cpp:24-540 (multicolour sweep order)
//   ProjectedConjugateGradient  .../quadratic_programming/utopia_ProjectedConjugateGradient.hpp:14-143
//   ProjectedGradient     .../quadratic_programming/utopia_ProjectedGradient.hpp:18-230
#pragma once

#include <cfloat>

#include "utopia_hip_coloring.hpp"
#include "utopia_hip_solvers.hpp"

namespace utopia {
// the solvers of the HIP backend (the tensor types, HipVector and HipCrsMatrix, are in utopia)
namespace hip {

struct BoxConstraints {
    std::shared_ptr<HipVector> lower, upper;
    bool has_bound() const { return lower || upper; }
    // BoxConstraints::fill_empty_bounds (utopia_BoxConstraints.hpp:281-300)
    void fill_empty_bounds(const HipContextPtr &ctx, int64_t n) {
        if (!lower || lower->size() != n) lower = std::make_shared<HipVector>(ctx, n, -DBL_MAX);
        if (!upper || upper->size() != n) upper = std::make_shared<HipVector>(ctx, n, DBL_MAX);
    }
};

class QPSolverBase : public IterativeSolver<HipCrsMatrix, HipVector> {
public:
    bool set_box_constraints(const BoxConstraints &box) {
        box_ = box;
        fill_ctx_ = nullptr;
        return true;
    }
    // after a solve, missing bounds are filled
    const BoxConstraints &get_box_constraints() const {
        if (fill_ctx_) box_.fill_empty_bounds(fill_ctx_, fill_n_);
        return box_;
    }

protected:
    // What a solve that takes its missing bounds as NULL (the kernels then use the filling's value and read nothing)
    // leaves to whoever asks for the bounds; from then on they are bounds as any other.
    void fill_when_asked(const HipCrsMatrix &A) {
        fill_ctx_ = A.context();
        fill_n_ = A.rows();
    }
    mutable BoxConstraints box_;

private:
    HipContextPtr fill_ctx_;
    int64_t fill_n_ = 0;
};

// ---------------------------------------------------------------------------
// MPRGP (non-"hardik" variant, no preconditioner), utopia_MPRGP.hpp:57-262
// ---------------------------------------------------------------------------
class MPRGP final : public QPSolverBase {
public:
    void set_eig_comp_tol(double v) { eps_eig_est_ = v; }
    void power_method_max_it(int64_t v) { power_method_max_it_ = v; }
    double alpha_bar() const { return alpha_bar_; }

    void update(const std::shared_ptr<const HipCrsMatrix> &op) override {
        QPSolverBase::update(op);
        const int64_t n = op->rows();
        if (fi_.size() != n || fi_.empty())
            for (HipVector *v : {&fi_, &p_, &Ap_, &g_, &h1_, &h2_}) *v = HipVector(op->context(), n, 0.0);
        reserve_work(*op);
    }

    bool apply(const HipVector &rhs, HipVector &x) override {
        const HipCrsMatrix &A = *this->op_;
        const int64_t n = A.rows();
        uhip_ctx c = A.c();
        if (x.empty() || x.size() != n) x.zeros_like(rhs);
        fill_when_asked(A);
        const auto bound = [n](const std::shared_ptr<HipVector> &v) -> const double * {
            return v && v->size() == n ? v->data() : nullptr;
        };
        const double *lb = bound(box_.lower), *ub = bound(box_.upper);
        alpha_bar_ = 1.95 / power_method(A);
        this->status_.clear();
        reserve_work(A);  // the operator may have another plan than at update
        hip_check(uhip_mprgp_begin_f64(c, &A.raw(), rhs.data(), lb, ub, x.data(), g_.data(), p_.data(), work_.data()),
                  "mprgp begin");
        // check_convergence stops after iteration it when it >= max_it, or at once with stol or rtol >= 1
        const int64_t most = this->stol_ >= 1 ? 1 : std::max<int64_t>(this->max_it_, 1);
        int64_t it = 0;
        double gnorm = 0, gnorm0 = 0;
        int reason = 0;
        while (it < most && reason == 0) {
            int64_t steps = 0;  // one at a time when every norm is to be printed
            hip_check(uhip_mprgp_run_f64(c, &A.raw(), rhs.data(), lb, ub, x.data(), g_.data(), p_.data(), Ap_.data(),
                                         work_.data(), alpha_bar_, this->atol_, this->rtol_, it,
                                         this->verbose_ ? 1 : most - it, &steps, &gnorm, &gnorm0, &reason),
                      "mprgp iterations");
            if (reason == 2) return true;  // negative curvature
            it += steps;
            this->print_iter(it, gnorm);
        }
        return this->check_convergence(it, gnorm, gnorm / gnorm0, 1);
    }

private:
    // the iterations' memory, by the number of partial sums of A's present plan
    void reserve_work(const HipCrsMatrix &A) {
        const int64_t n = (uhip_mprgp_work_bytes(&A.raw()) + 7) / 8;
        if (work_.size() < n) work_ = HipVector(A.context(), n);
    }

    // MPRGP::power_method (utopia_MPRGP.hpp:351-387)
    double power_method(const HipCrsMatrix &A) {
        h2_.set(1.0);
        int64_t it = 0;
        bool converged = false;
        double gnorm, lambda = 0.0, lambda_old;
        while (!converged) {
            h1_.copy_from(h2_);
            A.multiply(h1_, h2_);
            h2_.scale(1.0 / h2_.norm2());
            lambda_old = lambda;
            A.multiply(h2_, h1_);
            lambda = h2_.dot(h1_);
            hip_check(uhip_vec_waxpby_f64(A.c(), fi_.size(), 1.0, h2_.data(), -1.0, h1_.data(), fi_.data()), "fi");
            gnorm = fi_.norm2();
            converged = ((gnorm < eps_eig_est_) || (std::abs(lambda_old - lambda) < eps_eig_est_) ||
                         it > power_method_max_it_);
            it = it + 1;
        }
        return lambda;
    }

    double eps_eig_est_ = 1e-1, alpha_bar_ = 0;
    int64_t power_method_max_it_ = 10;
    HipVector fi_, p_, Ap_, g_, h1_, h2_, work_;
};

// ---------------------------------------------------------------------------
// ProjectedGaussSeidel: PETSc-specialisation semantics (apply/step, check of
// |x - x_old| every check_s_norm_each iterations, n_local_sweeps = 1, no line
// search), with the lexicographic sweep replaced by a multicolour one: colours
// forward, then backward for the symmetric sweep. Rows of one colour are not
// coupled, so each colour updates in parallel.
// ---------------------------------------------------------------------------
class ProjectedGaussSeidel final : public QPSolverBase {
public:
    void use_symmetric_sweep(bool v) { symmetric_ = v; }
    void check_s_norm_each(int64_t v) { check_each_ = v; }
    int32_t ncolors() const { return groups_ ? groups_->ncolors() : 0; }

    void update(const std::shared_ptr<const HipCrsMatrix> &op) override {
        QPSolverBase::update(op);
        const int64_t n = op->rows();
        auto ctx = op->context();
        for (HipVector *v : {&dinv_, &r_, &c_, &x_old_}) *v = HipVector(ctx, n, 0.0);
        hip_check(uhip_pgs_dinv(op->c(), &op->raw(), dinv_.data()), "pgs dinv");
        groups_ = std::make_shared<ColorGroups>();
        groups_->build(*op);
    }

    // ProjectedGaussSeidel::smooth (utopia_petsc_ProjectedGaussSeidel.cpp:111-132): with bounds,
    // `sweeps` projected steps; without, the reference loop
    // `while (unconstrained_step(...) && it++ < sweeps)` runs sweeps + 1 steps.
    bool smooth(const HipVector &b, HipVector &x, int64_t sweeps) {
        const HipCrsMatrix &A = *this->op_;
        if (x.empty() || x.size() != A.rows()) x.zeros_like(b);
        groups_->follow(A);
        const bool constrained = box_.has_bound();
        const int64_t steps = constrained ? sweeps : sweeps + 1;
        for (int64_t s = 0; s < steps; ++s) step(A, b, x, constrained);
        return true;
    }

    // apply (utopia_petsc_ProjectedGaussSeidel.cpp:134-178)
    bool apply(const HipVector &b, HipVector &x) override {
        const HipCrsMatrix &A = *this->op_;
        const int64_t n = A.rows();
        if (x.empty() || x.size() != n) x.zeros_like(b);
        groups_->follow(A);
        const bool constrained = box_.has_bound();
        this->status_.clear();
        x_old_.copy_from(x);
        bool converged = false;
        int64_t iteration = 0;
        while (!converged) {
            step(A, b, x, constrained);
            if (iteration % check_each_ == 0) {
                c_.copy_from(x);
                c_.axpy(-1.0, x_old_);
                const double diff = c_.norm2();
                this->print_iter(iteration, diff);
                converged = this->check_convergence(iteration, 1, 1, diff);
            }
            ++iteration;
            if (converged) break;
            if (iteration % check_each_ == 0) x_old_.copy_from(x);  // the next step is looked at
        }
        return converged;
    }

private:
    // step / unconstrained_step (utopia_petsc_ProjectedGaussSeidel.cpp:331-455)
    void step(const HipCrsMatrix &A, const HipVector &b, HipVector &x, bool constrained) {
        hip_check(uhip_spmv_residual_zero_f64(A.c(), &A.raw(), x.data(), b.data(), r_.data(), c_.data()),
                  "pgs residual");
        if (constrained) {
            if (groups_->has_plan()) fill_when_asked(A);
            else box_.fill_empty_bounds(A.context(), A.rows());
        }
        const auto bound = [&](const std::shared_ptr<HipVector> &v) -> const double * {
            return constrained && v && v->size() == x.size() ? v->data() : nullptr;
        };
        groups_->sweep(A, dinv_.data(), r_.data(), x.data(), bound(box_.lower), bound(box_.upper), c_.data(),
                       constrained, symmetric_, /*add=*/true);
    }

    bool symmetric_ = true;
    int64_t check_each_ = 10;
    std::shared_ptr<ColorGroups> groups_;
    HipVector dinv_, r_, c_, x_old_;
};

// ---------------------------------------------------------------------------
// ProjectedConjugateGradient::apply (utopia_ProjectedConjugateGradient.hpp:33-123),
// step for step; the second A*pk of the reference equals the first (pk is
// unchanged in between), so it is reused.
// ---------------------------------------------------------------------------
class ProjectedConjugateGradient final : public QPSolverBase {
public:
    void update(const std::shared_ptr<const HipCrsMatrix> &op) override {
        QPSolverBase::update(op);
        const int64_t n = op->rows();
        for (HipVector *v : {&x_old_, &x_half_, &uk_, &wk_, &zk_, &pk_, &Apk_, &d_}) *v = HipVector(op->context(), n, 0.0);
    }
    bool apply(const HipVector &b, HipVector &x) override {
        const HipCrsMatrix &A = *this->op_;
        const int64_t n = A.rows();
        uhip_ctx c = A.c();
        double *s = A.context()->scalars();
        if (x.empty() || x.size() != n) x.zeros_like(b);
        box_.fill_empty_bounds(A.context(), n);
        const double *lb = box_.lower->data(), *ub = box_.upper->data();
        this->status_.clear();
        x_old_.copy_from(x);
        A.residual(x, b, uk_);  // uk = b - A x
        zk_.set(0.0);           // init_memory: zk.zeros
        pk_.copy_from(uk_);
        pk_.scale(-1.0);        // pk = -uk
        bool converged = false;
        const int64_t check_each = 10;
        int64_t iteration = 0;
        while (!converged) {
            hip_check(uhip_spmv_dot(c, &A.raw(), pk_.data(), Apk_.data(), s + S_PAP), "Apk, pk.Apk");
            const double *u1[1] = {uk_.data()}, *p1[1] = {pk_.data()};
            hip_check(uhip_vec_dots_f64(c, n, 1, u1, p1, s + S_UP), "uk.pk");
            double h[2];
            A.context()->read_scalars(s + S_PAP, 2, h);  // S_PAP, S_UP adjacent
            const double alpha = h[1] / h[0];
            if (alpha == 0. || std::isinf(alpha) || std::isnan(alpha)) break;
            hip_check(uhip_vec_waxpby_f64(c, n, alpha, pk_.data(), 1.0, x_old_.data(), x_half_.data()), "x_half");
            hip_check(uhip_box_project_f64(c, n, x_half_.data(), lb, ub, x.data()), "project");
            A.residual(x, b, uk_);
            hip_check(uhip_pcg_wz_f64(c, n, uk_.data(), lb, ub, pk_.data(), zk_.data(), wk_.data()), "w, z");
            const double *w1[1] = {wk_.data()}, *a1[1] = {Apk_.data()};
            hip_check(uhip_vec_dots_f64(c, n, 1, w1, a1, s + S_WAP), "wk.Apk");
            double h3[3];
            A.context()->read_scalars(s + S_PAP, 3, h3);  // pk.Apk, uk.pk, wk.Apk
            const double beta = h3[2] / h3[0];
            hip_check(uhip_vec_waxpby_f64(c, n, 1.0, wk_.data(), beta, zk_.data(), pk_.data()), "pk = wk + beta zk");
            if (iteration % check_each == 0 || std::isinf(beta) || std::isnan(beta)) {
                d_.copy_from(x_old_);
                d_.axpy(-1.0, x);
                const double diff = d_.norm2();
                this->print_iter(iteration, diff);
                converged = this->check_convergence(iteration, 1, 1, diff);
            }
            ++iteration;
            if (converged) break;
            x_old_.copy_from(x);
        }
        return converged;
    }

private:
    enum { S_PAP = 20, S_UP = 21, S_WAP = 22 };
    HipVector x_old_, x_half_, uk_, wk_, zk_, pk_, Apk_, d_;
};

// ---------------------------------------------------------------------------
// ProjectedGradient::solve / solve_unconstrained (utopia_ProjectedGradient.hpp:54-213)
// ---------------------------------------------------------------------------
class ProjectedGradient final : public QPSolverBase {
public:
    void update(const std::shared_ptr<const HipCrsMatrix> &op) override {
        QPSolverBase::update(op);
        const int64_t n = op->rows();
        for (HipVector *v : {&x_old_, &x_half_, &p_, &u_, &Ap_, &d_}) *v = HipVector(op->context(), n, 0.0);
    }
    bool apply(const HipVector &b, HipVector &x) override {
        const HipCrsMatrix &A = *this->op_;
        const int64_t n = A.rows();
        uhip_ctx c = A.c();
        double *s = A.context()->scalars();
        if (x.empty() || x.size() != n) x.zeros_like(b);
        this->status_.clear();
        const bool bounded = box_.has_bound();
        if (bounded) box_.fill_empty_bounds(A.context(), n);
        const double *lb = bounded ? box_.lower->data() : nullptr, *ub = bounded ? box_.upper->data() : nullptr;
        x_old_.copy_from(x);
        A.residual(x, b, u_);  // u = b - A x
        p_.copy_from(u_);
        double alpha = 1.;
        bool converged = false;
        const int64_t check_each = 20;
        int64_t iteration = 0;
        while (!converged) {
            if (bounded) {
                hip_check(uhip_vec_waxpby_f64(c, n, 1.0, x.data(), alpha, p_.data(), x_half_.data()), "x_half");
                hip_check(uhip_box_project_f64(c, n, x_half_.data(), lb, ub, x.data()), "project");
                A.residual(x, b, u_);
                hip_check(uhip_pg_direction_f64(c, n, x.data(), u_.data(), lb, ub, p_.data()), "direction");
            } else {
                x.axpy(alpha, p_);
                A.residual(x, b, p_);  // p = b - A x
            }
            if (iteration % check_each == 0) {
                d_.copy_from(x_old_);
                d_.axpy(-1.0, x);
                const double diff = d_.norm2();
                this->print_iter(iteration, diff);
                converged = this->check_convergence(iteration, 1, 1, diff);
            }
            ++iteration;
            if (converged) break;
            x_old_.copy_from(x);
            hip_check(uhip_spmv_dot(c, &A.raw(), p_.data(), Ap_.data(), s + S_PAP), "Ap, p.Ap");
            const double *a1[1] = {bounded ? u_.data() : p_.data()}, *p1[1] = {p_.data()};
            hip_check(uhip_vec_dots_f64(c, n, 1, a1, p1, s + S_NUM), bounded ? "u.p" : "p.p");
            double h[2];
            A.context()->read_scalars(s + S_PAP, 2, h);
            alpha = h[1] / h[0];
            if (std::isinf(alpha) || alpha == 0. || std::isnan(alpha)) {
                d_.copy_from(x_old_);
                d_.axpy(-1.0, x);
                const double diff = d_.norm2();
                converged = this->check_convergence(iteration, 1, 1, diff);
                break;
            }
        }
        return converged;
    }

private:
    enum { S_PAP = 24, S_NUM = 25 };
    HipVector x_old_, x_half_, p_, u_, Ap_, d_;
};

}  // namespace hip
}  // namespace utopia
