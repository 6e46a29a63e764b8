// Rows of a matrix grouped by colour, and Gauss-Seidel sweeps over the groups: what the GaussSeidel smoother and
// ProjectedGaussSeidel share.
#pragma once

#include "utopia_hip_backend.hpp"

namespace utopia {
namespace hip {

// Jones-Plassmann colouring with a fixed seed: rows of one colour are not coupled, so a sweep updates a whole
// colour in parallel. The sweeps run from the colours' own copy of the matrix (uhip_color_plan); where that copy
// would be several times the matrix (very uneven rows), from the matrix itself.
class ColorGroups {
public:
    static constexpr uint64_t kSeed = 0x5eedull;
    ColorGroups() = default;
    ColorGroups(const ColorGroups &) = delete;
    ColorGroups &operator=(const ColorGroups &) = delete;
    ~ColorGroups() { release(); }
    void build(const HipCrsMatrix &A) {
        release();
        ctx_ = A.context();
        const int64_t n = A.rows();
        void *p = nullptr;
        hip_check(uhip_malloc(A.c(), &p, sizeof(int32_t) * (size_t)(n > 0 ? n : 1)), "alloc colors");
        color_ = (int32_t *)p;
        hip_check(uhip_malloc(A.c(), &p, sizeof(int32_t) * (size_t)(n > 0 ? n : 1)), "alloc rows");
        rows_ = (int32_t *)p;
        hip_check(uhip_graph_color(A.c(), &A.raw(), kSeed, color_, &ncolors_), "coloring");
        offsets_.assign((size_t)ncolors_ + 1, 0);
        hip_check(uhip_color_groups(A.c(), (int32_t)n, color_, ncolors_, rows_, offsets_.data()), "colour groups");
        make_plan(A);
    }
    // Ahead of sweeps with the residuals of A: the values as they are now. A matrix in a layout that copies the
    // values shows new ones when it is planned again, so does the colours' copy; the row-block form multiplies
    // with the matrix' own array, so the copy is filled from it.
    void follow(const HipCrsMatrix &A) {
        if (A.version() != version_) make_plan(A);
        else if (plan_ && A.raw().format == UHIP_FMT_ROWBLOCK)
            hip_check(uhip_color_plan_refresh(A.c(), plan_, &A.raw()), "colour plan values");
    }
    int32_t ncolors() const { return ncolors_; }
    const int32_t *color() const { return color_; }
    // whether the sweeps run from the colours' copy: a missing bound may be NULL then, otherwise not
    bool has_plan() const { return plan_ != nullptr; }
    // c = 0 on entry; forward over the colours, then (symmetric) backward:
    // c_i = d_inv_i (r_i - sum_{j != i} a_ij c_j), within lb - x and ub - x when constrained; add: x += c
    void sweep(const HipCrsMatrix &A, const double *dinv, const double *r, double *x, const double *lb,
               const double *ub, double *c, bool constrained, bool symmetric, bool add) const {
        if (plan_) {
            hip_check(uhip_color_plan_sweep(A.c(), plan_, dinv, r, x, lb, ub, c, constrained, symmetric, add),
                      "colour sweep");
            return;
        }
        for (int pass = 0; pass < (symmetric ? 2 : 1); ++pass)
            for (int32_t t = 0; t < ncolors_; ++t) {
                const int32_t k = pass == 0 ? t : ncolors_ - 1 - t;
                const int32_t o = offsets_[(size_t)k], cnt = offsets_[(size_t)k + 1] - o;
                hip_check(uhip_pgs_color_sweep(A.c(), &A.raw(), cnt, rows_ + o, dinv, r, x, lb, ub, c, constrained),
                          "colour sweep");
            }
        if (add) hip_check(uhip_vec_axpy_f64(A.c(), A.rows(), 1.0, c, x), "x += c");
    }

private:
    void make_plan(const HipCrsMatrix &A) {
        if (plan_) uhip_color_plan_destroy(A.c(), plan_);
        plan_ = nullptr;
        const int st = uhip_color_plan_create(A.c(), &A.raw(), ncolors_, rows_, offsets_.data(), &plan_);
        if (st != UHIP_ERR_UNSUPPORTED) hip_check(st, "colour plan");
        version_ = A.version();
    }
    void release() {
        if (ctx_) {
            if (color_) uhip_free(ctx_->get(), color_);
            if (rows_) uhip_free(ctx_->get(), rows_);
            uhip_color_plan_destroy(ctx_->get(), plan_);
        }
        color_ = rows_ = nullptr;
        plan_ = nullptr;
    }
    HipContextPtr ctx_;
    uhip_color_plan plan_ = nullptr;
    uint64_t version_ = 0;  // of the matrix that plan_ copies
    int32_t ncolors_ = 0;
    int32_t *color_ = nullptr, *rows_ = nullptr;
    std::vector<int32_t> offsets_;
};

}  // namespace hip
}  // namespace utopia
