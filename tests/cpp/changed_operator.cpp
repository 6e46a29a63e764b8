// Solvers of the host layer on an operator that changes between update and apply (new plan, new values in
// place), run by tests/test_gpu_cpp_surface.py with the name of one check. Exit status 0 = pass.
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

int main(int argc, char **argv) {
    const std::string name = argc > 1 ? argv[1] : "";
    auto ctx = std::make_shared<HipContext>(0);
    if (name == "mprgp_replanned") mprgp_replanned(ctx);
    else CHECK(!"a check of this name");
    std::printf(fails ? "FAILED (%d)\n" : "OK\n", fails);
    return fails ? 1 : 0;
}
