// Internal header shared by the HIP translation units of libutopia_hip.
// Not part of the public C ABI (that is include/utopia_hip.h).
#pragma once

#include <hip/hip_runtime.h>
#include <cstdint>
#include <cstdio>
#include <cstring>
#include <mutex>
#include <string>
#include <vector>

#include "../../include/utopia_hip.h"

namespace uhip {

// Launch geometry shared by all streaming kernels.
constexpr int kBlock = 256;          // 4 wavefronts of 64 lanes
constexpr int kMaxRedBlocks = 1024;  // upper bound on blocks of a grid-stride reduction
constexpr int kMaxDots = 4;          // fused dots per reduction launch
constexpr int kNumXcd = 8;           // MI355X: 8 XCDs, workgroups dispatched round-robin

// Record a message for uhip_last_error(); returns code.
int set_error(int code, const char *fmt, ...);

#define UHIP_CHECK_HIP(expr)                                                                  \
    do {                                                                                      \
        hipError_t e_ = (expr);                                                               \
        if (e_ != hipSuccess)                                                                 \
            return ::uhip::set_error(UHIP_ERR_HIP, "%s:%d %s -> %s", __FILE__, __LINE__, #expr, \
                                     hipGetErrorString(e_));                                  \
    } while (0)

#define UHIP_CHECK_LAUNCH() UHIP_CHECK_HIP(hipGetLastError())

#define UHIP_REQUIRE(cond, ...)                                                   \
    do {                                                                          \
        if (!(cond)) return ::uhip::set_error(UHIP_ERR_INVALID, __VA_ARGS__);     \
    } while (0)

#define UHIP_TRY(expr)              \
    do {                            \
        int s_ = (expr);            \
        if (s_ != UHIP_OK) return s_; \
    } while (0)

// Progress of a loop whose iterations decide on the device (CG with a Jacobi preconditioner, MPRGP).
// Kernels write it straight into pinned host memory, so the host, which stays a few iterations
// ahead, needs neither a copy nor an event per iteration to follow.
struct RunStatus {
    long long steps;   // iterations done
    int done;          // 0 running, else the loop's reason to stop
    int spare;
    double value[6];
};

// Device blocks kept between calls for temporaries of setup functions: a hipMalloc and hipFree pair
// takes 30 us at 8 MB and 350 us from 128 MB on, and a free waits for the device. Blocks are handed
// out again without a wait, so one cache serves the work of one stream only (each context has its
// own). At most kCacheBytes are kept; give_back() and the context's end return everything.
class BlockCache {
public:
    static constexpr size_t kCacheBytes = size_t(256) << 20;
    // a block of at least `bytes`; *held: its real size, to be given to put()
    int take(size_t bytes, void **ptr, size_t *held);
    // the block may still be read by work in the stream
    void put(void *ptr, size_t held);
    void give_back();

private:
    struct Block {
        void *ptr;
        size_t bytes;
    };
    std::mutex mu_;
    std::vector<Block> free_;
    size_t kept_ = 0;
};

}  // namespace uhip

// The context: one device, one stream, and the small device workspace every
// reduction writes its per-block partial sums into.
struct uhip_context_s {
    int device = 0;
    hipStream_t stream = nullptr;
    bool own_stream = false;
    int num_cus = 256;
    double *partials = nullptr;     // kMaxDots * max_partials doubles
    int64_t max_partials = 0;       // capacity per dot slot
    int64_t workspace_gen = 0;      // bumped whenever partials is (re)allocated
    const int32_t *gate = nullptr;  // device counter: batched kernels skip their work while it reads 0
    double *dev_scalars = nullptr;  // UHIP_NUM_SCALARS device scalar slots
    double *host_scalars = nullptr; // pinned mirror used for read-back
    double *host_fetch = nullptr;        // pinned targets of the asynchronous read-backs (2 slots)
    hipEvent_t fetch_done[2] = {nullptr, nullptr}; // recorded after each slot's read-back
    unsigned int *counters = nullptr;
    std::mutex ints_mu;             // read_ints: setup functions of several threads
    int32_t *host_ints = nullptr;   // pinned
    static constexpr int kHostInts = 16;
    int autotune_reps = 0;          // > 0: automatic SpMV plans are chosen by timing
    uhip::BlockCache cache;         // temporaries of setup functions, used on `stream` only
    // pinned: what the iterations of a device-paced loop report, a record for each depth of loops that run inside
    // another's iteration (as its preconditioner); the innermost one's is runs[run_depth]
    uhip::RunStatus *runs = nullptr;
    int run_depth = 0;
    static constexpr int kRunRecords = 8;
    // uhip_ctx_defer_sum: the next single dot whose result is wanted at defer_to may stay defer_most partial sums.
    // One that did is `left` of them in `partials`, wanted at left_for, until its consumer takes them or, ahead of
    // whatever else uses the workspace or reads scalars, finish_left.
    const double *defer_to = nullptr;
    int64_t defer_most = 0;
    double *left_for = nullptr;
    int left = 0;
};

namespace uhip {

inline hipStream_t stream_of(uhip_ctx ctx) { return ctx ? ctx->stream : nullptr; }

// Workgroup index remap so that each XCD walks a contiguous slice of the
// logical grid (the hardware hands workgroup b to XCD b % 8). Keeps
// neighbouring rows - and the x entries they share - in one XCD's L2.
__device__ __forceinline__ int xcd_remap(int b, int n) {
    const int xcd = b % kNumXcd;
    const int local = b / kNumXcd;
    const int per = n / kNumXcd;
    const int rem = n % kNumXcd;
    return xcd * per + (xcd < rem ? xcd : rem) + local;
}

// Wavefront (64-lane) sum via cross-lane shuffles.
template <typename T>
__device__ __forceinline__ T wave_sum(T v) {
#pragma unroll
    for (int off = 32; off > 0; off >>= 1) v += __shfl_xor(v, off, 64);
    return v;
}

// Block sum for blockDim.x == BS (multiple of 64); result valid in thread 0.
template <int BS, typename T>
__device__ __forceinline__ T block_sum(T v) {
    __shared__ T red[BS / 64];
    v = wave_sum(v);
    const int lane = threadIdx.x & 63, wid = threadIdx.x >> 6;
    if (lane == 0) red[wid] = v;
    __syncthreads();
    T s = T(0);
    if (threadIdx.x == 0) {
#pragma unroll
        for (int i = 0; i < BS / 64; ++i) s += red[i];
    }
    __syncthreads();
    return s;
}

// K block sums for blockDim.x == BS, the same values in every thread; one pair of barriers for all.
template <int BS, int K>
__device__ __forceinline__ void block_totals(double (&v)[K]) {
    __shared__ double red[K][BS / 64];
#pragma unroll
    for (int k = 0; k < K; ++k) {
        v[k] = wave_sum(v[k]);
        if ((threadIdx.x & 63) == 0) red[k][threadIdx.x >> 6] = v[k];
    }
    __syncthreads();
#pragma unroll
    for (int k = 0; k < K; ++k) {
        v[k] = 0.0;
#pragma unroll
        for (int i = 0; i < BS / 64; ++i) v[k] += red[k][i];
    }
    __syncthreads();
}

// A reduction finished by its consumer: every workgroup of the next kernel adds the producer's n partial
// sums (K dots, the k-th at parts + k * stride) for itself, in a fixed order (a finishing launch of its own
// costs 4 to 5 us of a short iteration). n is 1 where the sums are many and a finishing kernel has
// already run.
template <int BS, int K>
__device__ __forceinline__ void add_partials(const double *parts, int64_t stride, int n, double (&s)[K]) {
    double a[K][4];
#pragma unroll
    for (int k = 0; k < K; ++k)
#pragma unroll
        for (int u = 0; u < 4; ++u) a[k][u] = 0.0;
    int i = (int)threadIdx.x;
    for (; i + 3 * BS < n; i += 4 * BS) {
#pragma unroll
        for (int k = 0; k < K; ++k)
#pragma unroll
            for (int u = 0; u < 4; ++u) a[k][u] += parts[k * stride + i + u * BS];
    }
    for (; i < n; i += BS) {
#pragma unroll
        for (int k = 0; k < K; ++k) a[k][0] += parts[k * stride + i];
    }
#pragma unroll
    for (int k = 0; k < K; ++k) s[k] = (a[k][0] + a[k][1]) + (a[k][2] + a[k][3]);
}
template <int BS, int K>
__device__ __forceinline__ void sum_partials(const double *parts, int64_t stride, int n, double (&s)[K]) {
    add_partials<BS, K>(parts, stride, n, s);
    block_totals<BS, K>(s);
}
// most partial sums that consumers add for themselves in the loops that decide on the device (the MG-CG, whose
// consumers have fewer workgroups, has a line of its own)
constexpr int kConsumerSums = 2048;

inline int grid_for(int64_t n, int per_thread = 4, int cap = 1 << 20) {
    int64_t g = (n + (int64_t)kBlock * per_thread - 1) / ((int64_t)kBlock * per_thread);
    if (g < 1) g = 1;
    if (g > cap) g = cap;
    return (int)g;
}

// Deterministic second stage of all reductions: result[k] = sum_b partials[k*stride + b]
// summed in a fixed order (thread-strided, then a fixed tree); slot k is
// replaced by its square root when bit k of sqrt_mask is set.
int finish_sums(uhip_ctx ctx, int k, int64_t nparts, int64_t stride, double *result_d, unsigned sqrt_mask = 0);
// The same second stage over partial sums held elsewhere than ctx->partials.
int finish_sums_from(uhip_ctx ctx, const double *partials, int k, int64_t nparts, int64_t stride, double *result_d,
                     unsigned sqrt_mask = 0);
// y = A x (FP64, square) with the partial sums of x.y (and, z given, of z.x) left in parts, `cap` entries
// per dot; *count of them are written per dot.
int spmv_dots_into(uhip_ctx ctx, const uhip_csr *A, const double *x, double *y, const double *z, double *parts,
                   int64_t cap, int *count);
// MPRGP's two products (FP64): p.Ap and g.p with A p, g = A x - b with the dots of its state.
// Each leaves `spmv_parts(A)` partial sums per dot at stride cap. The second does nothing unless iteration j
// of the loop takes an expansion step.
struct MprgpScalars {
    double pap, gnorm0;
    long long last;     // the last iteration that counts
    int32_t kind;       // of the iteration in progress: 0 CG, 1 expansion, 2 proportioning step
    int32_t prop[2];    // [j & 1]: iteration j is a proportioning step (p holds beta)
};
int mprgp_product(uhip_ctx ctx, const uhip_csr *A, const double *p, double *Ap, const double *g, double *parts,
                  int64_t cap);
int mprgp_gradient(uhip_ctx ctx, const uhip_csr *A, const double *x, double *g, const double *b, const double *lb,
                   const double *ub, const MprgpScalars *s, long long j, double *parts, int64_t cap);

// MPRGP::get_fi and get_beta (utopia_MPRGP.hpp:266-287, 324-348)
__device__ __forceinline__ double free_grad(double x, double g, double l, double u) {
    return (l < x && x < u) ? g : 0.0;
}
__device__ __forceinline__ double chopped_grad(double x, double g, double l, double u) {
    return (fabs(l - x) < 1e-14) ? fmin(0.0, g) : ((fabs(u - x) < 1e-14) ? fmax(0.0, g) : 0.0);
}

// Partial sums of an SpMV launch on A.
inline int64_t spmv_parts(const uhip_csr *A) { return A->format == UHIP_FMT_ROWBLOCK ? A->nblocks : A->nparts; }
// The record of the loop that runs on the context, and one of its own for a loop while the scope lives.
inline RunStatus *run_record(uhip_ctx ctx) { return ctx->runs + ctx->run_depth; }
class RunScope {
public:
    explicit RunScope(uhip_ctx ctx) : ctx_(ctx), st_(uhip_ctx_enter_loop(ctx)) {}
    ~RunScope() {
        if (st_ == UHIP_OK) uhip_ctx_leave_loop(ctx_);
    }
    RunScope(const RunScope &) = delete;
    RunScope &operator=(const RunScope &) = delete;
    int status() const { return st_; }

private:
    uhip_ctx ctx_;
    int st_;
};
// Wait until the loop that reports to run_record(ctx) has done `steps` iterations or has stopped. Ends also
// when the stream has run out of work or failed (an error then).
int run_wait(uhip_ctx ctx, long long steps);
// Device address of the SpMV library's file-scope partial-sum scratch on `device` (the device
// must be current): looked up once per device at context creation.
int spmv_scratch_init(int device);

// Temporaries of one call, carved out of one block of the context's cache: sizes first (add), then
// allocate(), then the pointers. The block goes back when the object ends; work in the stream may still
// read it then.
class Scratch {
public:
    explicit Scratch(uhip_ctx ctx) : ctx_(ctx) {}
    ~Scratch() {
        if (base_) ctx_->cache.put(base_, held_);
    }
    Scratch(const Scratch &) = delete;
    Scratch &operator=(const Scratch &) = delete;
    size_t add(size_t bytes) {
        const size_t at = size_;
        size_ += (bytes + 255) & ~(size_t)255;
        return at;
    }
    int allocate() { return ctx_->cache.take(size_, &base_, &held_); }
    template <typename T>
    T *at(size_t offset) const {
        return (T *)((char *)base_ + offset);
    }

private:
    uhip_ctx ctx_;
    void *base_ = nullptr;
    size_t size_ = 0, held_ = 0;
};

// n int32 of device memory (n <= kHostInts) read through a pinned buffer of the context that serves nothing else,
// one thread at a time; waits for the stream.
int read_ints(uhip_ctx ctx, const int32_t *src_d, int n, int32_t *dst_h);

// A dot left as partial sums is finished (nothing where there is none).
int finish_left(uhip_ctx ctx);

// Ahead of every use of ctx->partials: a dot left there is finished, and the per-slot capacity grows to at
// least per_slot entries.
int ensure_partials(uhip_ctx ctx, int64_t per_slot);

}  // namespace uhip
