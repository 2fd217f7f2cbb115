// Internal helpers shared by every translation unit of libdopthip.so.
#pragma once

#include <hip/hip_runtime.h>

#include <cstdarg>
#include <cstddef>
#include <cstdint>
#include <cstdio>
#include <memory>
#include <string>
#include <vector>

#include "../../include/dopt_hip.h"

namespace dopt {

// Records the message returned by dopt_hip_last_error() and hands back `code`.
int fail(int code, const char *fmt, ...) __attribute__((format(printf, 2, 3)));
void clear_error();

// The library stream (created by dopt_hip_init; lazily initialises device 0 otherwise).
hipStream_t stream();
bool ensure_init();
bool is_initialised();   // dopt_hip_init (or a lazily initialising entry point) has run

// Process-wide scratch memory, grown on demand (the analogue of the single conv workspace at
// cuda/nnet/cudnn7.d:111).  Valid until the next call that asks for more; all users enqueue on
// the one library stream, so consecutive users never overlap.
void *workspace(size_t bytes);
// The same for callers that can do without: null, with no error recorded, where partial sums are parked in it (open_split_set) or
// it would have to grow while a graph is recorded.
void *workspace_if_free(size_t bytes);
// Changes whenever a workspace is reallocated (its address may have changed): whoever keeps the
// address beyond one call -- a recorded HIP graph -- compares generations before using it again.
unsigned long workspace_generation();
// A convolution that leaves its result open parks partial sums in the workspace until the next call adds
// them up; until open_split_clear, any other request for the workspace fails instead of overwriting them.
void open_split_set(const void *partial);
void open_split_clear(const void *partial);
// The library owns two in-order queues.  Everything enqueues on the main one unless a plan has
// switched to the side queue for a step it overlaps with its main chain (set_lane(1) ... set_lane(0));
// each queue has its own workspace.
void set_lane(int lane);
// While a plan records its kernels into a HIP graph, entry points that would allocate (from the
// driver or from the pool), fill device memory or grow the workspace fail instead (none of these can
// be replayed), and the plan runs its kernels directly.
void set_capturing(bool on);
bool capturing();
int scratch_alloc(void **ptr, size_t bytes);   // pooled block, NOT zero-filled; release with dopt_hip_free
// sgemm.hip: C = op(A) * op(B) (+ colbias[col >> bias_shift] per element when colbias is given and the
// shape takes a kernel with that epilogue; *biased says whether it did).
int sgemm_bias(int transA, int transB, size_t M, size_t N, size_t K, const float *A, const float *B, float *C,
               const float *colbias, int bias_shift, bool *biased);
// sgemm.hip: dopt_hip_sgemm_t, _rank1, _relu_grad, _batch and _order.  `written`, as a plan calls them: the reduction is cut the same
// however the operands are stored, so a product that reads a transposed matrix in place gives the bits of the product of its copy.
// Else it is cut as suits the storage ([52 x 2052] from 4403 steps, both operands across, 24 us; cut as the product of copies 31).
int product(bool written, int transA, int transB, size_t M, size_t N, size_t K, const float *A, const float *B, float *C);
int product_rank1(bool written, int transA, int transB, size_t M, size_t N, size_t K, const float *A, const float *B, const float *u, const float *v, int relu,
                  float *C);
int product_relu_grad(bool written, int transA, int transB, size_t M, size_t N, size_t K, const float *A, const float *B, const float *x, float *C);
int product_batch(bool written, int n, const int *transA, const int *transB, const size_t *M, const size_t *N, const size_t *K, const float *const *A,
                  const float *const *B, float *const *C);
uint64_t product_order(bool written, int transA, int transB, size_t M, size_t N, size_t K);
// sgemm.hip: dw[K][C][3][3] = filter gradient of a 3x3, pad-1 convolution over 2x2 images, from x[N][4C]
// and dy[N][4K] in one launch.  Returns false, with nothing launched, for shapes it does not take.
bool sgemm_fold2x2(size_t C, size_t K, size_t N, const float *x, const float *dy, float *dw, int *rc);
// The same for up to 8 layers in one launch; false, with nothing launched, unless every layer suits that kernel.
bool sgemm_fold2x2_batch(int n, const size_t *C, const size_t *K, const size_t *N, const float *const *x,
                         const float *const *dy, float *const *dw, int *rc);
// bn.hip: batchNormInference of [N, C, H, W] with what surrounds it in one launch: its operand x may be an open convolution
// result (`open`, value == x), relu != 0 clamps, `pooled` (or null) receives the 2 x 2 max-pool.  y receives the (clamped) value;
// with keep_y == 0 it is scratch that only the pool reads.
int bn_infer_fused(size_t N, size_t C, size_t H, size_t W, const float *x, const dopt_hip_split_sum *open, const float *scale, const float *bias,
                   const float *mean, const float *var, int relu, float *y, int keep_y, float *pooled);
// conv_smallc.hip: 3x3 pad-1 unit-stride convolutions over at most three input channels.  `done`
// stays false when the shape is not theirs (the caller then uses the general kernels).
bool conv_smallc_takes(const dopt_hip_conv_desc *d);
int conv_smallc_fwd(const dopt_hip_conv_desc *d, const float *x, const float *w, const float *bias, float *y, bool *done);
int conv_smallc_wgrad(const dopt_hip_conv_desc *d, const float *dy, const float *x, float *dw, bool *done);
// nn.hip: out[c] = sum_{n,i} in[n][c][i] in one launch; false, with nothing launched, for shapes it does not take.
bool channel_sum(size_t N, size_t C, size_t inner, const float *in, float *out, int *rc);
hipStream_t lane_stream(int lane);
// bn.hip: error report of the multi-block batch-norm kernels; call with the queues idle.
int bn_cluster_poll();
// bn.hip: how many such kernels have been enqueued so far (a plan samples it around a recording to learn whether the
// recording holds one), and the note a replay of such a recording leaves for the next synchronisation point.
unsigned long bn_cluster_launches();
void bn_cluster_mark_unchecked();
bool bn_cluster_pending();
// Per-device set-up done inside dopt_hip_init, with the device current: addresses of the file-scope device arrays
// (bn.hip: the records blocks of a channel exchange, filled with "absent"; nn.hip: the scratch of
// dopt_hip_bias_bwd_noalloc), so that no later call has to load a code object, fill memory or wait for the device.
int bn_device_setup();
int nn_device_setup();

// Number of compute units of the active device (256 on MI355X); used to size grids.
int num_cus();

// Workgroups of 256 threads that a launch of ours is given at most (a launch takes fewer than 2^32 threads along a dimension).
constexpr size_t kLaunchBlocks = (size_t)1 << 22;
inline size_t ceil_div(size_t a, size_t b) { return (a + b - 1) / b; }
inline bool aligned16(const void *p) { return (reinterpret_cast<uintptr_t>(p) & 15u) == 0; }

// rtc_ops.cpp: the same pointwise program over many tensors as one launch (more, when their addresses do not fit a launch's
// arguments).  Operand k < kind.size() of a node is input k - kind 0 an n-element tensor, 1 one element - and operand
// kind.size() + j is node j; `outs` are the nodes that are stored, each to a buffer of its own.  Every node rounds by itself, as
// the kernel of its operation does.
struct PointwiseProgram {
    std::vector<unsigned char> kind;
    struct Node { std::string op; int lhs, rhs; };
    std::vector<Node> nodes;
    std::vector<int> outs;
};
struct PointwiseItem {
    size_t n;
    std::vector<const void *> in;   // one per input of the program
    std::vector<void *> out;
};
constexpr int kGroupInputs = 48, kGroupNodes = 64, kGroupOuts = 8;
int pointwise_group(const PointwiseProgram &program, const std::vector<PointwiseItem> &items);

// rtc_ops.cpp: out[i] = the sum of the squares of the n[i] (more than 64) values at in[i], each the value that
// dopt_hip_reduce_squares gives.
int reduce_squares_batch(int count, const float *const *in, const size_t *n, float *const *out);

// tiny_rtc.cpp: a run of operations on tiny tensors (dopt_hip_tiny_graph's nodes) as a kernel of its own, compiled when it is first
// launched.  The results' buffers must overlap neither each other nor what is read from outside: a plan's own do not, and a plan
// that is given an argument in one of them (HIPPlan::mInOrder) does not call this.  `done` stays false, with nothing launched, for
// runs it does not take and where the kernel cannot be compiled or loaded (which is tried once): those are dopt_hip_tiny_graph's.
struct TinyRun {
    TinyRun(int nslots, const std::vector<dopt_hip_tiny_node> &nodes);
    ~TinyRun();
    TinyRun(const TinyRun &) = delete;
    TinyRun &operator=(const TinyRun &) = delete;
    int launch(void *const *slots, bool *done) const;
    struct Code;   // shared by the runs with one source

private:
    int compile() const;
    int slots, threads = 0;
    mutable bool refused = false;
    mutable std::shared_ptr<Code> code;
    std::string source;
};
void tiny_codes_trim();       // unloads the code of runs that are gone
void tiny_codes_shutdown();   // unloads all of it, with the queues idle; runs that are left compile theirs again

// hipRTC: compile `source`, load it and find the named kernels in it; wait for all that is queued; unload.
int rtc_load(const std::string &source, int n, const char *const *names, hipModule_t *module, hipFunction_t *fns);
void rtc_idle();
void rtc_unload(hipModule_t module);
// The same once per distinct `key`, for the life of the library.
int rtc_get(const std::string &key, const std::string &source, const char *kernel_name, hipFunction_t *fn);
// ... and several kernels of one source (under key:name), which is compiled once for all of them.
int rtc_get_all(const std::string &key, const std::string &source, int n, const char *const *names, hipFunction_t *fns);
bool rtc_find(const std::string &key, hipFunction_t *fn);   // a kernel compiled before (its source need not be put together again)
int rtc_compile_only(const std::string &source, const char *arch, std::string *log);
int rtc_launch(hipFunction_t fn, unsigned grid, unsigned block, void **args);

}  // namespace dopt

#define DOPT_HIP_CHECK(expr)                                                                       \
    do {                                                                                           \
        hipError_t e_ = (expr);                                                                    \
        if (e_ != hipSuccess)                                                                      \
            return ::dopt::fail(DOPT_HIP_ERR_RUNTIME, "%s:%d: %s failed: %s", __FILE__, __LINE__,  \
                                #expr, hipGetErrorString(e_));                                     \
    } while (0)

#define DOPT_LAUNCH_CHECK()                                                                        \
    do {                                                                                           \
        hipError_t e_ = hipGetLastError();                                                         \
        if (e_ != hipSuccess)                                                                      \
            return ::dopt::fail(DOPT_HIP_ERR_RUNTIME, "%s:%d: kernel launch failed: %s", __FILE__, \
                                __LINE__, hipGetErrorString(e_));                                  \
    } while (0)

#define DOPT_REQUIRE(cond, ...)                                                                    \
    do {                                                                                           \
        if (!(cond)) return ::dopt::fail(DOPT_HIP_ERR_INVALID, __VA_ARGS__);                       \
    } while (0)

#define DOPT_ENSURE_INIT()                                                                         \
    do {                                                                                           \
        if (!::dopt::ensure_init()) return DOPT_HIP_ERR_RUNTIME;                                   \
    } while (0)
