// Shared declarations of the gfx950 backward-pass library: error plumbing, scalar device
// functions with the reference's exact clamping rules, and the internal kernel launch API.
#pragma once

#include <hip/hip_runtime.h>

#include <cstdarg>
#include <cstdint>
#include <cstdio>
#include <functional>

#include "../../include/currennt_hip.h"

namespace cnt {

// ----- error plumbing: nothing throws across the C ABI ------------------------------------------
void set_error(const char *fmt, ...);
const char *last_error();

#define CNT_HIP(expr)                                                                        \
    do {                                                                                     \
        hipError_t _e = (expr);                                                              \
        if (_e != hipSuccess) {                                                              \
            ::cnt::set_error("%s failed: %s (%s:%d)", #expr, hipGetErrorString(_e), __FILE__, \
                             __LINE__);                                                      \
            return CNT_ERR_HIP;                                                              \
        }                                                                                    \
    } while (0)

#define CNT_REQUIRE(cond, ...)           \
    do {                                 \
        if (!(cond)) {                   \
            ::cnt::set_error(__VA_ARGS__); \
            return CNT_ERR_ARG;          \
        }                                \
    } while (0)

#define CNT_TRY(expr)            \
    do {                         \
        int _s = (expr);         \
        if (_s != CNT_OK) return _s; \
    } while (0)

// ----- scalar semantics ---------------------------------------------------------------------------
// Reference: activation_functions/{Logistic,Maxmin1,Tanh}.cuh, helpers/{limitedError,safeExp,
// NumericLimits}.cuh.  tanh is 2*logistic(2x)-1 and the logistic saturates outside +-88.722839.
namespace lim {
constexpr float kMin = 1.1754944e-038f;
constexpr float kMax = 3.4028235e+038f;
constexpr float kExpLimit = 88.722839f;
constexpr float kLogZero = -1e30f;
constexpr float kLSmall = -0.5e10f;
constexpr float kMinLarg = 1.1754944e-038f;
constexpr float kMinLogExp = -69.0776f;
}  // namespace lim

// 1 / (1 + exp(m)), m * log2(e) given as the sum of m * hi and m * lo (argument reduction by log2(e) as a float and its
// remainder, one Newton step for the quotient): exp2 of the hardware over [-1/2, 1/2], the integer
// part (the low bits of t, which has 1.5 * 2^23 added) put into the exponent, and a reciprocal with one Newton step that
// also takes in what 1 + e rounds away (REST): fourteen instructions with the clamp, eleven without REST.  expf and an fp32
// quotient take about forty (denormal results, exact rounding).  Against double precision over every float between 3e-8 and 87 of
// both signs: largest error 2.62 ulp with REST and without it (expf and quotient: 2.62), root mean square 0.34 and 0.56 (0.56); of
// the tanh functions 0.97e-7 and 1.79e-7 absolute (1.79e-7).  The callers clamp m * log2(e) to
// [-126, 128), which needs no branch and no select: a NaN becomes the lower limit, which gives 1 as it always did.
// Results below 1.2e-38 are zero.
template <bool REST>
__device__ __forceinline__ float logistic_of_negative(float m, float hi, float lo) {
    const float t = __builtin_fmaf(m, hi, 12582912.0f);
    const float p = __builtin_amdgcn_exp2f(__builtin_fmaf(m, lo, __builtin_fmaf(m, hi, -(t - 12582912.0f))));
    const float e = __uint_as_float(__float_as_uint(p) + (__float_as_uint(t) << 23));
    const float d = 1.0f + e, rest = e - (d - 1.0f);  // 1 + e = d + rest
    const float y = __builtin_amdgcn_rcpf(d), left = __builtin_fmaf(-d, y, 1.0f);
    return __builtin_fmaf(REST ? __builtin_fmaf(-rest, y, left) : left, y, y);
}
template <bool REST = true>
__device__ __forceinline__ float logistic(float x) {
    return logistic_of_negative<REST>(__builtin_amdgcn_fmed3f(-x, -87.3f, 88.72283f), 1.44269504088896341f, 1.92596303e-8f);
}
template <bool REST = true>
__device__ __forceinline__ float tanh_act(float x) {
    return 2.0f * logistic_of_negative<REST>(__builtin_amdgcn_fmed3f(-x, -43.65f, 44.361415f), 2.88539008177792681f, 3.85192606e-8f) - 1.0f;
}
// The same functions in the form of eleven instructions, for the forward recursion, where the five of them per cell and time step
// sit on the critical path of every step: an utterance of 800 steps through two layers of 512 cells 2074 us (2115 with REST), a
// pass of the acoustic model 3790 us (3787).
__device__ __forceinline__ float logistic_quick(float x) { return logistic<false>(x); }
__device__ __forceinline__ float tanh_quick(float x) { return tanh_act<false>(x); }
__device__ __forceinline__ float logistic_deriv(float y) { return y * (1.0f - y); }
__device__ __forceinline__ float tanh_deriv(float y) { return 1.0f - y * y; }
__device__ __forceinline__ float clip1(float e) { return e < -1.0f ? -1.0f : (e > 1.0f ? 1.0f : e); }
__device__ __forceinline__ float safe_exp(float x) {
    if (x <= lim::kLogZero) return 0.0f;
    if (x >= lim::kExpLimit) return lim::kMax;
    return expf(x);
}
__device__ __forceinline__ float safe_log(float x) { return x < lim::kMinLarg ? lim::kLogZero : logf(x); }
__device__ __forceinline__ float log_add(float x, float y) {
    const float hi = x > y ? x : y;
    const float lo = x > y ? y : x;
    if ((lo - hi) < lim::kMinLogExp) return hi < lim::kLSmall ? lim::kLogZero : hi;
    return (float)((double)hi + log(1.0 + (double)expf(lo - hi)));
}

enum Act { ACT_IDENTITY = 0, ACT_TANH = 1, ACT_LOGISTIC = 2, ACT_RELU = 3 };
__device__ __forceinline__ float act_fn(int act, float a) {
    switch (act) {
        case ACT_TANH: return tanh_act(a);
        case ACT_LOGISTIC: return logistic(a);
        case ACT_RELU: return a > 0.0f ? a : 0.0f;
        default: return a;
    }
}
__device__ __forceinline__ float act_deriv(int act, float y) {
    switch (act) {
        case ACT_TANH: return tanh_deriv(y);
        case ACT_LOGISTIC: return logistic_deriv(y);
        case ACT_RELU: return y > 0.0f ? 1.0f : 0.0f;
        default: return 1.0f;
    }
}

// ----- sum of a call's errors ---------------------------------------------------------------------
__device__ __forceinline__ double wave_sum_64(double v) {
    for (int o = 32; o > 0; o >>= 1) v += __shfl_xor(v, o);
    return v;
}

// Sum of the errors of a call, over the workgroups of all its units' launches.  It is formed in 64 bits: workgroups add in the
// order they finish in, and in 32 bits the last digits follow that order (over the same probabilities the error of 31 000 frames,
// 2.2e5, came out up to 0.36 apart).  The values added have 24 binary digits each, so their 64-bit sum
// is exact, or as good as, in any order.
// The workgroup that finishes last hands the sum to the caller and leaves accumulator and ticket counter at zero for the next
// call, so that no launch has to clear the caller's result first.
struct LossSum {
    double *acc;
    unsigned *ticket;     // workgroups that have added so far
    unsigned workgroups;  // of the call
    float *result;
};

// by one thread of a workgroup, once
__device__ __forceinline__ void add_loss(const LossSum &s, double v) {
    // No fence (a device-scope fence writes the L2 back, which costs more than the kernel): the ticket is taken
    // only after the add has returned its old value, i.e. has been performed where every XCD's atomics meet.
    const double before = __hip_atomic_fetch_add(s.acc, v, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    unsigned one = 1u;
    asm volatile("" : "+v"(one) : "v"(before));  // the ticket's operand depends on the returned value
    if (__hip_atomic_fetch_add(s.ticket, one, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) == s.workgroups - 1u) {
        *s.result = (float)__hip_atomic_exchange(s.acc, 0.0, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        __hip_atomic_store(s.ticket, 0u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    }
}

// every wave's value to the call's sum; all threads of the workgroup take part
template <int WAVES>
__device__ __forceinline__ void add_block_loss(const LossSum &s, double wave_total) {
    __shared__ double block_sum[WAVES];
    if ((threadIdx.x & 63) == 0) block_sum[threadIdx.x >> 6] = wave_total;
    __syncthreads();
    if (threadIdx.x == 0) {
        double v = 0.0;
#pragma unroll
        for (int w = 0; w < WAVES; ++w) v += block_sum[w];
        add_loss(s, v);
    }
}

// ----- optional per-kernel timing (capi.hip) -------------------------------------------------------
// When enabled through cnt_profile_enable, every ProfileScope brackets the launches made inside it
// with a pair of HIP events on the launch stream; cnt_profile_get sums them per label.
struct ProfileScope {
    ProfileScope(hipStream_t stream, const char *label);
    ~ProfileScope();
    hipStream_t stream_;
    int slot_;
};

// ----- GEMM (gemm.hip) ------------------------------------------------------------------------------
// C (m x n, column-major, ldc) = sum over segments of opA(A_i) * opB(B_i), optionally added to C.
// An operand is described by where element (row, kk) lives: row-contiguous (ptr[kk*ld + row]) or
// k-contiguous (ptr[row*ld + kk]).
constexpr int kGemmMaxSeg = 8;
constexpr int kGemmMaxProb = 8;

enum GemmEpilogue {
    EPI_STORE = 0,          // C = acc
    EPI_ADD = 1,            // C += acc
    EPI_ATOMIC = 2,         // atomicAdd(C, acc)   (split-K; C zeroed by the caller)
    EPI_BIAS_ACT = 3,       // C = act(acc + bias_scale * bias_vec[row])
    EPI_BIAS_ACT_SKIP = 4,  // as above, but columns whose pattern type is "none" are left untouched
    EPI_CONTEXT = 5,        // th = tanh(acc); aux_out = th; C = aux_in + th; both 0 on "none" columns
    EPI_PARTIAL = 6,        // split-K without atomics: every split stores its m x n partial product into the
                            // launcher's scratch, and a second kernel sums the splits into C (set by gemm_plan)
    EPI_STORE_DELTA = 8,    // C = acc * act'(aux_in): the product that writes a dense layer's output errors turns them
                            // into that layer's deltas on the way out (aux_in = the layer's outputs, layout of C)
    EPI_FAN = 7             // a skip layer's backward step in the epilogue of the product that writes the layer's
                            // errors: e = aux_in + acc (aux_in may be NULL), C = e, and e goes on to fan_n buffers of
                            // C's layout -- added to those flagged in fan_is_skip, stored over the others
};

struct GemmProblem {
    const float *A[kGemmMaxSeg];
    const float *B[kGemmMaxSeg];
    int b_shift[kGemmMaxSeg];  // masked mode: time-slot shift of the B operand per operand pair
    float *C;
    const float *bias_vec;
    const float *aux_in;  // EPI_CONTEXT, EPI_STORE_DELTA: same layout as C
    float *aux_out;       // EPI_CONTEXT, may be NULL
    float *rowsum_out;    // GemmArgs::rowsum: receives rowsum_scale * sum_k B(j, k), j < n
    float rowsum_scale;
    int k_trim;           // GemmArgs::k_order: 0 all listed k lines, 1 without those of the first time step, 2 without the last one's
    int k_shift;          // GemmArgs::k_order: added to every listed line (an operand pair that starts at a later slot)
};

// The slots of a fraction in the order "valid ones first, ascending; then the padding slots, ascending" (device
// memory: n_slots indices and three counts), made from the pattern types by slot_order_build.  The errors
// and deltas of every layer are zero on padding slots, so a sum over the slots may skip them.
struct SlotOrder {
    const int *order;
    const int *count;  // [0] valid slots, [1] those of the first time step, [2] those of the last time step
};
int slot_order_build(hipStream_t stream, const char *pat, int n_slots, int slots_per_step, int *order, int *count);

// Masked mode (dilated convolutions without a materialised column buffer): one index of the B operand is a
// time slot u -- its row index (b_time_on_k = 0) or its k index (b_time_on_k = 1).  The element is read from
// slot u + b_shift and counts only if pat[u] != 0, 0 <= u + b_shift < n_slots and pat[u + b_shift] != 0;
// otherwise it is 0.  This is exactly the set of entries the reference scatters into its column buffer
// (layers/CNNLayer.cu:182-237).
struct GemmArgs {
    int m, n, k;
    int lda, ldb, ldc;
    int a_kcontig, b_kcontig;  // 1: element (row,kk) at ptr[row*ld+kk]; 0: ptr[kk*ld+row]
    int nseg, nprob, splitk;
    int epilogue, act;
    float bias_scale;
    int masked, b_time_on_k, n_slots;
    const char *pat;  // masked mode and the *_SKIP / CONTEXT epilogues
    GemmProblem prob[kGemmMaxProb];
    const char *label;  // name under which the launch is timed when profiling is on (may be NULL)
    // Split-K products (EPI_ATOMIC, splitk = 0): `overwrite_ok` allows gemm_plan to choose EPI_PARTIAL, or EPI_STORE for a single
    // split, which overwrite C instead of adding to a cleared C.  With `rowsum` (one operand pair, unmasked)
    // the same pass also sums every problem's B operand over k into that problem's rowsum_out -- the bias gradient
    // of a dense layer; with EPI_ATOMIC it adds to what the caller has cleared.  gemm_plan clears `rowsum` where the
    // product cannot bring it along (operands that are not row-contiguous, several pairs).
    int overwrite_ok;
    int rowsum;
    int fan_n;                   // EPI_FAN: device tables of fan_n targets and their flags
    float *const *fan_targets;
    const int *fan_is_skip;
    // Columns of the output that may be left out (k-contiguous B, EPI_STORE and EPI_STORE_DELTA, one k range): column j of the product
    // is column cols[j] of B and C, and from cols_count[0] on the columns get zeros, which is what their products come to
    // (SlotOrder: the slots of a fraction, those of its padding behind the others).  The kernel for few blocks has no use for the list:
    // gemm_launch takes it away.
    const int *cols;
    const int *cols_count;
    float *partial;        // scratch of splitk * partial_stride floats: the stream's buffer (set by gemm_plan) or the caller's
    size_t partial_stride;  // floats per split: nprob * m * n (+ nprob * n with rowsum), rounded up to a multiple of four
    int xcd_map;            // set by gemm_launch: workgroups pick their tile by XCD (gemm_kernel.hpp)
    // A product over the slots of a fraction (weight gradients) that leaves the padding slots out (both in device memory,
    // or both NULL): only the k lines k_order[lo .. lo + n) of the operands are read, the others being all zero in at least
    // one operand.  k_count[0] = number of listed lines; with GemmProblem::k_trim = 1 the problem leaves out the first
    // k_count[1] of them (the lines of the first time step), with 2 the last k_count[2] (those of the last time step).  The
    // launcher uses the list where both operands are row-contiguous and 16-byte aligned, and
    // multiplies all k lines otherwise -- so the operands' base pointers must be valid for both readings.
    const int *k_order;
    const int *k_count;
};

// Resolves splitk = 0 (chosen by the launcher) and, where the arguments allow it, switches an
// EPI_ATOMIC product to EPI_PARTIAL or EPI_STORE.  A caller that needs to know whether C must be cleared first calls this
// before gemm_launch and looks at args.epilogue; gemm_launch calls it for everyone else.
void gemm_plan(GemmArgs &args, hipStream_t stream);
// The kernel for products that are too small for the tiled one (gemm_direct.hip): whether these arguments take it (masked
// products never do), and its launch
bool direct_product(const GemmArgs &args);
void gemm_direct_launch(const GemmArgs &args, hipStream_t stream);
// Weight gradients of few blocks, of any sizes, as one launch: the products of a small pass, whose results nothing but the optimizer
// waits for, and the two of a recurrent layer.  All through one list of k lines, or all without.  Their operands have to stay as they
// are until the launch.
constexpr int kGroupProducts = 32;
struct DirectProduct {
    const float *A[1], *B[1];
    float *C, *rowsum_out;
    int m, n, k, lda, ldb, ldc;
    float rowsum_scale;
    int rowsum, k_trim, k_shift;
};
struct DirectGroup {
    int count, blocks;
    const int *k_order, *k_count;
    int first[kGroupProducts];  // block of the launch at which a product begins
    DirectProduct product[kGroupProducts];
};
int gemm_group_add(hipStream_t stream, DirectGroup &group, const GemmArgs &planned);
int gemm_group_launch(hipStream_t stream, DirectGroup &group);
// whether a product with these operands can take the EPI_FAN epilogue (operand kinds, alignment)
bool gemm_fan_supported(const GemmArgs &args);
// group: a weight gradient that takes the few-block kernel waits there for others of its kind, until gemm_group_launch
int gemm_launch(hipStream_t stream, const GemmArgs &args, DirectGroup *group = nullptr);
// Frees the split-K scratch buffer that the launcher keeps for `stream` (for owners of a stream about to destroy
// it; the stream must be idle).  Buffers of streams never released stay until the process ends.
void gemm_release_stream(hipStream_t stream);
// Allocates the split-K scratch buffer of `stream` now instead of inside the first product that wants it.
int gemm_reserve_stream(hipStream_t stream);
// Sum over `count` parts, `stride` floats apart, of output e < total, by a workgroup of 256 for 32 consecutive outputs: the parts are
// dealt to eight groups of 32 threads whose sums meet in LDS, four loads in flight per thread.  The first 32 threads have the sums.
constexpr int kPartOutputs = 32;
__device__ __forceinline__ float sum_of_parts(const float *__restrict__ parts, size_t e, size_t total, int count, size_t stride) {
    constexpr int G = 256 / kPartOutputs;
    __shared__ float part[G][kPartOutputs];
    const int tx = threadIdx.x % kPartOutputs, g = threadIdx.x / kPartOutputs;
    float a0 = 0.0f, a1 = 0.0f, a2 = 0.0f, a3 = 0.0f;
    if (e < total) {
        const float *__restrict__ p = parts + e;
        int s = g;
        for (; s + 3 * G < count; s += 4 * G) {
            const float x0 = p[(size_t)s * stride], x1 = p[(size_t)(s + G) * stride];
            const float x2 = p[(size_t)(s + 2 * G) * stride], x3 = p[(size_t)(s + 3 * G) * stride];
            a0 += x0; a1 += x1; a2 += x2; a3 += x3;
        }
        for (; s < count; s += G) a0 += p[(size_t)s * stride];
    }
    part[g][tx] = (a0 + a1) + (a2 + a3);
    __syncthreads();
    float v = 0.0f;
    if (g == 0)
#pragma unroll
        for (int q = 0; q < G; ++q) v += part[q][tx];
    return v;
}
// Launches by other files whose parts meet in the stream's split-K scratch: calls `enqueue` with the buffer, and no product of the
// stream comes between what it launches.  false: no buffer of that size (as for gemm_plan), nothing was called.
constexpr size_t kSplitScratchFloats = (size_t)9 << 20;  // 36 MB per (device, stream)
bool with_split_scratch(hipStream_t stream, size_t floats, const std::function<void(float *)> &enqueue);
// While it lives, everything that this thread enqueues on `stream` and that would take the stream's split-K scratch takes `buffer` instead
// (kSplitScratchFloats floats, or null: nothing changes).  For a handle whose products run on a stream of the caller's, which it
// can neither reserve nor release: the buffer is the handle's, also in a graph that is captured meanwhile.
class ScratchLoan {
public:
    ScratchLoan(hipStream_t stream, float *buffer);
    ~ScratchLoan();
    ScratchLoan(const ScratchLoan &) = delete;
    ScratchLoan &operator=(const ScratchLoan &) = delete;

private:
    hipStream_t outer_stream_;
    float *outer_buffer_;
};
// number of split-K scratch buffers the library holds at the moment (one per stream that has needed or reserved one)
int gemm_scratch_buffers();
// cnt_dense_backward_weights with the partial products in a scratch array that is part of the code object
int gemm_dense_weights_static(hipStream_t stream, int P, int D, int N, float bias, const float *x, const float *err,
                              float *weight_updates);

// Convenience: single problem, BLAS-like transposes on column-major matrices.
int gemm_simple(hipStream_t stream, float *C, int m, int n, int k, const float *A, bool transA,
                const float *B, bool transB, bool accumulate);

// cnt_opt_step with a device flag in front of it: when *veto is non-zero at the time the kernel runs (a recursion of
// the pass that produced the gradients gave up), the step changes nothing.
int opt_step_guarded(hipStream_t stream, int option, long n, float *weights, const float *layer_updates, float *cur_updates,
                     float *stats, float *weight_deltas, const float *mask, float frac_length, float beta1_accum,
                     float beta2_accum, float learning_rate, float momentum, const int *veto, const float *accum_dev);
// Adam's bias-correction products (two floats in device memory, both 1 before the first step) advanced by one step,
// unless *veto is non-zero; opt_step_guarded reads them in place of its two float arguments when accum_dev is given.
int opt_adam_advance(hipStream_t stream, float *accum_dev, const int *veto);
// LSTM handles of a network share one such flag: a recursion that gives up also sets *veto (until the owner clears it).
void lstm_set_veto(cnt_lstm *h, int *veto);
// cnt_lstm_backward_weights; sums_done: the error half was lstm_backward_errors_sums.  group: products of few blocks wait there.
int lstm_backward_weights_grouped(cnt_lstm *h, hipStream_t stream, const float *x, float *weight_updates, bool sums_done,
                                  DirectGroup *group = nullptr);
// cnt_lstm_backward_errors whose recursion also sums up the bias and peephole gradients
int lstm_backward_errors_sums(cnt_lstm *h, hipStream_t stream, const float *weights, float *output_errors, float *prev_errors,
                              float *weight_updates);
// non-zero if a recursion of this handle has given up since the last report (no synchronisation: it only sees
// launches that have already ended); the report clears the mark
int lstm_take_failure(cnt_lstm *h);
// makes `other` wait for the recursion launched last on this handle's device (the event the library records behind
// every recursion launch anyway): what a stream needs that consumes the recursion's results, without another event
// record on the launching stream
int lstm_wait_recursion(cnt_lstm *h, hipStream_t other);
int lstm_is_persistent(const cnt_lstm *h);  // its recursions are launches behind which lstm_wait_recursion finds an event
int report_failure(cnt_network *net, hipStream_t stream);

// ----- error halves that also do the backward step of the skip layer in front of them ----------------
// A skip layer adds what its linkers left in its side buffer to the errors its following layer wrote, and hands the
// sum on (layers/SkipAddLayer.cu:305-346).  When that following layer is a dense or convolution layer, the sum and
// the hand-over happen in the epilogue of the product that computes those errors, instead of in a launch of their
// own.  `targets` / `is_skip` are device tables of `n` entries; `from_skip` is the side buffer or NULL.
struct FanOut {
    int n;
    float *const *targets;
    const int *is_skip;
    const float *from_skip;
};
// *fused tells whether the step was done (operands that the fan epilogue does not exist for, or a convolution
// with several filter groups, leave it to the caller).
int dense_backward_errors_fan(hipStream_t stream, int P, int D, int N, int act, const float *weights, const float *y,
                              float *err, float *prev_err, const FanOut *fan, bool *fused, int prev_act = ACT_IDENTITY,
                              const float *prev_y = nullptr, const SlotOrder *order = nullptr);
// (prev_act, prev_y): the preceding layer is a dense layer with that activation and those outputs, and nothing but
// this product writes its output errors: the product stores act'(prev_y) * error, the preceding layer's deltas, and
// that layer's own backward step then runs with ACT_IDENTITY.  The same for a recurrent layer's error product:
int lstm_prev_errors_delta(cnt_lstm *h, hipStream_t stream, const float *weights, float *prev_errors, int prev_act,
                           const float *prev_y);
// The slots of the fraction a recurrent layer has loaded, valid ones first (nullptr: none known); the layer's weight
// gradients then skip the padding slots.  cnt_lstm_load_sequences forgets it.
void lstm_set_slot_order(cnt_lstm *h, const SlotOrder *order);
// Forward pass of one WaveNet residual block in one launch: see wavenet_block_forward_kernel.
struct BlockForward {
    const float *x, *ctx;  // the block's input and the conditioning features
    const float *conv_weights, *ctx_weights, *out_weights, *skip_weights;  // the layers' weights, biases behind them
    float out_bias, skip_bias;
    float *conv, *core, *ctx_tanh, *gated, *out, *sum, *skip;
};
bool wavenet_block_forward_supported(const cnt_cnn *cnn, int R, int K, int C);
int wavenet_block_forward(hipStream_t stream, const cnt_cnn *cnn, int R, int K, int C, int N, const char *patTypes,
                          const BlockForward &block, int from, int to);
// Error path of one WaveNet residual block in one launch (skip 1x1 layer, the skip layer in front of it, the 1x1
// layer behind the gated unit, the gated unit): see wavenet_block_errors_kernel.
bool wavenet_block_errors_supported(int R, int K);
// `fold` (optional): the convolution layer above the block, whose error product (two live taps) is added to the
// block's summed errors inside the same launch instead of being written to the closing skip layer first.
// ctx_grad receives the gradient of the conditioning part: ctx_tanh itself (if core_buf is given) or a buffer of its own
bool cnn_foldable(const cnt_cnn *h, int R);
int wavenet_block_errors(hipStream_t stream, int R, int K, int N, const char *patTypes, const float *skip_weights,
                         const float *out_weights, const float *skip_errors, float *total, const FanOut *fan,
                         const float *core_buf, const float *ctx_tanh, float *ctx_grad, const float *conv_tanh_outputs, float *conv_errors,
                         const cnt_cnn *fold, const float *fold_weights, const float *fold_deltas, float *colsum_partial);
// workgroups of that launch = rows of `colsum_partial` ([rows][2R]: per-workgroup sums of conv_errors over the samples)
int wavenet_block_rows(int R, int N, bool fold);
int wavnetc_context_grad(hipStream_t stream, int D, int C, int N, const float *weights, const float *ctx_tanh,
                         float *ctx_grad);
int cnn_backward_errors_fan(cnt_cnn *h, hipStream_t stream, const char *patTypes, int curT, const float *weights,
                            const float *outputs, float *output_errors, float *prev_errors, int delta_applied,
                            const FanOut *fan, bool *fused);

// Weight gradients of up to kBlockGradients such blocks in one launch (wavenet_weights.hip): the convolution (two live taps of a
// window of three), the conditioning projection, the 1x1 layer behind the gate and the skip 1x1 layer, with the bias gradients.
constexpr int kBlockGradients = 8;
struct BlockGradients {
    const float *x, *gated, *sum;                                // inputs of the convolution and of the two 1x1 layers
    const float *deltas, *ctx_grad, *out_errors, *skip_errors;   // what their outputs receive, in that order
    float *conv, *conv_bias, *ctx, *out, *out_bias, *skip, *skip_bias;  // the weight updates
    float conv_scale, out_scale, skip_scale;                     // factors of the bias gradients
    int shift;                                                   // the earlier tap reads slot n - shift
};
bool wavenet_block_weights_supported(int R, int K, int C, long N);
size_t wavenet_block_weights_scratch(int R, int K, int C);  // floats; one launch at a time
int wavenet_block_weights(hipStream_t stream, int R, int K, int C, int N, int count, const BlockGradients *blocks, const float *ctx,
                          const char *patTypes, float *scratch);
// the shift, the bias gradient's place behind the weights and its factor, of a layer that cnn_foldable accepts
struct CnnTaps {
    int shift;
    size_t bias_at;
    float bias;
};
CnnTaps cnn_taps(const cnt_cnn *h);

// ----- weight-gradient halves of several layers of one shape in one launch --------------------------
// For the network sequencer: `count` (<= kGemmMaxProb) dense layers with the same P, D, N, or wavnetc layers with the
// same D, C, N and one context buffer, as the problems of one product.  Same results as `count` calls of
// cnt_dense_backward_weights / cnt_wavnetc_backward_weights.
int dense_backward_weights_batch(hipStream_t stream, int P, int D, int N, int count, const float *bias,
                                 const float *const *x, const float *const *err, float *const *weight_updates, const SlotOrder *order = nullptr,
                                 DirectGroup *group = nullptr);
bool dense_weights_direct(int P, int D, int N, int count);  // whether that is the kernel for few blocks
int wavnetc_backward_weights_batch(hipStream_t stream, int D, int C, int N, int count, const float *ctx,
                                   const float *const *ctx_tanh, float *const *weight_updates);
// Convolution layers with one filter group each and the same sizes, window and causality (dilations may differ):
// cnn_batch_taps gives the live taps of such a layer (0: not batchable, several filter groups), and `count` layers
// with count * taps <= kGemmMaxProb go into one product.
int cnn_batch_taps(const cnt_cnn *h);
bool cnn_batch_compatible(const cnt_cnn *a, const cnt_cnn *b);
int cnn_backward_weights_batch(cnt_cnn *const *h, int count, hipStream_t stream, const char *patTypes, int curT,
                               const float *const *x, const float *const *output_errors, float *const *weight_updates,
                               const float *const *colsum_partial = nullptr, const int *colsum_rows = nullptr);

// Flags of the events that order this library's streams among each other: what such an event orders is always a kernel of the same device, and a
// kernel's end makes its results visible to that.  The host only asks whether such an event is over (lstm_take_failure); what it then reads, a
// recursion's latch, is stored at system scope and needs no fence either.  Without the record's system-wide fence, which is for readers on the host
// or other devices, a launch behind a record starts 2 to 3 us earlier: acoustic model 2539 -> 2525 us per pass, one lstm layer 372 -> 368,
// eight small WaveNet blocks 298 -> 284.
constexpr unsigned kOrderEvent = hipEventDisableTiming | hipEventDisableSystemFence;

// whether the stream is being captured; a stream that cannot be asked (the null stream beside a capture) counts as captured
bool capturing(hipStream_t stream);

// ----- small streaming kernels (elementwise.hip) ----------------------------------------------------
int fill_zero(hipStream_t stream, float *p, size_t count);
// two buffers in one launch
int fill_zero_pair(hipStream_t stream, float *p, size_t count, float *q, size_t count_q);
// What a network does on the device when a fraction is loaded, as ONE launch: up to kLoadClears buffers zeroed (the
// recurrent layers' stored output-gate deltas), up to two copied (inputs and targets, from memory of this device) and, when
// `order` is given, the fraction's slot order built (as slot_order_build does).
constexpr int kLoadClears = 8, kLoadCopies = 2;
struct LoadClears {
    float *ptr[kLoadClears];
    unsigned long long count[kLoadClears];  // floats, multiples of four, 16-byte aligned buffers
    int n;
    const float *from[kLoadCopies];
    float *to[kLoadCopies];
    unsigned long long copy_count[kLoadCopies];  // floats
    int copies;
};
int load_clear_and_order(hipStream_t stream, const LoadClears &clears, const char *pat, int n_slots, int slots_per_step,
                         int *order, int *count);
// cnt_lstm_load_sequences without the clearing launch: the caller clears what `clears` lists afterwards (false: the list
// is full or a buffer does not qualify, and the handle has launched its own clear)
int lstm_load_sequences_collect(cnt_lstm *h, hipStream_t stream, const char *patTypes, int curMaxT, int curMinT,
                                LoadClears &clears);
int fill_words(hipStream_t stream, unsigned *p, size_t count, unsigned word);
// cnt_sse_error in one launch, summed in 64 bits; sum: 64 words of the caller's that are zero between calls
int sse_error_once(hipStream_t stream, int D, int N, const char *patTypes, const float *y, const float *target, float *result_dev,
                   float *sum);
// out[d] += scale * sum over the N columns of a D x N column-major matrix (out pre-zeroed by the caller), and the same with `=`, through
// the stream's scratch where it has one
int column_sum(hipStream_t stream, const float *v, int D, int N, float scale, float *out);
int column_sum_store(hipStream_t stream, const float *v, int D, int N, float scale, float *out);

}  // namespace cnt
