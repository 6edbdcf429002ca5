// Weight update of the training loop, as streaming kernels.
//
// Reference behaviour: optimizers/Optimizer.cu:186-198 (copy / accumulation of a layer's weight updates
// per fraction), optimizers/SteepestDescentOptimizer.cu:119-203 (AdaGrad / Adam / averaging functors),
// :312-405 (which of them runs for which optimizer option), :41-98 and :408-436 (the momentum update, with
// and without weight mask), MacroDefine.hpp:32-42 (option numbers, constants).
//
// The reference runs up to three passes over every weight vector (copy, adjust, update).  cnt_opt_step does
// the same arithmetic in one pass: per weight it reads the layer's gradient, the optimizer state and the
// weight and writes them back once (Adam: 20 B read + 20 B written).  The three separate entry points exist
// for callers that keep the reference's call structure.  The Adam moment updates use the reference's double
// constants (0.9, 0.999, 1e-8 are double literals there), so they are evaluated in double and rounded once.
// This file is compiled with -ffp-contract=off: every product and sum is rounded on its own, as in the
// reference, which makes the results bit-identical to a sequential host evaluation.
#include "common.hpp"

namespace cnt {
namespace {

constexpr double kBeta1 = 0.9, kBeta2 = 0.999, kEps = 0.00000001;

struct OptArgs {
    size_t n;
    const float *layer_updates;  // gradient of this fraction (step / accumulate)
    float *cur;                  // the optimizer's current weight updates
    float *stats;                // AdaGrad: n floats, Adam: n (m, v) pairs
    float *deltas;               // momentum state
    float *weights;
    const float *mask;           // optional weight mask
    int option;                  // 0 plain, 1 AdaGrad, 2 averaged, 3 stochastic AdaGrad, 5 Adam
    int add;                     // accumulate: add to cur instead of overwriting it
    float frac_length, beta1_accum, beta2_accum, learning_rate, momentum;
    const int *veto;             // optional device flag: non-zero means the gradients are invalid, nothing is touched
    const float *accum_dev;      // optional: Adam's two bias-correction products in device memory (replace the two floats)
};

__device__ __forceinline__ bool bad(float g) { return isnan(g) || isinf(g); }
// (the options that keep statistics, and how many floats of them per weight)
__device__ __forceinline__ bool with_statistics(const OptArgs &a) { return a.option == 1 || a.option == 3 || a.option == 5; }

// The gradient that the update uses; s: the weight's statistics (Adam: m and v).
__device__ __forceinline__ float adjust_one(const OptArgs &a, float g, float mask, float (&s)[2]) {
    if (a.option == 2) return g / a.frac_length;
    if (!with_statistics(a)) return g;
    if (bad(g)) g = 0.0f;
    if (mask < 1.0f) return g;
    const float ave = g / a.frac_length;
    if (a.option == 5) {
        const float m = (float)(s[0] * kBeta1 + ave * (1 - kBeta1));
        const float v = (float)(s[1] * kBeta2 + (double)(ave * ave) * (1 - kBeta2));
        s[0] = m;
        s[1] = v;
        const float b1 = a.accum_dev ? a.accum_dev[0] : a.beta1_accum, b2 = a.accum_dev ? a.accum_dev[1] : a.beta2_accum;
        const float mh = m / (1 - b1);
        const float vh = v / (1 - b2);
        return (float)(mh / (sqrtf(vh) + kEps));
    }
    const float acc = s[0] + (ave * ave);
    s[0] = acc;
    return a.option == 1 ? ave / sqrtf(acc) : g;
}

__device__ __forceinline__ float update_one(const OptArgs &a, float g, float mask, float &delta, float &w) {
    if (bad(g)) g = 0.0f;
    delta = a.momentum * delta - a.learning_rate * g;
    w = w + delta;
    if (a.mask) w = w * mask;
    return g;
}

// N neighbouring floats, at any address that a float may have
template <int N>
__device__ __forceinline__ void fetch(const float *p, float (&v)[N]) {
    typedef float vec __attribute__((ext_vector_type(N), aligned(4)));
    const vec x = *reinterpret_cast<const vec *>(p);
#pragma unroll
    for (int q = 0; q < N; ++q) v[q] = x[q];
}
template <int N>
__device__ __forceinline__ void put(float *p, const float (&v)[N]) {
    typedef float vec __attribute__((ext_vector_type(N), aligned(4)));
    vec x;
#pragma unroll
    for (int q = 0; q < N; ++q) x[q] = v[q];
    *reinterpret_cast<vec *>(p) = x;
}

// MODE 0 accumulate, 1 adjust, 2 update, 3 all three in one pass; N weights from i on: everything is asked for before anything is
// worked out, so that a wave has up to six accesses in flight.
template <int MODE, int N>
__device__ __forceinline__ void optimize(const OptArgs &a, size_t i) {
    constexpr bool LAYER = MODE == 0 || MODE == 3, ADJUST = MODE == 1 || MODE == 3, UPDATE = MODE == 2 || MODE == 3;
    float g[N], cur[N], mask[N], delta[N], w[N], s[N * 2];
    const bool moments = ADJUST && a.option == 5, squares = ADJUST && (a.option == 1 || a.option == 3);
    if (LAYER) fetch<N>(a.layer_updates + i, g);
    if (!LAYER || a.add) fetch<N>(a.cur + i, cur);
    if (moments) fetch<N * 2>(a.stats + 2 * i, s);
    if (squares) {
        float t[N];
        fetch<N>(a.stats + i, t);
#pragma unroll
        for (int q = 0; q < N; ++q) s[2 * q] = t[q];
    }
    if (UPDATE) { fetch<N>(a.deltas + i, delta); fetch<N>(a.weights + i, w); }
    if (a.mask) fetch<N>(a.mask + i, mask);
#pragma unroll
    for (int q = 0; q < N; ++q) {
        float x = !LAYER ? cur[q] : a.add ? g[q] + cur[q] : g[q];
        const float m = a.mask ? mask[q] : 1.0f;
        if (ADJUST) {
            float own[2] = {s[2 * q], s[2 * q + 1]};
            x = adjust_one(a, x, m, own);
            s[2 * q] = own[0];
            s[2 * q + 1] = own[1];
        }
        if (UPDATE) x = update_one(a, x, m, delta[q], w[q]);
        cur[q] = x;
    }
    if (moments) put<N * 2>(a.stats + 2 * i, s);
    if (squares) {
        float t[N];
#pragma unroll
        for (int q = 0; q < N; ++q) t[q] = s[2 * q];
        put<N>(a.stats + i, t);
    }
    if (UPDATE) { put<N>(a.deltas + i, delta); put<N>(a.weights + i, w); }
    put<N>(a.cur + i, cur);
}

// N weights per thread; those that are left over at the end go one by one.
template <int MODE, int N>
__global__ __launch_bounds__(256) void optimizer_kernel(const OptArgs a) {
    const size_t first = (size_t)blockIdx.x * blockDim.x + threadIdx.x, stride = (size_t)gridDim.x * blockDim.x;
    if (a.veto && *a.veto != 0) return;
    const size_t whole = a.n / N;
    for (size_t i = first; i < whole; i += stride) optimize<MODE, N>(a, i * N);
    if (first < a.n % N) optimize<MODE, 1>(a, whole * N + first);
}

// Adam's bias-correction products beta1^t, beta2^t kept in device memory, advanced in stream order in front of a step
// and under the same veto flag as the step: a step that the flag skips leaves them where they stood.
__global__ void adam_advance_kernel(float *accum, const int *veto) {
    if (veto && *veto != 0) return;
    accum[0] = (float)(accum[0] * kBeta1);
    accum[1] = (float)(accum[1] * kBeta2);
}

// One weight per thread while a full grid holds them, four beyond that.  What bounds a step is memory: with four-byte accesses and a
// second round of the grid a step in a training pass took 44.8 us (Adam, 4.8 million weights) and 21.0 (steepest descent, 3.0 million),
// in fours 38.1 and 19.4; one step after another 5.9 to 6.7 TB/s (two per thread 0 to 7 % less, eight 3 to 24 %).  Below the line
// the shorter threads finish first: Adam, 0.8 million 7.2 us and 8.6 in fours, 40 thousand in a small network's pass 3.2 and 3.6.
constexpr size_t kMostBlocks = 8192, kFours = kMostBlocks * 256;
template <int MODE>
int launch_optimizer(hipStream_t stream, const OptArgs &a) {
    const bool fours = a.n > kFours;
    const size_t blocks = ((fours ? a.n / 4 : a.n) + 255) / 256;
    void (*const kernel)(const OptArgs) = fours ? optimizer_kernel<MODE, 4> : optimizer_kernel<MODE, 1>;
    hipLaunchKernelGGL(kernel, dim3((unsigned)std::min(blocks, kMostBlocks)), dim3(256), 0, stream, a);
    CNT_HIP(hipGetLastError());
    return CNT_OK;
}

bool known_option(int o) { return o == 0 || o == 1 || o == 2 || o == 3 || o == 4 || o == 5; }

}  // namespace
}  // namespace cnt

extern "C" {

int cnt_opt_accumulate(void *stream, long n, const float *layer_updates, float *cur_updates, int add) {
    using namespace cnt;
    CNT_REQUIRE(n >= 0 && (n == 0 || (layer_updates && cur_updates)), "opt_accumulate: bad argument");
    if (n == 0) return CNT_OK;
    OptArgs a = {};
    a.n = (size_t)n; a.layer_updates = layer_updates; a.cur = cur_updates; a.add = add;
    ProfileScope prof(static_cast<hipStream_t>(stream), "opt_accumulate");
    return launch_optimizer<0>(static_cast<hipStream_t>(stream), a);
}

int cnt_opt_adjust_gradient(void *stream, int option, long n, float *cur_updates, float *stats, const float *mask,
                            float frac_length, float beta1_accum, float beta2_accum) {
    using namespace cnt;
    CNT_REQUIRE(n >= 0 && (n == 0 || cur_updates), "opt_adjust_gradient: bad argument");
    CNT_REQUIRE(known_option(option), "opt_adjust_gradient: unknown optimizer option %d", option);
    CNT_REQUIRE(!(option == 1 || option == 3 || option == 5) || stats, "opt_adjust_gradient: option %d needs a statistics buffer",
                option);
    if (n == 0 || option == 0 || option == 4) return CNT_OK;
    OptArgs a = {};
    a.n = (size_t)n; a.cur = cur_updates; a.stats = stats; a.mask = mask; a.option = option;
    a.frac_length = frac_length; a.beta1_accum = beta1_accum; a.beta2_accum = beta2_accum;
    ProfileScope prof(static_cast<hipStream_t>(stream), "opt_adjust_gradient");
    return launch_optimizer<1>(static_cast<hipStream_t>(stream), a);
}

int cnt_opt_update_weights(void *stream, long n, float *weights, float *cur_updates, float *weight_deltas,
                           const float *mask, float learning_rate, float momentum) {
    using namespace cnt;
    CNT_REQUIRE(n >= 0 && (n == 0 || (weights && cur_updates && weight_deltas)), "opt_update_weights: bad argument");
    // the reference skips the update altogether for a negative learning rate (SteepestDescentOptimizer.cu:283-285)
    if (n == 0 || learning_rate < 0) return CNT_OK;
    OptArgs a = {};
    a.n = (size_t)n; a.cur = cur_updates; a.deltas = weight_deltas; a.weights = weights; a.mask = mask;
    a.learning_rate = learning_rate; a.momentum = momentum;
    ProfileScope prof(static_cast<hipStream_t>(stream), "opt_update_weights");
    return launch_optimizer<2>(static_cast<hipStream_t>(stream), a);
}

int cnt_opt_step(void *stream, int option, long n, float *weights, const float *layer_updates, float *cur_updates,
                 float *stats, float *weight_deltas, const float *mask, float frac_length, float beta1_accum,
                 float beta2_accum, float learning_rate, float momentum) {
    return cnt::opt_step_guarded(static_cast<hipStream_t>(stream), option, n, weights, layer_updates, cur_updates, stats,
                                 weight_deltas, mask, frac_length, beta1_accum, beta2_accum, learning_rate, momentum, nullptr,
                                 nullptr);
}

extern "C++" int cnt::opt_adam_advance(hipStream_t stream, float *accum_dev, const int *veto) {
    hipLaunchKernelGGL(adam_advance_kernel, dim3(1), dim3(1), 0, stream, accum_dev, veto);
    CNT_HIP(hipGetLastError());
    return CNT_OK;
}

extern "C++" int cnt::opt_step_guarded(hipStream_t stream, int option, long n, float *weights, const float *layer_updates,
                                       float *cur_updates, float *stats, float *weight_deltas, const float *mask,
                                       float frac_length, float beta1_accum, float beta2_accum, float learning_rate,
                                       float momentum, const int *veto, const float *accum_dev) {
    using namespace cnt;
    CNT_REQUIRE(n >= 0 && (n == 0 || (weights && layer_updates && cur_updates && weight_deltas)), "opt_step: bad argument");
    CNT_REQUIRE(known_option(option), "opt_step: unknown optimizer option %d", option);
    CNT_REQUIRE(!(option == 1 || option == 3 || option == 5) || stats, "opt_step: option %d needs a statistics buffer", option);
    CNT_REQUIRE(learning_rate >= 0, "opt_step: negative learning rate (the reference skips the update; call cnt_opt_accumulate)");
    if (n == 0) return CNT_OK;
    OptArgs a = {};
    a.n = (size_t)n; a.layer_updates = layer_updates; a.cur = cur_updates; a.stats = stats; a.deltas = weight_deltas;
    a.weights = weights; a.mask = mask; a.option = option == 4 ? 0 : option;
    a.frac_length = frac_length; a.beta1_accum = beta1_accum; a.beta2_accum = beta2_accum;
    a.learning_rate = learning_rate; a.momentum = momentum;
    a.veto = veto;
    a.accum_dev = accum_dev;
    ProfileScope prof(stream, "opt_step");
    return launch_optimizer<3>(stream, a);
}

float cnt_opt_next_beta_accum(float accum, int which) { return (float)(accum * (which == 1 ? cnt::kBeta1 : cnt::kBeta2)); }

}  // extern "C"
