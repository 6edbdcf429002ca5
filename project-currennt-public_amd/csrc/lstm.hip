// LSTM layer for gfx950: forward recursion, BPTT error recursion, and the batched contractions.
//
// Reference behaviour: layers/LstmLayer.cu  (forward :57-208, :1743-1949; backward :210-648,
// :2066-2382; sequence loading :1488-1533; weight layout :1136-1169, :1218-1268).
//
// The reference launches four small matrix products and one elementwise functor per time step and
// direction.  Here a layer's whole recursion is ONE persistent launch, cut into independent jobs (a direction and at
// most four parallel sequences):
//   up to 64 cells per direction    a workgroup per job, nothing exchanged (lstm_solo.hpp);
//   up to 512 cells per direction   a team of workgroups on one XCD per job (lstm_local.hpp, lstm_local_fwd.hpp): each
//       owns a few cells for the whole sequence, keeps its slice of the recurrent weights in registers as MFMA operands,
//       carries the per-cell recurrent state in registers, and exchanges the only truly shared quantity of a step through
//       a small device-memory mailbox -- the block outputs h[t] (forward) or partial output errors (backward);
//   more cells                      step by step, the reference's own schedule.
// Mailbox words are plain 4-byte floats; a reserved NaN pattern means "not written yet", so a word validates
// itself and neither tags nor fences sit on the critical path.  Words are moved 16 bytes at a time, polled with
// loads that bypass the non-coherent caches, and handed back as empty after use; four slots rotate.  Every
// poll loop is bounded: when the bound is hit the workgroup raises a device flag and every workgroup drains
// out.  Inside a workgroup, waves specialise (polling waves that never store, product / cell waves that never
// wait for a store, a load and a store wave for all ordinary loads and stores), see the kernels' comments.
//
// The dense work that does not sit on the recursion is batched over all time steps on the MFMA
// GEMM: input projections (8 problems, one launch), the error to the preceding layer
// (one K-concatenated product), input and recurrent weight gradients (split-K), and one streaming
// reduction for bias and peephole gradients.
#include "common.hpp"

#include <cstdlib>
#include <cstring>
#include <new>
#include <type_traits>
#include <vector>
#include <utility>
#include <algorithm>
#include <mutex>

namespace cnt {
namespace {

typedef float f32x4 __attribute__((ext_vector_type(4)));
typedef unsigned long long u64;


struct DirPtrs {
    float *ni, *ig, *fg, *og, *c, *h;
    float *herr, *dni, *dig, *dfg, *dog, *cerr;
    const float *w_int;    // gate 0 block of this direction; gate g at + g*L*H
    const float *b[4];     // bias weights per gate
    const float *peep[3];  // ig, fg, og peepholes
};

struct ChainParams {
    int H, L, S, T, Tmin, ndir;
    float bias;
    const char *pat;
    DirPtrs d[2];
    float *out;           // forward: L x (T*S) layer outputs (NULL when it aliases d[0].h)
    const float *outerr;  // backward: L x (T*S) output errors
    float *herr_out;      // backward, unidirectional: where the summed error is written back
    unsigned spin_limit;
    int *abort_flag;
    int poll_delay, poll_limit, poll_gap;  // s_sleep units before the first poll of a step (-1: as the job's size wants it) and at most / between polls
    int mem_delay;             // XCD-local backward recursion: s_sleep units before the store wave's work of a step
    int poll_delay_fwd, poll_limit_fwd, mem_delay_fwd;  // forward: the same, and before the load wave's
    int *latch;  // host-visible mark "a recursion of this handle gave up" (pinned host memory), never cleared by kernels
    int *veto;   // optional device flag shared by a network's handles, set together with the latch
    // XCD-local recursions: jobs = (direction, group of sequences), see lstm_local.hpp
    unsigned job0;      // first job of this launch
    int njobs, groups;  // jobs of this launch; groups of sequences per direction
    int team;           // workgroups of a job's team
    int ctl_teams;
    unsigned *ctl;   // placement counters, zero at launch
    float *lmail;    // one mailbox per job
    float *flmail;   // the same for the XCD-local forward recursion
    // XCD-local backward recursion over a range of its steps: [step_begin, step_end) of 0 .. T.  A launch that starts
    // at a later step takes what the step before it left: the carried cell-state terms from the state arrays, the
    // partial errors from the mailbox (which nothing may touch in between).
    int step_begin, step_end;
    long long *clocks;  // of the kernels with CLOCKS
    // Backward: where the sums over the pass of the gates' deltas (times sum_scale) and of their products with the cell states go, or
    // null.  Sum k of cell u: [k * sum_k + direction * sum_dir + group * sum_group + u], the products' behind sum_peep.
    float *sum_bias, *sum_peep;
    int sum_k, sum_dir, sum_group;
    float sum_scale;
};

// A workgroup that gives up: every workgroup of the launch sees the device flag and drains; the host sees the latch
// at its next call into the handle, the optimizer step of a network sees the veto flag.
__device__ __forceinline__ void raise_abort(const ChainParams &p) {
    __hip_atomic_store(p.abort_flag, 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    __hip_atomic_store(p.latch, 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_SYSTEM);
    if (p.veto) __hip_atomic_store(p.veto, 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}

// Workgroup barrier that orders LDS traffic only.  __syncthreads() also drains every outstanding
// global load and store of the wave, which would put the HBM latency of the look-ahead loads and the
// acknowledgement of the result stores on the recursion's critical path.  No thread of a workgroup
// reads global data written by another thread of the same launch except through the mailbox.
__device__ __forceinline__ void lds_barrier() {
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "workgroup", "local");
    __builtin_amdgcn_s_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "workgroup", "local");
}

// ---------------------------------------------------------------------------------------------------
// Backward (error) recursion.
//
// The partial output errors travel through a mailbox of plain 4-byte words, laid out
// [slot][receiving workgroup][sending workgroup][sequence][cell of the receiver]:
//   * a word that holds kEmpty (an all-ones NaN pattern no product can yield) has not been written yet;
//     a sender stores the JB values of one (receiver, sequence) pair as 16-byte vectors, a receiver polls
//     its contiguous words with 16-byte loads and validates every word on its own;
//   * after reading, the receiving workgroup puts kEmpty back.  Four slots rotate (step % 4): a slot is used again three
//     steps later, by senders that have by then received something this workgroup published after its reset had
//     completed.
// A launch that runs to its end leaves every word empty, so the host fills the mailbox with kEmpty once and
// again only after a launch that gave up.
// ---------------------------------------------------------------------------------------------------
constexpr unsigned kEmpty = 0xFFFFFFFFu;
constexpr int kMailSlots = 4;
// Pauses of the XCD-local recursions, units of 64 clocks: before the first poll of a step (a pause that ends after the words have
// arrived costs a poll round less, one that ends too late its own length), and before the store wave's work of a backward and the
// load wave's of a forward step, which then stay out of the first poll's way.  Measured on MI355X, us per step.  Forward, 8 / 9 / 10 /
// 11 / 12 units: 256 cells 8 jobs of one sequence 0.785 / 0.769 / 0.776 / 0.798 / 0.832, of two 0.84 / 0.83 / 0.83 / 0.85 / 0.86, of three
// 0.93 / 0.91 / 0.92 / 0.92 / 0.92, 16 jobs of four (16 cells per workgroup) 1.14 / 1.14 / 1.13 / 1.12 / 1.12, 150 cells 0.96 / 0.93 /
// 0.96 / 0.98 / 1.00, 512 cells jobs of four 1.62 / 1.60 / 1.58 / 1.55 / 1.55.  Backward, 1 / 2 / 3 / 4 / 5 units: 0.68 / 0.67 / 0.70 / 0.75 / 0.76,
// 0.76 / 0.75 / 0.75 / 0.77 / 0.79, 0.84 / 0.83 / 0.81 / 0.82 / 0.86, 1.14 / 1.13 / 1.08 / 1.07 / 1.08, 0.85 / 0.86 / 0.86 / 0.89 / 0.90, 1.49 / 1.49 /
// 1.48 / 1.43 / 1.42.  Stores after 0 / 2 / 4 / 6 units: within 2 % of each other.
// EL = words of a message, cells per workgroup times sequences of the job.
constexpr int kStorePause = 4, kLoadPause = 4;
constexpr int backward_pause(int EL) { return EL <= 8 ? 2 : EL <= 32 ? 3 : 4; }
constexpr int forward_pause(int EL) { return EL <= 32 ? 9 : 11; }
typedef unsigned u32x4 __attribute__((ext_vector_type(4)));

// s_waitcnt vmcnt(0) (expcnt and lgkmcnt left at their maxima) as a builtin, so that the compiler's own wait
// insertion sees that nothing is outstanding afterwards and adds no waits of its own for older loads.
__device__ __forceinline__ void wait_all_vmem() { __builtin_amdgcn_s_waitcnt(0x0F70); }

// N 16-byte loads that bypass the non-coherent caches (device scope), all in flight together, then one wait.
// Inline assembly because the polled words change under the compiler's feet: the loads may neither be
// hoisted out of the polling loop nor merged.
template <int N>
__device__ __forceinline__ void poll_load(const float *base, unsigned byte_off, unsigned q_stride_bytes,
                                          unsigned last_byte_off, u32x4 (&w)[N]) {
#pragma unroll
    for (int q = 0; q < N; ++q) {
        const float *bq = reinterpret_cast<const float *>(reinterpret_cast<const char *>(base) +
                                                          (q + 1 < N ? (size_t)q * q_stride_bytes : 0));
        const unsigned off = q + 1 < N ? byte_off : last_byte_off;
        asm volatile("global_load_dwordx4 %0, %1, %2 sc1" : "=v"(w[q]) : "v"(off), "s"(bq) : "memory");
    }
    wait_all_vmem();
#pragma unroll
    for (int q = 0; q < N; ++q) asm volatile("" : "+v"(w[q]));  // consumers stay behind the wait
}

// After a poll that found a word empty: has this wave polled long enough, or another workgroup given up?  Uniform over the wave, as
// is the poll loop's way out: with every lane leaving for itself the masks of the loop were some twenty scalar instructions on
// the chain of a step.
__device__ __forceinline__ bool poll_gives_up(const ChainParams &p, unsigned spins) {
    if (spins > p.spin_limit) return true;
    return (spins & 255u) == 0u && __builtin_amdgcn_readfirstlane(__hip_atomic_load(p.abort_flag, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT)) != 0;
}

// Bias and peephole gradients of a whole pass, summed up by the backward recursions' store waves, which have the deltas in
// registers: per cell four sums of deltas and three of products with the cell state, in 64 bits (one addition per step of up to
// thousands).  A launch of their own read the four arrays of deltas and the cell states once more, 98 MB per layer with 32 sequences
// of 300 steps, 115 us beside the products; the recursion is as fast as without them (0 to 1 %).  Us per pass, with the launch / without:
// one lstm layer 368 / 362, a small network 119 / 115, 32 sequences 2483 / 2447.
constexpr int kSmallSums = 7;  // per cell: four biases, three peepholes (input, forget, output gate)
__device__ __forceinline__ void put_sum(const ChainParams &p, int dir, int group, int k, int u, float v) {
    float *const to = k < 4 ? p.sum_bias + k * p.sum_k : p.sum_peep + (k - 4) * p.sum_k;
    to[dir * p.sum_dir + group * p.sum_group + u] = k < 4 ? v * p.sum_scale : v;
}

// N neighbouring recurrent weights of a lane's row of H (at least four), from `from` on, zeros behind its end and in lanes without a
// row.  Every lane has a row of its own, so a load touches 64 lines however few values it takes of each: in fours, at any address, a
// quarter of the accesses of one by one.  A launch of 64 cells and 30 steps 27.7 -> 23.5 us, the pass around it 96 -> 92.  (Without a branch for
// rows of a multiple of four: with one, the 256-cell recursion took 597 us for 800 steps instead of 574.)
template <int N>
__device__ __forceinline__ void load_weight_row(const float *row, bool has_row, int from, int H, float (&w)[N]) {
    typedef float f32x4a4 __attribute__((ext_vector_type(4), aligned(4)));
#pragma unroll
    for (int i = 0; i < N; i += 4) {
        // the vector that would pass the row's end ends with it, and is moved into place
        const int at = from + i, last4 = H - 4, d = at - last4;
        const f32x4a4 v = *reinterpret_cast<const f32x4a4 *>(row + min(at, last4));
        const float x1 = d > 0 && (d & 1) ? v[1] : v[0], x2 = d > 0 && (d & 1) ? v[2] : v[1], x3 = d > 0 && (d & 1) ? v[3] : v[2];
        const bool two = d > 0 && (d & 2);
        w[i] = has_row && at < H ? (two ? x3 : x1) : 0.0f;
        w[i + 1] = has_row && at + 1 < H ? (two ? v[3] : x2) : 0.0f;
        w[i + 2] = has_row && at + 2 < H ? x3 : 0.0f;
        w[i + 3] = has_row && at + 3 < H ? v[3] : 0.0f;
    }
}

#include "lstm_local.hpp"
#include "lstm_local_fwd.hpp"
#include "lstm_solo.hpp"

// Runs in front of every recursion launch (one workgroup).  If the launch before gave up, the device flag is still
// set and mailbox words may be left over: refill the mailboxes and clear the flag, so that a handle heals without
// its owner's help.  Always: zero the placement counters of the XCD-local recursion.
struct GuardParams {
    int *abort_flag;
    unsigned *ctl;
    int nctl;
    unsigned *mail[2];
    size_t words[2];
};
// the work of one workgroup (any size)
__device__ __forceinline__ void guard_body(const GuardParams &g) {
    const bool heal = __hip_atomic_load(g.abort_flag, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) != 0;
    if (heal) {
        for (int m = 0; m < 2; ++m)
            for (size_t i = threadIdx.x; i < g.words[m]; i += blockDim.x) g.mail[m][i] = kEmpty;
    }
    for (int i = threadIdx.x; i < g.nctl; i += blockDim.x) g.ctl[i] = 0u;
    __syncthreads();
    if (heal && threadIdx.x == 0) __hip_atomic_store(g.abort_flag, 0, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}
__global__ __launch_bounds__(1024) void chain_guard(const GuardParams g) { guard_body(g); }

// ---------------------------------------------------------------------------------------------------
// Bias and peephole gradients: per (direction, gate, cell) sums over all patterns
// (LstmLayer.cu:524-541, 574-610, 625-646).  A thread owns V neighbouring cells (4, 2 or 1, what divides the cell count per
// direction: 16-byte loads where it can be), a wave walks whole rows of the state arrays, a workgroup's waves share a chunk of
// patterns and add up in LDS.  The chunks' sums meet in the stream's scratch in a fixed order (lstm_small_grads_sum); without one they
// are added atomically to gradients that the caller has cleared.  blockIdx.z is the direction.
// 150 cells in two directions over 10 000 patterns: 24 + 29 us with a thread per cell, a chunk of 32 patterns and a launch per
// direction, 23 us now.
// ---------------------------------------------------------------------------------------------------
struct SmallGradDirs {
    int H, L, S, N, chunk;
    float bias;
    const float *dni[2], *dig[2], *dfg[2], *dog[2], *c[2];
    float *g_bias;  // + g*L + dir*H + u
    float *g_peep;  // + k*L + dir*H + u
    float *parts;   // [chunk][direction][4 biases, 3 peepholes][cell]
};

template <int V>
__global__ __launch_bounds__(256) void lstm_small_grads(const SmallGradDirs p) {
    typedef float cells __attribute__((ext_vector_type(V)));
    __shared__ cells acc[kSmallSums][256];  // [row of patterns walked side by side][group of cells]
    const int dir = blockIdx.z;
    const int groups = p.H / V;
    const int gpb = min(groups, 256 / V);  // groups of cells per workgroup
    const int rows = 256 / gpb;            // pattern rows walked side by side
    const int tid = threadIdx.x;
    const int gl = tid % gpb, r = tid / gpb;
    const int q = blockIdx.x * gpb + gl;
    if (r < rows) {
        cells b0 = {}, b1 = b0, b2 = b0, b3 = b0, q_ig = b0, q_fg = b0, q_og = b0;
        if (q < groups) {
            const int i0 = blockIdx.y * p.chunk, i1 = min(p.N, i0 + p.chunk);
            const int S = p.S;
            const cells *dni = reinterpret_cast<const cells *>(p.dni[dir]), *dig = reinterpret_cast<const cells *>(p.dig[dir]);
            const cells *dfg = reinterpret_cast<const cells *>(p.dfg[dir]), *dog = reinterpret_cast<const cells *>(p.dog[dir]);
            const cells *c = reinterpret_cast<const cells *>(p.c[dir]);
#pragma unroll 4
            for (int i = i0 + r; i < i1; i += rows) {
                const size_t o = (size_t)i * groups + q;
                const cells d_ni = dni[o], d_ig = dig[o], d_fg = dfg[o], d_og = dog[o];
                b0 += d_ni; b1 += d_ig; b2 += d_fg; b3 += d_og;
                q_og += c[o] * d_og;
                // input/forget peepholes look at the cell state one step earlier in processing order
                const int ie = dir ? i + S : i - S;
                if (ie >= 0 && ie < p.N) {
                    const cells ce = c[(size_t)ie * groups + q];
                    q_ig += ce * d_ig;
                    q_fg += ce * d_fg;
                }
            }
        }
        const cells v[kSmallSums] = {b0 * p.bias, b1 * p.bias, b2 * p.bias, b3 * p.bias, q_ig, q_fg, q_og};
#pragma unroll
        for (int k = 0; k < kSmallSums; ++k) acc[k][tid] = v[k];
    }
    __syncthreads();
    const int mine = V * gpb, u0 = blockIdx.x * mine;
    for (int i = tid; i < kSmallSums * mine; i += 256) {
        const int k = i / mine, j = i % mine, u = u0 + j;
        if (u >= p.H) continue;
        const float *const sums = reinterpret_cast<const float *>(acc[k]) + j;
        float s0 = 0.0f, s1 = 0.0f, s2 = 0.0f, s3 = 0.0f;
        int row = 0;
        for (; row + 4 <= rows; row += 4) {
            s0 += sums[row * mine]; s1 += sums[(row + 1) * mine]; s2 += sums[(row + 2) * mine]; s3 += sums[(row + 3) * mine];
        }
        for (; row < rows; ++row) s0 += sums[row * mine];
        const float s = (s0 + s1) + (s2 + s3);
        if (p.parts) p.parts[(((size_t)blockIdx.y * gridDim.z + dir) * kSmallSums + k) * p.H + u] = s;
        else atomicAdd((k < 4 ? p.g_bias + (size_t)k * p.L : p.g_peep + (size_t)(k - 4) * p.L) + dir * p.H + u, s);
    }
}

__global__ __launch_bounds__(256) void lstm_small_grads_sum(const SmallGradDirs p, int ndir, int chunks) {
    const size_t total = (size_t)ndir * kSmallSums * p.H, e = (size_t)blockIdx.x * kPartOutputs + threadIdx.x % kPartOutputs;
    const float v = sum_of_parts(p.parts, e, total, chunks, total);
    if (threadIdx.x >= kPartOutputs || e >= total) return;
    const int u = (int)(e % p.H), k = (int)(e / p.H % kSmallSums), dir = (int)(e / p.H / kSmallSums);
    (k < 4 ? p.g_bias + (size_t)k * p.L : p.g_peep + (size_t)(k - 4) * p.L)[dir * p.H + u] = v;
}

// ---------------------------------------------------------------------------------------------------
// Step-by-step recursion for layers the persistent kernels do not cover (more than 512 cells per direction): per time step one batched recurrent product through the
// matrix-product kernel and one cell kernel, i.e. the reference's own schedule (LstmLayer.cu:1743-1949,
// :2066-2255).  One thread per (direction, sequence, cell).
// ---------------------------------------------------------------------------------------------------
__global__ void lstm_forward_step(const ChainParams p, int step) {
    const int H = p.H, S = p.S, n = S * H;
    const int idx = blockIdx.x * blockDim.x + threadIdx.x;
    if (idx >= p.ndir * n) return;
    const int dir = idx / n, r = idx % n, s = r / H, j = r % H;
    const DirPtrs &D = p.d[dir];
    const int t = dir ? (p.T - 1 - step) : step;
    const int prev = dir ? t + 1 : t - 1;
    const bool first = step == 0;
    const size_t i = (size_t)t * n + (size_t)s * H + j;
    float *out = p.out ? p.out + ((size_t)t * S + s) * p.L + dir * H + j : nullptr;
    // padding is only looked for at or after the shortest sequence's end (LstmLayer.cu:1800-1803)
    if (t >= p.Tmin && p.pat[t * S + s] == 0) {
        if (dir) D.c[i] = 0.0f;  // only the time-reversed direction clears the cell state
        D.h[i] = 0.0f;
        if (out) *out = 0.0f;
        return;
    }
    const size_t ip = (size_t)prev * n + (size_t)s * H + j;
    float a_ni = D.ni[i] + p.bias * D.b[0][j];
    float a_ig = D.ig[i] + p.bias * D.b[1][j];
    float a_fg = D.fg[i] + p.bias * D.b[2][j];
    float a_og = D.og[i] + p.bias * D.b[3][j];
    float cp = 0.0f;
    if (!first) {
        cp = D.c[ip];
        a_ig += cp * D.peep[0][j];
        a_fg += cp * D.peep[1][j];
    }
    const float ni = tanh_act(a_ni), ig = logistic(a_ig), fg = logistic(a_fg);
    D.ni[i] = ni; D.ig[i] = ig; D.fg[i] = fg;
    float c = ni * ig;
    if (!first) c += cp * fg;
    D.c[i] = c;
    a_og += c * D.peep[2][j];
    const float og = logistic(a_og);
    D.og[i] = og;
    const float hv = tanh_act(c) * og;
    D.h[i] = hv;
    if (out) *out = hv;
}

// herr of both directions from the interleaved output errors (LstmLayer.cu:210-235)
__global__ void lstm_split_errors(const ChainParams p, size_t count) {
    size_t i = (size_t)blockIdx.x * blockDim.x + threadIdx.x;
    const size_t stride = (size_t)gridDim.x * blockDim.x;
    for (; i < count; i += stride) {
        const size_t slot = i / p.L;
        const int v = (int)(i % p.L);
        const float e = p.outerr[i];
        if (v < p.H) p.d[0].herr[slot * p.H + v] = e;
        else p.d[1].herr[slot * p.H + v - p.H] = e;
    }
}

__global__ void lstm_backward_step(const ChainParams p, int step) {
    const int H = p.H, S = p.S, n = S * H;
    const int idx = blockIdx.x * blockDim.x + threadIdx.x;
    if (idx >= p.ndir * n) return;
    const int dir = idx / n, r = idx % n, s = r / H, j = r % H;
    const DirPtrs &D = p.d[dir];
    const int t = dir ? step : (p.T - 1 - step);
    const int later = dir ? t - 1 : t + 1;    // the slot handled one step before this one
    const int earlier = dir ? t + 1 : t - 1;  // the slot the forward pass came from
    const bool first = step == 0, last = step == p.T - 1;
    const size_t i = (size_t)t * n + (size_t)s * H + j;
    if (t >= p.Tmin && p.pat[t * S + s] == 0) {
        D.dni[i] = 0.0f; D.dig[i] = 0.0f; D.dfg[i] = 0.0f; D.dog[i] = 0.0f;
        D.cerr[i] = 0.0f;
        return;
    }
    const float e = D.herr[i];
    const float ni = D.ni[i], ig = D.ig[i], og = D.og[i], c = D.c[i];
    const float tc = tanh_act(c);
    // the stored output-gate delta is read back before it is overwritten (LstmLayer.cu:300-310)
    const float d_og = (logistic_deriv(og) * tc * e) + D.dog[i];
    float ce = og * tanh_deriv(tc) * e + D.peep[2][j] * d_og;
    if (!first) {
        const size_t il = (size_t)later * n + (size_t)s * H + j;
        ce += (D.fg[il] * D.cerr[il] + D.peep[0][j] * D.dig[il] + D.peep[1][j] * D.dfg[il]);
    }
    const float d_ni = ig * tanh_deriv(ni) * ce;
    float d_fg = 0.0f;
    if (!last) d_fg = logistic_deriv(D.fg[i]) * D.c[(size_t)earlier * n + (size_t)s * H + j] * ce;
    const float d_ig = logistic_deriv(ig) * ni * ce;
    D.dni[i] = clip1(d_ni);
    D.dig[i] = clip1(d_ig);
    D.dfg[i] = clip1(d_fg);
    D.dog[i] = clip1(d_og);
    D.cerr[i] = ce;
}

}  // namespace
}  // namespace cnt

// ---------------------------------------------------------------------------------------------------
// Host side
// ---------------------------------------------------------------------------------------------------
struct cnt_lstm {
    cnt_lstm_desc desc;
    int ndir, H;
    int T, Tmin;  // current fraction
    const char *pat;
    float *state[2][12];
    int *abort_flag;
    int device;
    unsigned spin_limit;
    int poll_gap;
    int bmail_dirty;       // the backward mailbox may hold words that are not empty
    int flmail_dirty;      // the same for the XCD-local forward recursion's mailbox
    cnt::SlotOrder slot_order;  // the loaded fraction's slots, valid ones first (set by the owner of the pattern types, or null)
    int *own_order;             // maxT * S indices + 4 counts: the list the handle makes itself for a fraction with much padding
    bool make_order;            // false inside a network, whose sequencer makes one list for all layers
    int stepwise;          // no persistent recursion kernel for this geometry: one product + one cell kernel per step
    int *latch_host, *latch_dev;  // pinned host word a kernel that gives up sets; read by the host without a sync
    int *veto;             // a network's shared flag (device), or NULL
    // XCD-local backward recursion
    int solo;              // 1: lstm_forward_solo and lstm_backward_solo run the recursions
    int local;             // 1: lstm_forward_local and lstm_backward_local run the recursions
    int njobs, groups;
    int launch_jobs;       // jobs of one launch: as many as complete teams fit the compute units at once
    int local_jb, team;    // cells per workgroup and workgroups of a team
    int local_most;        // sequences of a job at most: 1 or 4
    int ctl_teams;
    unsigned *ctl;
    float *lmail;
    size_t lmail_words;
    float *flmail;         // XCD-local forward recursion: one mailbox per job
    float *sums;           // the backward recursion's sums, [group][direction][kSmallSums][cell]
    size_t flmail_words;
    long long *clocks;     // CNT_LSTM_TIMING: kClockWords of the forward and of the backward recursion
    int warm;  // read the recursion's inputs once before the XCD-local backward recursion (off; CNT_LSTM_WARM=1: on)
    int spread_lds_most;
    int spread_lds;  // dynamic LDS the XCD-local recursion asks for so that a compute unit takes one of its workgroups
    int poll_delay_local, poll_limit_local;  // pause before the first poll of a step in the XCD-local recursion, units of 64 clocks (-1: the job's), and its limit
    int mem_delay_local;   // pause of that recursion's store wave after the step barrier, same units
    int poll_delay_fwd_local, poll_limit_fwd_local, mem_delay_fwd_local;  // XCD-local forward recursion: the same, and before the loads of a step
    // set by every recursion launch: the failure latch is taken only once the launch that may have set it has ended
    // (the device's recursion-order event, see launch_in_order), so that no workgroup of that launch can set it (or the
    // veto) again after the report
    int launch_pending;
    // backward recursion run as ranges of steps: the step the next range has to start at (0: a fresh pass)
    int next_step;
};

namespace cnt {
namespace {

typedef void (*chain_kernel_t)(const ChainParams);

size_t weight_count(int P, int L, int bidir) {
    const size_t H = L / (bidir ? 2 : 1);
    return (size_t)4 * P * L + (size_t)4 * L + (size_t)4 * L * H + (size_t)3 * L;
}

void fill_chain_params(const cnt_lstm *h, const float *weights, ChainParams &p) {
    const cnt_lstm_desc &d = h->desc;
    const int P = d.P, L = d.L, H = h->H;
    std::memset(&p, 0, sizeof(p));
    p.H = H; p.L = L; p.S = d.S; p.T = h->T; p.Tmin = h->Tmin; p.ndir = h->ndir; p.bias = d.bias;
    p.step_begin = 0; p.step_end = h->T;
    p.pat = h->pat;
    const size_t off_bias = (size_t)4 * P * L, off_int = off_bias + (size_t)4 * L;
    const size_t off_peep = off_int + (size_t)4 * L * H;
    for (int dir = 0; dir < h->ndir; ++dir) {
        DirPtrs &D = p.d[dir];
        float *const *s = h->state[dir];
        D.ni = s[0]; D.ig = s[1]; D.fg = s[2]; D.og = s[3]; D.c = s[4]; D.h = s[5];
        D.herr = s[6]; D.dni = s[7]; D.dig = s[8]; D.dfg = s[9]; D.dog = s[10]; D.cerr = s[11];
        D.w_int = weights + off_int + (size_t)dir * H * H;
        for (int g = 0; g < 4; ++g) D.b[g] = weights + off_bias + (size_t)g * L + dir * H;
        for (int k = 0; k < 3; ++k) D.peep[k] = weights + off_peep + (size_t)k * L + dir * H;
    }
    p.spin_limit = h->spin_limit;
    p.abort_flag = h->abort_flag;
    p.latch = h->latch_dev;
    p.veto = h->veto;
    p.groups = h->groups; p.team = h->team; p.ctl_teams = h->ctl_teams;
    p.ctl = h->ctl;
    p.lmail = h->lmail;
    p.flmail = h->flmail;
    p.poll_limit = h->poll_limit_local; p.poll_limit_fwd = h->poll_limit_fwd_local;
    p.poll_delay = h->poll_delay_local; p.poll_gap = h->poll_gap; p.poll_delay_fwd = h->poll_delay_fwd_local;
    p.mem_delay_fwd = h->mem_delay_fwd_local;
    p.mem_delay = h->mem_delay_local;
}

// Reads the arrays a backward recursion is going to read, at full memory bandwidth, so that they sit in the
// memory-side cache when the recursion asks for them row by row.  A compute unit returns its vector loads in order
// over all of its waves: a row that has to come from HBM holds back the mailbox polls issued behind it, which costs
// the XCD-local recursion about 0.25 us per step (measured with the states evicted against just read); the pass
// itself takes some 20 us for 84 MB.
struct WarmParams {
    const void *ptr[16];
    unsigned long long bytes[16];
    int count;
};

__global__ __launch_bounds__(256) void warm_cache(const WarmParams w, const GuardParams g) {
    if (blockIdx.x == 0) guard_body(g);  // the guard in front of the recursion rides along (a launch less)
    const size_t first = ((size_t)blockIdx.x * blockDim.x + threadIdx.x) * 16, pitch = (size_t)gridDim.x * blockDim.x * 16;
    for (int a = 0; a < w.count; ++a) {
        const char *base = static_cast<const char *>(w.ptr[a]);
        for (size_t i = first; i + 16 <= w.bytes[a]; i += pitch) {
            const uint4 v = *reinterpret_cast<const uint4 *>(base + i);
            asm volatile("" ::"v"(v.x), "v"(v.y), "v"(v.z), "v"(v.w));
        }
    }
}

int warm_backward_inputs(const cnt_lstm *h, hipStream_t stream, const ChainParams &p, const GuardParams &g) {
    WarmParams w = {};
    const size_t state_bytes = (size_t)h->T * p.S * p.H * sizeof(float);
    auto add = [&](const void *ptr, size_t bytes) {
        if (ptr && (reinterpret_cast<uintptr_t>(ptr) & 15u) == 0) { w.ptr[w.count] = ptr; w.bytes[w.count] = bytes; ++w.count; }
    };
    for (int dir = 0; dir < h->ndir; ++dir) {
        const DirPtrs &D = p.d[dir];
        add(D.ni, state_bytes); add(D.ig, state_bytes); add(D.fg, state_bytes); add(D.og, state_bytes);
        add(D.c, state_bytes); add(D.dog, state_bytes);
    }
    add(p.outerr, (size_t)h->T * p.S * p.L * sizeof(float));
    ProfileScope prof(stream, "lstm_warm_states");
    hipLaunchKernelGGL(warm_cache, dim3(2048), dim3(256), 0, stream, w, g);
    CNT_HIP(hipGetLastError());
    return CNT_OK;
}

template <int PW, int JB, int MOST>
chain_kernel_t local_pair(bool fwd, bool clocks) {
    if (clocks) return fwd ? (chain_kernel_t)lstm_forward_local<PW, JB, MOST, true> : (chain_kernel_t)lstm_backward_local<PW, JB, MOST, true>;
    return fwd ? (chain_kernel_t)lstm_forward_local<PW, JB, MOST, false> : (chain_kernel_t)lstm_backward_local<PW, JB, MOST, false>;
}
template <int PW, int JB>
chain_kernel_t local_pair(bool fwd, int most, bool clocks) {
    return most == 1 ? local_pair<PW, JB, 1>(fwd, clocks) : local_pair<PW, JB, kLocalSeqs>(fwd, clocks);
}

// Cells per workgroup of a layer with H cells per direction and `jobs` jobs; 0: no XCD-local kernel.  A team should fit
// the 32 compute units of an XCD one workgroup each, and two teams where there are more jobs than XCDs: 16 cells of 8
// per workgroup for up to 128 cells, 32 of 8 up to 256 cells -- or 16 of 16 when there are more than eight jobs --, 32
// of 16 up to 512.  Measured, us per step forward / backward, MI355X: 256 cells 8 jobs 0.99 / 0.87 with 8 and 1.09 / 1.03
// with 16 cells per workgroup, 16 jobs 1.33 / 1.33 (two workgroups per compute unit) and 1.19 / 1.14; 200 cells 0.95 / 0.85 and
// 1.08 / 1.01, 1.23 / 1.16 and 1.14 / 1.05.
int local_cells(int H, int jobs) {
    if (const char *e = std::getenv("CNT_LSTM_LOCAL_JB")) return std::atoi(e);
    return H > 512 ? 0 : H <= 128 ? 8 : H <= 256 ? (jobs <= kLocalXcds ? 8 : 16) : 16;
}

// Groups of sequences per direction.  A job of fewer sequences takes shorter steps, so as many as complete teams fit the compute
// units one workgroup each; at least what four sequences per job need.
int local_groups(int H, int JB, int S, int ndir, int cus_per_xcd) {
    const int least = (S + kLocalSeqs - 1) / kLocalSeqs;
    if (JB <= 0) return least;
    const int resident = kLocalXcds * std::max(1, cus_per_xcd / ((H + JB - 1) / JB));
    return std::max(least, std::min(resident / ndir, S));
}

// Sequences of a job at most, by which mailboxes, launches and kernels go alike: one where every sequence has a job of its own and
// kernels for that exist.  (Layers of 129 to 256 cells take 16 cells per workgroup with more than eight jobs of four, so there are none
// for them; CNT_LSTM_LOCAL_JB takes fewer jobs there.)
constexpr int local_most(int H, int JB, int groups, int S) { return groups < S || (JB == 16 && H <= 256) ? kLocalSeqs : 1; }

// nullptr: no such kernel
chain_kernel_t pick_local_kernel(bool fwd, int H, int JB, int most, bool clocks) {
    const int PW = (H + 63) / 64;
    if (JB == 8) {
        switch (PW) {
            case 2: return local_pair<2, 8>(fwd, most, clocks);
            case 3: return local_pair<3, 8>(fwd, most, clocks);
            case 4: return local_pair<4, 8>(fwd, most, clocks);
        }
    }
    if (JB == 16) {
        switch (PW) {
            case 3: return most == kLocalSeqs ? local_pair<3, 16, kLocalSeqs>(fwd, clocks) : nullptr;
            case 4: return most == kLocalSeqs ? local_pair<4, 16, kLocalSeqs>(fwd, clocks) : nullptr;
            case 5: return local_pair<5, 16>(fwd, most, clocks);
            case 6: return local_pair<6, 16>(fwd, most, clocks);
            case 7: return local_pair<7, 16>(fwd, most, clocks);
            case 8: return local_pair<8, 16>(fwd, most, clocks);
        }
    }
    return nullptr;
}

template <int NW, int CELLS>
chain_kernel_t solo_pair(bool fwd) {
    return fwd ? (chain_kernel_t)lstm_forward_solo<NW, CELLS> : (chain_kernel_t)lstm_backward_solo<NW, CELLS>;
}
chain_kernel_t pick_solo_kernel(bool fwd, int H) {
    const bool aligned = H % 4 == 0;
    switch ((H + 15) / 16) {
        case 1: return H < 4 ? solo_pair<1, kSingle>(fwd) : aligned ? solo_pair<1, kAligned>(fwd) : solo_pair<1, kOverlapping>(fwd);
        case 2: return aligned ? solo_pair<2, kAligned>(fwd) : solo_pair<2, kOverlapping>(fwd);
        case 3: return aligned ? solo_pair<3, kAligned>(fwd) : solo_pair<3, kOverlapping>(fwd);
        case 4: return aligned ? solo_pair<4, kAligned>(fwd) : solo_pair<4, kOverlapping>(fwd);
    }
    return nullptr;
}

// allows a kernel the dynamic LDS of the launches below (once per device and kernel)
int set_spread_lds(const cnt_lstm *h, const void *kernel) {
    if (h->spread_lds <= 0) return CNT_OK;
    static std::mutex mu;
    static std::vector<std::pair<int, const void *>> done;
    std::lock_guard<std::mutex> lock(mu);
    const std::pair<int, const void *> key(h->device, kernel);
    if (std::find(done.begin(), done.end(), key) == done.end()) {
        CNT_HIP(hipFuncSetAttribute(kernel, hipFuncAttributeMaxDynamicSharedMemorySize, h->spread_lds_most));
        done.push_back(key);
    }
    return CNT_OK;
}

// Persistent recursion launches of one process run one at a time on a device.  Every workgroup of a team has to be
// resident before the team can take a step, and an XCD-local launch takes a compute unit per workgroup: two such
// launches that start together on different streams can each hold half of an XCD's compute units with half a team and
// wait for the other half until their bounded waits give up.  A launch therefore waits, in stream order, for the
// recursion launched before it (from whatever handle or stream); launches on one stream are ordered anyway and skip
// the wait.  The mutex keeps wait, launch and record of one launch together when several host threads launch.
struct RecursionOrder {
    std::mutex mu;
    hipEvent_t done = nullptr;
    hipStream_t last = nullptr;
    bool any = false;
};
RecursionOrder &recursion_order(int device) {
    static RecursionOrder order[64];
    return order[device >= 0 && device < 64 ? device : 0];
}
template <typename Launch>
int launch_in_order(cnt_lstm *h, hipStream_t stream, Launch launch) {
    RecursionOrder &o = recursion_order(h->device);
    std::lock_guard<std::mutex> lock(o.mu);
    if (!o.done) CNT_HIP(hipEventCreateWithFlags(&o.done, kOrderEvent));
    if (o.any && o.last != stream) CNT_HIP(hipStreamWaitEvent(stream, o.done, 0));
    launch();
    CNT_HIP(hipGetLastError());
    // Also what lstm_take_failure asks: once this record (or a later one, which waited for it) has completed, every
    // recursion launched so far has ended.
    CNT_HIP(hipEventRecord(o.done, stream));
    o.last = stream; o.any = true;
    h->launch_pending = 1;
    return CNT_OK;
}

// enough workgroups that njobs complete teams form on any spread over the XCDs
int local_blocks(const cnt_lstm *h) { return (h->launch_jobs * h->team + kLocalXcds * (h->team - 1) + 7) / 8 * 8; }

int launch_chain(cnt_lstm *h, hipStream_t stream, bool fwd, ChainParams &p) {
    CNT_REQUIRE(!fwd || (p.step_begin == 0 && p.step_end == h->T), "lstm: only the backward recursion runs a range of steps");
    CNT_REQUIRE(p.step_begin >= 0 && p.step_begin < p.step_end && p.step_end <= h->T, "lstm: steps %d..%d of %d",
                p.step_begin, p.step_end, h->T);
    if (!fwd) {
        // A range that ends before T leaves its last partial errors in the mailbox for the range that continues it.  A
        // launch that starts over instead (the pass was abandoned) must not find them: the mailbox is refilled.
        CNT_REQUIRE(p.step_begin == 0 || p.step_begin == h->next_step, "lstm: the backward recursion stands at step %d, "
                    "a range cannot start at step %d", h->next_step, p.step_begin);
        if (p.step_begin == 0 && h->next_step != 0) h->bmail_dirty = 1;
        h->next_step = p.step_end < h->T ? p.step_end : 0;
    }
    if (h->solo) {
        ProfileScope prof(stream, fwd ? "lstm_forward_chain" : "lstm_backward_chain");
        hipLaunchKernelGGL(pick_solo_kernel(fwd, h->H), dim3(h->njobs), dim3(solo_threads((h->H + 15) / 16)), 0, stream, p);
        CNT_HIP(hipGetLastError());
        return CNT_OK;
    }
    chain_kernel_t k = pick_local_kernel(fwd, h->H, h->local_jb, h->local_most, h->clocks != nullptr);
    CNT_REQUIRE(k != nullptr, "lstm: no recursion kernel for H=%d JB=%d", h->H, h->local_jb);
    // heals the handle after a launch that gave up, zeroes the placement counters; in front of the backward recursion it
    // can be part of the cache-warming launch
    GuardParams g = {};
    g.abort_flag = h->abort_flag;
    g.ctl = h->ctl; g.nctl = ctl_words(h->ctl_teams);
    g.mail[0] = reinterpret_cast<unsigned *>(h->lmail); g.words[0] = h->lmail_words;
    g.mail[1] = reinterpret_cast<unsigned *>(h->flmail); g.words[1] = h->flmail_words;
    // a launch that continues a recursion in the middle: the counters are zeroed, nothing is refilled or warmed
    const bool resumes = !fwd && p.step_begin > 0;
    const bool guard_rides = !fwd && h->warm && !resumes && !h->bmail_dirty && h->njobs <= h->launch_jobs;
    auto guard = [&]() -> int {
        hipLaunchKernelGGL(chain_guard, dim3(1), dim3(1024), 0, stream, g);
        CNT_HIP(hipGetLastError());
        return CNT_OK;
    };
    if (!guard_rides) CNT_TRY(guard());
    // Every word of a mailbox starts out empty and the recursions hand every word back, so the fill is needed once (and
    // the guard above refills after a recursion that gave up).
    int &dirty = fwd ? h->flmail_dirty : h->bmail_dirty;
    if (dirty) CNT_TRY(fill_words(stream, reinterpret_cast<unsigned *>(fwd ? h->flmail : h->lmail),
                                  fwd ? h->flmail_words : h->lmail_words, kEmpty));
    dirty = 0;
    if (!fwd && h->warm && !resumes) {
        GuardParams none = {};
        none.abort_flag = h->abort_flag;  // with nothing to zero or refill the body only reads the flag
        CNT_TRY(warm_backward_inputs(h, stream, p, guard_rides ? g : none));
    }
    ProfileScope prof(stream, fwd ? "lstm_forward_chain" : "lstm_backward_chain");
    // One workgroup per compute unit while the teams of an XCD fit its 32 compute units.  A team's workgroups take a step
    // in lock-step, and two of them on one compute unit share its four matrix pipes and its path to the L2 at exactly
    // the same moments: the dispatcher, left to itself, puts the 32 workgroups of a 256-cell team on 16-17 compute units,
    // and a step then takes 1.55 us instead of 1.30 us (measured on MI355X, benchmark layer: 932 -> 781 us per launch).
    // What keeps a further workgroup of this kernel off a compute unit is its LDS request: the launch asks for a little
    // more than half of a compute unit's LDS (unused dynamic shared memory), which still leaves room for two workgroups
    // of a matrix product beside it.  CNT_LSTM_SPREAD_LDS sets the request in bytes (0: none).
    CNT_TRY(set_spread_lds(h, reinterpret_cast<const void *>(k)));
    p.clocks = h->clocks ? h->clocks + (fwd ? 0 : kClockWords) : nullptr;
    for (int job0 = 0; job0 < h->njobs; job0 += h->launch_jobs) {
        if (job0) CNT_TRY(guard());
        p.job0 = (unsigned)job0;
        p.njobs = std::min(h->launch_jobs, h->njobs - job0);
        CNT_TRY(launch_in_order(h, stream, [&] {
            hipLaunchKernelGGL(k, dim3(local_blocks(h)), dim3(local_threads((h->H + 63) / 64, h->local_jb, h->local_most)), (size_t)h->spread_lds, stream, p);
        }));
    }
    return CNT_OK;
}

// How many workgroups of the recursion a compute unit takes, the LDS request that holds it to that (see the launch), and
// how many jobs a launch may hold: no more than complete teams are resident at once.  One workgroup per compute unit
// where all jobs fit that way; else as many as hold all jobs, up to kLocalSlots.
constexpr int kLocalSlots = 2;
void local_placement(cnt_lstm *h, int lds_per_cu, int cus_per_xcd) {
    int most = kLocalSlots;
    for (int fwd = 0; fwd < 2; ++fwd) {
        int fit = 0;
        const void *k = reinterpret_cast<const void *>(pick_local_kernel(fwd != 0, h->H, h->local_jb, h->local_most, h->clocks != nullptr));
        if (hipOccupancyMaxActiveBlocksPerMultiprocessor(&fit, k, local_threads((h->H + 63) / 64, h->local_jb, h->local_most), 0) != hipSuccess) {
            (void)hipGetLastError();
            fit = 1;
        }
        most = std::max(1, std::min(most, fit));
    }
    if (const char *e = std::getenv("CNT_LSTM_SLOTS")) most = std::max(1, std::atoi(e));
    auto jobs = [&](int slots) { return kLocalXcds * std::max(1, cus_per_xcd * slots / h->team); };
    int slots = 1;
    while (slots < most && jobs(slots) < h->njobs) ++slots;
    h->launch_jobs = std::min(h->njobs, jobs(slots));
    h->spread_lds_most = lds_per_cu >= (64 << 10) ? lds_per_cu / 2 + 2048 : 0;
    h->spread_lds = lds_per_cu >= (64 << 10) ? lds_per_cu / (slots + 1) + 2048 : 0;
    if (const char *e = std::getenv("CNT_LSTM_SPREAD_LDS")) h->spread_lds = h->spread_lds_most = std::atoi(e);
}

// The recursions of both directions step by step (see lstm_forward_step): per step the recurrent products of all
// gates and directions are one launch of the matrix-product kernel, accumulating into the slices of that step.
int stepwise_forward(cnt_lstm *h, hipStream_t stream, ChainParams &p) {
    const int H = h->H, S = h->desc.S, L = h->desc.L, n = S * H;
    const int threads = h->ndir * n;
    ProfileScope prof(stream, "lstm_forward_steps");
    for (int step = 0; step < h->T; ++step) {
        if (step > 0) {
            GemmArgs ga = {};
            ga.m = H; ga.n = S; ga.k = H;
            ga.a_kcontig = 1; ga.lda = H;  // W_int block [from + to*H]: element (to, from) at [to*H + from]
            ga.b_kcontig = 1; ga.ldb = H;
            ga.ldc = H;
            ga.nseg = 1; ga.splitk = 1; ga.epilogue = EPI_ADD;
            ga.nprob = 4 * h->ndir;
            for (int dir = 0; dir < h->ndir; ++dir) {
                const int t = dir ? (h->T - 1 - step) : step, prev = dir ? t + 1 : t - 1;
                for (int g = 0; g < 4; ++g) {
                    GemmProblem &pb = ga.prob[dir * 4 + g];
                    pb.A[0] = p.d[dir].w_int + (size_t)g * L * H;
                    pb.B[0] = p.d[dir].h + (size_t)prev * n;
                    pb.C = h->state[dir][g] + (size_t)t * n;
                }
            }
            CNT_TRY(gemm_launch(stream, ga));
        }
        hipLaunchKernelGGL(lstm_forward_step, dim3((threads + 255) / 256), dim3(256), 0, stream, p, step);
        CNT_HIP(hipGetLastError());
    }
    return CNT_OK;
}

int stepwise_backward(cnt_lstm *h, hipStream_t stream, ChainParams &p) {
    const int H = h->H, S = h->desc.S, L = h->desc.L, n = S * H;
    const int threads = h->ndir * n;
    const size_t count = (size_t)L * h->T * S;
    ProfileScope prof(stream, "lstm_backward_steps");
    if (h->ndir == 2) {
        size_t blocks = (count + 255) / 256;
        if (blocks > 4096) blocks = 4096;
        hipLaunchKernelGGL(lstm_split_errors, dim3((unsigned)blocks), dim3(256), 0, stream, p, count);
        CNT_HIP(hipGetLastError());
    } else {
        CNT_HIP(hipMemcpyAsync(p.d[0].herr, p.outerr, count * sizeof(float), hipMemcpyDeviceToDevice, stream));
    }
    for (int step = 0; step < h->T; ++step) {
        if (step > 0) {
            // herr[t] += sum over gates of W_int[g] * delta_g[later]
            GemmArgs ga = {};
            ga.m = H; ga.n = S; ga.k = H;
            ga.a_kcontig = 0; ga.lda = H;
            ga.b_kcontig = 1; ga.ldb = H;
            ga.ldc = H;
            ga.nseg = 4; ga.splitk = 1; ga.epilogue = EPI_ADD;
            ga.nprob = h->ndir;
            for (int dir = 0; dir < h->ndir; ++dir) {
                const int t = dir ? step : (h->T - 1 - step), later = dir ? t - 1 : t + 1;
                GemmProblem &pb = ga.prob[dir];
                for (int g = 0; g < 4; ++g) {
                    pb.A[g] = p.d[dir].w_int + (size_t)g * L * H;
                    pb.B[g] = h->state[dir][7 + g] + (size_t)later * n;
                }
                pb.C = p.d[dir].herr + (size_t)t * n;
            }
            CNT_TRY(gemm_launch(stream, ga));
        }
        hipLaunchKernelGGL(lstm_backward_step, dim3((threads + 255) / 256), dim3(256), 0, stream, p, step);
        CNT_HIP(hipGetLastError());
    }
    // a unidirectional layer leaves the summed errors in the caller's buffer (LstmLayer.cu:2086-2087, :2378-2381)
    if (p.herr_out)
        CNT_HIP(hipMemcpyAsync(p.herr_out, p.d[0].herr, count * sizeof(float), hipMemcpyDeviceToDevice, stream));
    return CNT_OK;
}

}  // namespace
}  // namespace cnt

extern "C" {

long cnt_lstm_weight_count(int P, int L, int bidir) { return (long)cnt::weight_count(P, L, bidir); }

int cnt_lstm_create(const cnt_lstm_desc *desc, cnt_lstm **out) {
    using namespace cnt;
    CNT_REQUIRE(desc && out, "lstm_create: null argument");
    CNT_REQUIRE(desc->P > 0 && desc->L > 0 && desc->S > 0 && desc->maxT > 0, "lstm_create: non-positive size");
    // the reference refuses odd bidirectional sizes (LstmLayer.cu:1091-1092)
    CNT_REQUIRE(!desc->bidir || desc->L % 2 == 0, "Cannot create a bidirectional layer with an odd layer size");
    const int ndir = desc->bidir ? 2 : 1;
    const int H = desc->L / ndir;
    // up to 512 cells per direction run as persistent recursion kernels; everything else step by step
    int solo_cells = kSoloCells;
    if (const char *e = std::getenv("CNT_LSTM_SOLO")) solo_cells = std::min(std::atoi(e), kSoloCells);
    // (the one-workgroup kernels address their arrays by 31-bit byte offsets)
    const bool solo = H <= solo_cells && (size_t)desc->L * desc->maxT * desc->S < ((size_t)1 << 29) - 16;
    int per_cu = 0, cus = 0;  // LDS of a compute unit, compute units
    {
        int dev = 0;
        if (hipGetDevice(&dev) != hipSuccess ||
            hipDeviceGetAttribute(&per_cu, hipDeviceAttributeMaxSharedMemoryPerMultiprocessor, dev) != hipSuccess ||
            hipDeviceGetAttribute(&cus, hipDeviceAttributeMultiprocessorCount, dev) != hipSuccess) {
            (void)hipGetLastError();
            per_cu = cus = 0;
        }
    }
    // jobs of one direction and at most four sequences (the one-workgroup kernels gain nothing from smaller jobs)
    const int least = (desc->S + kLocalSeqs - 1) / kLocalSeqs;
    const int local_jb = local_cells(H, ndir * least);
    const int groups = solo ? least : local_groups(H, local_jb, desc->S, ndir, cus / kLocalXcds);
    const int most = local_most(H, local_jb, groups, desc->S);
    const bool stepwise = (!solo && pick_local_kernel(true, H, local_jb, most, false) == nullptr) || std::getenv("CNT_LSTM_STEPWISE") != nullptr;

    cnt_lstm *h = new (std::nothrow) cnt_lstm();
    CNT_REQUIRE(h != nullptr, "lstm_create: out of host memory");
    std::memset(h, 0, sizeof(*h));
    h->desc = *desc; h->ndir = ndir; h->H = H;
    h->stepwise = stepwise ? 1 : 0;
    h->solo = solo && !stepwise ? 1 : 0;
    h->local = !solo && !stepwise ? 1 : 0;
    h->local_jb = local_jb;
    h->local_most = most;
    h->bmail_dirty = 1;
    h->flmail_dirty = 1;
    h->spin_limit = 1u << 22;
    if (const char *e = std::getenv("CNT_LSTM_SPIN_LIMIT")) h->spin_limit = (unsigned)std::strtoul(e, nullptr, 10);
    h->poll_delay_local = h->poll_delay_fwd_local = -1;
    h->poll_limit_local = h->poll_limit_fwd_local = 1 << 20;
    h->mem_delay_local = kStorePause;
    if (const char *e = std::getenv("CNT_LSTM_MEM_DELAY")) h->mem_delay_local = std::atoi(e);
    // The full-bandwidth read of the recursion's inputs in front of it (warm_cache) was worth 0.15 ms per model pass
    // while loads were issued in front of the polls in every step; now it costs more than it gains.  CNT_LSTM_WARM=1 turns
    // it on.
    h->make_order = true;
    if (const char *e = std::getenv("CNT_LSTM_SKIP_PADDING")) h->make_order = std::atoi(e) != 0;
    h->warm = 0;
    if (const char *e = std::getenv("CNT_LSTM_WARM")) h->warm = std::atoi(e) != 0;
    if (const char *e = std::getenv("CNT_LSTM_POLL_DELAY")) h->poll_delay_local = std::atoi(e);
    h->mem_delay_fwd_local = kLoadPause;
    if (const char *e = std::getenv("CNT_LSTM_POLL_DELAY_FWD")) h->poll_delay_fwd_local = std::atoi(e);
    if (const char *e = std::getenv("CNT_LSTM_POLL_GAP")) h->poll_gap = std::atoi(e);
    hipError_t err = hipGetDevice(&h->device);
    const size_t nstate = (size_t)H * desc->maxT * desc->S;
    for (int dir = 0; dir < ndir && err == hipSuccess; ++dir) {
        for (int w = 0; w < 12 && err == hipSuccess; ++w) {
            err = hipMalloc(reinterpret_cast<void **>(&h->state[dir][w]), nstate * sizeof(float));
            if (err == hipSuccess) err = hipMemset(h->state[dir][w], 0, nstate * sizeof(float));
        }
    }
    h->groups = groups;
    h->njobs = ndir * groups;
    if (h->local) {
        h->team = (H + h->local_jb - 1) / h->local_jb;
        h->lmail_words = h->flmail_words = (size_t)h->njobs * local_job_words(h->team, h->local_jb, h->local_most);
        if (err == hipSuccess && std::getenv("CNT_LSTM_TIMING")) {
            err = hipMalloc(reinterpret_cast<void **>(&h->clocks), 2 * kClockWords * sizeof(long long));
            if (err == hipSuccess) err = hipMemset(h->clocks, 0, 2 * kClockWords * sizeof(long long));
        }
        local_placement(h, per_cu, cus / kLocalXcds);
        h->ctl_teams = local_blocks(h) / h->team + 1;
        if (err == hipSuccess) err = hipMalloc(reinterpret_cast<void **>(&h->lmail), h->lmail_words * sizeof(float));
        if (err == hipSuccess) err = hipMalloc(reinterpret_cast<void **>(&h->flmail), h->flmail_words * sizeof(float));
        if (err == hipSuccess) err = hipMalloc(reinterpret_cast<void **>(&h->ctl), ctl_words(h->ctl_teams) * sizeof(unsigned));
        if (err == hipSuccess) err = hipMemset(h->ctl, 0, ctl_words(h->ctl_teams) * sizeof(unsigned));
    }
    if (err == hipSuccess && !h->stepwise)
        err = hipMalloc(reinterpret_cast<void **>(&h->sums), (size_t)h->njobs * kSmallSums * H * sizeof(float));
    if (err == hipSuccess) err = hipMalloc(reinterpret_cast<void **>(&h->own_order), ((size_t)h->desc.maxT * h->desc.S + 4) * sizeof(int));
    if (err == hipSuccess) err = hipMalloc(reinterpret_cast<void **>(&h->abort_flag), sizeof(int));
    if (err == hipSuccess) err = hipMemset(h->abort_flag, 0, sizeof(int));
    // the word a kernel that gives up sets for the host: pinned, mapped, coherent host memory
    if (err == hipSuccess) err = hipHostMalloc(reinterpret_cast<void **>(&h->latch_host), sizeof(int), hipHostMallocMapped);
    if (err == hipSuccess) {
        *h->latch_host = 0;
        err = hipHostGetDevicePointer(reinterpret_cast<void **>(&h->latch_dev), h->latch_host, 0);
    }
    if (err != hipSuccess) {
        set_error("lstm_create: %s", hipGetErrorString(err));
        cnt_lstm_destroy(h);
        return CNT_ERR_HIP;
    }
    *out = h;
    return CNT_OK;
}

int cnt_lstm_destroy(cnt_lstm *h) {
    if (!h) return CNT_OK;
    for (int dir = 0; dir < 2; ++dir) {
        for (int w = 0; w < 12; ++w)
            if (h->state[dir][w]) (void)hipFree(h->state[dir][w]);
    }
    if (h->abort_flag) (void)hipFree(h->abort_flag);
    if (h->lmail) (void)hipFree(h->lmail);
    if (h->flmail) (void)hipFree(h->flmail);
    if (h->ctl) (void)hipFree(h->ctl);
    if (h->sums) (void)hipFree(h->sums);
    if (h->clocks) (void)hipFree(h->clocks);
    if (h->own_order) (void)hipFree(h->own_order);
    if (h->latch_host) (void)hipHostFree(h->latch_host);
    delete h;
    return CNT_OK;
}

namespace {
// everything cnt_lstm_load_sequences does; the stored output-gate deltas are cleared here, or listed in `collect` for the caller
int load_sequences_impl(cnt_lstm *h, hipStream_t stream, const char *patTypes, int curMaxT, int curMinT, cnt::LoadClears *collect) {
    using namespace cnt;
    CNT_REQUIRE(h && patTypes, "lstm_load_sequences: null argument");
    CNT_REQUIRE(curMaxT >= 1 && curMaxT <= h->desc.maxT, "lstm_load_sequences: curMaxT %d outside 1..%d", curMaxT,
                h->desc.maxT);
    CNT_REQUIRE(curMinT >= 0 && curMinT <= curMaxT, "lstm_load_sequences: curMinT %d outside 0..%d", curMinT, curMaxT);
    h->T = curMaxT; h->Tmin = curMinT; h->pat = patTypes;
    h->slot_order = SlotOrder{nullptr, nullptr};
    // A fraction with much padding (the shortest sequence at most 3/4 of the longest, and enough slots for the list's one
    // launch to pay): the weight gradients sum over its valid slots only (GemmArgs::k_order).  The owner of a network's
    // pattern types hands its own list over instead (lstm_set_slot_order).
    if (h->make_order && h->own_order && (long)curMaxT * h->desc.S >= 2048 && (curMaxT - curMinT) * 4 >= curMaxT) {
        const int n = curMaxT * h->desc.S;
        int *count = h->own_order + (size_t)h->desc.maxT * h->desc.S;
        CNT_TRY(slot_order_build(stream, patTypes, n, h->desc.S, h->own_order, count));
        h->slot_order = SlotOrder{h->own_order, count};
    }
    if (h->next_step != 0) { h->bmail_dirty = 1; h->next_step = 0; }  // an abandoned partial backward pass
    const size_t nstate = (size_t)h->H * h->desc.maxT * h->desc.S;
    if (collect && nstate % 4 == 0 && collect->n + h->ndir <= kLoadClears) {
        for (int dir = 0; dir < h->ndir; ++dir) {
            collect->ptr[collect->n] = h->state[dir][10];
            collect->count[collect->n] = nstate;
            ++collect->n;
        }
        return CNT_OK;
    }
    // stored output-gate deltas of both directions, one launch
    if (h->ndir == 2) CNT_TRY(fill_zero_pair(stream, h->state[0][10], nstate, h->state[1][10], nstate));
    else CNT_TRY(fill_zero(stream, h->state[0][10], nstate));
    return CNT_OK;
}
}  // namespace

int cnt_lstm_load_sequences(cnt_lstm *h, void *stream, const char *patTypes, int curMaxT, int curMinT) {
    return load_sequences_impl(h, static_cast<hipStream_t>(stream), patTypes, curMaxT, curMinT, nullptr);
}

extern "C++" int cnt::lstm_load_sequences_collect(cnt_lstm *h, hipStream_t stream, const char *patTypes, int curMaxT,
                                                  int curMinT, LoadClears &clears) {
    return load_sequences_impl(h, stream, patTypes, curMaxT, curMinT, &clears);
}

int cnt_lstm_set_wait_bounds(cnt_lstm *h, unsigned spin_limit, int poll_delay_backward, int poll_delay_forward) {
    using namespace cnt;
    CNT_REQUIRE(h, "lstm_set_wait_bounds: null handle");
    CNT_REQUIRE(poll_delay_backward >= 0 && poll_delay_backward <= 4096 && poll_delay_forward >= 0 &&
                poll_delay_forward <= 4096, "lstm_set_wait_bounds: poll delays must be within 0..4096");
    h->spin_limit = spin_limit;
    h->poll_limit_local = poll_delay_backward;
    h->mem_delay_local = std::min(poll_delay_backward, kStorePause);
    h->poll_limit_fwd_local = poll_delay_forward;
    return CNT_OK;
}

float *cnt_lstm_state(cnt_lstm *h, int dir, int which) {
    if (!h || dir < 0 || dir >= h->ndir || which < 0 || which >= 12) return nullptr;
    return h->state[dir][which];
}

static const char *kGaveUp = "lstm: a recursion kernel gave up waiting for a neighbouring workgroup; results are invalid";

extern "C++" void cnt::lstm_set_veto(cnt_lstm *h, int *veto) {
    if (h) h->veto = veto;
}

extern "C++" int cnt::lstm_is_persistent(const cnt_lstm *h) { return h && h->local ? 1 : 0; }

extern "C++" void cnt::lstm_set_slot_order(cnt_lstm *h, const SlotOrder *order) {
    if (!h) return;
    h->make_order = false;  // from now on the caller's lists (or none) are the ones that count: no list of the handle's own
    h->slot_order = order ? *order : SlotOrder{nullptr, nullptr};
}

extern "C++" int cnt::lstm_wait_recursion(cnt_lstm *h, hipStream_t other) {
    CNT_REQUIRE(h, "lstm_wait_recursion: null handle");
    RecursionOrder &o = recursion_order(h->device);
    std::lock_guard<std::mutex> lock(o.mu);
    if (o.done && o.any) CNT_HIP(hipStreamWaitEvent(other, o.done, 0));
    return CNT_OK;
}

extern "C++" int cnt::lstm_take_failure(cnt_lstm *h) {
    if (!h || !h->latch_host) return 0;
    volatile int *latch = h->latch_host;
    if (*latch == 0) return 0;
    if (h->launch_pending) {
        // the launch that set the mark may still be running: its other workgroups would set it again after the report
        RecursionOrder &o = recursion_order(h->device);
        std::lock_guard<std::mutex> lock(o.mu);
        if (o.done && hipEventQuery(o.done) != hipSuccess) {
            (void)hipGetLastError();
            return 0;  // reported by a later call, once the launch has ended
        }
        h->launch_pending = 0;
    }
    *latch = 0;
    return 1;
}

// Every entry point that launches or consumes a recursion starts with this: a recursion that gave up in an EARLIER
// call (and has ended by now) turns the current call into CNT_ERR_DEVICE, also for callers that never call
// cnt_lstm_check.  The handle itself is healed by the guard kernel in front of its next launch.  A handle that belongs to
// a network (it carries the network's veto flag) leaves the report to the network's entry points.
#define CNT_LSTM_REPORT_FAILURE(h)              \
    do {                                        \
        if (!(h)->veto && cnt::lstm_take_failure(h)) { \
            cnt::set_error("%s", kGaveUp);      \
            return CNT_ERR_DEVICE;              \
        }                                       \
    } while (0)

// CNT_LSTM_TIMING: means over the workgroups of the handle's last recursion in either direction of time, to stderr; then the
// counts start over.  CNT_LSTM_TRACE: the points of the steps, too.
static int print_clocks(cnt_lstm *h) {
    using namespace cnt;
    std::vector<long long> all(2 * kClockWords);
    CNT_HIP(hipMemcpy(all.data(), h->clocks, all.size() * sizeof(long long), hipMemcpyDeviceToHost));
    CNT_HIP(hipMemset(h->clocks, 0, all.size() * sizeof(long long)));
    for (int backward = 0; backward < 2; ++backward) {
        const long long *counts = all.data() + (backward ? kClockWords : 0), *traces = counts + (size_t)kClockBlocks * kClockCounts;
        double m[kClockCounts] = {};
        int active = 0;
        for (unsigned b = 0; b < kClockBlocks; ++b) {
            const long long *c = counts + (size_t)b * kClockCounts, *t = traces + (size_t)b * kTraceWords;
            if (c[CLK_LOOP] == 0) continue;
            ++active;
            for (int q = 0; q < kClockCounts; ++q) m[q] += (double)c[q];
            if (!std::getenv("CNT_LSTM_TRACE")) continue;
            std::fprintf(stderr, "trace %s block %u job %lld member %lld xcd %lld:", backward ? "backward" : "forward", b, t[0], t[1], t[2]);
            for (int q = 4; q < kTraceWords; ++q) std::fprintf(stderr, " %lld", t[q]);
            std::fprintf(stderr, "\n");
        }
        if (!active) continue;
        const double steps = std::max(m[CLK_STEPS], 1.0), us = 0.01 / steps;  // a job leaves out steps on which all its sequences are padding
        std::fprintf(stderr, "lstm %s per step [us]: %s wave pause+poll %.3f (%.2f rounds) %s %.3f barrier %.3f loop %.3f | load wave busy "
                     "%.3f store wave %.3f %s wave %.3f (T=%d, %.1f steps of a job, %d workgroups)\n", backward ? "backward" : "forward",
                     backward ? "cell" : "gather", m[CLK_WAIT] * us, m[CLK_ROUNDS] / steps, backward ? "update" : "product",
                     m[CLK_REST] * us, m[CLK_BARRIER] * us, m[CLK_LOOP] * us, m[CLK_LOAD] * us, m[CLK_STORE] * us,
                     backward ? "product" : "cell", m[CLK_OTHER] * us, h->T, steps / active, active);
    }
    return CNT_OK;
}

int cnt_lstm_check(cnt_lstm *h, void *stream) {
    using namespace cnt;
    CNT_REQUIRE(h, "lstm_check: null handle");
    CNT_HIP(hipStreamSynchronize(static_cast<hipStream_t>(stream)));
    if (h->clocks) CNT_TRY(print_clocks(h));
    if (lstm_take_failure(h)) {
        set_error("%s", kGaveUp);
        return CNT_ERR_DEVICE;
    }
    return CNT_OK;
}

int cnt_lstm_forward(cnt_lstm *h, void *stream_, const float *weights, const float *x, float *outputs) {
    using namespace cnt;
    CNT_REQUIRE(h && weights && x && outputs, "lstm_forward: null argument");
    CNT_REQUIRE(h->T > 0, "lstm_forward: load_sequences has not been called");
    CNT_LSTM_REPORT_FAILURE(h);
    if (h->next_step != 0) { h->bmail_dirty = 1; h->next_step = 0; }  // new states: a partial backward pass is void
    hipStream_t stream = static_cast<hipStream_t>(stream_);
    const cnt_lstm_desc &d = h->desc;
    const int P = d.P, L = d.L, H = h->H, N = h->T * d.S;

    // input projections of all gates and directions in one launch: a_g = W_in[g]^T x
    GemmArgs ga = {};
    ga.m = H; ga.n = N; ga.k = P;
    ga.a_kcontig = 1; ga.lda = P;  // W_in block is P x H column-major: element (unit, p) at [unit*P + p]
    ga.b_kcontig = 1; ga.ldb = P;
    ga.ldc = H;
    ga.nseg = 1; ga.splitk = 1; ga.epilogue = EPI_STORE;
    ga.nprob = 4 * h->ndir;
    for (int dir = 0; dir < h->ndir; ++dir)
        for (int g = 0; g < 4; ++g) {
            GemmProblem &pb = ga.prob[dir * 4 + g];
            pb.A[0] = weights + (size_t)g * P * L + (size_t)dir * P * H;
            pb.B[0] = x;
            pb.C = h->state[dir][g];
        }
    // (the recursion leaves padding slots out; what it finds there as pre-activations reaches nothing)
    ga.cols = h->slot_order.order; ga.cols_count = h->slot_order.count;
    ga.label = "gemm:lstm_input_projection";
    CNT_TRY(gemm_launch(stream, ga));

    ChainParams p;
    fill_chain_params(h, weights, p);
    // the reference lets a unidirectional layer write its outputs directly (buffer swap, :1747-1749)
    p.out = outputs;
    if (h->stepwise) return stepwise_forward(h, stream, p);
    return launch_chain(h, stream, true, p);
}

int cnt_lstm_backward_errors(cnt_lstm *h, void *stream_, const float *weights, float *output_errors,
                             float *prev_errors) {
    return cnt::lstm_backward_errors_sums(h, static_cast<hipStream_t>(stream_), weights, output_errors, prev_errors, nullptr);
}

// weight_updates: the bias and peephole gradients are summed up on the way, for lstm_backward_weights_grouped with sums_done; only within
// one call of this library's, between whose halves nobody can change the states
extern "C++" int cnt::lstm_backward_errors_sums(cnt_lstm *h, hipStream_t stream, const float *weights, float *output_errors,
                                                float *prev_errors, float *weight_updates) {
    CNT_REQUIRE(h && weights && output_errors, "lstm_backward_errors: null argument");
    CNT_REQUIRE(h->T > 0, "lstm_backward_errors: load_sequences has not been called");
    CNT_LSTM_REPORT_FAILURE(h);

    // 1. error recursion (splits the interleaved output errors on the fly)
    ChainParams p;
    fill_chain_params(h, weights, p);
    p.outerr = output_errors;
    p.herr_out = (h->ndir == 1) ? output_errors : nullptr;
    if (weight_updates && h->sums) {
        const size_t P = (size_t)h->desc.P, L = (size_t)h->desc.L, H = (size_t)h->H;
        p.sum_scale = h->desc.bias;
        if (h->groups == 1) {  // a job has all sequences of a direction: its sums are the gradients
            p.sum_bias = weight_updates + 4 * P * L;
            p.sum_peep = p.sum_bias + 4 * L + 4 * L * H;
            p.sum_k = (int)L; p.sum_dir = (int)H;
        } else {
            p.sum_bias = h->sums; p.sum_peep = h->sums + 4 * H;
            p.sum_k = (int)H; p.sum_dir = kSmallSums * (int)H; p.sum_group = h->ndir * kSmallSums * (int)H;
        }
    }
    if (h->stepwise) CNT_TRY(stepwise_backward(h, stream, p));
    else CNT_TRY(launch_chain(h, stream, false, p));

    // 2. error to the preceding layer
    if (prev_errors) return cnt_lstm_backward_prev_errors(h, stream, weights, prev_errors);
    return CNT_OK;
}

int cnt_lstm_backward_prev_errors(cnt_lstm *h, void *stream_, const float *weights, float *prev_errors) {
    CNT_REQUIRE(h, "lstm_backward_prev_errors: null argument");
    return cnt_lstm_backward_prev_errors_range(h, stream_, weights, prev_errors, 0, h->T);
}

int cnt_lstm_backward_steps_done(const cnt_lstm *h, int steps, int *t_begin, int *t_end) {
    using namespace cnt;
    CNT_REQUIRE(h && t_begin && t_end, "lstm_backward_steps_done: null argument");
    CNT_REQUIRE(h->T > 0 && steps >= 0 && steps <= h->T, "lstm_backward_steps_done: %d steps of %d", steps, h->T);
    // the first direction's recursion runs from the last time step down, the second one's from the first up
    *t_begin = h->T - steps;
    *t_end = h->ndir == 2 ? steps : h->T;
    if (*t_end < *t_begin) *t_end = *t_begin;
    return CNT_OK;
}

int cnt_lstm_backward_errors_range(cnt_lstm *h, void *stream_, const float *weights, float *output_errors, int step_begin,
                                   int step_end) {
    using namespace cnt;
    CNT_REQUIRE(h && weights && output_errors, "lstm_backward_errors_range: null argument");
    CNT_REQUIRE(h->T > 0, "lstm_backward_errors_range: load_sequences has not been called");
    CNT_REQUIRE(cnt_lstm_backward_can_split(h), "lstm_backward_errors_range: this layer's recursion cannot run a range of its "
                "steps (cnt_lstm_backward_can_split)");
    CNT_LSTM_REPORT_FAILURE(h);
    ChainParams p;
    fill_chain_params(h, weights, p);
    p.outerr = output_errors;
    p.herr_out = (h->ndir == 1) ? output_errors : nullptr;
    p.step_begin = step_begin; p.step_end = step_end;
    return launch_chain(h, static_cast<hipStream_t>(stream_), false, p);
}

int cnt_lstm_backward_can_split(const cnt_lstm *h) { return h && !h->stepwise && h->H >= 64 ? 1 : 0; }

int cnt_lstm_backward_prev_errors_range(cnt_lstm *h, void *stream_, const float *weights, float *prev_errors, int t_begin,
                                        int t_end) {
    using namespace cnt;
    CNT_REQUIRE(h && weights && prev_errors, "lstm_backward_prev_errors: null argument");
    CNT_REQUIRE(h->T > 0, "lstm_backward_prev_errors: load_sequences has not been called");
    CNT_REQUIRE(t_begin >= 0 && t_begin <= t_end && t_end <= h->T, "lstm_backward_prev_errors: time steps %d..%d of %d",
                t_begin, t_end, h->T);
    CNT_LSTM_REPORT_FAILURE(h);
    if (t_begin == t_end) return CNT_OK;
    hipStream_t stream = static_cast<hipStream_t>(stream_);
    const cnt_lstm_desc &d = h->desc;
    const int P = d.P, L = d.L, H = h->H, S = d.S, N = (t_end - t_begin) * S;
    const size_t first = (size_t)t_begin * S;  // slots are time-major
    // e_x = sum_{dir,g} W_in[g,dir] * delta[g,dir]  (overwrite)
    {
        GemmArgs ga = {};
        ga.m = P; ga.n = N; ga.k = H;
        ga.a_kcontig = 0; ga.lda = P;
        ga.b_kcontig = 1; ga.ldb = H;
        ga.ldc = P;
        ga.nseg = 4 * h->ndir; ga.nprob = 1; ga.splitk = 1; ga.epilogue = EPI_STORE;
        for (int dir = 0; dir < h->ndir; ++dir)
            for (int g = 0; g < 4; ++g) {
                ga.prob[0].A[dir * 4 + g] = weights + (size_t)g * P * L + (size_t)dir * P * H;
                ga.prob[0].B[dir * 4 + g] = h->state[dir][7 + g] + first * H;
            }
        ga.prob[0].C = prev_errors + first * P;
        if (t_begin == 0 && t_end == h->T) { ga.cols = h->slot_order.order; ga.cols_count = h->slot_order.count; }  // (no deltas on padding)
        ga.label = "gemm:lstm_prev_errors";
        CNT_TRY(gemm_launch(stream, ga));
    }
    return CNT_OK;
}

// cnt_lstm_backward_prev_errors whose product also applies the derivative of the preceding (dense) layer's activation
extern "C++" int cnt::lstm_prev_errors_delta(cnt_lstm *h, hipStream_t stream, const float *weights, float *prev_errors,
                                             int prev_act, const float *prev_y) {
    CNT_REQUIRE(h && weights && prev_errors && prev_y, "lstm_prev_errors_delta: null argument");
    CNT_REQUIRE(h->T > 0, "lstm_prev_errors_delta: load_sequences has not been called");
    CNT_LSTM_REPORT_FAILURE(h);
    const cnt_lstm_desc &d = h->desc;
    const int P = d.P, L = d.L, H = h->H, N = h->T * d.S;
    GemmArgs ga = {};
    ga.m = P; ga.n = N; ga.k = H;
    ga.a_kcontig = 0; ga.lda = P;
    ga.b_kcontig = 1; ga.ldb = H;
    ga.ldc = P;
    ga.nseg = 4 * h->ndir; ga.nprob = 1; ga.splitk = 1; ga.epilogue = EPI_STORE_DELTA;
    ga.act = prev_act;
    for (int dir = 0; dir < h->ndir; ++dir)
        for (int g = 0; g < 4; ++g) {
            ga.prob[0].A[dir * 4 + g] = weights + (size_t)g * P * L + (size_t)dir * P * H;
            ga.prob[0].B[dir * 4 + g] = h->state[dir][7 + g];
        }
    ga.prob[0].C = prev_errors;
    ga.prob[0].aux_in = prev_y;
    ga.cols = h->slot_order.order; ga.cols_count = h->slot_order.count;
    ga.label = "gemm:lstm_prev_errors";
    return gemm_launch(stream, ga);
}

int cnt_lstm_backward_weights(cnt_lstm *h, void *stream, const float *x, float *weight_updates) {
    return cnt::lstm_backward_weights_grouped(h, static_cast<hipStream_t>(stream), x, weight_updates, false);
}

extern "C++" int cnt::lstm_backward_weights_grouped(cnt_lstm *h, hipStream_t stream, const float *x, float *weight_updates, bool sums_done,
                                                    DirectGroup *group) {
    DirectGroup own;
    own.count = own.blocks = 0;
    if (!group) {
        // products of few blocks: both in one launch (a layer of 256 cells over 800 slots 14 + 9.5 us one after the other)
        CNT_TRY(lstm_backward_weights_grouped(h, stream, x, weight_updates, sums_done, &own));
        return gemm_group_launch(stream, own);
    }
    CNT_REQUIRE(h && x && weight_updates, "lstm_backward_weights: null argument");
    CNT_REQUIRE(h->T > 0, "lstm_backward_weights: load_sequences has not been called");
    CNT_LSTM_REPORT_FAILURE(h);
    const cnt_lstm_desc &d = h->desc;
    const int P = d.P, L = d.L, H = h->H, S = d.S, N = h->T * S;

    // 3. weight updates (overwritten every call, as the reference's transform-assign does)
    const size_t nW = weight_count(P, L, d.bidir);
    const size_t off_bias = (size_t)4 * P * L, off_int = off_bias + (size_t)4 * L;
    const size_t off_peep = off_int + (size_t)4 * L * H;
    if (sums_done && h->sums) {
        if (h->groups > 1) {
            SmallGradDirs sp = {};
            sp.H = H; sp.L = L; sp.parts = h->sums;
            sp.g_bias = weight_updates + off_bias;
            sp.g_peep = weight_updates + off_peep;
            const size_t sums = (size_t)h->ndir * kSmallSums * H;
            ProfileScope prof(stream, "lstm_small_grads");
            hipLaunchKernelGGL(lstm_small_grads_sum, dim3((unsigned)((sums + kPartOutputs - 1) / kPartOutputs)), dim3(256), 0, stream, sp,
                               h->ndir, h->groups);
            CNT_HIP(hipGetLastError());
        }
    } else {
        // In front of the products: reading all states is bound by memory and goes by beside another stream's products, while behind them,
        // at a pass's end, the card had nothing else to do (32 sequences 2485 -> 2448 us per pass, acoustic model 2572 -> 2559).
        SmallGradDirs sp;
        sp.H = H; sp.L = L; sp.S = S; sp.N = N; sp.bias = d.bias; sp.parts = nullptr;
        sp.chunk = N >= 4096 ? 64 : 16;  // a short fraction still fills some tens of workgroups
        for (int dir = 0; dir < 2; ++dir) {
            const int sd = dir < h->ndir ? dir : 0;
            sp.dni[dir] = h->state[sd][7]; sp.dig[dir] = h->state[sd][8]; sp.dfg[dir] = h->state[sd][9];
            sp.dog[dir] = h->state[sd][10]; sp.c[dir] = h->state[sd][4];
        }
        sp.g_bias = weight_updates + off_bias;
        sp.g_peep = weight_updates + off_peep;
        const int V = H % 4 == 0 ? 4 : H % 2 == 0 ? 2 : 1, groups = H / V, gpb = std::min(groups, 256 / V);
        // (very long fractions: as many chunks as the scratch holds sums of)
        const size_t sums = (size_t)h->ndir * kSmallSums * H, most = std::max<size_t>(kSplitScratchFloats / sums, 1);
        sp.chunk = std::max(sp.chunk, (int)((N + most - 1) / most));
        const dim3 grid((groups + gpb - 1) / gpb, (N + sp.chunk - 1) / sp.chunk, h->ndir);
        const auto small = V == 4 ? lstm_small_grads<4> : V == 2 ? lstm_small_grads<2> : lstm_small_grads<1>;
        ProfileScope prof(stream, "lstm_small_grads");
        const bool stored = with_split_scratch(stream, sums * grid.y, [&](float *buf) {
            sp.parts = buf;
            hipLaunchKernelGGL(small, grid, dim3(256), 0, stream, sp);
            hipLaunchKernelGGL(lstm_small_grads_sum, dim3((unsigned)((sums + kPartOutputs - 1) / kPartOutputs)), dim3(256), 0, stream, sp,
                               h->ndir, (int)grid.y);
        });
        if (!stored) {
            sp.parts = nullptr;
            CNT_TRY(fill_zero_pair(stream, weight_updates + off_bias, off_int - off_bias, weight_updates + off_peep, nW - off_peep));
            hipLaunchKernelGGL(small, grid, dim3(256), 0, stream, sp);
        }
        CNT_HIP(hipGetLastError());
    }
    {
        // input weights: dW_in[g,dir] (P x H) = x (P x N) * delta^T
        GemmArgs ga = {};
        ga.m = P; ga.n = H; ga.k = N;
        ga.a_kcontig = 0; ga.lda = P;
        ga.b_kcontig = 0; ga.ldb = H;
        ga.ldc = P;
        ga.nseg = 1; ga.nprob = 4 * h->ndir; ga.epilogue = EPI_ATOMIC;
        ga.splitk = 0;  // chosen by the launcher
        for (int dir = 0; dir < h->ndir; ++dir)
            for (int g = 0; g < 4; ++g) {
                GemmProblem &pb = ga.prob[dir * 4 + g];
                pb.A[0] = x;
                pb.B[0] = h->state[dir][7 + g];
                pb.C = weight_updates + (size_t)g * P * L + (size_t)dir * P * H;
            }
        if (h->slot_order.order) {
            // the deltas are zero on padding slots: the sum over the slots leaves them out
            ga.k_order = h->slot_order.order;
            ga.k_count = h->slot_order.count;
        }
        ga.label = "gemm:lstm_dW_input";
        ga.overwrite_ok = 1;  // the problems cover all input weights
        gemm_plan(ga, stream);
        if (ga.epilogue == EPI_ATOMIC) CNT_TRY(fill_zero(stream, weight_updates, off_bias));
        CNT_TRY(gemm_launch(stream, ga, group));
    }
    if (h->T > 1) {
        // recurrent weights: dW_int[g,dir][src + to*H] = sum h[src] at the earlier step * delta[to]
        GemmArgs ga = {};
        ga.m = H; ga.n = H; ga.k = N - S;
        ga.a_kcontig = 0; ga.lda = H;
        ga.b_kcontig = 0; ga.ldb = H;
        ga.ldc = H;
        ga.nseg = 1; ga.nprob = 4 * h->ndir; ga.epilogue = EPI_ATOMIC;
        ga.splitk = 0;  // chosen by the launcher
        for (int dir = 0; dir < h->ndir; ++dir)
            for (int g = 0; g < 4; ++g) {
                GemmProblem &pb = ga.prob[dir * 4 + g];
                const float *hbuf = h->state[dir][5];
                const float *dl = h->state[dir][7 + g];
                // forward states pair delta[t] with h[t-1]; backward states pair delta[t] with h[t+1]
                pb.A[0] = dir ? hbuf + (size_t)S * H : hbuf;
                pb.B[0] = dir ? dl : dl + (size_t)S * H;
                pb.C = weight_updates + off_int + (size_t)g * L * H + (size_t)dir * H * H;
                // with the list of valid slots: a forward state's pairs are the valid slots from the second time step on,
                // counted from there; a backward state's are the valid slots before the last time step
                pb.k_trim = dir ? 2 : 1;
                pb.k_shift = dir ? 0 : -S;
            }
        if (h->slot_order.order) {
            ga.k_order = h->slot_order.order;
            ga.k_count = h->slot_order.count;
        }
        ga.label = "gemm:lstm_dW_internal";
        ga.overwrite_ok = 1;  // the problems cover all recurrent weights
        gemm_plan(ga, stream);
        if (ga.epilogue == EPI_ATOMIC) CNT_TRY(fill_zero(stream, weight_updates + off_int, off_peep - off_int));
        CNT_TRY(gemm_launch(stream, ga, group));
    } else {
        CNT_TRY(fill_zero(stream, weight_updates + off_int, off_peep - off_int));
    }
    return CNT_OK;
}

int cnt_lstm_backward(cnt_lstm *h, void *stream, const float *weights, const float *x, const float *outputs,
                      float *output_errors, float *prev_errors, float *weight_updates) {
    using namespace cnt;
    CNT_REQUIRE(outputs, "lstm_backward: null argument");
    CNT_REQUIRE(x && weight_updates, "lstm_backward_weights: null argument");
    hipStream_t s = static_cast<hipStream_t>(stream);
    CNT_TRY(lstm_backward_errors_sums(h, s, weights, output_errors, prev_errors, weight_updates));
    return lstm_backward_weights_grouped(h, s, x, weight_updates, true);
}

}  // extern "C"
