// Forward pass of one WaveNet residual block in one launch: dilated causal convolution (two live taps, R -> 2R),
// conditioning projection (C -> 2R), gated unit, 1x1 layer behind it (R -> R), residual sum and skip 1x1 layer (R -> K).
//
// Reference behaviour: layers/CNNLayer.cu:1099-1224, layers/wavNetCore.cu:629-711, layers/FeedForwardLayer.cu (forward),
// layers/SkipAddLayer.cu:186-240.
#pragma once
#include "common.hpp"

namespace cnt {
namespace {

struct BlockFwdArgs {
    int N, K, C;             // (N: the end of the launch's slots)
    int shift;               // the earlier tap reads slot n - shift, the later one slot n
    const char *pat;
    const float *x;          // R x N: the block's input, also the residual
    const float *ctx;        // C x N conditioning features
    const float *conv_w[2];  // weight of (filter 0, channel 0) of the earlier and of the later tap
    int conv_ld;             // filter d at + d * conv_ld
    int first;               // the launch's first slot
    const float *conv_bias;
    const float *ctx_w;      // [2R][C]
    const float *out_w, *out_bias;    // [R][R]
    const float *skip_w, *skip_bias;  // [K][R]
    float conv_scale, out_scale, skip_scale;  // factors of the bias vectors
    int conv_tanh;
    float *conv, *core, *ctx_tanh, *gated, *out, *sum, *skip;  // core: null where the backward pass forms it again
};

typedef float f32x4 __attribute__((ext_vector_type(4)));
typedef unsigned u32x4 __attribute__((ext_vector_type(4)));
typedef float f32x4u __attribute__((ext_vector_type(4), aligned(4)));  // weights start wherever the layer before ends

constexpr int kBlockMaxContext = 112;  // conditioning features whose tile and operands a workgroup can hold
constexpr unsigned kDropped = 0x40000000u;  // offset of a store that the range of its buffer drops

// LDS of a workgroup, in 16-byte words: tiles [chunk of four channels][sample] of both taps' inputs and of the
// conditioning features.  One word of padding per row: the threads of a store take neighbouring chunks of one sample.
constexpr int block_forward_lds_words(int R, int st, int C) { return (3 * (R / 4) + (C + 15) / 16 * 4) * (16 * st + 1); }

// A workgroup owns 16 * ST samples and has one wave per 16 residual channels.  Every product is computed transposed,
// D[channel][sample] = sum_k W[channel][k] * X[sample][k], with v_mfma_f32_16x16x4f32, instruction (j, i) taking
// k = 16j + 4*(lane/16) + i from both operands.  All five weight matrices keep k contiguous, so the A operand of four
// instructions is one 16-byte load per lane straight from the layer's weights; a wave owns its channels for all samples
// of the workgroup, so no weight is read twice in a workgroup and none passes through LDS.  The samples' side does: the
// inputs arrive as contiguous rows, every wave reads them as B operands, and the accumulators (four consecutive channels
// of one sample per lane) go back into the same layout with one 16-byte write for the next product.  A wave holds
// channel c of the tanh half and channel R + c of the sigmoid half, so the gate needs no exchange.
//
// What bounds it: the chain of its phases.  64 residual, 128 skip channels, 80 conditioning features (per sample 78 kFLOP and 2.8 KB), 32 000
// samples in one launch, 39 us: FP32 matrix instructions 20 (without seven eighths of the convolution's 32), the gate's arithmetic 5, the stores of the
// activation buffers 2, the rest loads, barriers and the launch itself.
template <int R, int ST>
__global__ __launch_bounds__(R * 4, 2) void wavenet_block_forward_kernel(const BlockFwdArgs a) {
    constexpr int CJ = kBlockMaxContext / 16;
    constexpr int NT = R * 4, WAVES = R / 16, RC = R / 4, RJ = R / 16, NS = 16 * ST, ROW = NS + 1;
    extern __shared__ __attribute__((aligned(16))) f32x4 lds[];
    f32x4 *const now = lds, *const earlier = now + RC * ROW, *const zs = earlier + RC * ROW, *const cond = zs + RC * ROW;
    const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int quarter = lane >> 4, col = lane & 15;
    const int cj = (a.C + 15) / 16, last4 = a.C - 4;

    // four neighbouring values of a row of C values, which starts at any 4-byte boundary: the 16-byte piece that ends with
    // the row where k .. k+3 would pass its end, moved into place (zeros behind the row) when it is used
    auto piece_of_row = [&](const float *row, int k) -> f32x4 { return *reinterpret_cast<const f32x4u *>(row + min(k, last4)); };
    auto in_place = [&](f32x4 v, int k) {
        const int d = k - last4;
        const bool one = d > 0 && (d & 1), two = d > 0 && (d & 2), none = d > 3;
        v[0] = one ? v[1] : v[0]; v[1] = one ? v[2] : v[1]; v[2] = one ? v[3] : v[2]; v[3] = one ? 0.0f : v[3];
        v[0] = two ? v[2] : v[0]; v[1] = two ? v[3] : v[1]; v[2] = two ? 0.0f : v[2]; v[3] = two ? 0.0f : v[3];
#pragma unroll
        for (int i = 0; i < 4; ++i) v[i] = none ? 0.0f : v[i];
        return v;
    };

    // ---- the inputs: requested without branches, then put into LDS
    constexpr int XW = RC * NS, XF = (XW + NT - 1) / NT;
    constexpr int CB = (4 * CJ * NS + NT - 1) / NT;
    f32x4 x0[XF], x1[XF], xc[CB];
    char p1[XF], pc[CB], pl[ST];
    const int n0 = a.first + blockIdx.x * NS;
    {
#pragma unroll
        for (int q = 0; q < XF; ++q) {
            const int idx = q * NT + tid, s = idx / RC, ch = idx % RC;
            const int n = n0 + s, e = n - a.shift;
            const size_t s0 = n < a.N ? n : 0, s1 = ((n < a.N) & (e >= 0)) ? e : 0;
            x0[q] = *reinterpret_cast<const f32x4 *>(a.x + s0 * R + 4 * ch);
            x1[q] = *reinterpret_cast<const f32x4 *>(a.x + s1 * R + 4 * ch);
            p1[q] = a.pat[s1];
        }
#pragma unroll
        for (int s = 0; s < ST; ++s) pl[s] = a.pat[min(n0 + 16 * s + col, a.N - 1)];
        if (cj > 0)
#pragma unroll
            for (int q = 0; q < CB; ++q) {
                const int idx = q * NT + tid, s = idx / (4 * CJ), ch = idx % (4 * CJ), n = min(n0 + s, a.N - 1);
                xc[q] = piece_of_row(a.ctx + (size_t)n * a.C, 4 * ch);
                pc[q] = a.pat[n];
            }
    }
    auto place = [&] {
        const f32x4 zero = {0, 0, 0, 0};
#pragma unroll
        for (int q = 0; q < XF; ++q) {
            const int idx = q * NT + tid, s = idx / RC, ch = idx % RC, n = n0 + s;
            if (XW % NT == 0 || idx < XW) {
                now[ch * ROW + s] = n < a.N ? x0[q] : zero;
                earlier[ch * ROW + s] = ((n < a.N) & (n >= a.shift) & (p1[q] != 0)) ? x1[q] : zero;
            }
        }
        if (cj > 0)
#pragma unroll
            for (int q = 0; q < CB; ++q) {
                const int idx = q * NT + tid, s = idx / (4 * CJ), ch = idx % (4 * CJ);
                if (idx < 4 * CJ * NS && ch < 4 * cj) cond[ch * ROW + s] = pc[q] != 0 ? in_place(xc[q], 4 * ch) : zero;
            }
    };
    // ---- the weights of the convolution and of the conditioning projection
    const int f = 16 * wave + col;  // this lane's filter row in the A operands (tanh half; the sigmoid half is at + R)
    f32x4 wa[2][2][RJ];             // [half][tap][j]
#pragma unroll
    for (int h = 0; h < 2; ++h)
#pragma unroll
        for (int tap = 0; tap < 2; ++tap)
#pragma unroll
            for (int j = 0; j < RJ; ++j)
                wa[h][tap][j] = *reinterpret_cast<const f32x4u *>(a.conv_w[tap] + (size_t)(h * R + f) * a.conv_ld + 16 * j + 4 * quarter);
    f32x4 wc[2][CJ];
    if (cj > 0)
#pragma unroll
        for (int j = 0; j < CJ; ++j)
#pragma unroll
            for (int h = 0; h < 2; ++h)
                wc[h][j] = piece_of_row(a.ctx_w + (size_t)(h * R + f) * a.C, 16 * min(j, cj - 1) + 4 * quarter);
    const int own = 16 * wave + 4 * quarter;  // first of the four channels this lane holds per accumulator
    f32x4 bias_t = *reinterpret_cast<const f32x4u *>(a.conv_bias + own) * a.conv_scale;
    f32x4 bias_s = *reinterpret_cast<const f32x4u *>(a.conv_bias + R + own) * a.conv_scale;
    const f32x4 bias_o = *reinterpret_cast<const f32x4u *>(a.out_bias + own) * a.out_scale;
    __builtin_amdgcn_sched_barrier(0);
    place();
    if (a.C & 15)
#pragma unroll
        for (int j = 0; j < CJ; ++j)
#pragma unroll
            for (int h = 0; h < 2; ++h) wc[h][j] = in_place(wc[h][j], 16 * j + 4 * quarter);
    asm volatile("" : "+v"(bias_t), "+v"(bias_s));
    const int tiles_k = a.K / 16;

    bool live[ST];
#pragma unroll
    for (int s = 0; s < ST; ++s) live[s] = (n0 + 16 * s + col < a.N) & (pl[s] != 0);
    __syncthreads();
    // stores without branches: the tile's rows as buffers, what lies past the last sample is dropped by their range
    const int rows = min(NS, a.N - n0);
    auto rows_of = [&](float *p, int width) {
        return __builtin_amdgcn_make_buffer_rsrc(p + (size_t)n0 * width, 0, rows * width * 4, 0x00020000);
    };
    auto put = [](__amdgpu_buffer_rsrc_t to, unsigned offset, const f32x4 &v) {
        __builtin_amdgcn_raw_buffer_store_b128(__builtin_bit_cast(u32x4, v), to, offset, 0, 2);  // non-temporal: read in another pass
    };
    const auto to_conv = rows_of(a.conv, 2 * R), to_gated = rows_of(a.gated, R), nowhere = __builtin_amdgcn_make_buffer_rsrc(a.conv, 0, 0, 0x00020000);
    const auto to_core = a.core ? rows_of(a.core, 2 * R) : nowhere, to_ctx = a.ctx_tanh ? rows_of(a.ctx_tanh, 2 * R) : nowhere;

    // ---- convolution, conditioning projection and gate, one step of sixteen samples after the other.  The gate of a
    // step is evaluated between the matrix instructions of the next one's convolution: seven vector instructions fit
    // into the 32 cycles that one of those takes.
    // (without conditioning features `cond` has no words: what is read, and not used, then comes from the block's input)
    const f32x4 *const features = cj > 0 ? cond : now;
    f32x4 c0, c1, t0, t1;  // convolution and conditioning sums of the step, both halves
    auto gate = [&](int s, f32x4 p, f32x4 q, f32x4 tp, f32x4 tq) {
        const unsigned at = 4 * ((16 * s + col) * 2 * R + own);
        p += bias_t;
        q += bias_s;
        f32x4 z;
        // Evaluated first and chosen afterwards: as a branch it could not share the matrix instructions' cycles.  The
        // conditioning features of a padding slot are zeros in LDS, so tp and tq are tanh(0) there.
#pragma unroll
        for (int v = 0; v < 4; ++v) {
            float y0 = tanh_act(p[v]), y1 = tanh_act(q[v]);
            asm volatile("" : "+v"(y0), "+v"(y1));
            p[v] = a.conv_tanh ? y0 : p[v];
            q[v] = a.conv_tanh ? y1 : q[v];
            tp[v] = tanh_act(tp[v]);
            tq[v] = tanh_act(tq[v]);
        }
        // the convolution layer leaves padding slots as they are
        put(to_conv, live[s] ? at : kDropped, p);
        put(to_conv, live[s] ? at + 4 * R : kDropped, q);
#pragma unroll
        for (int v = 0; v < 4; ++v) {
            p[v] = live[s] ? p[v] + tp[v] : 0.0f;
            q[v] = live[s] ? q[v] + tq[v] : 0.0f;
            z[v] = tanh_act(p[v]) * logistic(q[v]);  // tanh(0) = 0 on padding
        }
        put(to_core, at, p);
        put(to_core, at + 4 * R, q);
        put(to_ctx, at, tp);
        put(to_ctx, at + 4 * R, tq);
        put(to_gated, 4 * ((16 * s + col) * R + own), z);
        zs[(4 * wave + quarter) * ROW + 16 * s + col] = z;
    };
#pragma unroll
    for (int s = 0; s < ST; ++s) {
        const f32x4 pc0 = c0, pc1 = c1, pt0 = t0, pt1 = t1;
        f32x4 b[2][RJ], x[CJ];
#pragma unroll
        for (int tap = 0; tap < 2; ++tap)
#pragma unroll
            for (int j = 0; j < RJ; ++j) b[tap][j] = (tap == 0 ? earlier : now)[(4 * j + quarter) * ROW + 16 * s + col];
#pragma unroll
        for (int j = 0; j < CJ; ++j) x[j] = features[(4 * min(j, max(cj - 1, 0)) + quarter) * ROW + 16 * s + col];
        c0 = f32x4{0, 0, 0, 0};
        c1 = f32x4{0, 0, 0, 0};
#pragma unroll
        for (int tap = 0; tap < 2; ++tap)
#pragma unroll
            for (int j = 0; j < RJ; ++j)
#pragma unroll
                for (int i = 0; i < 4; ++i) {
                    c0 = __builtin_amdgcn_mfma_f32_16x16x4f32(wa[0][tap][j][i], b[tap][j][i], c0, 0, 0, 0);
                    c1 = __builtin_amdgcn_mfma_f32_16x16x4f32(wa[1][tap][j][i], b[tap][j][i], c1, 0, 0, 0);
                }
        __builtin_amdgcn_sched_group_barrier(0x100, 2 * RJ + CJ, 0);
        if (s > 0) {
            gate(s - 1, pc0, pc1, pt0, pt1);
#pragma unroll
            for (int u = 0; u < 16 * RJ; ++u) {
                __builtin_amdgcn_sched_group_barrier(0x008, 1, 0);
                __builtin_amdgcn_sched_group_barrier(0x002, 7, 0);
            }
        }
        t0 = f32x4{0, 0, 0, 0};
        t1 = f32x4{0, 0, 0, 0};
#pragma unroll
        for (int j = 0; j < CJ; ++j) {
            if (j >= cj) break;
#pragma unroll
            for (int i = 0; i < 4; ++i) {
                t0 = __builtin_amdgcn_mfma_f32_16x16x4f32(wc[0][j][i], x[j][i], t0, 0, 0, 0);
                t1 = __builtin_amdgcn_mfma_f32_16x16x4f32(wc[1][j][i], x[j][i], t1, 0, 0, 0);
            }
        }
    }
    f32x4 wo[RJ], ws[RJ];
#pragma unroll
    for (int j = 0; j < RJ; ++j) wo[j] = *reinterpret_cast<const f32x4u *>(a.out_w + (size_t)f * R + 16 * j + 4 * quarter);
    auto skip_weights = [&](int t, f32x4 (&w)[RJ]) {
#pragma unroll
        for (int j = 0; j < RJ; ++j)
            w[j] = *reinterpret_cast<const f32x4u *>(a.skip_w + (size_t)(16 * t + col) * R + 16 * j + 4 * quarter);
    };
    skip_weights(min(wave, tiles_k - 1), ws);
    gate(ST - 1, c0, c1, t0, t1);
    __syncthreads();

    // ---- 1x1 layer and residual sum, which takes the place of the block's input in LDS
    f32x4 acc[ST], b[RJ][ST];
#pragma unroll
    for (int j = 0; j < RJ; ++j)
#pragma unroll
        for (int s = 0; s < ST; ++s) b[j][s] = zs[(4 * j + quarter) * ROW + 16 * s + col];
#pragma unroll
    for (int s = 0; s < ST; ++s) acc[s] = f32x4{0, 0, 0, 0};
#pragma unroll
    for (int j = 0; j < RJ; ++j)
#pragma unroll
        for (int i = 0; i < 4; ++i)
#pragma unroll
            for (int s = 0; s < ST; ++s) acc[s] = __builtin_amdgcn_mfma_f32_16x16x4f32(wo[j][i], b[j][s][i], acc[s], 0, 0, 0);
    const auto to_out = rows_of(a.out, R), to_sum = rows_of(a.sum, R), to_skip = rows_of(a.skip, a.K);
#pragma unroll
    for (int s = 0; s < ST; ++s) {
        const f32x4 o = acc[s] + bias_o;
        f32x4 &cell = now[(4 * wave + quarter) * ROW + 16 * s + col];
        const f32x4 sum = cell + o;
        cell = sum;
        put(to_out, 4 * ((16 * s + col) * R + own), o);
        __builtin_amdgcn_raw_buffer_store_b128(__builtin_bit_cast(u32x4, sum), to_sum, 4 * ((16 * s + col) * R + own), 0, 0);
    }
    __syncthreads();

    // ---- skip 1x1 layer
#pragma unroll
    for (int j = 0; j < RJ; ++j)
#pragma unroll
        for (int s = 0; s < ST; ++s) b[j][s] = now[(4 * j + quarter) * ROW + 16 * s + col];
    for (int t = wave; t < tiles_k; t += WAVES) {
        f32x4 next[RJ];
        skip_weights(min(t + WAVES, tiles_k - 1), next);
        const f32x4 bias_k = *reinterpret_cast<const f32x4u *>(a.skip_bias + 16 * t + 4 * quarter) * a.skip_scale;
#pragma unroll
        for (int s = 0; s < ST; ++s) acc[s] = f32x4{0, 0, 0, 0};
#pragma unroll
        for (int j = 0; j < RJ; ++j)
#pragma unroll
            for (int i = 0; i < 4; ++i)
#pragma unroll
                for (int s = 0; s < ST; ++s) acc[s] = __builtin_amdgcn_mfma_f32_16x16x4f32(ws[j][i], b[j][s][i], acc[s], 0, 0, 0);
#pragma unroll
        for (int s = 0; s < ST; ++s) put(to_skip, 4 * ((16 * s + col) * a.K + 16 * t + 4 * quarter), acc[s] + bias_k);
#pragma unroll
        for (int j = 0; j < RJ; ++j) ws[j] = next[j];
    }
}

typedef void (*block_fwd_kernel_t)(const BlockFwdArgs);
template <int R>
block_fwd_kernel_t block_forward_of(int st) {
    return st == 4 ? wavenet_block_forward_kernel<R, 4> : st == 2 ? wavenet_block_forward_kernel<R, 2> : wavenet_block_forward_kernel<R, 1>;
}
block_fwd_kernel_t pick_block_forward_kernel(int R, int st) {
    return R == 64 ? block_forward_of<64>(st) : R == 48 ? block_forward_of<48>(st) : R == 32 ? block_forward_of<32>(st) : nullptr;
}

}  // namespace
}  // namespace cnt
