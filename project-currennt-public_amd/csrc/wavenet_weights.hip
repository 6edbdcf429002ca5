// Weight gradients of the residual blocks of a WaveNet stack: all of a block's weight arrays, for several blocks, in one launch
// of products and one of sums.
//
// A block has four products over its slots: both taps of the convolution (2R x 2R sums), the conditioning projection (C x 2R), the
// 1x1 layer behind the gate (R x R) and the skip 1x1 layer (R x K).  As problems of the tiled product (gemm.hip, 64 x 64 tiles) an
// operand was read and split into its bf16 parts once per tile that needs it -- 1408 rows per slot at 64 residual, 128 skip
// channels and 80 features -- and every layer kind was a launch with a reduction of its own.  Here a workgroup takes all of a
// product's sums, up to 128 x 128, over a range of slots, so that every row is converted once (784 rows), both taps share the
// errors' rows, and the bias gradients are sums of rows on their way.  The arithmetic is the tiled product's: three bf16 parts,
// six part products, the small ones first.
//
// What bounds it: memory, conversions and matrix instructions about equally (30 blocks over 32 000 slots, per block 73 MB through
// the L2s, 18 us with the card idle before, 25 us inside the pass, where the clock is lower; before, 37 us and a reduction of 5
// to 20; pass 3850 -> 3580 us.  8 blocks of 32 channels over 2000 slots: 362 -> 325 us).
// A wave stages one segment of 64 rows, with two tiles of loads in flight.  Branches between a tile's loads cost all of that: the
// compiler then waits for every load in flight (40 us per block), which is why the kinds of segments are loops of their own.
// Two workgroups per compute unit (128 registers) rather than one, so that one's barriers fall into the other's work.
//
// Padding counts like any slot (the 1x1 products of before left it out): still the faster way where nearly half of a fraction is padding,
// 30 blocks over 2 x 16 000 slots with a sequence of 1000 3622 -> 3528 us per pass before the shares were dealt as they are now.
//
// Sums: a run of kTallRun tiles is added up by the matrix instructions, then joins the sums of earlier runs, then come the splits.
// 2-norm error against 64 bits, before / now, for the convolution, the projection, the 1x1 and the skip layer: 1.6 / 1.0, 4.0 /
// 2.3, 1.4 / 1.2, 1.1 / 0.9e-7 (32 000 slots); 1.8 / 1.3, 2.4 / 1.7, 1.7 / 1.2, 1.7 / 1.2e-7 (2001).  Without runs the 1x1 layers
// came out at 1.6 and 1.3e-7.  Every sum has a fixed order: the same gradients in every call.
//
// Reference behaviour: layers/CNNLayer.cu:1409-1597, layers/wavNetCore.cu:801-916, layers/FeedForwardLayer.cu (backward).
#include "gemm_kernel.hpp"

#include <algorithm>
#include <type_traits>

namespace cnt {
namespace {

constexpr int kTallDepth = 16;       // slots of a staged tile: one matrix instruction
constexpr int kTallThreads = 512;
constexpr int kTallGroup = 68;       // row 4c + r of a tile stands at r * kTallGroup + c
constexpr int kTallLine = 4 * kTallGroup;
constexpr int kTallPart = 2 * kTallLine;
constexpr int kTallUnits = 3 * kTallPart;
constexpr int kTallRun = 8;         // tiles added up before the sum joins the sums of earlier runs
constexpr int kTallWorkgroups = 512;
constexpr int kTallBlocks = 16;      // 32 x 32 blocks of sums of a workgroup
constexpr int kTallMaxJobs = 5;
constexpr int kTallTileCost = 8;     // of a tile of any size, see wavenet_block_weights

struct TallArgs {
    BlockGradients block[kBlockGradients];
    int n, R, K, C;         // slots, residual and skip channels, conditioning features
    int conv_ld;            // distance of two filters' weights
    int jobs;               // per block: convolution, conditioning projection, 1x1 layer, 128 skip channels each
    int sums;               // 32 x 32 blocks of sums that a workgroup has room for in `partial`
    int first[kTallMaxJobs + 1];  // workgroup of a block with which a job's splits begin
    const float *ctx;
    const char *pat;
    float *partial, *rows;  // a workgroup's blocks of sums; its sums of the B rows, per half of a tile's slots
};

// 64 rows of an operand tile: `rows` channels of a slot-major buffer, read `shift` slots back
struct Segment {
    const float *base;
    int ld, rows, shift;
    bool masked;  // both slots have to be inside the fraction and no padding
};

// segments 0 and 1 hold the A rows of a job, 2 and 3 the B rows
__device__ __forceinline__ Segment segment_of(const TallArgs &a, const BlockGradients &b, int job, int s) {
    const int D = 2 * a.R, at = 64 * (s & 1);
    const bool is_b = s >= 2;
    if (job == 0) {
        if (!is_b) return {b.x, a.R, a.R, s == 1 ? b.shift : 0, true};
        return {b.deltas + at, D, max(min(D - at, 64), 0), 0, false};
    }
    if (job == 1) {
        if (!is_b) return {a.ctx + at, a.C, max(min(a.C - at, 64), 0), 0, false};
        return {b.ctx_grad + at, D, max(min(D - at, 64), 0), 0, false};
    }
    if (!is_b) return {job == 2 ? b.gated : b.sum, a.R, s == 1 ? 0 : a.R, 0, false};
    if (job == 2) return {b.out_errors, a.R, s == 3 ? 0 : a.R, 0, false};
    const int col = 128 * (job - 3) + at;
    return {b.skip_errors + col, a.K, max(min(a.K - col, 64), 0), 0, false};
}

// the blocks of 32 rows that hold any, two bits per segment, and the i-th of them
__device__ __forceinline__ int row_blocks(int rows0, int rows1) {
    return (rows0 > 0 ? 1 : 0) | (rows0 > 32 ? 2 : 0) | (rows1 > 0 ? 4 : 0) | (rows1 > 32 ? 8 : 0);
}
__device__ __forceinline__ int ith_bit(int mask, int i) {
    int at = 0;
#pragma unroll
    for (int q = 0; q < 4; ++q) {
        const bool set = (mask >> q) & 1;
        if (set && i == 0) at = q;
        i -= set ? 1 : 0;
    }
    return at;
}

// What a thread has in flight of a tile: four rows of a segment at two neighbouring slots.  Every tile takes the same loads on every
// path, so that a tile's values are waited for without those of the next one: the kinds of segments differ at compile time.
// MASKED: padding counts as zeros.  RAGGED: rows that are no multiple of four.  SUMS: the rows' sums are a bias gradient.
struct TallLoader {
    const char *base, *pat;
    int rows, shift, ld, last_slot;  // uniform; ld in bytes
    int row, k;                      // the thread's first row and first slot inside a tile
    int at, lowest, highest;         // byte offset of its first vector at slot 0, those of the first and the last slot
    int end;

    __device__ __forceinline__ TallLoader(const Segment &s, const char *pat_, int n, int row_, int k_, int end_, bool ragged) {
        base = reinterpret_cast<const char *>(s.base); pat = pat_;
        rows = s.rows; shift = s.shift; ld = s.ld * (int)sizeof(float); last_slot = n - 1;
        row = row_; k = k_; end = end_;
        // (ragged: the last rows come in the vector that ends with them, which begins in front of a segment of fewer than four rows;
        // the base moves there, as the offset is an unsigned one)
        const int back = max(4 - rows, 0);
        base -= back * sizeof(float);
        lowest = 4 * (ragged ? min(row, rows - 4) + back : row < rows ? row : 0);
        at = (k - shift) * ld + lowest;
        highest = last_slot * ld + lowest;
    }
};
template <bool MASKED, bool RAGGED, bool SUMS>
struct TallStage {
    static constexpr bool kSums = SUMS;
    float v[2][4];
    unsigned src[2];  // pattern type of the slot that is read (the errors of a padding slot are zeros)

    __device__ __forceinline__ void load(const TallLoader &l, int n) {  // n = the tile's first slot
#pragma unroll
        for (int p = 0; p < 2; ++p) {
            if (MASKED) {
                src[p] = (unsigned char)l.pat[(unsigned)min(max(n + l.k + p - l.shift, 0), l.last_slot)];
            }
            const int off = (n + p) * l.ld + l.at;
            const f32x4u x = *reinterpret_cast<const f32x4u *>(l.base + (unsigned)min(MASKED ? max(off, l.lowest) : off, l.highest));
#pragma unroll
            for (int i = 0; i < 4; ++i) v[p][i] = x[i];
        }
    }
    __device__ __forceinline__ void put(uint4 *__restrict__ lds, const TallLoader &l, int n, int unit, int pair, float (&sums)[4]) {
        if (l.row >= l.rows) return;
        if (MASKED || RAGGED || n + kTallDepth > l.end) {
#pragma unroll
            for (int p = 0; p < 2; ++p) {
                const int to = n + l.k + p;
                const bool keep = to < l.end && (!MASKED || (to >= l.shift && src[p] != 0));
#pragma unroll
                for (int i = 0; i < 4; ++i) {
                    if (RAGGED) {
                        const int from = i + max(l.row - (l.rows - 4), 0);
                        float x = 0.0f;
#pragma unroll
                        for (int q = i; q < 4; ++q) x = q == from ? v[p][q] : x;
                        v[p][i] = x;
                    }
                    v[p][i] = keep ? v[p][i] : 0.0f;
                }
            }
        }
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            if (SUMS) sums[i] += v[0][i] + v[1][i];
            unsigned x[3];
            split_pair(v[0][i], v[1][i], x);
#pragma unroll
            for (int q = 0; q < 3; ++q) reinterpret_cast<unsigned *>(lds + unit + q * kTallPart + i * kTallGroup)[pair] = x[q];
        }
    }
};
struct NoStage {
    static constexpr bool kSums = false;
};

// 32 x 32 sums of a job over the slots [begin, end) on the fp32 instructions, straight from memory: where the split product left
// sums that are not finite (plain_sums, gemm_kernel.hpp)
__device__ __forceinline__ f32x16 plain_block(const Segment &sa, const Segment &sb, const char *pat, int row_a, int row_b,
                                                        int begin, int end, int half) {
    f32x16 acc;
#pragma unroll
    for (int r = 0; r < 16; ++r) acc[r] = 0.0f;
    auto value = [&](const Segment &s, int row, int n) {
        const int e = n - s.shift;
        const bool in = n < end && e >= 0 && row < s.rows;
        const float v = s.base[(size_t)(in ? e : 0) * s.ld + (in ? row : 0)];
        return in && !(s.masked && (pat[n] == 0 || pat[e] == 0)) ? v : 0.0f;
    };
#pragma unroll 1
    for (int n = begin; n < end; n += 2)
        acc = __builtin_amdgcn_mfma_f32_32x32x2f32(value(sb, row_b, n + half), value(sa, row_a, n + half), acc, 0, 0, 0);
    return acc;
}

// One job of one block over a range of slots per workgroup: up to 128 x 128 sums over the slots.  Wave w stages segment w % 4 for
// the eight slots w / 4 of every tile, two tiles ahead in registers, and takes the blocks of sums w and w + 8 of up to sixteen.
__global__ __launch_bounds__(kTallThreads, 4) void wavenet_block_weights_kernel(const TallArgs a) {
    __shared__ uint4 lds[2 * kTallUnits];
    const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int per_block = a.first[a.jobs];
    // The blocks' workgroups of one job and one range of slots follow each other on one XCD: the conditioning features and the skip
    // errors, which all blocks share, come out of its L2 for all but the first.
    const unsigned total = gridDim.x, per = total / 8, rem = total % 8, xcd = blockIdx.x % 8, slot = blockIdx.x / 8;
    const unsigned pos = xcd < rem ? xcd * (per + 1) + slot : rem * (per + 1) + (xcd - rem) * per + slot;
    const int blocks = (int)total / per_block, z = (int)pos % blocks, w = (int)pos / blocks;
    const size_t group = (size_t)z * per_block + w;
    int job = 0;
#pragma unroll
    for (int j = 1; j < kTallMaxJobs; ++j)
        if (j < a.jobs && w >= a.first[j]) job = j;
    const int splits = a.first[job + 1] - a.first[job], split = w - a.first[job];
    const BlockGradients &b = a.block[z];
    const int tiles = (a.n + kTallDepth - 1) / kTallDepth, per_split = (tiles + splits - 1) / splits;
    const int begin = min(split * per_split * kTallDepth, a.n), end = min(begin + per_split * kTallDepth, a.n);

    const int rows0 = segment_of(a, b, job, 0).rows, rows1 = segment_of(a, b, job, 1).rows;
    const int rows2 = segment_of(a, b, job, 2).rows, rows3 = segment_of(a, b, job, 3).rows;
    const int mask_m = row_blocks(rows0, rows1), mask_n = row_blocks(rows2, rows3);
    const int count_n = __builtin_popcount(mask_n), count = __builtin_popcount(mask_m) * count_n;

    // a quarter of the lanes along the rows, four pairs of slots, so that the lanes of a store fall on distinct banks
    const Segment seg = segment_of(a, b, job, wave & 3);
    const int quad = (lane & 7) | ((lane >> 2) & 8), pair = (lane >> 3) & 3, row = 4 * quad;
    const int k = 8 * (wave >> 2) + 2 * pair;
    const TallLoader loader(seg, a.pat, a.n, row, k, end, seg.rows % 4 != 0);
    const int unit = (wave >> 2) * kTallLine + 16 * (wave & 3) + quad;

    const int frag_row = lane & 31, half = lane >> 5;
    int pos_a[2], pos_b[2];
#pragma unroll
    for (int t = 0; t < 2; ++t) {
        const int at = min(wave + 8 * t, count - 1);
        const int m = ith_bit(mask_m, at / count_n), n = ith_bit(mask_n, at % count_n);
        const int common = half * kTallLine + (frag_row & 3) * kTallGroup + (frag_row >> 2);
        pos_a[t] = common + 8 * m;
        pos_b[t] = common + 32 + 8 * n;
    }
    f32x16 acc[2], sum[2];
#pragma unroll
    for (int t = 0; t < 2; ++t)
#pragma unroll
        for (int r = 0; r < 16; ++r) acc[t][r] = sum[t][r] = 0.0f;
    float run_rows[4] = {0.0f, 0.0f, 0.0f, 0.0f}, row_sums[4] = {0.0f, 0.0f, 0.0f, 0.0f};

    for (int i = tid; i < 2 * kTallUnits; i += kTallThreads) lds[i] = uint4{0, 0, 0, 0};  // rows that no segment holds
    auto multiply = [&](int buf) __attribute__((always_inline)) {
        const uint4 *const at = lds + buf * kTallUnits;
        constexpr int QA[6] = {0, 2, 1, 0, 1, 0}, QB[6] = {2, 0, 1, 1, 0, 0};  // the small terms first
#pragma unroll
        for (int t = 0; t < 2; ++t) {
            if (wave + 8 * t >= count) break;
            bf16x8 fa[3], fb[3];
#pragma unroll
            for (int q = 0; q < 3; ++q) {
                fa[q] = __builtin_bit_cast(bf16x8, at[pos_a[t] + q * kTallPart]);
                fb[q] = __builtin_bit_cast(bf16x8, at[pos_b[t] + q * kTallPart]);
            }
#pragma unroll
            for (int u = 0; u < 6; ++u) acc[t] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(fb[QB[u]], fa[QA[u]], acc[t], 0, 0, 0);
        }
    };
    // the walk along the slots, for every kind of segment a loop of its own: the waves of a workgroup meet at its barriers
    auto walk = [&](auto even) __attribute__((always_inline)) {
        typedef decltype(even) Stage;
        constexpr bool STAGING = !std::is_same<Stage, NoStage>::value;
        Stage odd;
        auto load = [&](Stage &s, int n) __attribute__((always_inline)) {
            if constexpr (STAGING) s.load(loader, n);
        };
        auto put = [&](Stage &s, int n, int buf) __attribute__((always_inline)) {
            if constexpr (STAGING) s.put(lds + buf * kTallUnits, loader, n, unit, pair, run_rows);
        };
        load(even, begin);
        load(odd, begin + kTallDepth);
        __syncthreads();
        put(even, begin, 0);
        load(even, begin + 2 * kTallDepth);
        lds_only_barrier();
        auto end_run = [&]() __attribute__((always_inline)) {
            if constexpr (Stage::kSums)
#pragma unroll
                for (int i = 0; i < 4; ++i) {
                    row_sums[i] += run_rows[i];
                    run_rows[i] = 0.0f;
                }
        };
        int run = 0;
#pragma unroll 1
        for (int n = begin; n < end; n += 2 * kTallDepth) {
            put(odd, n + kTallDepth, 1);
            load(odd, n + 3 * kTallDepth);
            multiply(0);
            lds_only_barrier();
            put(even, n + 2 * kTallDepth, 0);
            load(even, n + 4 * kTallDepth);
            multiply(1);
            lds_only_barrier();
            run += 2;
            if (run == kTallRun) {
                run = 0;
#pragma unroll
                for (int t = 0; t < 2; ++t) {
                    sum[t] += acc[t];
#pragma unroll
                    for (int r = 0; r < 16; ++r) acc[t][r] = 0.0f;
                }
                end_run();
            }
        }
        end_run();
    };
    if (seg.rows == 0) walk(NoStage());
    else if (seg.masked) walk(TallStage<true, false, false>());
    else if (seg.rows % 4 != 0) walk(TallStage<false, true, false>());
    else if ((wave & 2) && job != 1) walk(TallStage<false, false, true>());
    else walk(TallStage<false, false, false>());

    // a thread's rows over all pairs of slots of its wave, then per wave into the workgroup's sums
    if (wave & 2) {
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            row_sums[i] += __shfl_xor(row_sums[i], 8);
            row_sums[i] += __shfl_xor(row_sums[i], 16);
        }
        if (pair == 0)
            *reinterpret_cast<float4 *>(a.rows + (group * 2 + (wave >> 2)) * 128 + 64 * (wave & 1) + row) =
                float4{row_sums[0], row_sums[1], row_sums[2], row_sums[3]};
    }
#pragma unroll
    for (int t = 0; t < 2; ++t) {
        const int at = wave + 8 * t;
        if (at >= count) break;
        sum[t] += acc[t];
        bool finite = true;
#pragma unroll
        for (int r = 0; r < 16; ++r) finite = finite && __builtin_fabsf(sum[t][r]) <= lim::kMax;
#pragma unroll
        for (int r = 0; r < 16; ++r) sum[t][r] *= 1.0f / (kSplitScale * kSplitScale);
        if (__builtin_expect(__builtin_amdgcn_ballot_w64(!finite) != 0, 0)) {
            const int m = ith_bit(mask_m, at / count_n), n = ith_bit(mask_n, at % count_n);
            sum[t] = plain_block(segment_of(a, b, job, m >> 1), segment_of(a, b, job, 2 + (n >> 1)), a.pat, 32 * (m & 1) + frag_row,
                                 32 * (n & 1) + frag_row, begin, end, half);
        }
        float4 *const to = reinterpret_cast<float4 *>(a.partial) + (group * a.sums + at) * 256 + lane;
#pragma unroll
        for (int g = 0; g < 4; ++g) to[64 * g] = float4{sum[t][4 * g], sum[t][4 * g + 1], sum[t][4 * g + 2], sum[t][4 * g + 3]};
    }
}

// Adds up the splits of a block of sums, four neighbouring values per thread, and stores them where the layer's weight updates
// are; one workgroup more per job for the bias gradients.
__global__ __launch_bounds__(256) void wavenet_block_weights_sum_kernel(const TallArgs a) {
    const int job = blockIdx.x / (kTallBlocks + 1), at = blockIdx.x % (kTallBlocks + 1), z = blockIdx.y;
    const BlockGradients &b = a.block[z];
    const int tid = threadIdx.x, lane = tid & 63, g = tid >> 6;
    const int rows0 = segment_of(a, b, job, 0).rows, rows1 = segment_of(a, b, job, 1).rows;
    const int rows2 = segment_of(a, b, job, 2).rows, rows3 = segment_of(a, b, job, 3).rows;
    const int splits = a.first[job + 1] - a.first[job];
    const size_t first = (size_t)z * a.first[a.jobs] + a.first[job];
    const int col = 128 * max(job - 3, 0);
    if (at == kTallBlocks) {
        if (job == 1 || tid >= 128 || (tid & 63) >= (tid < 64 ? rows2 : rows3)) return;
        const float *const p = a.rows + first * 2 * 128 + tid;
        float v = 0.0f;
        int s = 0;
        for (; s + 4 <= splits; s += 4) {
            float x[8];
#pragma unroll
            for (int q = 0; q < 8; ++q) x[q] = p[(size_t)(2 * s + q) * 128];
            v += ((x[0] + x[1]) + (x[2] + x[3])) + ((x[4] + x[5]) + (x[6] + x[7]));
        }
        for (; s < splits; ++s) v += p[(size_t)(2 * s) * 128] + p[(size_t)(2 * s + 1) * 128];
        float *const to = job == 0 ? b.conv_bias : job == 2 ? b.out_bias : b.skip_bias;
        to[col + tid] = (job == 0 ? b.conv_scale : job == 2 ? b.out_scale : b.skip_scale) * v;
        return;
    }
    const int mask_m = row_blocks(rows0, rows1), mask_n = row_blocks(rows2, rows3);
    const int count_n = __builtin_popcount(mask_n), count = __builtin_popcount(mask_m) * count_n;
    if (at >= count) return;
    const float4 *const p = reinterpret_cast<const float4 *>(a.partial) + (first * a.sums + at) * 256 + tid;
    const auto add = [](const float4 &x, const float4 &y) { return float4{x.x + y.x, x.y + y.y, x.z + y.z, x.w + y.w}; };
    float4 v0 = {0, 0, 0, 0};
    int s = 0;
    for (; s + 8 <= splits; s += 8) {
        float4 x[8];
#pragma unroll
        for (int q = 0; q < 8; ++q) x[q] = p[(size_t)(s + q) * a.sums * 256];
        v0 = add(v0, add(add(add(x[0], x[1]), add(x[2], x[3])), add(add(x[4], x[5]), add(x[6], x[7]))));
    }
    float4 v1 = {0, 0, 0, 0};
    for (; s < splits; ++s) v1 = add(v1, p[(size_t)s * a.sums * 256]);
    v0 = add(v0, v1);
    const int mb = ith_bit(mask_m, at / count_n), nb = ith_bit(mask_n, at % count_n);
    const int m = 32 * (mb & 1) + (lane & 31), n = 32 * nb + 8 * g + 4 * (lane >> 5);
    if (m >= (mb < 2 ? rows0 : rows1)) return;
    const float v[4] = {v0.x, v0.y, v0.z, v0.w};
#pragma unroll
    for (int i = 0; i < 4; ++i) {
        const int nn = n + i;
        if ((nn & 63) >= (nn < 64 ? rows2 : rows3)) continue;
        if (job == 0) {
            float *const filter = b.conv + (size_t)nn * a.conv_ld + m;  // the taps: one step back, now, the one ahead (dead)
            filter[mb < 2 ? a.R : 0] = v[i];
            if (mb < 2) filter[2 * a.R] = 0.0f;
        } else if (job == 1) {
            b.ctx[(size_t)nn * a.C + 64 * (mb >> 1) + m] = v[i];
        } else if (job == 2) {
            b.out[(size_t)nn * a.R + m] = v[i];
        } else {
            b.skip[(size_t)(col + nn) * a.R + m] = v[i];
        }
    }
}

}  // namespace

bool wavenet_block_weights_supported(int R, int K, int C, long N) {
    // (32-bit byte offsets, one window of shifts ahead of the first slot and a few tiles behind the last)
    return (N + 8 * kTallDepth) * std::max({2 * R, K, C}) * (long)sizeof(float) < (1L << 30) && R >= 4 && R <= 64 && R % 4 == 0 &&
           K >= 4 && K <= 256 && K % 4 == 0 && C >= 4 && C <= 128;
}

// 32 x 32 blocks of sums of the job that has the most: 16 with 64 residual channels, 12 with 48
static int most_sums(int R, int K, int C) {
    const auto blocks_of = [](int rows) { return (rows + 31) / 32; };
    return std::max({2 * blocks_of(R) * blocks_of(2 * R), blocks_of(C) * blocks_of(2 * R), blocks_of(R) * blocks_of(R),
                     blocks_of(R) * blocks_of(std::min(K, 128))});
}
size_t wavenet_block_weights_scratch(int R, int K, int C) { return (size_t)kTallWorkgroups * (most_sums(R, K, C) * 1024 + 256); }

int wavenet_block_weights(hipStream_t stream, int R, int K, int C, int N, int count, const BlockGradients *blocks, const float *ctx,
                          const char *patTypes, float *scratch) {
    CNT_REQUIRE(wavenet_block_weights_supported(R, K, C, N) && N > 0 && count >= 1 && count <= kBlockGradients && blocks && ctx &&
                patTypes && scratch, "wavenet_block_weights: bad argument");
    TallArgs a = {};
    for (int z = 0; z < count; ++z) {
        a.block[z] = blocks[z];
        a.block[z].shift = std::min(blocks[z].shift, N);  // further back there is nothing
    }
    a.n = N; a.R = R; a.K = K; a.C = C;
    a.conv_ld = 3 * R;
    a.jobs = 3 + (K + 127) / 128;
    a.ctx = ctx; a.pat = patTypes;
    a.partial = scratch;
    a.sums = most_sums(R, K, C);
    a.rows = scratch + (size_t)kTallWorkgroups * a.sums * 1024;
    // The launch is one generation, two workgroups per compute unit; a block's share is dealt to its jobs by what a tile of theirs
    // takes: 16 rows to convert weigh about as much as a block of sums to multiply, and a tile's barriers and the wait for its loads
    // about eight times that.  Pass without this constant / with 3 / 5 / 8, us: 20 blocks of 32 and 32 channels, 80 features, 24 000
    // slots 1088 / 1015 / 1011 / 994 (the tiled products took 1060 to 1075 there), 32 and 64 channels, 50 features 1073 / - / - / 1033, 64 and
    // 256 channels 2270 / 2263 / 2270 / 2266, 30 blocks of 64 and 128 over 32 000 3407 / 3352 / 3334 / 3328; with 16 to 30 the wide ones lose
    // 1 to 2 % again.
    const int per_block = kTallWorkgroups / count;
    const auto blocks_of = [](int rows) { return (rows + 31) / 32; };
    int cost[kTallMaxJobs], total = 0;
    for (int j = 0; j < a.jobs; ++j) {
        const int skip = std::min(K - 128 * (j - 3), 128);
        const int m = j == 0 ? 2 * R : j == 1 ? C : R, n = j < 2 ? 2 * R : j == 2 ? R : skip;
        cost[j] = kTallTileCost + (m + n + 15) / 16 + (j == 0 ? 2 * blocks_of(R) : blocks_of(m)) * blocks_of(n);
        total += cost[j];
    }
    const int tiles = (N + kTallDepth - 1) / kTallDepth;
    for (int j = 0; j < a.jobs; ++j)
        a.first[j + 1] = a.first[j] + std::max(1, std::min(per_block * cost[j] / total, (tiles + 3) / 4));
    ProfileScope prof(stream, "wavenet_block_weights");
    hipLaunchKernelGGL(wavenet_block_weights_kernel, dim3((unsigned)(count * a.first[a.jobs])), dim3(kTallThreads), 0, stream, a);
    hipLaunchKernelGGL(wavenet_block_weights_sum_kernel, dim3((unsigned)(a.jobs * (kTallBlocks + 1)), (unsigned)count), dim3(256), 0,
                       stream, a);
    CNT_HIP(hipGetLastError());
    return CNT_OK;
}

}  // namespace cnt
