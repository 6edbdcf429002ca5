// fp32 matrix product for launches that cannot fill the machine with the tiles of gemm_split_kernel.
//
// Small layers, short fractions and a single utterance make products of a few tiles with hundreds of k: there a tile's serial
// chain -- load, convert, LDS, barrier, matrix instructions, barrier, 0.7 to 1.1 us per 32 k -- is the launch's time.  Here a
// workgroup owns a 32 x 32 block of the output and its eight waves deal the k positions among themselves, sixteen at a time.  A
// wave stages its share through a piece of LDS of its own: vectors of four floats, requested two steps ahead, are converted
// (split_pair, the same three bf16 parts and six part products as there), laid down in 16-byte units of eight consecutive k
// and read back as fragments, without a barrier; two waves per SIMD, so that one converts while the other's matrix instructions
// run.  The waves meet once, when the eight partial sums are added through LDS.  With fragments loaded straight from memory, one
// float per lane and k, the address unit (sixteen clocks per load and wave) took 0.85 us per 128 k.
//
// What bounds it: a compute unit gets 50 GB/s through its outstanding misses, 0.66 us per 128 k (twice as many waves, or loads
// three and four steps ahead: the same).
// What it costs: operands are read and converted once per 32 rows of the other operand instead of 64 or 128, so it is the faster
// one only up to a size (direct_product below).
#include "gemm_kernel.hpp"

#include <cstdlib>
#include <limits>

namespace cnt {
namespace {

constexpr int kDirectWaves = 8;
constexpr int kChunk = 16;  // k positions of a step: one matrix instruction deep
constexpr int kAhead = 2;   // steps whose loads are in flight

// A wave's 32-row x 16-k piece of an operand: what a lane loads of it and where that lies in the wave's LDS.
// LDS: 16-byte units of eight consecutive k of one row, [part][k / 8][position of the row].
// k-contiguous operands: a vector holds four k of one row, four lanes a row; position = row.
// Row-contiguous: a vector holds four rows of one k, a lane two consecutive k; position (row % 4) * 8 + row / 4, so that the lanes of
// a store fall on distinct banks.  At the matrix's last rows the vectors overlap instead of reaching beyond the line.
// Rows of the block outside the matrix hold the last row again, or whatever was there: they reach only sums that are not stored.
template <bool KCONTIG>
struct Piece {
    static constexpr int LINE = KCONTIG ? 32 : 40, PART = 2 * LINE, UNITS = 3 * PART;
    unsigned voff[2];  // bytes from the operand's first value to the lane's vectors at k = 0
    int at[KCONTIG ? 2 : 4];  // byte offset in LDS of vector p's / row q's first part
    int row[2], ld;

    static __device__ __forceinline__ int k(int lane, int p) { return KCONTIG ? lane % 4 * 4 : lane / 8 * 2 + p; }
    __device__ __forceinline__ void init(int ld_, int row0, int rows_total, int lane) {
        ld = ld_;
#pragma unroll
        for (int p = 0; p < 2; ++p) {
            row[p] = KCONTIG ? min(row0 + lane / 4 + 16 * p, rows_total - 1) : min(row0 + lane % 8 * 4, rows_total - 4);
            voff[p] = (unsigned)((KCONTIG ? (size_t)row[p] * ld + k(lane, p) : (size_t)k(lane, p) * ld + row[p]) * sizeof(float));
            if (KCONTIG) at[p] = 16 * (lane % 4 / 2 * LINE + lane / 4 + 16 * p) + 8 * (lane & 1);
        }
        if constexpr (!KCONTIG) {
#pragma unroll
            for (int q = 0; q < 4; ++q) {
                const int r = row[0] - row0 + q;  // below 0: the row belongs to the block before this one
                const int position = r >= 0 ? r % 4 * 8 + r / 4 : 32 + (lane & 7);  // (the pad of the line takes it)
                at[q] = 16 * (lane / 32 * LINE + position) + 4 * (lane / 8 % 4);
            }
        }
    }
    // the vectors of sixteen k positions from `base` on (uniform)
    __device__ __forceinline__ void load(const float *__restrict__ base, float (&v)[2][4]) const {
#pragma unroll
        for (int p = 0; p < 2; ++p) {
            const f32x4u x = *reinterpret_cast<const f32x4u *>(reinterpret_cast<const char *>(base) + voff[p]);
#pragma unroll
            for (int q = 0; q < 4; ++q) v[p][q] = x[q];
        }
    }
    // the same of sixteen listed k lines (row-contiguous operands): idx = the lane's two
    __device__ __forceinline__ void load_listed(const float *__restrict__ base, const int (&idx)[2], float (&v)[2][4]) const {
#pragma unroll
        for (int p = 0; p < 2; ++p) {
            const f32x4u x = *reinterpret_cast<const f32x4u *>(base + (size_t)idx[p] * ld + row[0]);
#pragma unroll
            for (int q = 0; q < 4; ++q) v[p][q] = x[q];
        }
    }
    // load where the operand ends after `left` of them: zeros behind its end
    __device__ __forceinline__ void load_end(const float *__restrict__ base, int left, int lane, float (&v)[2][4]) const {
#pragma unroll
        for (int p = 0; p < 2; ++p)
#pragma unroll
            for (int q = 0; q < 4; ++q) {
                const int kk = k(lane, p) + (KCONTIG ? q : 0), kc = kk < left ? kk : 0;
                const float x = base[KCONTIG ? (size_t)row[p] * ld + kc : (size_t)kc * ld + row[p] + q];
                v[p][q] = kk < left ? x : 0.0f;
            }
    }
    __device__ __forceinline__ void put(uint4 *lds, const float (&v)[2][4]) const {
        char *const to = reinterpret_cast<char *>(lds);
        if constexpr (KCONTIG) {
#pragma unroll
            for (int p = 0; p < 2; ++p) {
                unsigned x[2][3];
                split_pair(v[p][0], v[p][1], x[0]);
                split_pair(v[p][2], v[p][3], x[1]);
#pragma unroll
                for (int q = 0; q < 3; ++q) *reinterpret_cast<uint2 *>(to + at[p] + 16 * q * PART) = uint2{x[0][q], x[1][q]};
            }
        } else {
#pragma unroll
            for (int r = 0; r < 4; ++r) {
                unsigned x[3];
                split_pair(v[0][r], v[1][r], x);
#pragma unroll
                for (int q = 0; q < 3; ++q) *reinterpret_cast<unsigned *>(to + at[r] + 16 * q * PART) = x[q];
            }
        }
    }
    // lane = 32 * half + row: k positions 8 * half .. + 7 of the row
    static __device__ __forceinline__ void fragment(const uint4 *lds, int lane, bf16x8 (&f)[3]) {
        const int r = lane & 31;
        const uint4 *from = lds + lane / 32 * LINE + (KCONTIG ? r : r % 4 * 8 + r / 4);
#pragma unroll
        for (int q = 0; q < 3; ++q) f[q] = __builtin_bit_cast(bf16x8, from[q * PART]);
    }
};

// One block.  GATHER: the k lines of both (row-contiguous) operands are those a list names (GemmArgs::k_order).  ARGS and PROBLEM: GemmArgs
// and one of its problems, or a group of weight gradients (one operand pair, EPI_STORE) and one of those.
template <bool AK, bool BK_, bool GATHER, typename ARGS, typename PROBLEM>
__device__ __forceinline__ void direct_block(const ARGS &args, const PROBLEM &pb, unsigned block) {
    constexpr bool GROUP = std::is_same<ARGS, DirectGroup>::value;
    typedef Piece<AK> PA;
    typedef Piece<BK_> PB;
    constexpr int STAGE = PA::UNITS + PB::UNITS;
    static_assert(STAGE >= 4 * 64, "a wave's sums fit its staging buffer");
    __shared__ uint4 lds[kDirectWaves][STAGE];
    __shared__ float row_sums[kDirectWaves][32];

    const int lane = threadIdx.x & 63;
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    uint4 *const mine_a = lds[wave], *const mine_b = lds[wave] + PA::UNITS;
    const auto &size = sizes_of(args, pb);
    int nseg = 1, has_sums = 0;
    if constexpr (GROUP) has_sums = pb.rowsum;
    else { nseg = args.nseg; has_sums = args.rowsum; }
    const int tiles_m = (size.m + 31) / 32;
    const int m0 = (int)(block % (unsigned)tiles_m) * 32, n0 = (int)(block / (unsigned)tiles_m) * 32;

    PA oa;
    PB ob;
    oa.init(size.lda, m0, size.m, lane);
    ob.init(size.ldb, n0, size.n, lane);
    const size_t ka = kChunk * (AK ? 1 : (size_t)size.lda), kb = kChunk * (BK_ ? 1 : (size_t)size.ldb);  // floats per chunk
    const bool rowsum = !AK && !BK_ && has_sums != 0 && m0 == 0;
    float rs[4] = {0.0f, 0.0f, 0.0f, 0.0f};  // of the lane's four rows, over the k positions it loads

    f32x16 acc;
#pragma unroll
    for (int r = 0; r < 16; ++r) acc[r] = 0.0f;
    auto multiply = [&](const float (&a)[2][4], const float (&b)[2][4], auto meanwhile) __attribute__((always_inline)) {
        if (!AK && !BK_ && rowsum) {
#pragma unroll
            for (int q = 0; q < 4; ++q) rs[q] += b[0][q] + b[1][q];
        }
        oa.put(mine_a, a);
        ob.put(mine_b, b);
        meanwhile();
        bf16x8 fa[3], fb[3];
        __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
        __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
        PA::fragment(mine_a, lane, fa);
        PB::fragment(mine_b, lane, fb);
        __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
        __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
        __builtin_amdgcn_sched_barrier(0);  // one wait for all six
        // h*l, l*h, m*m, h*m, m*h, h*h: the small terms first
        constexpr int QA[6] = {0, 2, 1, 0, 1, 0}, QB[6] = {2, 0, 1, 1, 0, 0};
#pragma unroll
        for (int t = 0; t < 6; ++t) acc = __builtin_amdgcn_mfma_f32_32x32x16_bf16(fb[QB[t]], fa[QA[t]], acc, 0, 0, 0);
    };
    // the k positions this problem takes: all of them, or the listed lines, all but the first / last time step's
    int k_extent = size.k, k_lo = 0;
    if (GATHER) {
        k_extent = args.k_count[0];
        if (pb.k_trim == 1) { k_lo = args.k_count[1]; k_extent -= k_lo; }
        else if (pb.k_trim == 2) k_extent -= args.k_count[2];
        k_extent = max(k_extent, 0);
    }
    // the whole chunks of the concatenated operand pairs: wave, wave + 8, ...
    const int per_seg = k_extent / kChunk, total = per_seg * nseg;
    const int *const lines = GATHER ? args.k_order + k_lo : nullptr;
    const int shift = GATHER ? pb.k_shift : 0;
    auto lines_of = [&](int chunk, int (&idx)[2]) __attribute__((always_inline)) {
#pragma unroll
        for (int p = 0; p < 2; ++p) idx[p] = lines[chunk * kChunk + PA::k(lane, p)] + shift;
    };
    if (wave < total) {
        const int mine = (total - wave + kDirectWaves - 1) / kDirectWaves;
        int seg = wave / per_seg, kin = wave % per_seg, left = mine - 1;
        const float *pa = pb.A[seg], *pbb = pb.B[seg];
        float a[kAhead][2][4], b[kAhead][2][4];
        int idx[2];
        if constexpr (GATHER) lines_of(kin, idx);
        // the next of the wave's chunks; after the last one that one again, so that as many loads are in flight on every path
        auto fetch = [&](float (&va)[2][4], float (&vb)[2][4]) __attribute__((always_inline)) {
            const int at = kin;
            const float *const qa = pa, *const qb = pbb;
            if (left > 0) {
                --left;
                kin += kDirectWaves;
                if (kin >= per_seg) {
                    do { kin -= per_seg; ++seg; } while (kin >= per_seg);
                    pa = pb.A[seg]; pbb = pb.B[seg];
                }
            }
            if constexpr (GATHER) {
                // the next chunk's lines in front of this one's data: waiting for them does not wait for the data
                const int now[2] = {idx[0], idx[1]};
                lines_of(kin, idx);
                oa.load_listed(qa, now, va);
                ob.load_listed(qb, now, vb);
            } else {
                oa.load(qa + at * ka, va);
                ob.load(qb + at * kb, vb);
            }
        };
#pragma unroll
        for (int d = 0; d < kAhead; ++d) fetch(a[d], b[d]);
        for (int i = 0; i < mine; i += kAhead) {
#pragma unroll
            for (int d = 0; d < kAhead; ++d) {
                if (d > 0 && i + d >= mine) break;
                multiply(a[d], b[d], [&]() __attribute__((always_inline)) { fetch(a[d], b[d]); });
            }
        }
    }
    // what is left of each pair, one wave each
    const int rest = k_extent % kChunk;
    if (rest != 0 && wave < nseg) {
        float a[2][4], b[2][4];
        if constexpr (GATHER) {
            int idx[2];
            bool on[2];
#pragma unroll
            for (int p = 0; p < 2; ++p) {
                on[p] = PA::k(lane, p) < rest;
                idx[p] = lines[per_seg * kChunk + (on[p] ? PA::k(lane, p) : 0)] + shift;
            }
            oa.load_listed(pb.A[0], idx, a);
            ob.load_listed(pb.B[0], idx, b);
#pragma unroll
            for (int p = 0; p < 2; ++p)
#pragma unroll
                for (int q = 0; q < 4; ++q) { a[p][q] = on[p] ? a[p][q] : 0.0f; b[p][q] = on[p] ? b[p][q] : 0.0f; }
        } else {
            oa.load_end(pb.A[wave] + per_seg * ka, rest, lane, a);
            ob.load_end(pb.B[wave] + per_seg * kb, rest, lane, b);
        }
        multiply(a, b, [] {});
    }

    auto leave = [&](const f32x16 &x) __attribute__((always_inline)) {
#pragma unroll
        for (int r = 0; r < 16; r += 4)
            lds[wave][r / 4 * 64 + lane] = uint4{__float_as_uint(x[r]), __float_as_uint(x[r + 1]), __float_as_uint(x[r + 2]), __float_as_uint(x[r + 3])};
    };
    // of the sixteen sums of a lane, wave w takes the registers MINE * w and on
    constexpr int MINE = 16 / kDirectWaves;
    static_assert(kDirectWaves == 8, "the sums below");
    auto gather = [&](float (&v)[MINE]) __attribute__((always_inline)) {
        constexpr int PER_UNIT = 4 / MINE;  // waves that share a 16-byte unit
        float x[kDirectWaves][MINE];
#pragma unroll
        for (int q = 0; q < kDirectWaves; ++q)
#pragma unroll
            for (int r = 0; r < MINE; ++r)
                x[q][r] = (reinterpret_cast<const float *>(&lds[q][wave / PER_UNIT * 64 + lane]) + wave % PER_UNIT * MINE)[r];
#pragma unroll
        for (int r = 0; r < MINE; ++r)
            v[r] = ((x[0][r] + x[1][r]) + (x[2][r] + x[3][r])) + ((x[4][r] + x[5][r]) + (x[6][r] + x[7][r]));
    };
    leave(acc);
    if (rowsum) {
        // the lanes that loaded other k positions of the same four rows differ in lane / 8
#pragma unroll
        for (int q = 0; q < 4; ++q) {
            float t = rs[q];
            t += __shfl_xor(t, 8); t += __shfl_xor(t, 16); t += __shfl_xor(t, 32);
            const int r = ob.row[0] - n0 + q;
            if (lane < 8 && r >= 0) row_sums[wave][r] = t;
        }
    }
    __syncthreads();
    float v[MINE];
    gather(v);
    // what came out infinite or not a number is formed again, by all waves (plain_sums)
    const int m = m0 + (lane & 31), half = lane >> 5;
    bool finite = true;
#pragma unroll
    for (int q = 0; q < MINE; ++q) {
        const int r = MINE * wave + q, n = n0 + 8 * (r >> 2) + 4 * half + (r & 3);
        finite = finite && (m >= size.m || n >= size.n || __builtin_fabsf(v[q]) <= lim::kMax);
    }
#pragma unroll
    for (int r = 0; r < MINE; ++r) v[r] *= 1.0f / (kSplitScale * kSplitScale);
    if (__builtin_expect(__syncthreads_or(!finite), 0)) {
        const int kt = (k_extent + BK - 1) / BK, all = kt * nseg, each = (all + kDirectWaves - 1) / kDirectWaves;
        // (every wave has read the sums above before this: the barrier in __syncthreads_or)
        leave(plain_sums<AK, BK_, false, GATHER>(args, pb, m0, n0, lane, min(all, wave * each), min(all, (wave + 1) * each), kt,
                                                   k_extent, k_lo));
        __syncthreads();
        gather(v);
    }

    if (rowsum && threadIdx.x < 32 && n0 + (int)threadIdx.x < size.n) {
        float x[kDirectWaves];
#pragma unroll
        for (int q = 0; q < kDirectWaves; ++q) x[q] = row_sums[q][threadIdx.x];
        const float s = ((x[0] + x[1]) + (x[2] + x[3])) + ((x[4] + x[5]) + (x[6] + x[7]));
        pb.rowsum_out[n0 + threadIdx.x] = pb.rowsum_scale * s;
    }
    if (m >= size.m) return;
    if constexpr (GROUP) {
#pragma unroll
        for (int q = 0; q < MINE; ++q) {
            const int r = MINE * wave + q, n = n0 + 8 * (r >> 2) + 4 * half + (r & 3);
            if (n < size.n) pb.C[(size_t)n * size.ldc + m] = v[q];
        }
        return;
    } else {
    float bterm = 0.0f;
    if (args.epilogue == EPI_BIAS_ACT || args.epilogue == EPI_BIAS_ACT_SKIP) bterm = args.bias_scale * pb.bias_vec[m];
#pragma unroll
    for (int q = 0; q < MINE; ++q) {
        const int r = MINE * wave + q, n = n0 + 8 * (r >> 2) + 4 * half + (r & 3);
        if (n >= size.n) continue;
        const size_t idx = (size_t)n * size.ldc + m;
        float *dst = pb.C + idx;
        const float x = v[q];
        switch (args.epilogue) {
            case EPI_STORE: *dst = x; break;
            case EPI_STORE_DELTA: *dst = x * act_deriv(args.act, pb.aux_in[idx]); break;
            case EPI_ADD: *dst = *dst + x; break;
            case EPI_ATOMIC: atomicAdd(dst, x); break;
            case EPI_BIAS_ACT: *dst = act_fn(args.act, x + bterm); break;
            case EPI_BIAS_ACT_SKIP:
                if (args.pat[n] != 0) *dst = act_fn(args.act, x + bterm);
                break;
            case EPI_FAN: {
                const float e = pb.aux_in ? pb.aux_in[idx] + x : x;
                *dst = e;
                for (int f = 0; f < args.fan_n; ++f) {
                    float *t = args.fan_targets[f] + idx;
                    *t = args.fan_is_skip[f] ? e + *t : e;
                }
            } break;
            default: {  // EPI_CONTEXT
                const bool valid = args.pat[n] != 0;
                const float th = valid ? tanh_act(x) : 0.0f;
                if (pb.aux_out) pb.aux_out[idx] = th;
                *dst = valid ? pb.aux_in[idx] + th : 0.0f;
            } break;
        }
    }
    }
}

template <bool AK, bool BK_, bool GATHER>
__global__ __launch_bounds__(64 * kDirectWaves, 4) void gemm_direct_kernel(const GemmArgs args) {
    direct_block<AK, BK_, GATHER>(args, args.prob[blockIdx.z], blockIdx.x);
}

// The weight gradients of a small pass, or a recurrent layer's two, as one launch (DirectGroup).  One after the other each took 5 to 16 us
// for blocks that leave most of the compute units idle; side by side they take little longer than the longest.  blstm 128 with dense
// layers over 120 slots, four such launches: 115 -> 96 us per pass; one lstm layer of 256 cells over 800 slots, two: 362 -> 359.
template <bool GATHER>
__global__ __launch_bounds__(64 * kDirectWaves, 4) void gemm_direct_group_kernel(const DirectGroup group) {
    // (the starts are a few scalar loads side by side; a search along them would wait for one after the other)
    int i = 0;
#pragma unroll
    for (int q = 1; q < kGroupProducts; ++q) i += (int)blockIdx.x >= group.first[q] ? 1 : 0;
    direct_block<false, false, GATHER>(group, group.product[i], blockIdx.x - (unsigned)group.first[i]);
}

}  // namespace

// Measured on MI355X, us, tiled kernel / this one (weight gradients: with the clear and the column sum that the tiled one needs).
// Products: 32 x 120 over 64 / 512 values of k 5.7 / 4.3, 16.4 / 6.7; 256 x 400 over 256 / 1024 11.6 / 5.7, 28.6 / 9.9 (104 blocks);
// 382 x 800 over 1024 28.3 / 15.7 (300); 512 x 800 over 512 16.6 / 10.5 (400); 300 x 2000 over 1200 33.0 / 24.9 (630); 600 x 1000 over
// 2048 52.5 / 37.5 (608); 200 x 3000 over 200 10.9 / 10.4 (658); 512 x 2000 over 512 18.6 / 19.3 (1008); 1936 x 600 over 256 14.1 /
// 14.9 (1159); 1936 x 6000 over 256 52.9 / 101.6: up to 640 blocks, five for two compute units.
// Weight gradients, which the tiled kernel cuts along k: 32 x 128 over 120 14.5 / 5.8; 256 x 256 over 500 / 2000 / 8000 18.9 / 7.4, 19.5 /
// 15.5, 22.0 / 47.6; 512 x 512 over 400 / 1600 / 6000 22.6 / 7.3, 22.3 / 14.7, 41.6 / 41.8; 64 x 64 over 2000 18.7 / 15.1; 400 x 60 over
// 3000 16.2 / 20.4; 1024 x 1024 over 4000 79.4 / 92.4: up to 512 blocks and 2048 values of k, which take sixteen rounds of 0.66.
constexpr long kDirectBlocks = 640, kDirectGradientBlocks = 512, kDirectGradientDepth = 2048;
bool direct_product(const GemmArgs &a) {
    static const int forced = [] { const char *e = std::getenv("CNT_GEMM_DIRECT"); return e ? std::atoi(e) : -1; }();
    // (a row-contiguous operand is read in vectors of four rows)
    if (a.masked || (a.a_kcontig && !a.b_kcontig) || (!a.a_kcontig && a.m < 4) || (!a.b_kcontig && a.n < 4)) return false;
    if (forced >= 0) return forced != 0;
    const long blocks = (long)((a.m + 31) / 32) * ((a.n + 31) / 32) * a.nprob;
    return a.splitk == 0 ? blocks <= kDirectGradientBlocks && (long)a.k * a.nseg <= kDirectGradientDepth : blocks <= kDirectBlocks;
}

int gemm_group_add(hipStream_t stream, DirectGroup &g, const GemmArgs &a) {
    const bool listed = a.k_order && a.k_count;
    const int *const order = listed ? a.k_order : nullptr;
    if (g.count > 0 && (g.count + a.nprob > kGroupProducts || order != g.k_order)) CNT_TRY(gemm_group_launch(stream, g));
    g.k_order = order; g.k_count = listed ? a.k_count : nullptr;
    const int blocks = ((a.m + 31) / 32) * ((a.n + 31) / 32);
    for (int z = 0; z < a.nprob; ++z) {
        const GemmProblem &p = a.prob[z];
        g.first[g.count] = g.blocks;
        g.product[g.count] = {{p.A[0]}, {p.B[0]}, p.C, p.rowsum_out, a.m, a.n, a.k, a.lda, a.ldb, a.ldc, p.rowsum_scale, a.rowsum, p.k_trim,
                              p.k_shift};
        ++g.count;
        g.blocks += blocks;
    }
    return CNT_OK;
}

int gemm_group_launch(hipStream_t stream, DirectGroup &g) {
    if (g.count == 0) return CNT_OK;
    for (int q = g.count; q < kGroupProducts; ++q) g.first[q] = std::numeric_limits<int>::max();
    ProfileScope prof(stream, "gemm:weight_gradients");
    const dim3 grid((unsigned)g.blocks), block(64 * kDirectWaves);
    if (g.k_order) hipLaunchKernelGGL(gemm_direct_group_kernel<true>, grid, block, 0, stream, g);
    else hipLaunchKernelGGL(gemm_direct_group_kernel<false>, grid, block, 0, stream, g);
    g.count = g.blocks = 0;
    CNT_HIP(hipGetLastError());
    return CNT_OK;
}

void gemm_direct_launch(const GemmArgs &a, hipStream_t s) {
    const dim3 grid((unsigned)(((a.m + 31) / 32) * ((a.n + 31) / 32)), 1, (unsigned)a.nprob), block(64 * kDirectWaves);
    if (a.a_kcontig) hipLaunchKernelGGL((gemm_direct_kernel<true, true, false>), grid, block, 0, s, a);
    else if (a.b_kcontig) hipLaunchKernelGGL((gemm_direct_kernel<false, true, false>), grid, block, 0, s, a);
    else if (a.k_order && a.k_count && a.nseg == 1) hipLaunchKernelGGL((gemm_direct_kernel<false, false, true>), grid, block, 0, s, a);
    else hipLaunchKernelGGL((gemm_direct_kernel<false, false, false>), grid, block, 0, s, a);
}

}  // namespace cnt
