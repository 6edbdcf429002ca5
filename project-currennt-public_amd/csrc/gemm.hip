// fp32 matrix product for gfx950 on the bf16 matrix instructions.
//
// This is the seam that the reference reaches through helpers::Matrix::assignProduct/addProduct
// (helpers/Matrix.cu:353-377 -> helpers/cublas.cu:52-84).  One kernel covers every operand
// orientation, K-concatenated accumulation over several operand pairs (the eight W_in * delta
// products of a BLSTM become one pass), several independent problems per launch, split-K for the
// long-K weight-gradient shapes, and a fused bias + activation epilogue for the dense forward.
//
// Arithmetic: the fp32 matrix instructions end at 157 TFLOP/s and reached 88 here, with the matrix units 56% busy.  Every
// operand value is therefore split into three bf16 parts, 2^16 x = h + m + l (round to nearest, so m <= 2^-9 of it and
// l <= 2^-18), and a product is the sum of the six part products h*h, h*m, m*h, m*m, h*l, l*h, which the bf16
// instructions form exactly and add in fp32, the small ones first.  What is left out (m*l, l*m, l*l) is below 2^-25 of
// |a||b|, less than the rounding of one fp32 product.  An instruction adds sixteen products before it rounds, where the fp32 one
// adds two, so the result is closer to a 64-bit product than before: 2-norm error 4.9e-7 against 5.7e-7 at k = 1024, 1.2e-6
// against 1.4e-6 at k = 6000, 1.6e-7 against 2.0e-7 at k = 128.
// Range: the split is exact for every fp32 value below 2^112, subnormal ones included, which is what the factor 2^16 is for
// (without it values below 2^-110 lose their low parts, and products of values around 2^-126 were off by 2^-9); it costs a
// multiplication per operand value and load, 1-3% of a product's time.  Operands from 2^112 on, infinite ones and sums
// from 2^96 on leave infinities or infinity minus infinity behind; a block of sums of which one is not finite is formed again on
// the fp32 instructions (plain_sums).
//   1024 x 12000 x 1024: 283 -> 140 us (180 TFLOP/s), 512 x 6000 x 512: 40 -> 29 us, 1024 x 6000 x 512: 74 -> 51 us,
//   1024 x 32000 x 128: 108 -> 73 us, 425 x 12000 x 1024: 141 -> 96 us, 300 x 10000 x 425: 47 -> 34 us.
// Operands whose lines are no multiple of four long are read in vectors of four as well (FastStage); with one float per
// lane and load the last two sizes took 100 and 43 us.
// What bounds it now: the matrix instructions under the card's power limit.  With random operands one takes 20 to 24 ns of a SIMD
// (15 with zeros), which is 105 us of the first size's 138; leaving out five of the six part products gives 80 us, the
// conversions 130, the loads 122.  With 64 x 64 tiles (512 x 9600 x 1024, 77 us: 48, 68, 60) the loads through the L2s and the
// conversions weigh twice as much.  Measured and not taken: the conversion of the next tile between the matrix instructions of
// this one, with two LDS buffers and one or two tiles of loads in flight (245 us: one wave per SIMD issues a vector
// instruction every eight clocks, not four); 128 x 64 tiles (182 us); 256 x 192 tiles of eight waves, half of them converting
// in turn (162 us); LDS stores without bank conflicts (a third of the LDS clocks less, no difference); instructions of
// 16 x 16 x 32, which alone run a third faster (150 us: twice as many of them hold the vector instructions up).
//
// Tiling: T x T x 32 per workgroup with T = 128 or 64, four 64-lane waves in a 2 x 2 arrangement, each wave
// owning a T/2 x T/2 block as tiles of v_mfma_f32_32x32x16_bf16.  The parts lie in LDS in the order the instruction takes
// them (TileLayout); 50 KB (T = 128) and 26 KB (T = 64) per workgroup leave room for three and five of them per compute unit, whose
// phases overlap.  Two workgroups of T = 128 instead of three: 197 us at the first size above.  A launch of few large tiles
// takes eight waves for each of them, 2 x 4 of 64 x 32 (same sums, bit for bit; eight_waves below).
// The MFMA operands are swapped (the B tile feeds the instruction's A port) so that lane%32 walks
// along the column-major output's contiguous dimension and every store is a 128-byte segment.
#include "gemm_kernel.hpp"

#include <algorithm>
#include <cstdlib>
#include <mutex>
#include <vector>

namespace cnt {
namespace {

inline int pick_vec(const GemmArgs &a, bool for_a) {
    const int ld = for_a ? a.lda : a.ldb;
    const bool kc = for_a ? a.a_kcontig : a.b_kcontig;
    const int extent = kc ? a.k : (for_a ? a.m : a.n);
    int v = 4;
    while (v > 1) {
        bool ok = (ld % v == 0) && (extent % v == 0);
        for (int p = 0; ok && p < a.nprob; ++p)
            for (int s = 0; ok && s < a.nseg; ++s) {
                const float *ptr = for_a ? a.prob[p].A[s] : a.prob[p].B[s];
                ok = (reinterpret_cast<uintptr_t>(ptr) % (4 * v)) == 0;
            }
        if (ok) break;
        v >>= 1;
    }
    return v;
}

// Tile edge, and the waves of a workgroup.  128 x 128 tiles convert and read half as much per matrix instruction as 64 x 64 ones.
// On four waves three of them fill a compute unit, and a launch needs some 600 of them to hide a tile's chain of load, conversion,
// barrier and products behind the others'.  On eight waves (kEightWaves) the chain is half as long, so that ONE per compute unit
// is worth having: a launch then takes as long as its busiest compute unit, and what decides is how full the last level of
// one tile per compute unit is.  Times as fast on eight waves as the better of 64 x 64 and 128 x 128 on four (1024 rows, both
// operands k-contiguous; a row-contiguous A and operands of odd length within 5 % of it or better):
//   tiles     192  208  256  264  320  336  400  512  520  640  680  768  800  960 1024 1040 1200 1280 1536 2048
//   level     .75  .81   1   .52  .62  .66  .78   1   .68  .83  .89   1   .78  .94   1   .81  .94   1    1    1
//   k = 384   .93 1.07 1.08  .87  .90 1.03 1.13 1.19  .94 1.03 1.05 1.07 1.05 1.16 1.21 1.05 1.18 1.21 1.10 1.17
//   512       .94 1.11 1.09  .88  .92 1.05 1.09 1.19  .96 1.01 1.01 1.05 1.06 1.19 1.19 1.02 1.04 1.14 1.05 1.06
//   768       .97 1.15 1.16  .90  .92 1.06 1.07 1.10  .94  .99  .98 1.00 1.08 1.13 1.10  .96 1.00 1.08  .98  .99
//   1024      .98 1.18 1.14  .91  .94 1.02 1.01 1.05  .93  .96  .97  .98 1.08 1.09 1.06  .95  .98 1.00  .98  .97
//   2048     1.02 1.21 1.22  .93  .95  .96  .98 1.00  .92  .94  .94  .96 1.05 1.06 1.03  .95
// (512 x 8192 x 2048, 256 tiles: 123 us with 64 x 64, 128 on four waves, 103 on eight.)  From 768 values on, three levels and more
// than four are better off on four waves (a generation of those is 768), and the lines below give away at most 5 %.  Below 384
// values the launch is its stores: back to back eight waves gain up to 15 % there, too, but inside a pass, with operands that have
// left the caches, 1024 x 32000 x 128 takes 99 instead of 79 us, 1936 x 6000 x 256 61 instead of 53, 1024 x 12000 x 187 101 instead of
// 94 (x 425: 100 either way, 2048 x 9600 x 512 123 instead of 125 to 156).
inline bool eight_waves(long tiles, long run) {
    const long levels = (tiles + 255) / 256, percent = 100 * tiles / (256 * levels);
    if (run >= 1536) return levels == 1 ? percent >= 80 : levels == 4;
    if (run >= 768) return levels == 1 ? percent >= 80 : levels == 2 ? percent >= 65 : levels == 4;
    return run >= 384 && (levels == 2 ? percent >= 65 : levels == 3 ? percent >= 77 : levels == 4 || percent >= 80);
}
// Elsewhere, 64 x 64 or 128 x 128 on four waves.  Between 256 and 383 values the large tile pays where it fills the last generation
// of 768 to nine tenths: 64 / 128, us, for 1024 rows and a k-contiguous A: 752 tiles (0.98) 54 / 49, 704 (0.92) 1.05 times as fast,
// 1360 (0.89) 1.02, 2000 (0.87) 0.97, 640 (0.83) 1.04, 1040 (0.68) 0.87; k = 192 no gain anywhere.  With 768 values and more: the
// large tile from 336 tiles on, where the small ones begin a second generation (1280 of them at a time); times as fast with 304 /
// 320 / 336 / 400 / 600 / 768 / 800 / 1040 large tiles
// (least and most over 512, 1024 and 2048 rows and both orders of A): k = 768 0.84-0.87 / 0.86-0.89 / 1.00-1.04 / 1.08-1.13 / 1.04 /
// 1.23-1.25 / 0.97-0.99 / 1.10-1.12, k = 3072 0.95-1.01 / 0.96-1.02 / 1.12-1.18 / 1.22-1.28 / 1.12 / 1.32-1.35 / 1.06 / 1.17-1.20.  Lines
// of odd length (loads of single values at the edges): from 600 tiles and 512 values on.
inline long large_tiles(const GemmArgs &a) { return (long)((a.m + 127) / 128) * ((a.n + 127) / 128) * a.nprob; }

// The weight gradient of one dense layer of 64 to 256 large tiles (1024 x 1024 weights and more) also takes the large tile, and
// as many splits of k as make two workgroups per compute unit (the parts of two row-contiguous operands take 55 KB of LDS, so more
// do not fit), as long as a split has at least 768 values of k: below that, filling and draining the pipeline and the atomic sums
// of the tiles outweigh what the large tile saves, and three times as many small workgroups share them better.  64 / 128, us,
// with the clear and a column sum behind it, which the product brings along by now: 1024 x 1024 over 2000 / 5000 / 8000 /
// 12 000 slots (250 / 625 / 1000 / 1500 per split) 43 / 58, 88 / 89, 134 / 121, 193 / 162; 1300 x 1300 over 3000 / 4000 (750 / 1000) 98 / 101, 125 / 120; 2048 x 2048 over
// 1000 / 3000 (500 / 1500) 73 / 79, 187 / 159.  (Below 64 tiles the line is further up, 896 x 896 over 2000 / 6000 / 12 000
// 41 / 57, 92 / 86, 173 / 136, and layers of 32 tiles gain nothing; they keep the small tile.)  The feed-forward model of five
// such layers: 2320 -> 2224 us per pass, with 768 workgroups 2230; on eight waves 2228 -> 2152.
constexpr long kWideGradientGroups = 512;
constexpr long kWideGradientSplit = 768;
inline bool wide_gradient(const GemmArgs &a) {
    const long tiles = large_tiles(a);
    return a.nprob == 1 && !a.masked && !a.a_kcontig && !a.b_kcontig && tiles >= 64 && tiles <= kWideGradientGroups / 2 &&
           (long)a.k * a.nseg * tiles >= kWideGradientSplit * kWideGradientGroups;
}

// The gradients of a recurrent layer, several problems per launch, on eight waves and one tile per compute unit: at least 32 large
// tiles that the outputs fill, cut into as many splits as make 256 workgroups, of at least 704 values of k.  64 x 64 tiles cut to
// 768 workgroups / 192, 256, 384, 512 workgroups of eight waves, us per pass: 32 sequences 2463 / 2410, 2373, 2357, 2376; the
// acoustic model, where they run beside the recursion of the layer below, 2587 / 2582, 2569, 2620, 2599.  A layer of 2 x 256 cells
// by itself over 2048 / 3200 / 6400 / 9600 slots (512, 800, 1600 and 2400 per split of the input weights) 454 / 464, 626 / 620, 837 /
// 817, 1189 / 1161, of 2 x 512 cells over 2048 / 9600 757 / 743, 3008 / 2886.  Around the line,
// 2 x 256 cells over 2048 / 2304 / 2560 / 2752 / 3008 / 3200 / 3840 slots (512 to 960 per split) 613 / 611, 667 / 670, 720 / 724, 763 / 766,
// 815 / 817, 855 / 855, 990 / 986; 2 x 512 over 1536 / 2048 / 2560 / 3200 (768 to 1600) 784 / 776, 963 / 943, 1190 / 1157, 1435 / 1397: what
// lies on the wrong side of it is 0.5 %.  (300 and 200 cells leave a quarter of the large tiles' rows empty: 2264 -> 2315 with
// them.)
constexpr long kLevelGradientGroups = 256;
constexpr long kLevelGradientSplit = 704;
inline bool level_gradient(const GemmArgs &a) {
    const long tiles = large_tiles(a);
    return a.nprob > 1 && !a.masked && !a.a_kcontig && !a.b_kcontig && tiles >= 32 && tiles <= kLevelGradientGroups &&
           20L * a.m * a.n * a.nprob >= 19L * 16384 * tiles && (long)a.k * a.nseg * tiles >= kLevelGradientSplit * kLevelGradientGroups;
}

int pick_tile(const GemmArgs &a) {
    static const int forced = [] { const char *e = std::getenv("CNT_GEMM_TILE"); return e ? std::atoi(e) : 0; }();
    if (a.masked || a.epilogue == EPI_FAN) return 64;
    if (forced == 64 || forced == 128 || forced == kEightWaves) return forced;
    const long t128 = large_tiles(a) * a.splitk;
    if ((wide_gradient(a) && t128 >= kWideGradientGroups / 2) || (level_gradient(a) && t128 >= kLevelGradientGroups / 2)) return kEightWaves;
    const long run = (long)a.k * a.nseg / a.splitk;
    const long t64 = (long)((a.m + 63) / 64) * ((a.n + 63) / 64) * a.nprob * a.splitk;
    // (outputs that leave more than a twelfth of the large tiles' rows and columns empty stay on the small ones: 300 x 10 000 x 425
    // and the like, 2207 -> 2276 us per pass with them on the large ones.  Up to an eighth empty, 600 tiles and more of 512 to 767
    // values are better off on the large ones, us with 64 x 64 / 128 on four waves / on eight: 430 rows, k = 640, 608 tiles 89 / 85 / 87,
    // 680 94 / 86 / 88, 760 103 / 90 / 90, 980 129 / 133 / 116, 1100 145 / 141 / 142, 1300 165 / 164 / 168, 1400 181 / 168 / 170; k = 760, 680 tiles
    // 115 / 104 / 105, 1100 179 / 167 / 171; 550 rows the same within 1 %; 300 rows, a sixth empty, k = 512 to 760, 609 to 1300 tiles 67 to 194 /
    // 71 to 196 / 72 to 201.)
    const bool filled = 12 * t64 >= 11 * 4 * t128;
    if ((a.a_kcontig || a.b_kcontig) && filled && eight_waves(t128, run)) return kEightWaves;
    if ((a.a_kcontig || a.b_kcontig) && !filled && 8 * t64 >= 7 * 4 * t128 && t128 >= 600 && run >= 512 && run < 768)
        return t128 > 768 && t128 <= 1024 ? kEightWaves : 128;
    const bool quads = (a.a_kcontig ? a.k : a.m) % 4 == 0 && a.b_kcontig && a.k % 4 == 0;
    if (!quads) return t128 >= 600 && run >= 512 ? 128 : 64;
    if (run >= 768) return t128 >= 336 ? 128 : 64;
    return t128 >= 600 && run >= 256 && 10 * t128 >= 9 * ((t128 + 767) / 768 * 768) ? 128 : 64;
}

// ----- split-K through partial products ---------------------------------------------------------------------
// Weight gradients sum over all slots of a fraction, so their products are cut along k, and the splits' sums have to meet.  Every
// split stores its partial product with plain stores into a scratch buffer and a second, small kernel adds the splits up in a fixed
// order, the row sums of B (a dense layer's bias gradient) with them.  Nothing has to be cleared and nothing is added atomically.
// Outputs of a few hundred splits (64 x 128 summed over 32 000 slots) would be bound by their atomic additions.  Wide outputs of a
// few splits take as long either way (five 1024 x 1024 layers over 10 000 slots: pass 2143 us with clears and atomic additions,
// 2152 so, of 33 MB of partial products a layer; the acoustic model 2610 and 2559, 32 sequences 2458 and 2448), but a clear in front of
// atomic additions has once been seen to take a split's additions with it: on one run the bias gradient of a 1024 x 1028 layer came
// out without its first split's share.  Nothing in the launches' order explains it, so no layer's weight gradient rests on it any
// more, and all of them are the same bits in every call.
// (kSplitScratchFloats holds kWideGradientGroups large tiles and their row sums)
constexpr long kManySplits = 8;                          // from here on, and up to kFewOutputs sums, eight threads share a sum's splits
constexpr long kFewOutputs = 128 << 10;

struct SplitScratch {
    int device;
    hipStream_t stream;
    float *buf;
};
std::mutex g_split_mu;  // held while a product and its reduction are enqueued, so that they stay adjacent
std::vector<SplitScratch> g_split_scratch;

// CNT_GEMM_PARTIAL=0: no scratch, everything adds atomically
bool partial_on() {
    static const bool on = [] { const char *e = std::getenv("CNT_GEMM_PARTIAL"); return !e || std::atoi(e) != 0; }();
    return on;
}

thread_local hipStream_t t_loan_stream = nullptr;
thread_local float *t_loan_buffer = nullptr;  // of the thread's ScratchLoan, or null

// One scratch buffer per stream: launches on a stream execute in order, so the next product on the same stream
// cannot overwrite partial sums that a reduction has yet to read.  Kept until gemm_release_stream.
float *split_scratch_find(hipStream_t stream) {
    if (t_loan_buffer && t_loan_stream == stream) return t_loan_buffer;
    int dev = 0;
    if (hipGetDevice(&dev) != hipSuccess) return nullptr;
    for (const SplitScratch &e : g_split_scratch)
        if (e.device == dev && e.stream == stream) return e.buf;
    return nullptr;
}

// the stream's buffer, allocated now if the stream has none; NULL when the allocation is refused (out of memory,
// a stream under capture): the caller then takes the atomic path
float *split_scratch(hipStream_t stream) {
    if (float *buf = split_scratch_find(stream)) return buf;
    int dev = 0;
    if (hipGetDevice(&dev) != hipSuccess) return nullptr;
    float *buf = nullptr;
    if (hipMalloc(reinterpret_cast<void **>(&buf), kSplitScratchFloats * sizeof(float)) != hipSuccess) {
        (void)hipGetLastError();
        return nullptr;
    }
    g_split_scratch.push_back({dev, stream, buf});
    return buf;
}

// ----- scratch that is part of the loaded code object, for callers that must not allocate ---------------------
// Every device the library runs on holds its own copy of this array at its own address until the process ends.
// In host code the array's name is only a handle for hipGetSymbolAddress: the address a kernel may use is looked
// up once per device and kept in g_static_ptr.
constexpr size_t kStaticScratchFloats = (size_t)2 << 20;  // 8 MB
constexpr int kMaxDevices = 64;
static __device__ __align__(256) float scratch[kStaticScratchFloats];
float *g_static_ptr[kMaxDevices];

// device address of the current device's copy of `scratch` (NULL with the error text set on failure)
float *static_scratch() {
    int dev = 0;
    if (hipGetDevice(&dev) != hipSuccess || dev < 0 || dev >= kMaxDevices) {
        set_error("static scratch: no current device");
        return nullptr;
    }
    std::lock_guard<std::mutex> lock(g_split_mu);
    if (!g_static_ptr[dev]) {
        void *ptr = nullptr;
        const hipError_t err = hipGetSymbolAddress(&ptr, HIP_SYMBOL(scratch));
        if (err != hipSuccess || !ptr) {
            set_error("static scratch: hipGetSymbolAddress: %s", hipGetErrorString(err));
            return nullptr;
        }
        g_static_ptr[dev] = static_cast<float *>(ptr);
    }
    return g_static_ptr[dev];
}

__global__ __launch_bounds__(256) void splitk_reduce_kernel(const GemmArgs args) {
    const size_t mn = (size_t)args.m * args.n;
    const size_t products = mn * args.nprob;
    const size_t total = products + (args.rowsum ? (size_t)args.n * args.nprob : 0);
    const size_t e = (size_t)blockIdx.x * kPartOutputs + threadIdx.x % kPartOutputs;
    const float v = sum_of_parts(args.partial, e, total, args.splitk, args.partial_stride);
    if (threadIdx.x < kPartOutputs && e < total) {
        if (e < products) {
            const size_t z = e / mn, r = e % mn;
            args.prob[z].C[(r / args.m) * args.ldc + r % args.m] = v;
        } else {
            const size_t z = (e - products) / args.n, j = (e - products) % args.n;
            args.prob[z].rowsum_out[j] = args.prob[z].rowsum_scale * v;
        }
    }
}

// Outputs large enough to fill the chip with a thread per four neighbouring sums, or with few splits: a thread adds up all splits of
// its sums, eight loads in flight.
constexpr int kReduceThreads = 256;
__global__ __launch_bounds__(kReduceThreads) void splitk_reduce_quads_kernel(const GemmArgs args) {
    const size_t mn = (size_t)args.m * args.n;
    const size_t products = mn * args.nprob;
    const size_t total = products + (args.rowsum ? (size_t)args.n * args.nprob : 0);
    const size_t e = 4 * ((size_t)blockIdx.x * kReduceThreads + threadIdx.x);
    if (e >= total) return;
    const float4 *__restrict__ p = reinterpret_cast<const float4 *>(args.partial + e);
    const size_t st = args.partial_stride / 4;  // (a multiple of four floats, so that every split's quads are aligned)
    const auto add = [](const float4 &x, const float4 &y) { return float4{x.x + y.x, x.y + y.y, x.z + y.z, x.w + y.w}; };
    float4 v = {0.0f, 0.0f, 0.0f, 0.0f};
    int s = 0;
    for (; s + 8 <= args.splitk; s += 8) {
        float4 x[8];
#pragma unroll
        for (int q = 0; q < 8; ++q) x[q] = p[(size_t)(s + q) * st];
        v = add(v, add(add(add(x[0], x[1]), add(x[2], x[3])), add(add(x[4], x[5]), add(x[6], x[7]))));
    }
    for (; s + 2 <= args.splitk; s += 2) {
        const float4 x = p[(size_t)s * st], y = p[(size_t)(s + 1) * st];
        v = add(v, add(x, y));
    }
    if (s < args.splitk) v = add(v, p[(size_t)s * st]);
    const size_t z = e / mn, r = e - z * mn;
    if (e + 4 <= products && r + 4 <= mn && args.ldc == args.m) {
        float *const to = args.prob[z].C + r;
        if ((reinterpret_cast<uintptr_t>(to) & 15) == 0) {
            *reinterpret_cast<float4 *>(to) = v;
            return;
        }
    }
    const float x[4] = {v.x, v.y, v.z, v.w};
#pragma unroll
    for (int i = 0; i < 4; ++i) {
        const size_t at = e + i;
        if (at < products) {
            const size_t zi = at / mn, ri = at % mn;
            args.prob[zi].C[(ri / args.m) * args.ldc + ri % args.m] = x[i];
        } else if (at < total) {
            const size_t zi = (at - products) / args.n, j = (at - products) % args.n;
            args.prob[zi].rowsum_out[j] = args.prob[zi].rowsum_scale * x[i];
        }
    }
}

}  // namespace

bool gemm_fan_supported(const GemmArgs &a) {
    return !a.a_kcontig && a.b_kcontig && a.nprob == 1 && pick_vec(a, true) == 4 && pick_vec(a, false) == 4;
}

void gemm_release_stream(hipStream_t stream) {
    int dev = 0;
    if (hipGetDevice(&dev) != hipSuccess) return;
    std::lock_guard<std::mutex> lock(g_split_mu);
    for (size_t i = 0; i < g_split_scratch.size(); ++i)
        if (g_split_scratch[i].device == dev && g_split_scratch[i].stream == stream) {
            (void)hipFree(g_split_scratch[i].buf);
            g_split_scratch.erase(g_split_scratch.begin() + (long)i);
            return;
        }
}

int gemm_reserve_stream(hipStream_t stream) {
    std::lock_guard<std::mutex> lock(g_split_mu);
    CNT_REQUIRE(split_scratch(stream) != nullptr, "gemm: no memory for the split-K scratch buffer");
    return CNT_OK;
}

bool with_split_scratch(hipStream_t stream, size_t floats, const std::function<void(float *)> &enqueue) {
    if (!partial_on() || floats > kSplitScratchFloats) return false;
    std::lock_guard<std::mutex> lock(g_split_mu);
    float *buf = split_scratch_find(stream);
    if (!buf && !capturing(stream)) buf = split_scratch(stream);
    if (buf) enqueue(buf);
    return buf != nullptr;
}

ScratchLoan::ScratchLoan(hipStream_t stream, float *buffer) : outer_stream_(t_loan_stream), outer_buffer_(t_loan_buffer) {
    t_loan_stream = stream;
    t_loan_buffer = buffer;
}

ScratchLoan::~ScratchLoan() {
    t_loan_stream = outer_stream_;
    t_loan_buffer = outer_buffer_;
}

int gemm_scratch_buffers() {
    std::lock_guard<std::mutex> lock(g_split_mu);
    return (int)g_split_scratch.size();
}

namespace {
// floats of a split's partial products and row sums, a multiple of four
size_t partial_stride(const GemmArgs &a) {
    return ((size_t)a.m * a.n * a.nprob + (a.rowsum ? (size_t)a.n * a.nprob : 0) + 3) / 4 * 4;
}
}  // namespace

void gemm_plan(GemmArgs &args, hipStream_t stream) {
    if (args.splitk != 0) return;
    if (direct_product(args)) {
        // one workgroup sums over all of k: nothing to add to, and the row sums come along
        args.splitk = 1;
        if (args.epilogue == EPI_ATOMIC && args.overwrite_ok) args.epilogue = EPI_STORE;
        else args.rowsum = 0;
        return;
    }
    // Long-K products with a small output (weight gradients): cut K so that the launch has about
    // `target` workgroups of 64 x 64 tiles, but leave every workgroup at least eight k-iterations -- each
    // one ends with an atomic add (or a store) of its whole tile, and those, not the products, dominate short
    // ranges.
    // Outputs of one or two tiles per problem (the WaveNet layers' 64 x 64 ... 80 x 128 weights) take twice the
    // workgroups: measured on MI355X next to the error chain of the same pass, 1024 workgroups end the stack's backward
    // pass 4% sooner than 512, and 1536 or more (whose partial products did not fit the scratch buffer of then, so that the
    // launch added atomically) 4-8% later; the acoustic model's wide outputs are best at 768 (2.249 / 2.232 / 2.219 / 2.246 /
    // 2.243 ms at 512 / 640 / 768 / 896 / 1024 with the loader of constant offsets; they were best at 512 before it).
    static const int forced_target = [] { const char *e = std::getenv("CNT_GEMM_SPLIT_TARGET"); return e ? std::atoi(e) : 0; }();
    const long tiles = (long)((args.m + 63) / 64) * ((args.n + 63) / 64) * args.nprob;
    // (768 only where a launch has at least 64 tiles to begin with: the WaveNet stack's 256 x 256 output layers over
    // 32 000 samples, 16 tiles, are better off with 512: 2.724 against 2.736 ms)
    const int target = forced_target > 0 ? forced_target : ((long)args.m * args.n <= 16384 ? 1024 : tiles >= 64 ? 768 : 512);
    const long kt = ((long)args.k + BK - 1) / BK * args.nseg;
    long s = (target + tiles - 1) / tiles;
    if (forced_target == 0 && wide_gradient(args))
        s = kWideGradientGroups / large_tiles(args);
    else if (forced_target == 0 && level_gradient(args))
        s = kLevelGradientGroups / large_tiles(args);
    s = std::min(s, std::max(1L, kt / 8));
    s = std::max(1L, s);
    const size_t stride = partial_stride(args);
    const bool rowsum_ok = !args.rowsum || (args.nseg == 1 && !args.masked);
    bool partial = partial_on() && args.epilogue == EPI_ATOMIC && args.overwrite_ok && rowsum_ok;
    if (partial) s = std::max(1L, std::min(s, (long)(kSplitScratchFloats / stride)));
    // no empty split: every split of the partial-product path has to write its share
    while (s > 1 && (s - 1) * ((kt + s - 1) / s) >= kt) --s;
    args.splitk = (int)s;
    const bool sums_with_store = !args.rowsum || (!args.a_kcontig && !args.b_kcontig);
    if (partial && s == 1 && sums_with_store) {
        args.epilogue = EPI_STORE;
        return;
    }
    if (partial && !args.partial) {
        // the stream's scratch buffer: reserved by its owner, else allocated on first use; without one (allocation refused, a
        // stream under capture, whose graph may outlive a buffer that nobody has reserved) the product adds atomically
        std::lock_guard<std::mutex> lock(g_split_mu);
        args.partial = split_scratch_find(stream);
        if (!args.partial && !capturing(stream)) args.partial = split_scratch(stream);
        partial = args.partial != nullptr;
    }
    if (partial) {
        args.epilogue = EPI_PARTIAL;
        args.partial_stride = stride;
    } else if (!rowsum_ok || args.epilogue != EPI_ATOMIC || args.a_kcontig || args.b_kcontig) {
        args.rowsum = 0;  // the caller sums the rows itself
    }
}

int gemm_launch(hipStream_t stream, const GemmArgs &args_in, DirectGroup *group) {
    GemmArgs args = args_in;
    CNT_REQUIRE(args.m > 0 && args.n > 0 && args.k > 0, "gemm: empty problem %d x %d x %d", args.m, args.n,
                args.k);
    CNT_REQUIRE(args.nseg >= 1 && args.nseg <= kGemmMaxSeg, "gemm: %d operand pairs, supported 1..%d",
                args.nseg, kGemmMaxSeg);
    CNT_REQUIRE(args.nprob >= 1 && args.nprob <= kGemmMaxProb, "gemm: %d problems, supported 1..%d",
                args.nprob, kGemmMaxProb);
    CNT_REQUIRE(!args.a_kcontig || args.b_kcontig, "gemm: a k-contiguous A with a row-contiguous B is not supported");
    CNT_REQUIRE(args.splitk >= 0 && (args.splitk == 1 || args.epilogue == EPI_ATOMIC || args.epilogue == EPI_PARTIAL),
                "gemm: split-K needs the atomic epilogue");
    CNT_REQUIRE(args.epilogue != EPI_STORE_DELTA || (args.splitk == 1 && args.prob[0].aux_in != nullptr),
                "gemm: the delta epilogue needs the preceding layer's outputs and no split");
    CNT_REQUIRE((args.epilogue != EPI_BIAS_ACT && args.epilogue != EPI_BIAS_ACT_SKIP && args.epilogue != EPI_CONTEXT) || args.a_kcontig,
                "gemm: the forward epilogues are for two k-contiguous operands");
    CNT_REQUIRE((args.epilogue != EPI_BIAS_ACT_SKIP || args.masked) && (args.epilogue != EPI_CONTEXT || !args.masked),
                "gemm: an epilogue that goes by the pattern types has one loader");
    CNT_REQUIRE(args.epilogue != EPI_STORE_DELTA || (!args.a_kcontig && args.b_kcontig),
                "gemm: the delta epilogue is for a row-contiguous A and a k-contiguous B");
    CNT_REQUIRE(args.epilogue != EPI_FAN || (gemm_fan_supported(args) && args.splitk == 1),
                "gemm: the fan epilogue exists for one unsplit problem with 16-byte row-contiguous A and k-contiguous B");
    CNT_REQUIRE(args.epilogue != EPI_PARTIAL || (args.splitk >= 1 && args.partial_stride > 0 && args.partial),
                "gemm: the partial-product epilogue is chosen by gemm_plan only");
    for (int p = 0; p < args.nprob; ++p) {
        CNT_REQUIRE(args.prob[p].C != nullptr, "gemm: null output");
        for (int s = 0; s < args.nseg; ++s)
            CNT_REQUIRE(args.prob[p].A[s] && args.prob[p].B[s], "gemm: null operand");
    }
    // the unmasked loaders address an operand through 32-bit byte offsets beside a base that moves along k
    const auto reachable = [](long rows, long ld, int kcontig) {
        return (kcontig ? rows * ld : BK * ld + rows) * (long)sizeof(float) < (1L << 32);
    };
    CNT_REQUIRE(args.masked || (reachable(args.m, args.lda, args.a_kcontig) && reachable(args.n, args.ldb, args.b_kcontig)),
                "gemm: operands of 4 GiB and more are not supported (%d x %d x %d, lda %d, ldb %d)", args.m, args.n, args.k,
                args.lda, args.ldb);
    int va = pick_vec(args, true), vb = pick_vec(args, false);
    const bool aligned = va == 4 && vb == 4;
    if (!args.masked && args.epilogue != EPI_FAN) {  // the unmasked loader goes by the length of the lines alone
        va = (args.a_kcontig ? args.k : args.m) % 4 == 0 ? 4 : 1;
        vb = (args.b_kcontig ? args.k : args.n) % 4 == 0 ? 4 : 1;
    }
    gemm_plan(args, stream);
    static const bool use_lines = [] { const char *e = std::getenv("CNT_GEMM_K_ORDER"); return !e || std::atoi(e) != 0; }();
    if (!use_lines) args.k_order = nullptr;
    if (args.splitk == 1 && args.epilogue != EPI_PARTIAL && direct_product(args)) {
        if (group && !args.a_kcontig && !args.b_kcontig && args.nseg == 1 && args.epilogue == EPI_STORE)
            return gemm_group_add(stream, *group, args);
        // It multiplies all columns, each in its place, and so do the sums it forms again in fp32, which go by the list where there is one.
        args.cols = args.cols_count = nullptr;
        ProfileScope prof(stream, args.label ? args.label : "gemm");
        gemm_direct_launch(args, stream);
        CNT_HIP(hipGetLastError());
        return CNT_OK;
    }
    if (args.epilogue != EPI_PARTIAL && args.epilogue != EPI_ATOMIC && args.epilogue != EPI_STORE) args.rowsum = 0;
    if (args.masked || !args.b_kcontig || args.splitk != 1 || (args.epilogue != EPI_STORE && args.epilogue != EPI_STORE_DELTA)) args.cols = nullptr;
    const int tile = pick_tile(args);
    const int edge = tile == kEightWaves ? 128 : tile;
    // a list of k lines is used where the kernel that reads through it exists, and ignored otherwise (the lines it leaves
    // out are zero)
    if (args.k_order && !(args.k_count && !args.masked && !args.a_kcontig && !args.b_kcontig && aligned &&
                          args.epilogue != EPI_FAN && args.k < (1 << 24) && args.lda < (1 << 22) && args.ldb < (1 << 22)))
        args.k_order = nullptr;
    const int tiles = ((args.m + edge - 1) / edge) * ((args.n + edge - 1) / edge);
    dim3 grid(tiles, args.splitk, args.nprob);
    // XCD-aware placement (gemm_kernel.hpp): measured with FETCH_SIZE on MI355X it cuts what the L2s fetch 2.2-2.6x for the
    // WaveNet stack's batched weight gradients (a convolution's two taps and a stack's conditioning projections share an
    // operand) and 2-4x for single problems (the acoustic model's weight gradients: 270 -> 68 MB).  Since the products run on the
    // bf16 instructions they feel it: the feed-forward model's pass takes 2283 us with single problems mapped, 2363 without, the
    // models with recurrent layers 0.1-0.5% less.
    static const bool xcd_map = [] { const char *e = std::getenv("CNT_GEMM_XCD_MAP"); return !e || std::atoi(e) != 0; }();
    args.xcd_map = xcd_map && (long)tiles * args.splitk * args.nprob >= 16 ? 1 : 0;
    ProfileScope prof(stream, args.label ? args.label : "gemm");
    std::unique_lock<std::mutex> split_lock(g_split_mu, std::defer_lock);
    // a product and its reduction stay adjacent on the stream
    if (args.epilogue == EPI_PARTIAL) split_lock.lock();
    if (va == 4) gemm_dispatch_va4(args, grid, stream, args.a_kcontig, vb, args.b_kcontig, tile);
    else if (va == 2) gemm_dispatch_va2(args, grid, stream, args.a_kcontig, vb, args.b_kcontig, tile);
    else if (args.a_kcontig) gemm_dispatch_va1k(args, grid, stream, vb, args.b_kcontig, tile);
    else gemm_dispatch_va1r(args, grid, stream, vb, args.b_kcontig, tile);
    CNT_HIP(hipGetLastError());
    if (args.epilogue == EPI_PARTIAL) {
        const size_t total = args.partial_stride;
        if (args.splitk >= kManySplits && total <= (size_t)kFewOutputs)
            hipLaunchKernelGGL(splitk_reduce_kernel, dim3((unsigned)((total + kPartOutputs - 1) / kPartOutputs)), dim3(256), 0,
                               stream, args);
        else
            hipLaunchKernelGGL(splitk_reduce_quads_kernel, dim3((unsigned)((total / 4 + kReduceThreads - 1) / kReduceThreads)),
                               dim3(kReduceThreads), 0, stream, args);
        CNT_HIP(hipGetLastError());
    }
    return CNT_OK;
}

// A dense layer's weight gradient (dW = x * delta^T, P x D, plus the bias part: bias * row sums of delta) as a
// split-K product whose partial products go through the code object's own scratch array: no allocation at all.
int gemm_dense_weights_static(hipStream_t stream, int P, int D, int N, float bias, const float *x, const float *err,
                              float *weight_updates) {
    const size_t sums = (size_t)P * D + D, stride = (sums + 3) / 4 * 4;
    CNT_REQUIRE(stride <= kStaticScratchFloats,
                "dense_backward_weights_static: %d x %d weights + %d biases = %zu floats exceed the static scratch of %zu "
                "floats; use cnt_dense_backward_weights", P, D, D, sums, kStaticScratchFloats);
    float *buf = static_scratch();
    if (!buf) return CNT_ERR_HIP;
    GemmArgs ga = {};
    ga.m = P; ga.n = D; ga.k = N;
    ga.a_kcontig = 0; ga.lda = P;
    ga.b_kcontig = 0; ga.ldb = D;
    ga.ldc = P;
    ga.nseg = 1; ga.nprob = 1;
    ga.prob[0].A[0] = x; ga.prob[0].B[0] = err; ga.prob[0].C = weight_updates;
    ga.prob[0].rowsum_out = weight_updates + (size_t)P * D;
    ga.prob[0].rowsum_scale = bias;
    ga.label = "gemm:dense_dW_static";
    ga.rowsum = 1;
    if (direct_product(ga)) {
        ga.splitk = 1;
        ga.epilogue = EPI_STORE;
        return gemm_launch(stream, ga);
    }
    // as many splits as the usual plan takes, as far as their partial products fit into the array
    GemmArgs probe = ga;
    probe.epilogue = EPI_ATOMIC; probe.splitk = 0; probe.overwrite_ok = 0;
    gemm_plan(probe, stream);
    size_t splits = (size_t)probe.splitk;
    if (splits * stride > kStaticScratchFloats) splits = kStaticScratchFloats / stride;
    const long kt = ((long)N + BK - 1) / BK;
    while (splits > 1 && ((long)splits - 1) * ((kt + (long)splits - 1) / (long)splits) >= kt) --splits;  // no empty split
    ga.splitk = (int)splits;
    ga.epilogue = EPI_PARTIAL;
    ga.partial = buf;
    ga.partial_stride = stride;
    return gemm_launch(stream, ga);
}

int gemm_simple(hipStream_t stream, float *C, int m, int n, int k, const float *A, bool transA,
                const float *B, bool transB, bool accumulate) {
    GemmArgs a = {};
    a.m = m; a.n = n; a.k = k;
    // column-major A (m x k, lda=m) is row-contiguous; transposed storage (k x m, lda=k) is k-contiguous
    a.a_kcontig = transA ? 1 : 0;
    a.lda = transA ? k : m;
    // column-major B (k x n, ldb=k) is k-contiguous; transposed storage (n x k, ldb=n) is row-contiguous
    a.b_kcontig = transB ? 0 : 1;
    a.ldb = transB ? n : k;
    a.ldc = m;
    a.nseg = 1; a.nprob = 1; a.splitk = 1;
    a.epilogue = accumulate ? EPI_ADD : EPI_STORE;
    a.prob[0].A[0] = A;
    a.prob[0].B[0] = B;
    a.prob[0].C = C;
    return gemm_launch(stream, a);
}

}  // namespace cnt

extern "C" int cnt_probe_product_of_halves(void *stream, float *C, int m, int n, int k, const float *A, int transA, const float *B, int transB) {
    return cnt_matrix_product(stream, C, m, n, k, A, transA, B, transB, 0);
}

extern "C" int cnt_probe_gemm_plan(int m, int n, int k, int problems, int a_kcontig, int b_kcontig, int weight_gradient, int *plan) {
    using namespace cnt;
    CNT_REQUIRE(plan && m > 0 && n > 0 && k > 0 && problems >= 1 && problems <= kGemmMaxProb && (!a_kcontig || b_kcontig),
                "probe_gemm_plan: bad argument");
    GemmArgs a = {};
    a.m = m; a.n = n; a.k = k;
    a.a_kcontig = a_kcontig != 0; a.lda = a_kcontig ? k : m;
    a.b_kcontig = b_kcontig != 0; a.ldb = b_kcontig ? k : n;
    a.ldc = m;
    a.nseg = 1; a.nprob = problems;
    a.epilogue = weight_gradient ? EPI_ATOMIC : EPI_STORE;
    a.splitk = weight_gradient ? 0 : 1;
    a.overwrite_ok = 1;
    float nothing = 0.0f;
    a.partial = &nothing;  // (a plan is made for the stream's scratch; none is asked for here)
    gemm_plan(a, nullptr);
    const bool direct = a.splitk == 1 && a.epilogue != EPI_PARTIAL && direct_product(a);
    const int tile = direct ? 32 : pick_tile(a);
    plan[0] = tile == kEightWaves ? 128 : tile;
    plan[1] = direct || tile == kEightWaves ? 8 : 4;
    plan[2] = a.splitk;
    return CNT_OK;
}
