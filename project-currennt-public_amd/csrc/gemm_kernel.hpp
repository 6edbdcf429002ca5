// Kernel template and launch ladder of the fp32 matrix product (design notes: gemm.hip).
#pragma once

#include "common.hpp"

#include <type_traits>

namespace cnt {

namespace {

constexpr int BK = 32;  // k depth of a staged tile: two matrix instructions deep
constexpr int NTHREADS = 256;
constexpr int kEightWaves = 129;  // "tile" of a launch: 128 x 128, on eight waves

typedef float f32x16 __attribute__((ext_vector_type(16)));
typedef float f32x2 __attribute__((ext_vector_type(2)));
typedef __bf16 bf16x2 __attribute__((ext_vector_type(2)));
typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));

// workgroup barrier that orders LDS traffic only; global loads issued before it stay in flight
__device__ __forceinline__ void lds_only_barrier() {
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "workgroup", "local");
    __builtin_amdgcn_s_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "workgroup", "local");
}

template <int V>
struct VecT;
template <>
struct VecT<1> { typedef float type; };
template <>
struct VecT<2> { typedef float2 type; };
template <>
struct VecT<4> { typedef float4 type; };

// Two fp32 values as three bf16 pairs (the lower half of a word belongs to x0): kSplitScale * x = h + m + l exactly, each part
// the nearest bf16 value to what the parts before it leave (8 + 8 + 8 bits of significand hold the 24 of x).  bf16 ends at
// 2^-133, fp32 at 2^-149: without the factor the low parts of values below 2^-110 are cut off, and one near 2^-126 keeps eight
// bits.  With it the parts of every fp32 value below 2^112 are exact, and sums up to 2^96 come out finite; those above are
// formed again (plain_sums).
constexpr float kSplitScale = 65536.0f;
__device__ __forceinline__ unsigned nearest_bf16(float x0, float x1) {
    return __builtin_bit_cast(unsigned, __builtin_convertvector((f32x2{x0, x1}), bf16x2));
}
__device__ __forceinline__ void split_pair(float x0, float x1, unsigned (&part)[3]) {
    x0 *= kSplitScale; x1 *= kSplitScale;
#pragma unroll
    for (int q = 0; q < 3; ++q) {
        part[q] = nearest_bf16(x0, x1);
        if (q == 2) break;
        x0 -= __uint_as_float(part[q] << 16);
        x1 -= __uint_as_float(part[q] & 0xffff0000u);
    }
}

// Where the parts of a ROWS-row x BK-k operand tile lie in LDS.  The 16-byte unit is what one lane of a matrix instruction
// takes: eight consecutive k of one row.  Units are ordered [part][k / 8][position of the row]; the position of a row is the
// row itself where a thread loads along k, and r * GROUP + t for row VEC * t + r where it loads VEC rows at once, so that in
// both cases the lanes of one store, and those of one read, fall on distinct banks (the pads of GROUP and LINE see to it).
template <int VEC, bool KCONTIG, int ROWS, int NT = NTHREADS>
struct TileLayout {
    static constexpr int NLOAD = (ROWS * BK) / (NT * VEC);  // vectors per thread
    static_assert(NLOAD >= 1, "tile too small for this vector width");
    static constexpr int GROUP = ROWS / VEC + (VEC == 4 ? 4 : VEC == 2 ? 8 : 0);
    static constexpr int LINE = KCONTIG ? ROWS + 4 : VEC * GROUP;  // units per k / 8
    static constexpr int PART = (BK / 8) * LINE;                   // units per part
    static constexpr int UNITS = 3 * PART;
    typedef typename VecT<VEC>::type vec_t;

    // k-contiguous: the thread's vectors start at k position first_k of the rows row(p); row-contiguous: they hold the VEC
    // rows from first_row on, of the NLOAD consecutive k positions from first_k on
    static constexpr int TPR = BK / VEC, RPP = NT / TPR;
    static constexpr int TPK = ROWS / VEC;
    static __device__ __forceinline__ int column(int tid) {  // t above
        if (TPK == 32) return (tid & 15) | ((tid & 32) >> 1);  // sixteen lanes along the rows, two halves of a unit
        return tid % TPK;
    }
    static __device__ __forceinline__ int first_k(int tid) {
        if (KCONTIG) return (tid % TPR) * VEC;
        if (TPK == 32) return (2 * (tid >> 6) + ((tid >> 4) & 1)) * NLOAD;
        return (tid / TPK) * NLOAD;
    }
    static __device__ __forceinline__ int first_row(int tid) { return KCONTIG ? tid / TPR : column(tid) * VEC; }
    static __device__ __forceinline__ int row(int tid, int p) { return KCONTIG ? tid / TPR + p * RPP : column(tid) * VEC; }

    static __device__ __forceinline__ void put(uint4 *__restrict__ lds, int tid, const vec_t (&v)[NLOAD]) {
        const int k = first_k(tid);
        if (KCONTIG) {
            char *at = reinterpret_cast<char *>(lds + (k / 8) * LINE + tid / TPR) + 2 * (k % 8);
            if constexpr (VEC == 1) {
#pragma unroll
                for (int p = 0; p < NLOAD; p += 2) {
                    unsigned x[3];
                    split_pair(v[p], v[p + 1], x);
#pragma unroll
                    for (int q = 0; q < 3; ++q) {
                        *reinterpret_cast<unsigned short *>(at + 16 * (q * PART + p * RPP)) = (unsigned short)x[q];
                        *reinterpret_cast<unsigned short *>(at + 16 * (q * PART + (p + 1) * RPP)) = (unsigned short)(x[q] >> 16);
                    }
                }
            } else {
#pragma unroll
                for (int p = 0; p < NLOAD; ++p) {
                    const float *e = reinterpret_cast<const float *>(&v[p]);
                    unsigned x[VEC / 2][3];
#pragma unroll
                    for (int j = 0; j < VEC / 2; ++j) split_pair(e[2 * j], e[2 * j + 1], x[j]);
#pragma unroll
                    for (int q = 0; q < 3; ++q) {
                        char *to = at + 16 * (q * PART + p * RPP);
                        if constexpr (VEC == 4) *reinterpret_cast<uint2 *>(to) = uint2{x[0][q], x[1][q]};
                        else *reinterpret_cast<unsigned *>(to) = x[0][q];
                    }
                }
            }
        } else {
            char *at = reinterpret_cast<char *>(lds + (k / 8) * LINE + column(tid)) + 2 * (k % 8);
#pragma unroll
            for (int r = 0; r < VEC; ++r) {
                unsigned x[NLOAD / 2][3];
#pragma unroll
                for (int p = 0; p < NLOAD; p += 2)
                    split_pair(reinterpret_cast<const float *>(&v[p])[r], reinterpret_cast<const float *>(&v[p + 1])[r], x[p / 2]);
#pragma unroll
                for (int q = 0; q < 3; ++q) {
                    char *to = at + 16 * (q * PART + r * GROUP);
                    if constexpr (NLOAD == 2) *reinterpret_cast<unsigned *>(to) = x[0][q];
                    else if constexpr (NLOAD == 4) *reinterpret_cast<uint2 *>(to) = uint2{x[0][q], x[1][q]};
                    else {
#pragma unroll
                        for (int u = 0; u < NLOAD / 8; ++u)
                            *reinterpret_cast<uint4 *>(to + 16 * u * LINE) =
                                uint4{x[4 * u][q], x[4 * u + 1][q], x[4 * u + 2][q], x[4 * u + 3][q]};
                    }
                }
            }
        }
    }

    // the three parts of k positions [8 * k8, 8 * k8 + 8) of tile row `row`
    static __device__ __forceinline__ void fragment(const uint4 *__restrict__ lds, int row, int k8, bf16x8 (&f)[3]) {
        const uint4 *at = lds + k8 * LINE + (KCONTIG ? row : (row % VEC) * GROUP + row / VEC);
#pragma unroll
        for (int q = 0; q < 3; ++q) f[q] = __builtin_bit_cast(bf16x8, at[q * PART]);
    }
};

// Stages one ROWS-row x BK-k operand tile: global -> registers -> LDS.
//
// A load always executes, on a clamped address, and what decides whether its vector counts (inside the matrix; in
// masked mode: both pattern bytes non-zero and the shifted slot inside the fraction) is only LOOKED AT in store(),
// one k-iteration later.  Nothing between a load and the LDS store a whole iteration later touches the loaded
// registers -- neither the data nor the two pattern bytes -- so the only wait the loop needs is "all but the newest
// tile have arrived"; zeroing the vector right after the load would make every iteration wait for its own loads.
template <int VEC, bool KCONTIG, int ROWS>
struct TileStage {
    typedef TileLayout<VEC, KCONTIG, ROWS> L;
    static constexpr int NLOAD = L::NLOAD;
    typename VecT<VEC>::type r[NLOAD];
    bool inside_[NLOAD];      // known at load time (indices only)
    char pat_own_[NLOAD], pat_src_[NLOAD];  // masked mode: loaded next to the data, looked at in store()

    // shift / pat / n_slots: masked mode (pat == nullptr switches it off); time_on_k selects which index is
    // the time slot
    __device__ __forceinline__ void load(const float *__restrict__ base, int ld, int row0, int k0,
                                         int rows_total, int k_total, int tid, const char *__restrict__ pat = nullptr,
                                         int shift = 0, int n_slots = 0, bool time_on_k = false) {
        // Addresses are formed here, tile by tile, where keeping them through the loop would push the data or the pattern bytes out
        // of the registers (the kernels for sizes that are no multiple of four spilled 2 to 27 of them): 63 -> 126 channels over 2 x 8000
        // slots 22.1 -> 19.4 us forward, 31 -> 62 over 16 000 14.3 -> 12.5, 63 -> 128 over 2 x 16 000 30.4 -> 26.0.  A bound of three
        // workgroups per compute unit instead of four gave the first two and took 28.0 instead of 22.1 for 62 -> 124 over 2 x 16 000.
        if (KCONTIG && VEC < 4 && pat) asm volatile("" : "+s"(ld));
        if (!KCONTIG && pat) asm volatile("" : "+s"(row0));
        if (KCONTIG) {
            const int kq = L::first_k(tid);
#pragma unroll
            for (int p = 0; p < NLOAD; ++p) {
                const int row = row0 + L::row(tid, p);
                typename VecT<VEC>::type v = {};
                pat_own_[p] = 1; pat_src_[p] = 1;
                if (!pat) {
                    inside_[p] = row < rows_total && (k0 + kq) < k_total;
                    const int rc = min(row, rows_total - 1), kc = (k0 + kq) < k_total ? k0 + kq : 0;
                    v = *reinterpret_cast<const typename VecT<VEC>::type *>(base + (size_t)rc * ld + kc);
                } else if (!time_on_k) {
                    // the row is the time slot, so the whole vector is kept or dropped
                    const int rc = min(row, rows_total - 1), kc = (k0 + kq) < k_total ? k0 + kq : 0;
                    const int src = rc + shift;
                    const int sc = min(max(src, 0), n_slots - 1);
                    inside_[p] = row < rows_total && (k0 + kq) < k_total && src == sc;
                    v = *reinterpret_cast<const typename VecT<VEC>::type *>(base + (size_t)sc * ld + kc);
                    pat_own_[p] = pat[rc]; pat_src_[p] = pat[sc];
                } else {
                    inside_[p] = true;
                    if (row < rows_total && (k0 + kq) < k_total) {
                        // vector along k = consecutive time slots: element-wise masking
                        float *e = reinterpret_cast<float *>(&v);
#pragma unroll
                        for (int j = 0; j < VEC; ++j) {
                            const int u = k0 + kq + j, src = u + shift;
                            if (pat[u] != 0 && src >= 0 && src < n_slots && pat[src] != 0)
                                e[j] = base[(size_t)row * ld + src];
                        }
                    }
                }
                r[p] = v;
            }
        } else {
            const int rq = L::first_row(tid);
            const int kk = L::first_k(tid);
#pragma unroll
            for (int p = 0; p < NLOAD; ++p) {
                const int k = k0 + kk + p;
                typename VecT<VEC>::type v = {};
                pat_own_[p] = 1; pat_src_[p] = 1;
                if (!pat) {
                    inside_[p] = k < k_total && (row0 + rq) < rows_total;
                    const int kc = min(k, k_total - 1), rc = (row0 + rq) < rows_total ? row0 + rq : 0;
                    v = *reinterpret_cast<const typename VecT<VEC>::type *>(base + (size_t)kc * ld + rc);
                } else if (time_on_k) {
                    // the k line is the time slot
                    const int kc = min(k, k_total - 1), rc = (row0 + rq) < rows_total ? row0 + rq : 0;
                    const int src = kc + shift;
                    const int sc = min(max(src, 0), n_slots - 1);
                    inside_[p] = k < k_total && (row0 + rq) < rows_total && src == sc;
                    v = *reinterpret_cast<const typename VecT<VEC>::type *>(base + (size_t)sc * ld + rc);
                    pat_own_[p] = pat[kc]; pat_src_[p] = pat[sc];
                } else {
                    inside_[p] = true;
                    if (k < k_total && (row0 + rq) < rows_total) {
                        float *e = reinterpret_cast<float *>(&v);
#pragma unroll
                        for (int j = 0; j < VEC; ++j) {
                            const int u = row0 + rq + j, src = u + shift;
                            if (pat[u] != 0 && src >= 0 && src < n_slots && pat[src] != 0)
                                e[j] = base[(size_t)k * ld + src];
                        }
                    }
                }
                r[p] = v;
            }
        }
    }

    __device__ __forceinline__ typename VecT<VEC>::type kept(int p) const {
        const bool keep = inside_[p] && pat_own_[p] != 0 && pat_src_[p] != 0;
        return keep ? r[p] : typename VecT<VEC>::type{};
    }

    __device__ __forceinline__ void store(uint4 *__restrict__ lds, int tid) const {
        typename VecT<VEC>::type v[NLOAD];
#pragma unroll
        for (int p = 0; p < NLOAD; ++p) v[p] = kept(p);
        L::put(lds, tid, v);
    }
};

// The unmasked loader, in vectors of four floats at any float's address (the hardware loads 16 bytes from a multiple of 4; a
// vector that is not aligned costs at most a second cache line, where one float per lane costs four times the instructions).
// What a thread loads differs from tile to tile only by the tile's k offset, so everything per thread is computed once:
// `voff`, the byte offset of its vector inside the operand at k = 0 (row clamped into the matrix), as a 32-bit offset beside
// a 64-bit base that is uniform over the workgroup -- the address form that costs no vector arithmetic per load.  A vector may
// reach beyond its own line only where it still ends inside the operand: rows outside the matrix reach only sums that are not
// stored, and the tiles where a vector could leave the operand or hold k values beyond its end take a path of their own
// (uniform over the workgroup), one float at a time unless the lines are a multiple of four long.
typedef float f32x4u __attribute__((ext_vector_type(4), aligned(4)));
// adds a thread's share of a tile, NLOAD k positions of four rows, to its sums of those rows: the positions among themselves
// first, so that a sum's chain of additions has one link per tile
template <int NLOAD>
__device__ __forceinline__ void add_tile_rows(float (&sum)[4], const float4 (&r)[NLOAD]) {
    float4 v = r[0];
    if constexpr (NLOAD == 4) {
        v.x = (r[0].x + r[1].x) + (r[2].x + r[3].x); v.y = (r[0].y + r[1].y) + (r[2].y + r[3].y);
        v.z = (r[0].z + r[1].z) + (r[2].z + r[3].z); v.w = (r[0].w + r[1].w) + (r[2].w + r[3].w);
    } else {
#pragma unroll
        for (int p = 1; p < NLOAD; ++p) { v.x += r[p].x; v.y += r[p].y; v.z += r[p].z; v.w += r[p].w; }
    }
    sum[0] += v.x; sum[1] += v.y; sum[2] += v.z; sum[3] += v.w;
}

// WHOLE: the lines are a multiple of four long, so that no vector crosses the end of one.
template <bool WHOLE, bool KCONTIG, int ROWS, int NT>
struct FastStage {
    typedef TileLayout<4, KCONTIG, ROWS, NT> L;
    static constexpr int NLOAD = L::NLOAD;
    float4 r[NLOAD];
    unsigned voff[NLOAD];
    int ld, row0, rows_total;  // uniform

    // rows: where the operand's rows of this tile stand, or null (k-contiguous operands)
    __device__ __forceinline__ void init(int ld_, int row0_, int rows_total_, int tid, const int *rows = nullptr) {
        ld = ld_; row0 = row0_; rows_total = rows_total_;
#pragma unroll
        for (int p = 0; p < NLOAD; ++p) {
            const int row = row0 + L::row(tid, p), k = kpos(tid, p);
            int rc = KCONTIG ? min(row, rows_total - 1) : row < rows_total ? row : 0;
            if (KCONTIG && rows) rc = rows[L::row(tid, p)];
            voff[p] = (unsigned)((KCONTIG ? (size_t)rc * ld + k : (size_t)k * ld + rc) * sizeof(float));
        }
    }
    static __device__ __forceinline__ int kpos(int tid, int p) { return L::first_k(tid) + (KCONTIG ? 0 : p); }
    // base = the operand at the tile's first k, left = k values from there to the operand's end (both uniform)
    __device__ __forceinline__ void load(const float *__restrict__ base, int left, int tid) {
        const char *b = reinterpret_cast<const char *>(base);
        // (row-contiguous: a vector that crosses ends at most three floats behind its line, hence three lines behind at most)
        if (left >= (KCONTIG || WHOLE ? BK : BK + 3)) {
#pragma unroll
            for (int p = 0; p < NLOAD; ++p) {
                const f32x4u v = *reinterpret_cast<const f32x4u *>(b + voff[p]);
                r[p] = float4{v[0], v[1], v[2], v[3]};
            }
        } else if (WHOLE) {
#pragma unroll
            for (int p = 0; p < NLOAD; ++p) {
                const int k = kpos(tid, p);
                const unsigned back = (unsigned)(k * (KCONTIG ? 1 : ld)) * (unsigned)sizeof(float);  // to k position 0
                const f32x4u v = *reinterpret_cast<const f32x4u *>(b + (k < left ? voff[p] : voff[p] - back));
                r[p] = k < left ? float4{v[0], v[1], v[2], v[3]} : float4{0.0f, 0.0f, 0.0f, 0.0f};
            }
        } else {
            int line = ld;
            asm volatile("" : "+s"(line));  // the addresses below are formed here, not kept in registers through the loop
#pragma unroll
            for (int p = 0; p < NLOAD; ++p) {
                float e[4];
                const float *const line_start = reinterpret_cast<const float *>(b + voff[p]) - kpos(tid, p);  // (k-contiguous)
#pragma unroll
                for (int q = 0; q < 4; ++q) {
                    const int k = kpos(tid, p) + (KCONTIG ? q : 0), kc = k < left ? k : 0;
                    const int row = min(row0 + L::row(tid, p) + (KCONTIG ? 0 : q), rows_total - 1);
                    const float v = KCONTIG ? line_start[kc] : base[(size_t)kc * line + row];
                    e[q] = k < left ? v : 0.0f;
                }
                r[p] = float4{e[0], e[1], e[2], e[3]};
            }
        }
    }
    __device__ __forceinline__ void store(uint4 *__restrict__ lds, int tid) const { L::put(lds, tid, r); }
    // adds the tile in registers to the sums of the thread's four rows (row-contiguous operands)
    __device__ __forceinline__ void add_rows(float (&sum)[4]) const { add_tile_rows<NLOAD>(sum, r); }
};

// The unmasked loader for row-contiguous operands whose k lines are picked through a list (16-byte vectors only): tile k
// line j is line idx[j] of the operand.  The indices of a tile are loaded one iteration ahead by the kernel (both operands
// share them) and handed to load(); everything else is FastStage.
template <int ROWS, int NT>
struct GatherStage {
    typedef TileLayout<4, false, ROWS, NT> L;
    static constexpr int NLOAD = L::NLOAD;
    float4 r[NLOAD];
    unsigned roff;   // byte offset of the thread's four rows inside a k line (clamped into the matrix)
    int kk;          // the thread's first k line inside a tile; its others follow
    int k_valid;     // uniform: k lines of the tile in registers that are listed

    __device__ __forceinline__ void init(int row0, int rows_total, int tid) {
        const int rq = L::first_row(tid);
        kk = L::first_k(tid);
        roff = (unsigned)(((row0 + rq) < rows_total ? row0 + rq : 0) * sizeof(float));
    }
    // line_bytes and the indices are below 2^24 and the operand below 4 GiB (checked by the launcher): a 24-bit multiply-add
    // gives the 32-bit offset beside the uniform base
    __device__ __forceinline__ void load(const float *__restrict__ operand, unsigned line_bytes, const int (&idx)[NLOAD], int kv) {
        k_valid = kv;
        const char *b = reinterpret_cast<const char *>(operand);
#pragma unroll
        for (int p = 0; p < NLOAD; ++p)
            r[p] = *reinterpret_cast<const float4 *>(b + (__umul24((unsigned)idx[p], line_bytes) + roff));
    }
    __device__ __forceinline__ void store(uint4 *__restrict__ lds, int tid) const {
        if (k_valid < BK) {
            float4 v[NLOAD];
#pragma unroll
            for (int p = 0; p < NLOAD; ++p) v[p] = kk + p < k_valid ? r[p] : float4{0.0f, 0.0f, 0.0f, 0.0f};
            L::put(lds, tid, v);
        } else {
            L::put(lds, tid, r);
        }
    }
    __device__ __forceinline__ void add_rows(float (&sum)[4]) const {
        float4 v[NLOAD];
#pragma unroll
        for (int p = 0; p < NLOAD; ++p) v[p] = kk + p < k_valid ? r[p] : float4{0.0f, 0.0f, 0.0f, 0.0f};
        add_tile_rows<NLOAD>(sum, v);
    }
};

// where a product's sizes and leading dimensions stand
__device__ __forceinline__ const GemmArgs &sizes_of(const GemmArgs &args, const GemmProblem &) { return args; }
__device__ __forceinline__ const DirectProduct &sizes_of(const DirectGroup &, const DirectProduct &product) { return product; }

// 32 x 32 sums of the product over the k tiles [it_begin, it_end), by one wave on the fp32 matrix instructions and straight
// from memory, where the split product left sums that are not finite: scaled, an operand from 2^112 on is infinite and has
// infinity minus infinity in its parts, and a sum from 2^96 on overflows.  Infinities and NaN come out as fp32 arithmetic has them.
// A pass of a network that has diverged is full of NaN, which stay what they are: the walk along k ends when all sums are.  1024 x 6000 x 1024,
// usually 107 us: 107 us with NaN throughout, 756 with one at the end of every sum; one thread per sum took 11 400.
// ARGS and PROBLEM: GemmArgs and one of its problems, or a group of products and one of those.
template <bool AK, bool BK_, bool MASKED, bool GATHER, typename ARGS, typename PROBLEM>
__device__ __forceinline__ f32x16 plain_sums(const ARGS &args, const PROBLEM &pb, int m0, int n0, int lane, int it_begin,
                                             int it_end, int kt_per_seg, int k_extent, int k_lo) {
    constexpr int AHEAD = 4;  // matrix instructions whose operands are in flight together
    const int half = lane >> 5;
    const auto &size = sizes_of(args, pb);
    const int m = min(m0 + (lane & 31), size.m - 1);  // past an edge: sums that are not stored
    int n = min(n0 + (lane & 31), size.n - 1);
    if constexpr (BK_ && !MASKED && std::is_same<ARGS, GemmArgs>::value)
        if (args.cols) n = args.cols[max(min(n, args.cols_count[0] - 1), 0)];
    f32x16 acc;
#pragma unroll
    for (int r = 0; r < 16; ++r) acc[r] = 0.0f;
#pragma unroll 1
    for (int it = it_begin; it < it_end; ++it) {
        const int seg = it / kt_per_seg, k0 = (it % kt_per_seg) * BK, k1 = min(k0 + BK, k_extent);
#pragma unroll 1
        for (int kk = k0; kk < k1; kk += 2 * AHEAD) {
            float a[AHEAD], b[AHEAD];
#pragma unroll
            for (int u = 0; u < AHEAD; ++u) {
                const int at = kk + 2 * u + half;
                const bool on = at < k1;  // a lane without a k position takes the tile's first one, times zero
                const int k = GATHER ? args.k_order[k_lo + (on ? at : k0)] + pb.k_shift : on ? at : k0;
                int bk = k, bn = n;
                bool keep = on;
                if constexpr (MASKED) if (args.pat) {
                    const int slot = args.b_time_on_k ? k : n, from = slot + pb.b_shift[seg], src = min(max(from, 0), args.n_slots - 1);
                    keep = on && args.pat[slot] != 0 && src == from && args.pat[src] != 0;
                    if (args.b_time_on_k) bk = src; else bn = src;
                }
                const float x = pb.A[seg][AK ? (size_t)m * size.lda + k : (size_t)k * size.lda + m];
                const float y = pb.B[seg][BK_ ? (size_t)bn * size.ldb + bk : (size_t)bk * size.ldb + bn];
                a[u] = on ? x : 0.0f;
                b[u] = keep ? y : 0.0f;
            }
#pragma unroll
            for (int u = 0; u < AHEAD; ++u) acc = __builtin_amdgcn_mfma_f32_32x32x2f32(b[u], a[u], acc, 0, 0, 0);
        }
        bool open = false;
#pragma unroll
        for (int r = 0; r < 16; ++r) open = open || acc[r] == acc[r];
        if (__builtin_amdgcn_ballot_w64(open) == 0) break;
    }
    return acc;
}

// step(the activation function as a constant)
template <typename STEP>
__device__ __forceinline__ void by_activation(int act, STEP &&step) {
    switch (act) {
        case ACT_TANH: step(std::integral_constant<int, ACT_TANH>()); break;
        case ACT_LOGISTIC: step(std::integral_constant<int, ACT_LOGISTIC>()); break;
        case ACT_RELU: step(std::integral_constant<int, ACT_RELU>()); break;
        default: step(std::integral_constant<int, ACT_IDENTITY>()); break;
    }
}

// VA, VB: vector widths of the masked loader, 16-byte alignment included; unmasked: 4 where the operand's lines are a
// multiple of four long, at any alignment, else 1.
// MASKED selects the time-shifted, padding-masked B loader at compile time: its per-element predication is a lot
// of code, which inside the plain kernels would
// push their hot loop out of the instruction cache.
// FAN: the EPI_FAN epilogue, a kernel of its own (instantiated for 16-byte row-contiguous A and k-contiguous B only,
// the shapes of the error products that use it) so that its registers and code stay out of every other product.
// GATHER: the k lines of both (row-contiguous, 16-byte aligned) operands are those a list names (GemmArgs::k_order).
// The workgroups a compute unit is to hold (by registers; LDS allows as many) are what hides one's loads and conversions
// behind another's matrix instructions.  128 x 128 tiles of two row-contiguous operands take 55 KB each, so two: where three were
// asked for, the compiler held operands in accumulator registers and a small change made it miss two as well (the feed-forward
// model 2213 -> 2293 us per pass).
template <int VA, bool AK, int VB, bool BK_, bool MASKED, int TILE, bool FAN = false, bool GATHER = false, int WAVES = 4>
__global__ __launch_bounds__(64 * WAVES, WAVES == 8 ? 4 : TILE == 128 ? (VA * VB == 16 && (AK || BK_) ? 3 : 2) : VA * VB == 16 ? 5 : 4) void gemm_split_kernel(const GemmArgs args) {
    constexpr int BM = TILE, BN = TILE;
    constexpr int NT = 64 * WAVES;
    static_assert(WAVES == 4 || !MASKED, "the masked loader is for four waves");
    constexpr int WM = TILE / 2, WN = 2 * TILE / WAVES;  // a wave's block (waves are arranged 2 x 2 or 2 x 4)
    constexpr int NBM = WM / 32, NBN = WN / 32;          // 32 x 32 MFMA tiles per wave and dimension
    typedef TileLayout<MASKED ? VA : 4, AK, TILE, NT> LA;
    typedef TileLayout<MASKED ? VB : 4, BK_, TILE, NT> LB;
    __shared__ uint4 lds[LA::UNITS + LB::UNITS];
    uint4 *const lds_a = lds, *const lds_b = lds + LA::UNITS;

    const int tid = threadIdx.x;
    const int lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int wm = wave & 1, wn = wave >> 1;

    // Which tile, k range and problem this workgroup takes.  Workgroups go to the eight XCDs in turn, in launch
    // order, and each XCD has its own L2: the workgroups one XCD receives take CONSECUTIVE positions of the order
    // (tile, problem, k range), with the tiles of one output walked in bands of eight rows of tiles.  What runs on one XCD
    // at a time is then a compact block of tiles of one k range (its operand panels are fetched into that L2 once
    // instead of once per XCD) and, for several problems per launch, the same k range of neighbouring problems
    // (which share an operand where a layer's taps or a stack's layers read the same input).
    const int tiles_m = (args.m + BM - 1) / BM;
    int tile = blockIdx.x, split_id = blockIdx.y, prob_id = blockIdx.z;
    // Listed columns: the tiles that hold some of them are dealt as if there were no others, the rest, behind them, store zeros.  A
    // k-contiguous operand's offsets are per row and formed once, so the list costs a load in front of the loop.  Input projections
    // 512 -> 2 x 4 x 256 over 9600 slots of which 7200 are valid: 141 -> 108 us; the errors of such a layer 168 -> 143 beside its weight
    // gradients; the pass of 32 sequences 2443 -> 2296, 150 and 200 cells with twenty sequences (71 % valid) 2165 -> 2133.
    constexpr bool LISTS = BK_ && !MASKED && !FAN && !GATHER;
    __shared__ int col_of[LISTS ? BN : 1];
    const bool listed = LISTS && args.cols != nullptr;
    unsigned tiles = gridDim.x;
    int listed_n = args.n;
    if (listed) {
        listed_n = args.cols_count[0];
        const unsigned at = blockIdx.x + gridDim.x * blockIdx.z;
        tiles = (unsigned)(tiles_m * ((listed_n + BN - 1) / BN));
        const unsigned live = tiles * gridDim.z;
        if (at >= live) {
            const unsigned others = gridDim.x - tiles, in_output = tiles + (at - live) % others;
            const int z0 = (int)(in_output % (unsigned)tiles_m) * BM, c0 = (int)(in_output / (unsigned)tiles_m) * BN;
            float *__restrict__ const C = args.prob[(at - live) / others].C;
            for (int i = tid; i < BM * BN; i += NT) {
                const int m = z0 + i % BM, n = c0 + i / BM;
                if (m < args.m && n < args.n) C[(size_t)args.cols[n] * args.ldc + m] = 0.0f;
            }
            return;
        }
        tile = (int)(at % tiles);
        prob_id = (int)(at / tiles);
    }
    if (args.xcd_map) {
        const unsigned total = tiles * gridDim.y * gridDim.z;
        const unsigned at = blockIdx.x + gridDim.x * (blockIdx.y + gridDim.y * blockIdx.z);
        const unsigned per = total / 8, rem = total % 8, xcd = at % 8, slot = at / 8;
        const unsigned pos = xcd < rem ? xcd * (per + 1) + slot : rem * (per + 1) + (xcd - rem) * per + slot;
        const unsigned in_output = pos % tiles, rest = pos / tiles;
        prob_id = (int)(rest % gridDim.z);
        split_id = (int)(rest / gridDim.z);
        const int tiles_n = (int)tiles / tiles_m;
        const int band = (int)in_output / (8 * tiles_n), off = (int)in_output % (8 * tiles_n);
        const int rows = min(tiles_m - 8 * band, 8);
        tile = (8 * band + off % rows) + (off / rows) * tiles_m;
    }
    const int m0 = (tile % tiles_m) * BM;
    const int n0 = (tile / tiles_m) * BN;
    const GemmProblem &pb = args.prob[prob_id];
    if (listed) {
        if (tid < BN) col_of[tid] = args.cols[min(n0 + tid, args.n - 1)];
        __syncthreads();
    }

    // iteration space: segments x k-tiles, cut into splitk contiguous ranges
    // the listed k lines this problem takes: all of them, or all but the first / last time step's
    int k_extent = args.k, k_lo = 0;
    if (GATHER) {
        k_extent = args.k_count[0];
        if (pb.k_trim == 1) { k_lo = args.k_count[1]; k_extent -= k_lo; }
        else if (pb.k_trim == 2) k_extent -= args.k_count[2];
        k_extent = max(k_extent, 0);
    }
    const int kt_per_seg = max((k_extent + BK - 1) / BK, 1);  // (1 where the list is empty: no k tile, and nothing divided by zero)
    const int total_it = k_extent > 0 ? kt_per_seg * args.nseg : 0;
    const int per_split = (total_it + args.splitk - 1) / args.splitk;
    const int it_begin = split_id * per_split;
    const int it_end = min(total_it, it_begin + per_split);
    // (a split left without k lines by a short list still has its zeros to write)
    if (it_begin >= it_end && !(GATHER && args.epilogue != EPI_ATOMIC)) return;

    f32x16 acc[NBM][NBN];
#pragma unroll
    for (int i = 0; i < NBM; ++i)
#pragma unroll
        for (int j = 0; j < NBN; ++j)
#pragma unroll
            for (int r = 0; r < 16; ++r) acc[i][j][r] = 0.0f;

    const char *mask_pat = MASKED ? args.pat : nullptr;

    // sum of the B operand over this split's k range, per row (dense bias gradient), by the workgroups of the first row of
    // tiles: taken from the fp32 values on their way to LDS, because an infinite value cannot be put together again from its
    // parts.  Those workgroups run a loop of their own, and only the operand kinds of a weight gradient have one.
    const bool rowsum = !AK && !BK_ && !MASKED && args.rowsum != 0 && m0 == 0;
    float rs[4] = {0.0f, 0.0f, 0.0f, 0.0f};  // the rows of one of the thread's vectors, over the k positions it loads

    const int frag_row = lane & 31;
    const int half = lane >> 5;

    // `fetch_next(a, b)` loads the next tile of the walk into the register sets; after the last tile it loads that one
    // again, so that the count of loads in flight is the same on every path.  The loads of tile it+1 are in flight during
    // the matrix instructions of tile it; the barriers order LDS only (__syncthreads() would also wait for those loads).
    auto loop = [&](auto &ra, auto &rb, auto &fetch_next, auto sums) __attribute__((always_inline)) {
        fetch_next(ra, rb);
        for (int it = it_begin; it < it_end; ++it) {
            if constexpr (decltype(sums)::value) rb.add_rows(rs);
            ra.store(lds_a, tid);
            rb.store(lds_b, tid);
            fetch_next(ra, rb);
            lds_only_barrier();
#pragma unroll
            for (int s = 0; s < BK / 16; ++s) {
                bf16x8 fa[NBM][3], fb[NBN][3];
#pragma unroll
                for (int i = 0; i < NBM; ++i) LA::fragment(lds_a, wm * WM + i * 32 + frag_row, 2 * s + half, fa[i]);
#pragma unroll
                for (int j = 0; j < NBN; ++j) LB::fragment(lds_b, wn * WN + j * 32 + frag_row, 2 * s + half, fb[j]);
                // h*l, l*h, m*m, h*m, m*h, h*h: the small terms first
                constexpr int QA[6] = {0, 2, 1, 0, 1, 0}, QB[6] = {2, 0, 1, 1, 0, 0};
#pragma unroll
                for (int t = 0; t < 6; ++t)
#pragma unroll
                    for (int i = 0; i < NBM; ++i)
#pragma unroll
                        for (int j = 0; j < NBN; ++j)
                            acc[i][j] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(fb[j][QB[t]], fa[i][QA[t]], acc[i][j], 0, 0, 0);
            }
            lds_only_barrier();
        }
    };
    auto run = [&](auto &ra, auto &rb, auto &fetch_next) __attribute__((always_inline)) {
        if constexpr (!AK && !BK_ && !MASKED) {
            if (rowsum) {
                loop(ra, rb, fetch_next, std::true_type());
                return;
            }
        }
        loop(ra, rb, fetch_next, std::false_type());
    };
    if constexpr (GATHER) {
        static_assert(VA == 4 && VB == 4 && !AK && !BK_ && !MASKED, "the gathering loader is for two row-contiguous operands");
        GatherStage<TILE, NT> ga, gb;
        ga.init(m0, args.m, tid);
        gb.init(n0, args.n, tid);
        constexpr int NL = GatherStage<TILE, NT>::NLOAD;
        const int *__restrict__ order = args.k_order + k_lo;
        const int k_shift = pb.k_shift;
        const unsigned a_line = (unsigned)(args.lda * sizeof(float)), b_line = (unsigned)(args.ldb * sizeof(float));
        int seg = min(it_begin / kt_per_seg, args.nseg - 1), kin = it_begin % kt_per_seg, left = it_end - it_begin - 1;
        const float *pa = pb.A[seg], *pbb = pb.B[seg];
        // the k lines of the cursor's tile, loaded while the tile before it is being requested
        int idx[NL];
        auto lines_of = [&](int tile) __attribute__((always_inline)) {
#pragma unroll
            for (int p = 0; p < NL; ++p) idx[p] = order[max(min(tile * BK + ga.kk + p, k_extent - 1), 0)] + k_shift;
        };
        lines_of(kin);
        auto fetch_next = [&](GatherStage<TILE, NT> &qa, GatherStage<TILE, NT> &qb) __attribute__((always_inline)) {
            const int kv = min(BK, k_extent - kin * BK);
            qa.load(pa, a_line, idx, kv);
            qb.load(pbb, b_line, idx, kv);
            if (left > 0) {
                --left;
                if (++kin == kt_per_seg) {
                    kin = 0; ++seg;
                    pa = pb.A[seg]; pbb = pb.B[seg];
                }
            }
            lines_of(kin);
        };
        if (it_begin < it_end) run(ga, gb, fetch_next);
    } else if constexpr (MASKED) {
        TileStage<VA, AK, TILE> sa;
        TileStage<VB, BK_, TILE> sb;
        int next_it = it_begin;
        auto fetch_next = [&](TileStage<VA, AK, TILE> &ra, TileStage<VB, BK_, TILE> &rb) __attribute__((always_inline)) {
            const int it = min(next_it, it_end - 1);
            ++next_it;
            const int seg = it / kt_per_seg;
            const int k0 = (it % kt_per_seg) * BK;
            ra.load(pb.A[seg], args.lda, m0, k0, args.m, args.k, tid);
            rb.load(pb.B[seg], args.ldb, n0, k0, args.n, args.k, tid, mask_pat, pb.b_shift[seg], args.n_slots,
                    args.b_time_on_k != 0);
        };
        run(sa, sb, fetch_next);
    } else {
        // the tile cursor: operand pair `seg`, k tile `kin` inside it; the operands' base pointers are looked up only
        // when the pair changes
        FastStage<VA == 4, AK, TILE, NT> sa;
        FastStage<VB == 4, BK_, TILE, NT> sb;
        sa.init(args.lda, m0, args.m, tid);
        sb.init(args.ldb, n0, args.n, tid, listed ? col_of : nullptr);
        int seg = it_begin / kt_per_seg, kin = it_begin % kt_per_seg, left = it_end - it_begin - 1;
        const float *pa = pb.A[seg], *pbb = pb.B[seg];
        const size_t ka = AK ? 1 : (size_t)args.lda, kb = BK_ ? 1 : (size_t)args.ldb;  // floats per k step
        auto fetch_next = [&](FastStage<VA == 4, AK, TILE, NT> &qa, FastStage<VB == 4, BK_, TILE, NT> &qb) __attribute__((always_inline)) {
            qa.load(pa + (size_t)kin * BK * ka, args.k - kin * BK, tid);
            qb.load(pbb + (size_t)kin * BK * kb, args.k - kin * BK, tid);
            if (left > 0) {
                --left;
                if (++kin == kt_per_seg) {
                    kin = 0; ++seg;
                    pa = pb.A[seg]; pbb = pb.B[seg];
                }
            }
        };
        run(sa, sb, fetch_next);
    }

    // what came out infinite or not a number is formed again (plain_sums)
#pragma unroll
    for (int i = 0; i < NBM; ++i)
#pragma unroll
        for (int j = 0; j < NBN; ++j) {
            bool finite = true;
#pragma unroll
            for (int r = 0; r < 16; ++r) finite = finite && __builtin_fabsf(acc[i][j][r]) <= lim::kMax;
#pragma unroll
            for (int r = 0; r < 16; ++r) acc[i][j][r] *= 1.0f / (kSplitScale * kSplitScale);
            if (__builtin_expect(__builtin_amdgcn_ballot_w64(!finite) != 0, 0))
                acc[i][j] = plain_sums<AK, BK_, MASKED, GATHER>(args, pb, m0 + wm * WM + 32 * i, n0 + wn * WN + 32 * j, lane, it_begin,
                                                                it_end, kt_per_seg, k_extent, k_lo);
        }

    // epilogue: lane%32 runs along m (contiguous), the 16 accumulators along n
    float *__restrict__ C = pb.C;
    if constexpr (!AK && !BK_ && !MASKED) {
        if (rowsum) {
            // the threads that loaded different k positions of the same rows add up through LDS, in a fixed order
            constexpr int PARTS = BK / LB::NLOAD;
            static_assert(PARTS * BN * sizeof(float) <= sizeof(lds), "the row sums fit the tile's buffer");
            float *const sums = reinterpret_cast<float *>(lds);
            __syncthreads();
            *reinterpret_cast<float4 *>(sums + LB::first_k(tid) / LB::NLOAD * BN + LB::first_row(tid)) = float4{rs[0], rs[1], rs[2], rs[3]};
            __syncthreads();
            if (tid < BN && n0 + tid < args.n) {
                float s = 0.0f;
#pragma unroll
                for (int q = 0; q < PARTS; ++q) s += sums[q * BN + tid];
                if (args.epilogue == EPI_PARTIAL)
                    args.partial[(size_t)split_id * args.partial_stride + (size_t)args.nprob * args.m * args.n +
                                 (size_t)prob_id * args.n + n0 + tid] = s;
                else if (args.epilogue == EPI_STORE)
                    pb.rowsum_out[n0 + tid] = pb.rowsum_scale * s;
                else
                    atomicAdd(pb.rowsum_out + n0 + tid, pb.rowsum_scale * s);
            }
        }
    }
    if (FAN) {
        // All loads of a 32 x 32 tile's sixteen values per lane are issued before anything is stored: the compiler
        // cannot know that the buffers do not overlap and would otherwise wait for memory once per value.
#pragma unroll
        for (int i = 0; i < NBM; ++i) {
            const int m = m0 + wm * WM + i * 32 + frag_row;
#pragma unroll
            for (int j = 0; j < NBN; ++j) {
                size_t idx[16];
                bool ok[16];
                float e[16], old[16];
#pragma unroll
                for (int r = 0; r < 16; ++r) {
                    const int n = n0 + wn * WN + j * 32 + 8 * (r >> 2) + 4 * half + (r & 3);
                    ok[r] = m < args.m && n < args.n;
                    idx[r] = ok[r] ? (size_t)n * args.ldc + m : 0;
                    old[r] = (ok[r] && pb.aux_in) ? pb.aux_in[idx[r]] : 0.0f;
                }
#pragma unroll
                for (int r = 0; r < 16; ++r) {
                    e[r] = pb.aux_in ? old[r] + acc[i][j][r] : acc[i][j][r];
                    if (ok[r]) C[idx[r]] = e[r];
                }
                for (int q = 0; q < args.fan_n; ++q) {
                    float *__restrict__ t = args.fan_targets[q];
                    if (args.fan_is_skip[q]) {
#pragma unroll
                        for (int r = 0; r < 16; ++r) old[r] = ok[r] ? t[idx[r]] : 0.0f;
#pragma unroll
                        for (int r = 0; r < 16; ++r)
                            if (ok[r]) t[idx[r]] = e[r] + old[r];
                    } else {
#pragma unroll
                        for (int r = 0; r < 16; ++r)
                            if (ok[r]) t[idx[r]] = e[r];
                    }
                }
            }
        }
        return;
    }
    // The other epilogues: what becomes of the sums first, in registers, one kind of step after the other, then the stores.  Every step is
    // straight code over a wave's sums with the choices outside.  With a switch and the edges' conditions per sum the kernels were 7 to
    // 28 thousand instructions, and what bounded a tile's end was fetching them: 1024 x 32000 x 128 103 -> 58 us (128 x 128 tiles, four
    // waves), 79 -> 72 (64 x 64), 1936 x 6000 x 256 51 -> 42, 1024 x 12000 x 1024 161 -> 151, 512 x 6000 x 512 33 -> 31; the feed-forward
    // model's pass 2018 -> 1924, mixture output 171 -> 158.
    const int epilogue = args.epilogue;
    int ldc = args.ldc;
    if (epilogue == EPI_PARTIAL) {
        // this split's partial product, m x n column-major without padding, after those of the problems before it
        C = args.partial + (size_t)split_id * args.partial_stride + (size_t)prob_id * args.m * args.n;
        ldc = args.m;
    }
    const int wave_m = m0 + wm * WM, wave_n = wn * WN;  // the wave's first row, its first column inside the tile
    auto in_tile = [&](int j, int r) __attribute__((always_inline)) { return wave_n + 32 * j + 8 * (r >> 2) + 4 * half + (r & 3); };
    // the column of C for a column of the tile (clamped into the matrix)
    auto column = [&](int at) __attribute__((always_inline)) { return listed ? col_of[at] : min(n0 + at, args.n - 1); };
    auto all_sums = [&](auto &&step) __attribute__((always_inline)) {
#pragma unroll
        for (int i = 0; i < NBM; ++i)
#pragma unroll
            for (int j = 0; j < NBN; ++j)
#pragma unroll
                for (int r = 0; r < 16; ++r) acc[i][j][r] = step(acc[i][j][r], i, j, r);
    };
    if (listed && n0 + BN > listed_n)  // behind the listed columns there are zeros
        all_sums([&](float v, int, int j, int r) { return n0 + in_tile(j, r) < listed_n ? v : 0.0f; });
    // (which operand kinds come with which epilogue: gemm_launch)
    constexpr bool FORWARD = AK && BK_, BACKWARD = !AK && BK_;
    if (FORWARD && (epilogue == EPI_BIAS_ACT || epilogue == EPI_BIAS_ACT_SKIP)) {
#pragma unroll
        for (int i = 0; i < NBM; ++i) {
            const float bterm = args.bias_scale * pb.bias_vec[min(wave_m + 32 * i + frag_row, args.m - 1)];
#pragma unroll
            for (int j = 0; j < NBN; ++j)
#pragma unroll
                for (int r = 0; r < 16; ++r) acc[i][j][r] += bterm;
        }
        by_activation(args.act, [&](auto act) { all_sums([&](float v, int, int, int) { return act_fn(decltype(act)::value, v); }); });
    } else if ((BACKWARD && epilogue == EPI_STORE_DELTA) || (FORWARD && !MASKED && epilogue == EPI_CONTEXT) || epilogue == EPI_ADD) {
        // What the sums meet in memory is requested for sixteen of them at a time: the compiler cannot know that it does not
        // overlap the output and would wait for one load per sum (a dense layer's deltas in the epilogue of the product above
        // it: the feed-forward model's pass, four such products, 2260 -> 2183 us).
        const float *const old = epilogue == EPI_ADD ? C : pb.aux_in;
#pragma unroll
        for (int j = 0; j < NBN; ++j)
#pragma unroll
            for (int i = 0; i < NBM; ++i) {
                const int m = min(wave_m + 32 * i + frag_row, args.m - 1);
                float met[16];
#pragma unroll
                for (int r = 0; r < 16; ++r) met[r] = old[(size_t)column(in_tile(j, r)) * ldc + m];
                f32x16 &v = acc[i][j];
                if (epilogue == EPI_ADD) {
#pragma unroll
                    for (int r = 0; r < 16; ++r) v[r] = met[r] + v[r];
                } else if constexpr (BACKWARD) {
                    by_activation(args.act, [&](auto act) {
#pragma unroll
                        for (int r = 0; r < 16; ++r) v[r] *= act_deriv(decltype(act)::value, met[r]);
                    });
                } else if constexpr (FORWARD && !MASKED) {
                    bool valid[16];
#pragma unroll
                    for (int r = 0; r < 16; ++r) valid[r] = args.pat[column(in_tile(j, r))] != 0;
#pragma unroll
                    for (int r = 0; r < 16; ++r) {
                        const float th = valid[r] ? tanh_act(v[r]) : 0.0f;
                        met[r] = valid[r] ? met[r] + th : 0.0f;
                        v[r] = th;
                    }
                    if (pb.aux_out)
#pragma unroll
                        for (int r = 0; r < 16; ++r) {
                            const int n = n0 + in_tile(j, r);
                            if (n < args.n && wave_m + 32 * i + frag_row < args.m) pb.aux_out[(size_t)n * ldc + m] = v[r];
                        }
#pragma unroll
                    for (int r = 0; r < 16; ++r) v[r] = met[r];
                }
            }
    }
    // A wave whose sums all lie inside the matrix stores them through one offset per lane beside an address per sum that is uniform.
    if (epilogue != EPI_ATOMIC && epilogue != EPI_BIAS_ACT_SKIP && !listed && wave_m + WM <= args.m && n0 + wave_n + WN <= args.n) {
        const unsigned mine = ((unsigned)(4 * half) * (unsigned)ldc + (unsigned)frag_row) * (unsigned)sizeof(float);
        char *at = reinterpret_cast<char *>(C + (size_t)(n0 + wave_n) * ldc + wave_m);
        const size_t line = (size_t)ldc * sizeof(float);
#pragma unroll
        for (int j = 0; j < NBN; ++j)
#pragma unroll
            for (int r = 0; r < 16; ++r) {
#pragma unroll
                for (int i = 0; i < NBM; ++i) *reinterpret_cast<float *>(at + mine + 128 * i) = acc[i][j][r];
                at += (r & 3) == 3 ? 5 * line : line;
                asm volatile("" : "+s"(at));  // (one address that moves along, not one per column)
            }
        return;
    }
#pragma unroll
    for (int j = 0; j < NBN; ++j) {
        bool keep[16];
#pragma unroll
        for (int r = 0; r < 16; ++r) {
            keep[r] = n0 + in_tile(j, r) < args.n;
            if constexpr (FORWARD && MASKED)
                if (epilogue == EPI_BIAS_ACT_SKIP) keep[r] = keep[r] && args.pat[column(in_tile(j, r))] != 0;
        }
#pragma unroll
        for (int i = 0; i < NBM; ++i) {
            const int m = wave_m + 32 * i + frag_row;
            if (m >= args.m) continue;
            if (epilogue == EPI_ATOMIC) {
#pragma unroll
                for (int r = 0; r < 16; ++r)
                    if (keep[r]) atomicAdd(C + (size_t)column(in_tile(j, r)) * ldc + m, acc[i][j][r]);
            } else {
#pragma unroll
                for (int r = 0; r < 16; ++r)
                    if (keep[r]) C[(size_t)column(in_tile(j, r)) * ldc + m] = acc[i][j][r];
            }
        }
    }
}

template <int VA, bool AK, int VB, bool BK_>
void launch_t(const GemmArgs &a, dim3 grid, hipStream_t s, int tile) {
    // gemm_launch has checked the operand kinds of the two special products and that they, and the masked one, come with
    // the small tile
    if (a.epilogue == EPI_FAN) {
        if constexpr (VA == 4 && !AK && VB == 4 && BK_) {
            if (a.masked)
                hipLaunchKernelGGL((gemm_split_kernel<VA, AK, VB, BK_, true, 64, true>), grid, dim3(NTHREADS), 0, s, a);
            else
                hipLaunchKernelGGL((gemm_split_kernel<VA, AK, VB, BK_, false, 64, true>), grid, dim3(NTHREADS), 0, s, a);
        }
    } else if (a.k_order) {
        if constexpr (VA == 4 && !AK && VB == 4 && !BK_) {
            if (tile == kEightWaves)
                hipLaunchKernelGGL((gemm_split_kernel<VA, AK, VB, BK_, false, 128, false, true, 8>), grid, dim3(2 * NTHREADS), 0, s, a);
            else if (tile == 128)
                hipLaunchKernelGGL((gemm_split_kernel<VA, AK, VB, BK_, false, 128, false, true>), grid, dim3(NTHREADS), 0, s, a);
            else
                hipLaunchKernelGGL((gemm_split_kernel<VA, AK, VB, BK_, false, 64, false, true>), grid, dim3(NTHREADS), 0, s, a);
        }
    } else if (a.masked) {
        hipLaunchKernelGGL((gemm_split_kernel<VA, AK, VB, BK_, true, 64>), grid, dim3(NTHREADS), 0, s, a);
    } else if constexpr (VA != 2 && VB != 2) {
        if (tile == kEightWaves)
            hipLaunchKernelGGL((gemm_split_kernel<VA, AK, VB, BK_, false, 128, false, false, 8>), grid, dim3(2 * NTHREADS), 0, s, a);
        else if (tile == 128) hipLaunchKernelGGL((gemm_split_kernel<VA, AK, VB, BK_, false, 128>), grid, dim3(NTHREADS), 0, s, a);
        else hipLaunchKernelGGL((gemm_split_kernel<VA, AK, VB, BK_, false, 64>), grid, dim3(NTHREADS), 0, s, a);
    }
}
template <int VA, bool AK, int VB>
void launch_b(const GemmArgs &a, dim3 grid, hipStream_t s, bool bk, int tile) {
    if (bk) launch_t<VA, AK, VB, true>(a, grid, s, tile);
    else if constexpr (!AK) launch_t<VA, AK, VB, false>(a, grid, s, tile);  // (no product has a k-contiguous A and a row-contiguous B)
}
template <int VA, bool AK>
void launch_vb(const GemmArgs &a, dim3 grid, hipStream_t s, int vb, bool bk, int tile) {
    if (vb == 4) launch_b<VA, AK, 4>(a, grid, s, bk, tile);
    else if (vb == 2) launch_b<VA, AK, 2>(a, grid, s, bk, tile);
    else launch_b<VA, AK, 1>(a, grid, s, bk, tile);
}
template <int VA>
void launch_ak(const GemmArgs &a, dim3 grid, hipStream_t s, bool ak, int vb, bool bk, int tile) {
    if (ak) launch_vb<VA, true>(a, grid, s, vb, bk, tile);
    else launch_vb<VA, false>(a, grid, s, vb, bk, tile);
}

}  // namespace

// One translation unit per A-operand vector width instantiates its share of the kernels (they compile in
// parallel); gemm.hip dispatches on the width.
void gemm_dispatch_va4(const GemmArgs &a, dim3 grid, hipStream_t s, bool ak, int vb, bool bk, int tile);
void gemm_dispatch_va2(const GemmArgs &a, dim3 grid, hipStream_t s, bool ak, int vb, bool bk, int tile);
void gemm_dispatch_va1k(const GemmArgs &a, dim3 grid, hipStream_t s, int vb, bool bk, int tile);
void gemm_dispatch_va1r(const GemmArgs &a, dim3 grid, hipStream_t s, int vb, bool bk, int tile);

}  // namespace cnt
