// Multi-resolution STFT spectral loss (seven amplitude / spectrum distances) and its gradient for gfx950, with
// an in-house radix-4 FFT.
//
// Reference behaviour: helpers/FFTMat.cu (FrameSignal :282-312, distances :473-628, gradients :760-900,
// cleanDummyGradients :456-471, collectGrad :965-1006, drivers :1246-1274, :1350-1475, :1637-1770,
// :1833-1886) and layers/DFTErrorPostoutputLayer.cu (:1186-1244, :1699-1714, :1782-1885).  The reference
// runs about a dozen launches and three cuFFT calls per resolution and waveform, with every intermediate
// (framed signals, spectra, per-bin differences, framed gradients) in device memory.
//
// Here a frame stays in one workgroup's registers and LDS end to end, all resolutions of a call are one launch, and nothing
// but the waveforms and the gradient touches HBM:
//   frame + window source and target  ->  ONE complex FFT of z = source + i*target in LDS (both real
//   spectra are recovered from Z[b] and Z[N-b])  ->  per-bin distance, loss partial and gradient spectrum,
//   written back as its Hermitian extension  ->  inverse FFT in LDS  ->  windowed overlap-add straight into
//   the per-sample gradient with float atomics.
// A workgroup of 256 threads holds 2048 points, one frame of 2048 or as many shorter ones as that makes, eight points per
// thread in registers; frames of up to 512 points lie inside one wave and need no barrier.  It adds its loss partial to the
// per-waveform sums once at its end.
// What bounds it is the chain of a frame: loads, LOGN/2 - 1 exchanges through LDS, the bins, the exchanges back, the atomics.
// Eight waveforms of 16 000 samples at 2048 / 512 / 128 points: 23 us with four points per butterfly read from and written to
// LDS, a barrier per radix-4 step, tables in LDS and two or three passes of a workgroup; 16 us now (16 points per thread, four
// stages per exchange: 19 us; three stages of eight: 15 us, but its rounding differs and the log distance's gradient, which
// divides by amplitudes close to zero, moves by 5e-5).  The registers decide: 119 of them let four workgroups share a compute
// unit, with a loop over several frames per workgroup (145, three workgroups) the same call takes 24.5 instead of 18.7 us.
// The forward transform is decimation-in-frequency (natural order in, bit-reversed out), the per-bin stage
// addresses bins through the bit-reversal, and the inverse is decimation-in-time (bit-reversed in, natural
// out), so no reordering pass exists; two butterfly stages share a barrier as one radix-4 butterfly.  Twiddles
// (one run per stage, so that a wave reads consecutive words) and the window (with the reference's
// constant 3.141215) are tabulated in double on the host.  Transform conventions are cuFFT's: unnormalised,
// N/2+1 bins, the imaginary parts of the DC and Nyquist bins do not enter the inverse.
#include "common.hpp"

#include <algorithm>
#include <cmath>
#include <cstring>
#include <new>
#include <vector>

namespace cnt {
namespace {

constexpr int kMaxRes = 3;
constexpr int kMaxWavesPerLaunch = 32;
constexpr int kMaxThreads = 512;  // eight points per thread: a workgroup holds a frame of 4096

struct DftParams {
    // per resolution: log2 of the fft length, frame length, frame shift, blocks along x that carry frames
    int logn[kMaxRes], Nw[kMaxRes], Hs[kMaxRes], nblocks[kMaxRes];
    const float2 *twiddle[kMaxRes];  // N entries, stage by stage: entry 2^s + k = exp(-2*pi*i*k / 2^(s+1)), k < 2^s
    const float *window[kMaxRes];    // Nw entries
    int max_length;      // samples per waveform buffer
    int n_waves, n_res;

    int lengths[kMaxWavesPerLaunch];
    float gamma, log_floor;
    float zeta;          // weight of the cosine phase distance; 0 = not evaluated
    const float *source, *target;
    float *grad;    // n_waves x max_length, accumulated over resolutions
    float *errors;  // n_waves x n_res amplitude distances, followed by n_waves x n_res phase distances if zeta > 0
};

__host__ __device__ inline int frame_count(int length, int Nw, int Hs) {
    return length < Nw ? 1 : 1 + (length - Nw) / Hs;
}

// The reference's floors and constants (helpers/FFTMat.hpp: FFT_KLD_FLOOR_NUM, FFT_IS_FLOOR_NUM,
// FFT_SPEC_LOG_MSE_CONST)
constexpr float kKldFloor = 0.00001f;
constexpr float kIsFloor = 0.00001f;
constexpr float kSpecLogMseConst = 1.0f;

// Distance of one bin and the gradient spectrum of that bin, for source spectrum (sx, sy) and target spectrum
// (tx, ty).  Distance functors: helpers/FFTMat.cu:473-628; gradient functors: :760-900.  DIS is the reference's
// specDisType: 0 log-amplitude MSE, 1 KLD of amplitudes, 2 MSE of squared amplitudes, 3 log of the complex
// spectral distance, 4 complex spectral MSE, 5 amplitude ratio, 6 Itakura-Saito.
template <int DIS>
__device__ inline void bin_distance(float sx, float sy, float tx, float ty, float log_floor, float &e, float &gx,
                                    float &gy) {
    const float s2 = sx * sx + sy * sy, t2 = tx * tx + ty * ty;
    if (DIS == 1) {
        const float s = sqrtf(s2 + kKldFloor), t = sqrtf(t2 + kKldFloor);
        e = t * safe_log(t / s) - t + s;
        const float aux = 1.0f - t / s;
        gx = aux * sx / s;
        gy = aux * sy / s;
    } else if (DIS == 2) {
        const float aux = s2 - t2;
        e = aux * aux;
        gx = aux * sx;
        gy = aux * sy;
    } else if (DIS == 3) {
        const float dx = sx - tx, dy = sy - ty;
        const float aux = dx * dx + dy * dy + kSpecLogMseConst;
        e = safe_log(aux);
        gx = dx / aux;
        gy = dy / aux;
    } else if (DIS == 4) {
        const float dx = sx - tx, dy = sy - ty;
        e = dx * dx + dy * dy;
        gx = dx;
        gy = dy;
    } else if (DIS == 5) {
        const float tf = t2 + kKldFloor;
        const float aux = (s2 + kKldFloor) / tf - 1.0f;
        e = aux * aux;
        gx = aux * sx / tf;
        gy = aux * sy / tf;
    } else if (DIS == 6) {
        const float sf = s2 + kIsFloor;
        const float aux = sqrtf(t2 + kIsFloor) / sqrtf(sf);
        e = aux - safe_log(aux) - 1.0f;
        gx = sx / sf * (1.0f - aux);
        gy = sy / sf * (1.0f - aux);
    } else {
        const float spec = s2 + log_floor;
        const float d = safe_log(spec) - safe_log(t2 + log_floor);
        e = d * d;
        gx = d * sx / spec;
        gy = d * sy / spec;
    }
}

// Cosine phase distance 1 - cos(arg S - arg T) of one bin and its gradient spectrum (helpers/FFTMat.cu:630-656
// phaseDistance, :862-878 PhaseGrad; FFT_AMP_MIN_NUM floors the amplitude product, FFT_KLD_FLOOR_NUM the
// gradient's denominator).
constexpr float kAmpMin = 0.0000001f;
__device__ inline void bin_phase(float sx, float sy, float tx, float ty, float &e, float &gx, float &gy) {
    float amp = sqrtf(sx * sx + sy * sy) * sqrtf(tx * tx + ty * ty);
    if (amp < kAmpMin) {
        e = 0.0f;
        amp = kAmpMin;
    } else {
        e = 1.0f - (sx * tx + sy * ty) / amp;
    }
    const float spec = sx * sx + sy * sy + kKldFloor;
    const float fac = (sy * tx - sx * ty) / amp;
    gx = -fac * sy / spec;
    gy = fac * sx / spec;
}

constexpr int kMaxLogN = 12;

// ---- the transform: radix 4, eight points per thread ----
// In-place decimation in frequency over T = N/8 threads.  Stage s, from LOGN - 1 down, combines points 2^s apart; the stages s and
// s - 1 are one radix-4 butterfly on the points base + {0, q, 2q, 3q}, q = 2^(s-1).  In a pass a thread takes the butterflies t
// and t + T, in the first one, q = N/4, that is the points t + j*T, which is how the samples arrive; in the last one it takes the
// points 8t + r, in three stages for odd LOGN, in two for even.  A pass leaves its results where it took its points, so one
// exchange through LDS lies between two passes.  Point p is then bin bitrev(p).  The inverse walks the same stages backwards
// with conjugated twiddles and ends with the samples t + j*T.
struct Twiddles4 {
    float2 w1, w2;  // of the butterfly's first stage (its second pair takes -i times that) and of its second
};
// Which products are rounded is written out: a spectrum's small amplitudes, by which some distances divide, are what their
// rounding leaves, and the log distance's gradient moves by up to 5e-5 with it.
__device__ __forceinline__ float2 turned(float2 a, float2 w) {  // a * w
    return make_float2(__builtin_fmaf(a.x, w.x, -(a.y * w.y)), __builtin_fmaf(a.y, w.x, a.x * w.y));
}
__device__ __forceinline__ float2 turned_back(float2 a, float2 w) {  // a * conj(w)
    return make_float2(__builtin_fmaf(a.x, w.x, a.y * w.y), __builtin_fmaf(a.y, w.x, -(a.x * w.y)));
}
// what enters and leaves a butterfly is rounded, whatever the compiler could join across it
__device__ __forceinline__ void settle(float2 &x) { asm volatile("" : "+v"(x.x), "+v"(x.y)); }

__device__ __forceinline__ void butterfly4(float2 &x0, float2 &x1, float2 &x2, float2 &x3, const Twiddles4 &w) {
    const float2 w1 = w.w1, w2 = w.w2;
    const float2 y0 = make_float2(x0.x + x2.x, x0.y + x2.y), d02 = make_float2(x0.x - x2.x, x0.y - x2.y);
    const float2 y1 = make_float2(x1.x + x3.x, x1.y + x3.y), d13 = make_float2(x1.y - x3.y, x3.x - x1.x);
    const float2 y2 = turned(d02, w1), y3 = turned(d13, w1);
    const float2 e01 = make_float2(y0.x - y1.x, y0.y - y1.y), e23 = make_float2(y2.x - y3.x, y2.y - y3.y);
    x0 = make_float2(y0.x + y1.x, y0.y + y1.y);
    x1 = turned(e01, w2);
    x2 = make_float2(y2.x + y3.x, y2.y + y3.y);
    x3 = make_float2(__builtin_fmaf(e23.x, w2.x, -(e23.y * w2.y)), __builtin_fmaf(e23.x, w2.y, e23.y * w2.x));
    settle(x0); settle(x1); settle(x2); settle(x3);
}
__device__ __forceinline__ void inverse_butterfly4(float2 &x0, float2 &x1, float2 &x2, float2 &x3, const Twiddles4 &w) {
    const float2 w1 = w.w1, w2 = w.w2;
    const float2 v1 = turned_back(x1, w2), v3 = turned_back(x3, w2);
    const float2 y0 = make_float2(x0.x + v1.x, x0.y + v1.y), y1 = make_float2(x0.x - v1.x, x0.y - v1.y);
    const float2 y2 = make_float2(x2.x + v3.x, x2.y + v3.y), y3 = make_float2(x2.x - v3.x, x2.y - v3.y);
    const float2 u2 = turned_back(y2, w1), t3 = turned_back(y3, w1);
    const float2 u3 = make_float2(-t3.y, t3.x);  // conj(-i * w1) = i * conj(w1)
    x0 = make_float2(y0.x + u2.x, y0.y + u2.y);
    x1 = make_float2(y1.x + u3.x, y1.y + u3.y);
    x2 = make_float2(y0.x - u2.x, y0.y - u2.y);
    x3 = make_float2(y1.x - u3.x, y1.y - u3.y);
    settle(x0); settle(x1); settle(x2); settle(x3);
}
__device__ __forceinline__ void butterfly2(float2 &a, float2 &b) {
    const float2 d = make_float2(a.x - b.x, a.y - b.y);
    a = make_float2(a.x + b.x, a.y + b.y);
    b = d;
    settle(a); settle(b);
}

// One block = passes of FPB frames of resolution `res` of one waveform.  lds: 9 complex words per thread.
template <int LOGN, int DIS>
__device__ __forceinline__ void dft_frames(const DftParams &p, const int res, float2 *__restrict__ lds,
                                           float (*err_part)[kMaxThreads / 64]) {
    constexpr int N = 1 << LOGN, HALF = N / 2, TPF = N / 8;
    constexpr bool ODD = LOGN & 1;
    constexpr int PASSES = LOGN / 2;  // the last one included
    const int tid = threadIdx.x, fpb = blockDim.x / TPF;
    const int fl = tid / TPF, t = tid % TPF;  // frame slot in the block, thread within the frame
    float2 *const zf = lds + fl * (N + N / 8);  // this frame's storage; a word of padding every eight
    const int Nw = p.Nw[res], Hs = p.Hs[res];
    const int wave_id = blockIdx.y;
    const int length = p.lengths[wave_id];
    const int Kvalid = frame_count(length, Nw, Hs);
    const float *__restrict__ win = p.window[res];
    const float *__restrict__ src = p.source + (size_t)wave_id * p.max_length;
    const float *__restrict__ tgt = p.target + (size_t)wave_id * p.max_length;
    float *g = p.grad + (size_t)wave_id * p.max_length;
    const bool phase = p.zeta > 0.0f;
    const float inv = 1.0f / (float)((HALF + 1) * Kvalid);
    const float scale = phase ? inv : p.gamma * inv;
    float err = 0.0f, err_ph = 0.0f;

    if ((int)blockIdx.x * fpb >= Kvalid) return;  // the same for every thread
    const int k = blockIdx.x * fpb + fl;
    const bool active = k < Kvalid;
    const int start = active ? k * Hs : 0;

    // frames of up to 64 threads lie inside one wave, whose LDS accesses run in order
    auto exchange = [] {
        if (TPF > 64) {
            __syncthreads();
        } else {
            __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
            __builtin_amdgcn_wave_barrier();
        }
    };
    auto at = [](int pos) { return pos + (pos >> 3); };
    // windowed samples, source in x and target in y; zero outside the window, the waveform and Kvalid
    float2 v[8];  // point m of the pass's butterfly b in v[2m + b]
    float w[8];
#pragma unroll
    for (int e = 0; e < 8; ++e) {
        const int j = t + e * TPF, pos = start + j, from = min(max(pos, 0), length - 1);
        w[e] = win[min(j, Nw - 1)];
        const float s = src[from] * w[e], r = tgt[from] * w[e];
        v[e] = active && j < Nw && pos < length ? make_float2(s, r) : make_float2(0.0f, 0.0f);
    }
    // The table holds exp(-2 pi i k / 2^(s+1)) at 2^s + k for stage s.  A thread's two butterflies share their twiddles but in the
    // first pass; those of the last pass are the same for all threads.
    const float2 *__restrict__ table = p.twiddle[res];
    Twiddles4 tw[PASSES - 1];
    const Twiddles4 tw_second = {table[N / 2 + TPF + t], table[N / 4 + TPF + t]};
#pragma unroll
    for (int c = 0; c + 1 < PASSES; ++c) {
        const int q = N / 4 >> 2 * c, j = t & (q - 1);
        tw[c] = {table[2 * q + j], table[q + j]};
    }
    const Twiddles4 last0 = ODD ? Twiddles4{table[4], table[2]} : Twiddles4{table[2], table[1]}, last1 = {table[5], table[3]};
    // the place of point m of butterfly b (0: t, 1: t + T) of pass c; in the last pass of the point 8t + r, r = 2m + b
    auto place = [&](int c, int b, int m) {
        if (c == PASSES - 1) return 9 * t + 2 * m + b;
        const int q = N / 4 >> 2 * c, i = t + b * TPF;
        return at(i / q * 4 * q + i % q + m * q);
    };
    // The thread that holds the bins N - b of this thread's bins b = bitrev(8t + r), r even, in register 7 - r.  Thread 0, whose
    // bins are the multiples of N/8, holds its own: bin 0 (register 0) and N/2 (1) pair with themselves, register 4 with
    // 7, 2 with 3, 6 with 5.
    constexpr int TLOG = LOGN - 3;
    const unsigned bin_t = __brev((unsigned)t) >> (32 - TLOG);
    const int partner = (int)(__brev((TPF - bin_t) & (TPF - 1)) >> (32 - TLOG));
    auto mirror = [&](int r) { return t == 0 ? (r == 4 ? 7 : r == 2 ? 3 : r == 6 ? 5 : 1) : 9 * partner + 7 - r; };

#pragma unroll
    for (int e = 0; e < 8; ++e) settle(v[e]);
    // from the places of one pass to those of another
    auto move = [&](int from, int to) {
#pragma unroll
        for (int e = 0; e < 8; ++e) zf[place(from, e & 1, e >> 1)] = v[e];
        exchange();
#pragma unroll
        for (int e = 0; e < 8; ++e) v[e] = zf[place(to, e & 1, e >> 1)];
    };
#pragma unroll
    for (int c = 0; c + 1 < PASSES; ++c) {
        butterfly4(v[0], v[2], v[4], v[6], tw[c]);
        butterfly4(v[1], v[3], v[5], v[7], c == 0 ? tw_second : tw[c]);
        move(c, c + 1);
    }
    if (ODD) {
        butterfly4(v[0], v[2], v[4], v[6], last0);
        butterfly4(v[1], v[3], v[5], v[7], last1);
#pragma unroll
        for (int r = 0; r < 8; r += 2) butterfly2(v[r], v[r + 1]);
    } else {
        butterfly4(v[0], v[1], v[2], v[3], last0);
        butterfly4(v[4], v[5], v[6], v[7], last0);
    }

    // Per-bin stage on the pairs (b, N - b).  The bins below N/2 are this thread's even registers, their partners another
    // thread's odd ones: those are put into LDS, and what the pair leaves there is taken back.
    // With the phase term both gradient spectra are weighted here and share the inverse transform (the
    // reference runs a second framing / FFT / inverse FFT / overlap-add for it,
    // layers/DFTErrorPostoutputLayer.cu:1246-1295).
    auto bin = [&](const float2 zb, const float2 zn) {
        // S = (Z[b] + conj(Z[N-b])) / 2,  T = (Z[b] - conj(Z[N-b])) / (2i)
        const float sx = 0.5f * (zb.x + zn.x), sy = 0.5f * (zb.y - zn.y);
        const float tx = 0.5f * (zb.y + zn.y), ty = -0.5f * (zb.x - zn.x);
        float e, gx, gy;
        bin_distance<DIS>(sx, sy, tx, ty, p.log_floor, e, gx, gy);
        if (active) err += e;
        if (phase) {
            float pe, px, py;
            bin_phase(sx, sy, tx, ty, pe, px, py);
            if (active) err_ph += pe;
            gx = p.gamma * gx + p.zeta * px;
            gy = p.gamma * gy + p.zeta * py;
        }
        return make_float2(gx, gy);
    };
#pragma unroll
    for (int r = 1; r < 8; r += 2) zf[9 * t + r] = v[r];
    exchange();
    float2 zn[4];
#pragma unroll
    for (int r = 0; r < 8; r += 2) zn[r / 2] = zf[mirror(r)];
    if (t == 0) {
        zn[0] = v[0];
        v[1] = make_float2(bin(v[1], v[1]).x, 0.0f);
    }
#pragma unroll
    for (int r = 0; r < 8; r += 2) {
        v[r] = bin(v[r], zn[r / 2]);
        settle(v[r]);
        if (t == 0 && r == 0) v[0].y = 0.0f;
        else zf[mirror(r)] = make_float2(v[r].x, -v[r].y);
    }
    exchange();
#pragma unroll
    for (int r = 1; r < 8; r += 2)
        if (t != 0 || r != 1) v[r] = zf[9 * t + r];

    // inverse, unnormalised
    if (ODD) {
#pragma unroll
        for (int r = 0; r < 8; r += 2) butterfly2(v[r], v[r + 1]);
        inverse_butterfly4(v[0], v[2], v[4], v[6], last0);
        inverse_butterfly4(v[1], v[3], v[5], v[7], last1);
    } else {
        inverse_butterfly4(v[0], v[1], v[2], v[3], last0);
        inverse_butterfly4(v[4], v[5], v[6], v[7], last0);
    }
#pragma unroll
    for (int c = PASSES - 2; c >= 0; --c) {
        move(c + 1, c);
        inverse_butterfly4(v[0], v[2], v[4], v[6], tw[c]);
        inverse_butterfly4(v[1], v[3], v[5], v[7], c == 0 ? tw_second : tw[c]);
    }

    // windowed overlap-add; frames at or beyond Kvalid contribute nothing
    if (active) {
#pragma unroll
        for (int e = 0; e < 8; ++e) {
            const int j = t + e * TPF, pos = start + j;
            if (j < Nw && pos < length) atomicAdd(&g[pos], scale * v[e].x * w[e]);
        }
    }

    for (int o = 32; o > 0; o >>= 1) {
        err += __shfl_xor(err, o);
        err_ph += __shfl_xor(err_ph, o);
    }
    if ((tid & 63) == 0) {
        err_part[0][tid >> 6] = err;
        err_part[1][tid >> 6] = err_ph;
    }
    __syncthreads();
    if (tid < 2 && (tid == 0 || phase)) {
        float e = 0.0f;
        for (int q = 0; q < (int)blockDim.x / 64; ++q) e += err_part[tid][q];
        e *= inv;
        if (e != 0.0f) atomicAdd(&p.errors[tid * p.n_waves * p.n_res + wave_id * p.n_res + res], e);
    }
}

// All resolutions of a call in one launch: blockIdx.z selects the resolution, blockIdx.x the group of frames
// (blocks beyond a resolution's last frame leave at once), blockIdx.y the waveform.
template <int DIS>
__global__ __launch_bounds__(kMaxThreads) void dft_loss_kernel(const DftParams p) {
    // sized by the launch for the call's longest transform; every instantiation places its tables at fixed offsets
    extern __shared__ __attribute__((aligned(16))) float2 dft_lds[];
    __shared__ float err_part[2][kMaxThreads / 64];
    const int res = blockIdx.z;
    if ((int)blockIdx.x >= p.nblocks[res]) return;
    switch (p.logn[res]) {
        case 5: dft_frames<5, DIS>(p, res, dft_lds, err_part); break;
        case 6: dft_frames<6, DIS>(p, res, dft_lds, err_part); break;
        case 7: dft_frames<7, DIS>(p, res, dft_lds, err_part); break;
        case 8: dft_frames<8, DIS>(p, res, dft_lds, err_part); break;
        case 9: dft_frames<9, DIS>(p, res, dft_lds, err_part); break;
        case 10: dft_frames<10, DIS>(p, res, dft_lds, err_part); break;
        case 11: dft_frames<11, DIS>(p, res, dft_lds, err_part); break;
        default: dft_frames<12, DIS>(p, res, dft_lds, err_part); break;
    }
}

__global__ void dft_backward_kernel(int max_length, int n_waves, DftParams p, float *__restrict__ prev_errors) {
    const size_t count = (size_t)max_length * n_waves;
    size_t i = (size_t)blockIdx.x * blockDim.x + threadIdx.x;
    const size_t stride = (size_t)gridDim.x * blockDim.x;
    for (; i < count; i += stride) {
        const int w = (int)(i / max_length), t = (int)(i % max_length);
        prev_errors[i] = t < p.lengths[w] ? p.grad[i] : 0.0f;
    }
}

typedef void (*dft_kernel_t)(const DftParams);
dft_kernel_t pick_dft_kernel(int dis_type) {
    switch (dis_type) {
        case 0: return dft_loss_kernel<0>;
        case 1: return dft_loss_kernel<1>;
        case 2: return dft_loss_kernel<2>;
        case 3: return dft_loss_kernel<3>;
        case 4: return dft_loss_kernel<4>;
        case 5: return dft_loss_kernel<5>;
        case 6: return dft_loss_kernel<6>;
        default: return nullptr;
    }
}

}  // namespace
}  // namespace cnt

struct cnt_dft {
    cnt_dft_desc desc;
    int logn[cnt::kMaxRes];
    float2 *twiddle[cnt::kMaxRes];
    float *window[cnt::kMaxRes];
    float *grad;  // max_waves x max_length
    int lengths[cnt::kMaxWavesPerLaunch];
    int n_waves;  // of the last forward
};

extern "C" {

int cnt_dft_destroy(cnt_dft *h) {
    if (!h) return CNT_OK;
    for (int r = 0; r < cnt::kMaxRes; ++r) {
        if (h->twiddle[r]) (void)hipFree(h->twiddle[r]);
        if (h->window[r]) (void)hipFree(h->window[r]);
    }
    if (h->grad) (void)hipFree(h->grad);
    delete h;
    return CNT_OK;
}

int cnt_dft_create(const cnt_dft_desc *desc, cnt_dft **out) {
    using namespace cnt;
    CNT_REQUIRE(desc && out, "dft_create: null argument");
    CNT_REQUIRE(desc->n_res >= 1 && desc->n_res <= kMaxRes, "dft_create: %d resolutions, supported 1..%d", desc->n_res,
                kMaxRes);
    CNT_REQUIRE(desc->max_length > 0 && desc->max_waves >= 1 && desc->max_waves <= kMaxWavesPerLaunch,
                "dft_create: max_length must be positive and max_waves in 1..%d", kMaxWavesPerLaunch);
    // the reference implements the Hann window (default) and the square window, and the amplitude / spectrum
    // distances 0..6; its phase distances are a separate driver and are not built
    CNT_REQUIRE(desc->spec_dis_type >= 0 && desc->spec_dis_type <= 6, "dft_create: specDisType %d outside 0..6",
                desc->spec_dis_type);
    CNT_REQUIRE(desc->zeta >= 0.0f, "dft_create: negative zeta");
    CNT_REQUIRE(desc->zeta == 0.0f || desc->phase_dis_type == 0,
                "dft_create: phaseDisType %d; only 0 (cosine distance) is built", desc->phase_dis_type);
    cnt_dft *h = new (std::nothrow) cnt_dft();
    CNT_REQUIRE(h != nullptr, "dft_create: out of host memory");
    std::memset(h, 0, sizeof(*h));
    h->desc = *desc;
    hipError_t err = hipSuccess;
    for (int r = 0; r < desc->n_res && err == hipSuccess; ++r) {
        const int N = desc->fft_length[r], Nw = desc->frame_length[r], Hs = desc->frame_shift[r];
        int logn = 0;
        while ((1 << logn) < N) ++logn;
        if ((1 << logn) != N || logn < 5 || logn > kMaxLogN || Nw < 2 || Nw > N || Hs < 1) {
            set_error("dft_create: resolution %d has fftLength %d, frameLength %d, frameShift %d; supported: fftLength a "
                      "power of two in 32..4096, 2 <= frameLength <= fftLength, frameShift >= 1", r, N, Nw, Hs);
            cnt_dft_destroy(h);
            return CNT_ERR_ARG;
        }
        h->logn[r] = logn;
        // one run of twiddles per butterfly stage, so that a stage reads consecutive LDS words
        std::vector<float2> tw((size_t)N, make_float2(1.0f, 0.0f));
        for (int half = 1; half < N; half *= 2)
            for (int k2 = 0; k2 < half; ++k2) {
                const double a = -3.14159265358979323846 * k2 / half;
                tw[(size_t)(half + k2)] = make_float2((float)std::cos(a), (float)std::sin(a));
            }
        std::vector<float> win((size_t)Nw);
        for (int j = 0; j < Nw; ++j)
            win[(size_t)j] = desc->window_type[r] == 1 ? 1.0f
                                                       : (float)(0.5 * (1 - std::cos(2.0 * 3.141215 * j / (Nw - 1))));
        err = hipMalloc(reinterpret_cast<void **>(&h->twiddle[r]), tw.size() * sizeof(float2));
        if (err == hipSuccess) err = hipMemcpy(h->twiddle[r], tw.data(), tw.size() * sizeof(float2), hipMemcpyHostToDevice);
        if (err == hipSuccess) err = hipMalloc(reinterpret_cast<void **>(&h->window[r]), win.size() * sizeof(float));
        if (err == hipSuccess) err = hipMemcpy(h->window[r], win.data(), win.size() * sizeof(float), hipMemcpyHostToDevice);
    }
    if (err == hipSuccess)
        err = hipMalloc(reinterpret_cast<void **>(&h->grad), (size_t)desc->max_waves * desc->max_length * sizeof(float));
    if (err != hipSuccess) {
        set_error("dft_create: %s", hipGetErrorString(err));
        cnt_dft_destroy(h);
        return CNT_ERR_HIP;
    }
    *out = h;
    return CNT_OK;
}

static void fill_params(const cnt_dft *h, cnt::DftParams &p) {
    std::memset(&p, 0, sizeof(p));
    p.max_length = h->desc.max_length;
    p.n_waves = h->n_waves;
    p.n_res = h->desc.n_res;
    for (int w = 0; w < h->n_waves; ++w) p.lengths[w] = h->lengths[w];
    p.gamma = h->desc.gamma;
    p.log_floor = h->desc.log_floor;
    p.zeta = h->desc.zeta;
    p.grad = h->grad;
    for (int r = 0; r < h->desc.n_res; ++r) {
        p.logn[r] = h->logn[r];
        p.Nw[r] = h->desc.frame_length[r];
        p.Hs[r] = h->desc.frame_shift[r];
        p.twiddle[r] = h->twiddle[r];
        p.window[r] = h->window[r];
    }
}

int cnt_dft_forward(cnt_dft *h, void *stream_, int n_waves, const int *lengths, const float *source,
                    const float *target, float *errors_dev) {
    using namespace cnt;
    CNT_REQUIRE(h && lengths && source && target && errors_dev, "dft_forward: null argument");
    CNT_REQUIRE(n_waves >= 1 && n_waves <= h->desc.max_waves, "dft_forward: %d waveforms, handle allows 1..%d", n_waves,
                h->desc.max_waves);
    for (int w = 0; w < n_waves; ++w)
        CNT_REQUIRE(lengths[w] >= 1 && lengths[w] <= h->desc.max_length, "dft_forward: length %d of waveform %d outside 1..%d",
                    lengths[w], w, h->desc.max_length);
    hipStream_t stream = static_cast<hipStream_t>(stream_);
    h->n_waves = n_waves;
    for (int w = 0; w < n_waves; ++w) h->lengths[w] = lengths[w];
    CNT_TRY(fill_zero_pair(stream, h->grad, (size_t)n_waves * h->desc.max_length, errors_dev,
                           (size_t)n_waves * h->desc.n_res * (h->desc.zeta > 0.0f ? 2 : 1)));
    int max_len = 0;
    for (int w = 0; w < n_waves; ++w) max_len = lengths[w] > max_len ? lengths[w] : max_len;
    DftParams p;
    fill_params(h, p);
    p.source = source; p.target = target; p.errors = errors_dev;
    // a workgroup transforms eight points per thread, whatever the transforms' length
    int threads = 256, gx = 1;
    for (int r = 0; r < h->desc.n_res; ++r) threads = p.logn[r] > 11 ? kMaxThreads : threads;
    for (int r = 0; r < h->desc.n_res; ++r) {
        const int fpb = threads * 8 >> p.logn[r];
        p.nblocks[r] = (frame_count(max_len, p.Nw[r], p.Hs[r]) + fpb - 1) / fpb;
        gx = std::max(gx, p.nblocks[r]);
    }
    const size_t lds_bytes = (size_t)threads * 9 * sizeof(float2);
    {
        ProfileScope prof(stream, "dft_loss");
        hipLaunchKernelGGL(pick_dft_kernel(h->desc.spec_dis_type), dim3(gx, n_waves, h->desc.n_res), dim3(threads), lds_bytes, stream,
                           p);
        CNT_HIP(hipGetLastError());
    }
    return CNT_OK;
}

int cnt_dft_backward(cnt_dft *h, void *stream_, float *prev_errors) {
    using namespace cnt;
    CNT_REQUIRE(h && prev_errors, "dft_backward: null argument");
    CNT_REQUIRE(h->n_waves > 0, "dft_backward: forward has not been called");
    DftParams p;
    fill_params(h, p);
    const size_t count = (size_t)h->desc.max_length * h->n_waves;
    size_t blocks = (count + 255) / 256;
    if (blocks > 4096) blocks = 4096;
    ProfileScope prof(static_cast<hipStream_t>(stream_), "dft_backward");
    hipLaunchKernelGGL(dft_backward_kernel, dim3((unsigned)blocks), dim3(256), 0, static_cast<hipStream_t>(stream_),
                       h->desc.max_length, h->n_waves, p, prev_errors);
    CNT_HIP(hipGetLastError());
    return CNT_OK;
}

}  // extern "C"
