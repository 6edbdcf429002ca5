// Recursions of small layers (up to 64 cells per direction) inside one workgroup (included by lstm.hip inside its
// anonymous namespace, after lstm_local.hpp).
//
// The recurrent weights of such a layer fit the registers of one compute unit, so a job -- a direction and up to four
// sequences, as in lstm_local.hpp -- needs no exchange between workgroups: no mailbox, no polling, nothing that has to be
// resident at the same time, and jobs may run in any number and order.  What bounds a step is the chain barrier -> LDS
// read -> 16*NW v_mfma_f32_4x4x1 -> cell update -> LDS write -> barrier.
//
// NW = ceil(cells / 16) cell waves.  A wave owns sixteen cells for the job's four sequences, and a lane owns ONE (cell,
// sequence) for the whole recursion: the matrix instructions leave the lane's own sums in its accumulator, so gates,
// cell state, deltas and carried terms never leave registers, and a step has one LDS-only barrier.
// A block of the matrix instruction holds four cells of one gate for the four sequences; lane swaps afterwards transpose
// the gates into registers (forward) or add the gates' shares (backward) and leave each lane with its own element.
// Two more waves do all global accesses: one requests a step's inputs kSoloAhead steps ahead and hands them over through LDS,
// the other stores the step before's results.  They take four neighbouring cells per lane in one access, so that an array
// takes one access per step instead of one per cell wave: an access occupies the compute unit's address path for sixteen
// clocks whatever its width, and twelve to fourteen of each of four waves, issued between the LDS reads and the matrix
// instructions, held those up by 700 clocks a step (64 / 48 / 32 / 16 cells, us per step forward 0.77 /
// 0.65 / 0.54 / 0.44, backward 0.74 / 0.63 / 0.52 / 0.40; now 0.60 / 0.53 / 0.47 / 0.37 and 0.65 / 0.50 / 0.50 / 0.35).
// Global accesses are buffer accesses whose range check drops what a lane or a step has no part in: every step issues
// the same number of loads and stores and no branch, so that the compiler's wait for the loads of a step does not wait for
// those of later ones.

constexpr int kSoloCells = 64;
constexpr int kSoloAhead = 4;   // even: the step parity of every unrolled step is a constant
constexpr int solo_threads(int NW) { return (NW + 2) * 64; }
// The sequences are dealt to the groups as evenly as possible, in order.
struct SoloJob { int dir, seq0, nseq; };
__device__ __forceinline__ SoloJob solo_job(const ChainParams &p, int job) {
    const int dir = job / p.groups, q = job % p.groups;
    const int each = p.S / p.groups, more = p.S % p.groups;
    return SoloJob{dir, q * each + min(q, more), each + (q < more ? 1 : 0)};
}
constexpr unsigned kSoloNowhere = 0x7FFFFFFCu;  // an offset past every array: loads give zero, stores go nowhere

__device__ __forceinline__ __amdgpu_buffer_rsrc_t solo_array(const void *base, size_t bytes) {
    return __builtin_amdgcn_make_buffer_rsrc(const_cast<void *>(base), 0, (int)bytes, 0x00020000);
}
__device__ __forceinline__ float solo_load(__amdgpu_buffer_rsrc_t r, unsigned off, int at) {
    return __builtin_bit_cast(float, __builtin_amdgcn_raw_buffer_load_b32(r, (int)off, at, 0));
}
__device__ __forceinline__ void solo_store(__amdgpu_buffer_rsrc_t r, unsigned off, int at, float v) {
    __builtin_amdgcn_raw_buffer_store_b32(__builtin_bit_cast(unsigned, v), r, (int)off, at, 0);
}
// How the helper waves take four neighbouring cells of a sequence per lane: in vectors of a layer whose cells are a multiple of four
// (kAligned), in vectors of which the last begins at the fourth cell from the end (kOverlapping), and one by one below
// four cells (kSingle).
enum { kSingle = 0, kOverlapping = 1, kAligned = 2 };
typedef float f32x4a4 __attribute__((ext_vector_type(4), aligned(4)));
template <int CELLS>
__device__ __forceinline__ f32x4 lds_load4(const float *p) {
    if (CELLS == kAligned) return *reinterpret_cast<const f32x4 *>(p);
    return *reinterpret_cast<const f32x4a4 *>(p);
}
template <int CELLS>
__device__ __forceinline__ void lds_store4(float *p, const f32x4 &v) {
    if (CELLS == kAligned) *reinterpret_cast<f32x4 *>(p) = v;
    else *reinterpret_cast<f32x4a4 *>(p) = v;
}
// off = the first cell's byte offset in a time step, or nowhere; `last` = how many of the four exist (kSingle)
template <int CELLS>
__device__ __forceinline__ f32x4 solo_load4(__amdgpu_buffer_rsrc_t r, unsigned off, int last, int at) {
    if (CELLS != kSingle) return __builtin_bit_cast(f32x4, __builtin_amdgcn_raw_buffer_load_b128(r, (int)off, at, 0));
    f32x4 v;
#pragma unroll
    for (int q = 0; q < 4; ++q) v[q] = solo_load(r, q < last ? off + 4u * q : kSoloNowhere, at);
    return v;
}
template <int CELLS>
__device__ __forceinline__ void solo_store4(__amdgpu_buffer_rsrc_t r, unsigned off, int last, int at, const f32x4 &v) {
    if (CELLS != kSingle) {
        __builtin_amdgcn_raw_buffer_store_b128(__builtin_bit_cast(u32x4, v), r, (int)off, at, 0);
        return;
    }
#pragma unroll
    for (int q = 0; q < 4; ++q) solo_store(r, q < last ? off + 4u * q : kSoloNowhere, at, v[q]);
}
// One step's recurrent sums.  The step's LDS values are the A operand, one 16-byte read per lane for 4 * BLOCKS of the K
// source values: v_mfma's operand broadcast (2^CBSZ neighbouring blocks take block I of the operand) hands each of them
// to all blocks that need it, where a broadcast read from LDS would move every value sixteen times and take longer than
// the matrix instructions.  wreg[16 * x + 4 * I + r] belongs to source value 4 * BLOCKS * x + 4 * I + r; the four values
// of a read feed four accumulator chains.
template <int CBSZ, int BLOCKS, int K, int... I>
__device__ __forceinline__ void solo_piece(const float (&wreg)[K], int base, const f32x4 &v, f32x4 (&acc)[4],
                                           std::integer_sequence<int, I...>) {
    auto one = [&](auto block) __attribute__((always_inline)) {
        constexpr int b = decltype(block)::value;
#pragma unroll
        for (int r = 0; r < 4; ++r)
            acc[r] = __builtin_amdgcn_mfma_f32_4x4x1f32(v[r], wreg[base + 4 * b + r], acc[r], CBSZ, b, 0);
    };
    (one(std::integral_constant<int, I>{}), ...);
}
template <int CBSZ, int K>
__device__ __forceinline__ f32x4 solo_product(const float (&wreg)[K], const float *mine) {
    constexpr int BLOCKS = 1 << CBSZ, SPAN = 4 * BLOCKS, NX = (K + SPAN - 1) / SPAN;
    f32x4 v[NX];
#pragma unroll
    for (int x = 0; x < NX; ++x) v[x] = *reinterpret_cast<const f32x4 *>(mine + SPAN * x);
    f32x4 acc[4] = {{0, 0, 0, 0}, {0, 0, 0, 0}, {0, 0, 0, 0}, {0, 0, 0, 0}};
#pragma unroll
    for (int x = 0; x < K / SPAN; ++x)
        solo_piece<CBSZ, BLOCKS, K>(wreg, SPAN * x, v[x], acc, std::make_integer_sequence<int, BLOCKS>{});
    if (K % SPAN) solo_piece<CBSZ, BLOCKS, K>(wreg, K / SPAN * SPAN, v[NX - 1], acc, std::make_integer_sequence<int, K % SPAN / 4>{});
    return (acc[0] + acc[1]) + (acc[2] + acc[3]);
}
// exchanges the upper half of the wave in a with the lower half in b / odd with even rows of sixteen lanes
__device__ __forceinline__ void swap_halves(float &a, float &b) {
    const auto r = __builtin_amdgcn_permlane32_swap(__builtin_bit_cast(unsigned, a), __builtin_bit_cast(unsigned, b), false, false);
    a = __builtin_bit_cast(float, (unsigned)r[0]); b = __builtin_bit_cast(float, (unsigned)r[1]);
}
__device__ __forceinline__ void swap_rows(float &a, float &b) {
    const auto r = __builtin_amdgcn_permlane16_swap(__builtin_bit_cast(unsigned, a), __builtin_bit_cast(unsigned, b), false, false);
    a = __builtin_bit_cast(float, (unsigned)r[0]); b = __builtin_bit_cast(float, (unsigned)r[1]);
}

template <int NW, int CELLS>
__global__ __launch_bounds__(solo_threads(NW)) __attribute__((amdgpu_waves_per_eu(2))) void lstm_forward_solo(const ChainParams p) {
    constexpr int K = 16 * NW;      // cells, padded
    constexpr int PITCH = (K + 63) / 64 * 64 + 4;
    constexpr int ROW = 80;         // pitch of a sequence's values that the helper waves move: four rows on different banks
    __shared__ __attribute__((aligned(16))) float hs[2][kLocalSeqs][PITCH];
    __shared__ __attribute__((aligned(16))) float inputs[2][4][kLocalSeqs][ROW];   // input projections of the step, by gate
    __shared__ __attribute__((aligned(16))) float results[2][6][kLocalSeqs][ROW];  // ni, ig, fg, og, cell state, output
    __shared__ unsigned pads[2][kLocalSeqs];

    const int H = p.H, S = p.S, T = p.T;
    const SoloJob part = solo_job(p, blockIdx.x);
    const int dir = part.dir;
    const DirPtrs &D = p.d[dir];
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    const int j = lane >> 4, s = part.seq0 + j;
    const int steps = (T + kSoloAhead - 1) / kSoloAhead * kSoloAhead;
    const int row = S * H * 4, out_row = S * p.L * 4;  // bytes of a time step
    const size_t bytes = (size_t)row * T;
    auto t_of = [&](int step) { return dir ? (T - 1 - step) : step; };

    if (wave >= NW) {
        // (lanes past the last cells move those once more: no branch, into which the compiler would sink the loads)
        const int cells = min(4 * (lane & 15), max(H - 4, 0)), last = H - cells;
        const bool valid = j < part.nseq;
        const unsigned off = valid ? (unsigned)(s * H + cells) * 4u : kSoloNowhere;
        const __amdgpu_buffer_rsrc_t r_ni = solo_array(D.ni, bytes), r_ig = solo_array(D.ig, bytes), r_fg = solo_array(D.fg, bytes),
                                     r_og = solo_array(D.og, bytes);
        if (wave == NW) {
            // -------------------------------------------------------------- load wave
            const __amdgpu_buffer_rsrc_t r_pat = solo_array(p.pat, (size_t)S * T);
            const unsigned pat_off = j < part.nseq ? (unsigned)s : kSoloNowhere;
            struct StepIn { f32x4 a[4]; unsigned pat; };
            auto request = [&](int step, StepIn &v) __attribute__((always_inline)) {
                const bool on = step < T;
                const int t = on ? t_of(step) : 0;
                const unsigned o = on ? off : kSoloNowhere;
                v.a[0] = solo_load4<CELLS>(r_ni, o, last, t * row);
                v.a[1] = solo_load4<CELLS>(r_ig, o, last, t * row);
                v.a[2] = solo_load4<CELLS>(r_fg, o, last, t * row);
                v.a[3] = solo_load4<CELLS>(r_og, o, last, t * row);
                v.pat = __builtin_amdgcn_raw_buffer_load_b8(r_pat, (int)pat_off, t * S, 0);
            };
            auto put = [&](int step, int parity, const StepIn &v) __attribute__((always_inline)) {
#pragma unroll
                for (int g = 0; g < 4; ++g) lds_store4<CELLS>(&inputs[parity][g][j][cells], v.a[g]);
                pads[parity][j] = step < T && t_of(step) >= p.Tmin && (v.pat & 0xFFu) == 0 ? 1u : 0u;
            };
            StepIn in[kSoloAhead];
#pragma unroll
            for (int i = 0; i < kSoloAhead; ++i) request(i, in[i]);
            put(0, 0, in[0]);
            request(kSoloAhead, in[0]);
            __syncthreads();
            for (int step = 0; step < steps; step += kSoloAhead) {
#pragma unroll
                for (int i = 0; i < kSoloAhead; ++i) {
                    StepIn &next = in[(i + 1) % kSoloAhead];
                    put(step + i + 1, (i + 1) & 1, next);
                    request(step + i + 1 + kSoloAhead, next);
                    lds_barrier();
                }
            }
            return;
        }
        // ------------------------------------------------------------------ store wave
        const __amdgpu_buffer_rsrc_t r_c = solo_array(D.c, bytes), r_h = solo_array(D.h, bytes), r_out = solo_array(p.out, (size_t)out_row * T);
        const unsigned out_off = valid ? (unsigned)(s * p.L + dir * H + cells) * 4u : kSoloNowhere;
        bool pad = false;  // of the step whose results are stored
        auto store = [&](int step, int parity) __attribute__((always_inline)) {
            const bool on = step >= 0 && step < T;
            const int t = on ? t_of(step) : 0;
            // a padding slot keeps its input projections, and its cell state unless the direction is the time-reversed one
            // (the reference clears it there)
            const unsigned gate_off = on && !pad ? off : kSoloNowhere, c_off = on && (!pad || dir) ? off : kSoloNowhere;
            auto value = [&](int k) { return lds_load4<CELLS>(&results[parity][k][j][cells]); };
            solo_store4<CELLS>(r_ni, gate_off, last, t * row, value(0));
            solo_store4<CELLS>(r_ig, gate_off, last, t * row, value(1));
            solo_store4<CELLS>(r_fg, gate_off, last, t * row, value(2));
            solo_store4<CELLS>(r_og, gate_off, last, t * row, value(3));
            solo_store4<CELLS>(r_c, c_off, last, t * row, value(4));
            const f32x4 h = value(5);
            solo_store4<CELLS>(r_h, on ? off : kSoloNowhere, last, t * row, h);
            solo_store4<CELLS>(r_out, on ? out_off : kSoloNowhere, last, t * out_row, h);
        };
        __syncthreads();
        for (int step = 0; step < steps; ++step) {
            store(step - 1, (step + 1) & 1);
            pad = pads[step & 1][j] != 0;
            lds_barrier();
        }
        store(steps - 1, (steps + 1) & 1);
        return;
    }

    // ---------------------------------------------------------------------- cell waves
    __builtin_amdgcn_s_setprio(3);  // before the helper wave on the same SIMD
    const int cell = 16 * wave + (lane & 15);
    const bool valid = cell < H && j < part.nseq;
    // B operand: lane = 16 * gate + cell of the wave
    float wreg[K];
    {
        const float *wg = D.w_int + (size_t)(lane >> 4) * p.L * H + (size_t)(cell < H ? cell : 0) * H;
        if constexpr (CELLS == kSingle) {
#pragma unroll
            for (int k = 0; k < K; ++k) wreg[k] = cell < H && k < H ? wg[k] : 0.0f;
        } else {
            load_weight_row(wg, cell < H, 0, H, wreg);
        }
    }
    f32x4 bias = {0, 0, 0, 0};
    float p_ig = 0, p_fg = 0, p_og = 0;
    if (valid) {
#pragma unroll
        for (int g = 0; g < 4; ++g) bias[g] = p.bias * D.b[g][cell];
        p_ig = D.peep[0][cell]; p_fg = D.peep[1][cell]; p_og = D.peep[2][cell];
    }
    for (int i = threadIdx.x; i < 2 * kLocalSeqs * PITCH; i += 64 * NW) (&hs[0][0][0])[i] = 0.0f;
    // cells past the layer's (zero weights) start from zeros; nothing else writes there
    if (cell >= H)
#pragma unroll
        for (int i = 0; i < 8; ++i) inputs[i / 4][i % 4][j][cell] = 0.0f;

    float c_prev = 0.0f;
    auto run = [&](int parity) __attribute__((always_inline)) {
        f32x4 start = bias;
#pragma unroll
        for (int g = 0; g < 4; ++g) start[g] += inputs[parity][g][j][cell];
        const bool padding = pads[parity][j] != 0;
        // A operand: lane = 4 * (four source cells) + sequence; the sums come out as lane = 16 * gate + cell with one
        // sequence per register and are transposed to lane = 16 * sequence + cell with one gate per register
        f32x4 x = solo_product<4, K>(wreg, &hs[parity][lane & 3][lane & ~3]);
        {
            float x0 = x[0], x1 = x[1], x2 = x[2], x3 = x[3];
            swap_halves(x0, x2); swap_halves(x1, x3);
            swap_rows(x0, x1); swap_rows(x2, x3);
            x = f32x4{x0, x1, x2, x3} + start;
        }
        const float ni = tanh_quick(x[0]), ig = logistic_quick(x[1] + c_prev * p_ig), fg = logistic_quick(x[2] + c_prev * p_fg);
        float c = ni * ig + c_prev * fg;
        const float og = logistic_quick(x[3] + c * p_og);
        float hval = tanh_quick(c) * og;
        hval = padding ? 0.0f : hval;
        hs[parity ^ 1][j][cell] = hval;
        c = padding ? (dir ? 0.0f : c_prev) : c;
        c_prev = c;
        float *const to = &results[parity][0][j][cell];
        constexpr int NEXT = kLocalSeqs * ROW;
        to[0] = ni; to[NEXT] = ig; to[2 * NEXT] = fg; to[3 * NEXT] = og; to[4 * NEXT] = c; to[5 * NEXT] = hval;
        lds_barrier();
    };
    __syncthreads();
    for (int step = 0; step < steps; step += 2) {
        run(0);
        run(1);
    }
}

template <int NW, int CELLS>
__global__ __launch_bounds__(solo_threads(NW)) __attribute__((amdgpu_waves_per_eu(2))) void lstm_backward_solo(const ChainParams p) {
    constexpr int K = 16 * NW;
    constexpr int PITCH = K + 4;          // one gate's deltas of a sequence; 4 * PITCH per sequence keeps the sixteen
                                          // (gate, sequence) pieces of a read on different banks
    constexpr int ROW = 80;
    enum { I_E = 0, I_NI, I_IG, I_FG, I_OG, I_DOG, I_C, I_CNEXT, NK };
    // what a cell wave needs of a step: the error, the coefficients of e in d_og and in the cell error, the stored d_og, the
    // coefficients of the cell error in the other deltas, the forget gate's activation
    enum { K_E = 0, K_OG, K_CE, K_DOG, K_NI, K_IG, K_FG, K_FGACT };
    // ... which the load wave computes where it has a SIMD to itself, beside three cell waves, and the cell waves otherwise (load / cell
    // waves, us per step at 64 / 48 / 16 cells 0.69 / 0.65, 0.50 / 0.59, 0.44 / 0.35).
    // Beyond the last step the cell state reads as zero, which is what makes the forget gate's last delta zero.  (Fused
    // multiply-adds are written out here and below: the copies of a body, for even and odd steps, have to round alike, or a
    // pass run as ranges of steps would depend on where it is cut.)
    constexpr bool LOADER = NW == 3;
    auto coefficients = [](const float (&in)[NK], float (&k)[NK]) __attribute__((always_inline)) {
        const float tc = tanh_act(in[I_C]);
        k[K_E] = in[I_E]; k[K_DOG] = in[I_DOG]; k[K_FGACT] = in[I_FG];
        k[K_OG] = logistic_deriv(in[I_OG]) * tc;
        k[K_CE] = in[I_OG] * __builtin_fmaf(-tc, tc, 1.0f);
        k[K_NI] = in[I_IG] * __builtin_fmaf(-in[I_NI], in[I_NI], 1.0f);
        k[K_IG] = logistic_deriv(in[I_IG]) * in[I_NI];
        k[K_FG] = logistic_deriv(in[I_FG]) * in[I_CNEXT];
    };
    __shared__ __attribute__((aligned(16))) float ds[2][kLocalSeqs][4][PITCH];
    __shared__ __attribute__((aligned(16))) float coef[2][NK][kLocalSeqs][ROW];
    __shared__ __attribute__((aligned(16))) float results[2][6][kLocalSeqs][ROW];  // d_ni, d_ig, d_fg, d_og, cell error, output error
    __shared__ __attribute__((aligned(16))) float cells_ahead[4][kLocalSeqs][ROW];  // cell states of four steps, for the store wave's sums
    __shared__ unsigned pads[2][kLocalSeqs];

    const int H = p.H, S = p.S, T = p.T;
    const SoloJob part = solo_job(p, blockIdx.x);
    const int dir = part.dir;
    const DirPtrs &D = p.d[dir];
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    const int j = lane >> 4, s = part.seq0 + j;
    const int row = S * H * 4, out_row = S * p.L * 4;  // bytes of a time step
    const size_t bytes = (size_t)row * T;
    const int sb = p.step_begin, se = p.step_end;
    const int steps = (se - sb + kSoloAhead - 1) / kSoloAhead * kSoloAhead;
    auto t_of = [&](int step) { return dir ? step : (T - 1 - step); };

    if (wave >= NW) {
        // (lanes past the last cells move those once more: no branch, into which the compiler would sink the loads)
        const int cells = min(4 * (lane & 15), max(H - 4, 0)), last = H - cells;
        const bool valid = j < part.nseq;
        const unsigned off = valid ? (unsigned)(s * H + cells) * 4u : kSoloNowhere;
        const __amdgpu_buffer_rsrc_t r_dog = solo_array(D.dog, bytes);
        if (wave == NW) {
            // -------------------------------------------------------------- load wave
            const __amdgpu_buffer_rsrc_t r_e = solo_array(p.outerr, (size_t)out_row * T), r_pat = solo_array(p.pat, (size_t)S * T),
                                         r_ni = solo_array(D.ni, bytes), r_ig = solo_array(D.ig, bytes), r_fg = solo_array(D.fg, bytes),
                                         r_og = solo_array(D.og, bytes), r_c = solo_array(D.c, bytes);
            const unsigned out_off = valid ? (unsigned)(s * p.L + dir * H + cells) * 4u : kSoloNowhere;
            const unsigned pat_off = j < part.nseq ? (unsigned)s : kSoloNowhere;
            struct StepIn { f32x4 v[NK]; unsigned pat; };
            auto request = [&](int step, StepIn &x) __attribute__((always_inline)) {
                const bool on = step < T;
                const int t = on ? t_of(step) : 0;
                const unsigned o = on ? off : kSoloNowhere;
                x.v[I_E] = solo_load4<CELLS>(r_e, on ? out_off : kSoloNowhere, last, t * out_row);
                x.v[I_NI] = solo_load4<CELLS>(r_ni, o, last, t * row);
                x.v[I_IG] = solo_load4<CELLS>(r_ig, o, last, t * row);
                x.v[I_FG] = solo_load4<CELLS>(r_fg, o, last, t * row);
                x.v[I_OG] = solo_load4<CELLS>(r_og, o, last, t * row);
                x.v[I_DOG] = solo_load4<CELLS>(r_dog, o, last, t * row);
                x.v[I_C] = solo_load4<CELLS>(r_c, o, last, t * row);
                x.v[I_CNEXT] = solo_load4<CELLS>(r_c, step + 1 < T ? off : kSoloNowhere, last, (step + 1 < T ? t_of(step + 1) : 0) * row);
                x.pat = __builtin_amdgcn_raw_buffer_load_b8(r_pat, (int)pat_off, t * S, 0);
            };
            auto put = [&](int step, int i, const StepIn &x) __attribute__((always_inline)) {  // i: the launch's step, of kSoloAhead
                const int parity = i & 1;
                f32x4 v[NK];
#pragma unroll
                for (int q = 0; q < 4; ++q) {
                    float in[NK], k[NK];
#pragma unroll
                    for (int i = 0; i < NK; ++i) in[i] = x.v[i][q];
                    if (LOADER) coefficients(in, k);
#pragma unroll
                    for (int i = 0; i < NK; ++i) v[i][q] = LOADER ? k[i] : in[i];
                }
#pragma unroll
                for (int n = 0; n < NK; ++n) lds_store4<CELLS>(&coef[parity][n][j][cells], v[n]);
                lds_store4<CELLS>(&cells_ahead[i & 3][j][cells], x.v[I_C]);
                pads[parity][j] = step < T && t_of(step) >= p.Tmin && (x.pat & 0xFFu) == 0 ? 1u : 0u;
            };
            StepIn in[kSoloAhead];
#pragma unroll
            for (int i = 0; i < kSoloAhead; ++i) request(sb + i, in[i]);
            put(sb, 0, in[0]);
            request(sb + kSoloAhead, in[0]);
            __syncthreads();
            for (int step = 0; step < steps; step += kSoloAhead) {
#pragma unroll
                for (int i = 1; i <= kSoloAhead; ++i) {
                    StepIn &now = in[i % kSoloAhead];
                    put(sb + step + i, i, now);
                    request(sb + step + i + kSoloAhead, now);
                    lds_barrier();
                }
            }
            return;
        }
        // ------------------------------------------------------------------ store wave
        const __amdgpu_buffer_rsrc_t r_dni = solo_array(D.dni, bytes), r_dig = solo_array(D.dig, bytes), r_dfg = solo_array(D.dfg, bytes),
                                     r_ce = solo_array(D.cerr, bytes), r_herr = solo_array(p.herr_out ? p.herr_out : D.herr, bytes);
        double sums[kSmallSums][4] = {};
        auto store = [&](int step, int parity) __attribute__((always_inline)) {
            const bool on = step >= 0 && sb + step < se;
            const int t = on ? t_of(sb + step) : 0;
            const unsigned o = on ? off : kSoloNowhere;
            auto value = [&](int k) { return lds_load4<CELLS>(&results[parity][k][j][cells]); };
            const f32x4 d_ni = value(0), d_ig = value(1), d_fg = value(2), d_og = value(3);
            solo_store4<CELLS>(r_dni, o, last, t * row, d_ni);
            solo_store4<CELLS>(r_dig, o, last, t * row, d_ig);
            solo_store4<CELLS>(r_dfg, o, last, t * row, d_fg);
            solo_store4<CELLS>(r_dog, o, last, t * row, d_og);
            solo_store4<CELLS>(r_ce, o, last, t * row, value(4));
            solo_store4<CELLS>(r_herr, o, last, t * row, value(5));
            if (!p.sum_bias || !on) return;
            // the load wave is two steps ahead of this one; the last step has no earlier state, and a zero in its place would be NaN with a
            // delta that is not finite
            const bool has_earlier = sb + step + 1 < se;
            const f32x4 c = lds_load4<CELLS>(&cells_ahead[step & 3][j][cells]), earlier = lds_load4<CELLS>(&cells_ahead[(step + 1) & 3][j][cells]);
#pragma unroll
            for (int q = 0; q < 4; ++q) {
                const double ig = d_ig[q], fg = d_fg[q], og = d_og[q], before = earlier[q];
                sums[0][q] += (double)d_ni[q]; sums[1][q] += ig; sums[2][q] += fg; sums[3][q] += og;
                sums[6][q] += (double)c[q] * og;
                if (has_earlier) { sums[4][q] += before * ig; sums[5][q] += before * fg; }
            }
        };
        __syncthreads();
        for (int step = 0; step < steps; ++step) {
            store(step - 1, (step + 1) & 1);
            lds_barrier();
        }
        store(steps - 1, (steps + 1) & 1);
        if (p.sum_bias) {
#pragma unroll
            for (int k = 0; k < kSmallSums; ++k)
#pragma unroll
                for (int q = 0; q < 4; ++q) {
                    float v = valid ? (float)sums[k][q] : 0.0f;
                    v += __shfl_xor(v, 16);
                    v += __shfl_xor(v, 32);
                    // (of cells that two lanes take both write the same)
                    if (j == 0 && q < last) put_sum(p, dir, (int)blockIdx.x % p.groups, k, cells + q, v);
                }
        }
        return;
    }

    // ---------------------------------------------------------------------- cell waves
    __builtin_amdgcn_s_setprio(3);  // before the helper wave on the same SIMD
    const int cell = 16 * wave + (lane & 15);
    const bool valid = cell < H && j < part.nseq;
    // B operand: lane = 16 * gate + receiving cell of the wave
    float wreg[K];
    {
        const float *wg = D.w_int + (size_t)(lane >> 4) * p.L * H + cell;
#pragma unroll
        for (int k = 0; k < K; ++k) wreg[k] = cell < H && k < H ? wg[(size_t)k * H] : 0.0f;
    }
    float p_ig = 0, p_fg = 0, p_og = 0;
    if (valid) { p_ig = D.peep[0][cell]; p_fg = D.peep[1][cell]; p_og = D.peep[2][cell]; }
    float fg_later = 0, cerr_later = 0, dig_later = 0, dfg_later = 0;
    float (*const first)[PITCH] = ds[0][j];
    if (sb > 0 && valid) {
        // a launch that starts in the middle: what the step before carried over stands in the state arrays
        const size_t gi = (size_t)t_of(sb - 1) * S * H + (size_t)s * H + cell;
        fg_later = D.fg[gi]; cerr_later = D.cerr[gi]; dig_later = D.dig[gi]; dfg_later = D.dfg[gi];
        first[0][cell] = D.dni[gi]; first[1][cell] = dig_later; first[2][cell] = dfg_later; first[3][cell] = D.dog[gi];
    } else {
        first[0][cell] = 0.0f; first[1][cell] = 0.0f; first[2][cell] = 0.0f; first[3][cell] = 0.0f;
    }

    // cells past the layer's (zero weights) start from zeros; nothing else writes there
    if (cell >= H)
#pragma unroll
        for (int i = 0; i < 2 * NK; ++i) coef[i / NK][i % NK][j][cell] = 0.0f;

    auto run = [&](int parity) __attribute__((always_inline)) {
        float in[NK], k[NK];
#pragma unroll
        for (int i = 0; i < NK; ++i) in[i] = coef[parity][i][j][cell];
        if (!LOADER) coefficients(in, k);
#pragma unroll
        for (int i = 0; i < NK; ++i) k[i] = LOADER ? in[i] : k[i];
        const bool padding = pads[parity][j] != 0;
        const float carry = __builtin_fmaf(fg_later, cerr_later, __builtin_fmaf(p_ig, dig_later, p_fg * dfg_later));
        // A operand: lane = 16 * gate + 4 * (four source cells) + sequence; the sums come out as lane = 16 * gate + cell
        // with one sequence per register: the gates' shares meet in the lane of their sequence
        f32x4 x = solo_product<2, K>(wreg, &ds[parity][lane & 3][lane >> 4][lane & 12]);
        float e = k[K_E];
        {
            float x0 = x[0], x1 = x[1], x2 = x[2], x3 = x[3];
            swap_halves(x0, x2); swap_halves(x1, x3);
            float even = x0 + x2, odd = x1 + x3;
            swap_rows(even, odd);
            e += even + odd;
        }
        const float d_og = __builtin_fmaf(k[K_OG], e, k[K_DOG]);
        float ce = __builtin_fmaf(k[K_CE], e, p_og * d_og) + carry;
        float s_ni = clip1(k[K_NI] * ce), s_ig = clip1(k[K_IG] * ce), s_fg = clip1(k[K_FG] * ce), s_og = clip1(d_og);
        s_ni = padding ? 0.0f : s_ni; s_ig = padding ? 0.0f : s_ig; s_fg = padding ? 0.0f : s_fg; s_og = padding ? 0.0f : s_og;
        ce = padding ? 0.0f : ce;
        float (*d)[PITCH] = ds[parity ^ 1][j];
        d[0][cell] = s_ni; d[1][cell] = s_ig; d[2][cell] = s_fg; d[3][cell] = s_og;
        fg_later = k[K_FGACT]; cerr_later = ce; dig_later = s_ig; dfg_later = s_fg;
        float *const to = &results[parity][0][j][cell];
        constexpr int NEXT = kLocalSeqs * ROW;
        to[0] = s_ni; to[NEXT] = s_ig; to[2 * NEXT] = s_fg; to[3 * NEXT] = s_og; to[4 * NEXT] = ce; to[5 * NEXT] = e;
        lds_barrier();
    };
    __syncthreads();
    for (int step = 0; step < steps; step += 2) {
        run(0);
        run(1);
    }
}
