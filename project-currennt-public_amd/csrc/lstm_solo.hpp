// Recursions of small layers (up to 64 cells per direction) inside one workgroup (included by lstm.hip inside its
// anonymous namespace, after lstm_local.hpp).
//
// The recurrent weights of such a layer fit the registers of one compute unit, so a job -- a direction and up to four
// sequences, as in lstm_local.hpp -- needs no exchange between workgroups: no mailbox, no polling, nothing that has to be
// resident at the same time, and jobs may run in any number and order.  What bounds a step is the chain barrier -> LDS
// read -> 16*NW v_mfma_f32_4x4x1 -> cell update -> LDS write -> barrier.
//
// NW = ceil(cells / 16) waves.  A wave owns sixteen cells for the job's four sequences, and a lane owns ONE (cell,
// sequence) for the whole recursion: the matrix instructions leave the lane's own sums in its accumulator, so gates,
// cell state, deltas and carried terms never leave registers, and a step has one LDS-only barrier.
// A block of the matrix instruction holds four cells of one gate for the four sequences; lane swaps afterwards transpose
// the gates into registers (forward) or add the gates' shares (backward) and leave each lane with its own element.
// Global accesses are buffer accesses whose range check drops what a lane or a step has no part in: every step issues
// the same number of loads and stores and no branch, so that the compiler's wait for the loads of a step, requested
// kSoloAhead steps earlier, does not wait for the stores issued since.

constexpr int kSoloCells = 64;
constexpr int kSoloAhead = 4;   // even: the step parity of every unrolled step is a constant
constexpr int solo_threads(int NW) { return NW * 64; }
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
// One step's recurrent sums.  The step's LDS values are the A operand, one 16-byte read per lane for 4 * BLOCKS of the K
// source values: v_mfma's operand broadcast (2^CBSZ neighbouring blocks take block I of the operand) hands each of them
// to all blocks that need it, where a broadcast read from LDS would move every value sixteen times and take longer than
// the matrix instructions.  wreg[16 * x + 4 * I + r] belongs to source value 4 * BLOCKS * x + 4 * I + r; the four values
// of a read feed four accumulator chains.  `meanwhile` runs while the reads are under way.
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
template <int CBSZ, int K, class F>
__device__ __forceinline__ f32x4 solo_product(const float (&wreg)[K], const float *mine, F meanwhile) {
    constexpr int BLOCKS = 1 << CBSZ, SPAN = 4 * BLOCKS, NX = (K + SPAN - 1) / SPAN;
    f32x4 v[NX];
#pragma unroll
    for (int x = 0; x < NX; ++x) v[x] = *reinterpret_cast<const f32x4 *>(mine + SPAN * x);
    __builtin_amdgcn_sched_barrier(0);
    meanwhile();
    __builtin_amdgcn_sched_barrier(0);
    f32x4 acc[4] = {{0, 0, 0, 0}, {0, 0, 0, 0}, {0, 0, 0, 0}, {0, 0, 0, 0}};
#pragma unroll
    for (int x = 0; x < K / SPAN; ++x)
        solo_piece<CBSZ, BLOCKS, K>(wreg, SPAN * x, v[x], acc, std::make_integer_sequence<int, BLOCKS>{});
    if (K % SPAN) solo_piece<CBSZ, BLOCKS, K>(wreg, K / SPAN * SPAN, v[NX - 1], acc, std::make_integer_sequence<int, K % SPAN / 4>{});
    // a wave's matrix instructions of this size issue every sixteen clocks: what the caller computes beside them fits between
#pragma unroll
    for (int i = 0; i < K; ++i) {
        __builtin_amdgcn_sched_group_barrier(0x8, 1, 0);
        __builtin_amdgcn_sched_group_barrier(0x2, 2, 0);
    }
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

template <int NW>
__global__ __launch_bounds__(solo_threads(NW)) __attribute__((amdgpu_waves_per_eu(2))) void lstm_forward_solo(const ChainParams p) {
    constexpr int K = 16 * NW;      // cells, padded
    constexpr int PITCH = (K + 63) / 64 * 64 + 4;
    __shared__ __attribute__((aligned(16))) float hs[2][kLocalSeqs][PITCH];

    const int H = p.H, S = p.S, T = p.T;
    const LocalJob part = local_job(p, blockIdx.x);
    const int dir = part.dir;
    const DirPtrs &D = p.d[dir];
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    const int cell = 16 * wave + (lane & 15), j = lane >> 4, s = part.seq0 + j;
    const bool valid = cell < H && j < part.nseq;
    const int row = S * H * 4, out_row = S * p.L * 4;  // bytes of a time step
    const unsigned off = valid ? (unsigned)(s * H + cell) * 4u : kSoloNowhere;
    const unsigned out_off = valid ? (unsigned)(s * p.L + dir * H + cell) * 4u : kSoloNowhere;
    const unsigned pat_off = j < part.nseq ? (unsigned)s : kSoloNowhere;
    const size_t bytes = (size_t)row * T;
    const __amdgpu_buffer_rsrc_t r_ni = solo_array(D.ni, bytes), r_ig = solo_array(D.ig, bytes), r_fg = solo_array(D.fg, bytes),
                                 r_og = solo_array(D.og, bytes), r_c = solo_array(D.c, bytes), r_h = solo_array(D.h, bytes),
                                 r_out = solo_array(p.out, (size_t)out_row * T), r_pat = solo_array(p.pat, (size_t)S * T);

    // B operand: lane = 16 * gate + cell of the wave
    float wreg[K];
    {
        const float *wg = D.w_int + (size_t)(lane >> 4) * p.L * H + (size_t)cell * H;
#pragma unroll
        for (int k = 0; k < K; ++k) wreg[k] = cell < H && k < H ? wg[k] : 0.0f;
    }
    f32x4 bias = {0, 0, 0, 0};
    float p_ig = 0, p_fg = 0, p_og = 0;
    if (valid) {
#pragma unroll
        for (int g = 0; g < 4; ++g) bias[g] = p.bias * D.b[g][cell];
        p_ig = D.peep[0][cell]; p_fg = D.peep[1][cell]; p_og = D.peep[2][cell];
    }
    for (int i = threadIdx.x; i < 2 * kLocalSeqs * PITCH; i += solo_threads(NW)) (&hs[0][0][0])[i] = 0.0f;

    struct StepIn { f32x4 a; unsigned pat; };
    struct StepOut { float ni, ig, fg, og, c, h; unsigned gate_off, c_off, off, out_off; int t; };
    auto t_of = [&](int step) { return dir ? (T - 1 - step) : step; };
    auto request = [&](int step, StepIn &v) __attribute__((always_inline)) {
        const bool on = step < T;
        const int t = on ? t_of(step) : 0;
        const unsigned o = on ? off : kSoloNowhere;
        v.a[0] = solo_load(r_ni, o, t * row);
        v.a[1] = solo_load(r_ig, o, t * row);
        v.a[2] = solo_load(r_fg, o, t * row);
        v.a[3] = solo_load(r_og, o, t * row);
        v.pat = __builtin_amdgcn_raw_buffer_load_b8(r_pat, (int)pat_off, t * S, 0);
    };
    StepOut done = {0, 0, 0, 0, 0, 0, kSoloNowhere, kSoloNowhere, kSoloNowhere, kSoloNowhere, 0};
    auto store_done = [&]() __attribute__((always_inline)) {
        solo_store(r_ni, done.gate_off, done.t * row, done.ni);
        solo_store(r_ig, done.gate_off, done.t * row, done.ig);
        solo_store(r_fg, done.gate_off, done.t * row, done.fg);
        solo_store(r_og, done.gate_off, done.t * row, done.og);
        solo_store(r_c, done.c_off, done.t * row, done.c);
        solo_store(r_h, done.off, done.t * row, done.h);
        solo_store(r_out, done.out_off, done.t * out_row, done.h);
    };
    float c_prev = 0.0f;
    auto run = [&](int step, int parity, StepIn &in) __attribute__((always_inline)) {
        const bool on = step < T;
        const int t = on ? t_of(step) : 0;
        const bool padding = t >= p.Tmin && (in.pat & 0xFFu) == 0;
        const f32x4 start = in.a + bias;
        // A operand: lane = 4 * (four source cells) + sequence; the sums come out as lane = 16 * gate + cell with one
        // sequence per register and are transposed to lane = 16 * sequence + cell with one gate per register
        f32x4 x = solo_product<4, K>(wreg, &hs[parity][lane & 3][lane & ~3], [&]() __attribute__((always_inline)) {
            store_done();  // the step before's results leave while the LDS reads are under way
            request(step + kSoloAhead, in);
        });
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
        // a padding slot keeps its input projections, and its cell state unless the direction is the time-reversed one
        // (the reference clears it there)
        done = StepOut{ni, ig, fg, og, c, hval, on && !padding ? off : kSoloNowhere, on && (!padding || dir) ? off : kSoloNowhere,
                       on ? off : kSoloNowhere, on ? out_off : kSoloNowhere, t};
        lds_barrier();
    };
    StepIn in[kSoloAhead];
#pragma unroll
    for (int i = 0; i < kSoloAhead; ++i) {
        // (with the stores, which go nowhere yet, as many accesses are in flight here as at the loop's back edge, and the
        // compiler's waits in the loop are not tightened to the lower count)
        store_done();
        request(i, in[i]);
        __builtin_amdgcn_sched_barrier(0);
    }
    __syncthreads();
    for (int step = 0; step < T; step += kSoloAhead) {
#pragma unroll
        for (int i = 0; i < kSoloAhead; ++i) run(step + i, i & 1, in[i]);
    }
    store_done();
}

template <int NW>
__global__ __launch_bounds__(solo_threads(NW)) __attribute__((amdgpu_waves_per_eu(2))) void lstm_backward_solo(const ChainParams p) {
    constexpr int K = 16 * NW;
    constexpr int PITCH = K + 4;          // one gate's deltas of a sequence; 4 * PITCH per sequence keeps the sixteen
                                          // (gate, sequence) pieces of a read on different banks
    __shared__ __attribute__((aligned(16))) float ds[2][kLocalSeqs][4][PITCH];

    const int H = p.H, S = p.S, T = p.T;
    const LocalJob part = local_job(p, blockIdx.x);
    const int dir = part.dir;
    const DirPtrs &D = p.d[dir];
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    const int cell = 16 * wave + (lane & 15), j = lane >> 4, s = part.seq0 + j;
    const bool valid = cell < H && j < part.nseq;
    const int row = S * H * 4, out_row = S * p.L * 4;  // bytes of a time step
    const unsigned off = valid ? (unsigned)(s * H + cell) * 4u : kSoloNowhere;
    const unsigned out_off = valid ? (unsigned)(s * p.L + dir * H + cell) * 4u : kSoloNowhere;
    const unsigned pat_off = j < part.nseq ? (unsigned)s : kSoloNowhere;
    const size_t bytes = (size_t)row * T;
    const __amdgpu_buffer_rsrc_t r_e = solo_array(p.outerr, (size_t)out_row * T), r_pat = solo_array(p.pat, (size_t)S * T),
                                 r_ni = solo_array(D.ni, bytes), r_ig = solo_array(D.ig, bytes), r_fg = solo_array(D.fg, bytes),
                                 r_og = solo_array(D.og, bytes), r_c = solo_array(D.c, bytes), r_dni = solo_array(D.dni, bytes),
                                 r_dig = solo_array(D.dig, bytes), r_dfg = solo_array(D.dfg, bytes), r_dog = solo_array(D.dog, bytes),
                                 r_ce = solo_array(D.cerr, bytes), r_herr = solo_array(p.herr_out ? p.herr_out : D.herr, bytes);

    // B operand: lane = 16 * gate + receiving cell of the wave
    float wreg[K];
    {
        const float *wg = D.w_int + (size_t)(lane >> 4) * p.L * H + cell;
#pragma unroll
        for (int k = 0; k < K; ++k) wreg[k] = cell < H && k < H ? wg[(size_t)k * H] : 0.0f;
    }
    float p_ig = 0, p_fg = 0, p_og = 0;
    if (valid) { p_ig = D.peep[0][cell]; p_fg = D.peep[1][cell]; p_og = D.peep[2][cell]; }
    for (int i = threadIdx.x; i < 2 * kLocalSeqs * 4 * PITCH; i += solo_threads(NW)) (&ds[0][0][0][0])[i] = 0.0f;
    __syncthreads();

    auto t_of = [&](int step) { return dir ? step : (T - 1 - step); };
    float fg_later = 0, cerr_later = 0, dig_later = 0, dfg_later = 0;
    const int sb = p.step_begin, se = p.step_end;
    if (sb > 0 && valid) {
        // a launch that starts in the middle: what the step before carried over stands in the state arrays
        const size_t gi = (size_t)t_of(sb - 1) * S * H + (size_t)s * H + cell;
        fg_later = D.fg[gi]; cerr_later = D.cerr[gi]; dig_later = D.dig[gi]; dfg_later = D.dfg[gi];
        float (*d)[PITCH] = ds[0][j];
        d[0][cell] = D.dni[gi]; d[1][cell] = dig_later; d[2][cell] = dfg_later; d[3][cell] = D.dog[gi];
    }

    struct StepIn { float e, ni, ig, fg, og, dog_old, c; unsigned pat; };
    struct StepOut { float ni, ig, fg, og, ce, e; unsigned off; int t; };
    auto request = [&](int step, StepIn &v) __attribute__((always_inline)) {
        const bool on = step < T;
        const int t = on ? t_of(step) : 0;
        const unsigned o = on ? off : kSoloNowhere;
        v.e = solo_load(r_e, on ? out_off : kSoloNowhere, t * out_row);
        v.ni = solo_load(r_ni, o, t * row);
        v.ig = solo_load(r_ig, o, t * row);
        v.fg = solo_load(r_fg, o, t * row);
        v.og = solo_load(r_og, o, t * row);
        v.dog_old = solo_load(r_dog, o, t * row);
        v.c = solo_load(r_c, o, t * row);
        v.pat = __builtin_amdgcn_raw_buffer_load_b8(r_pat, (int)pat_off, t * S, 0);
    };
    StepOut done = {0, 0, 0, 0, 0, 0, kSoloNowhere, 0};
    auto store_done = [&]() __attribute__((always_inline)) {
        solo_store(r_dni, done.off, done.t * row, done.ni);
        solo_store(r_dig, done.off, done.t * row, done.ig);
        solo_store(r_dfg, done.off, done.t * row, done.fg);
        solo_store(r_dog, done.off, done.t * row, done.og);
        solo_store(r_ce, done.off, done.t * row, done.ce);
        solo_store(r_herr, done.off, done.t * row, done.e);
    };
    auto run = [&](int step, int parity, StepIn &in, const StepIn &next) __attribute__((always_inline)) {
        const bool on = step < se;
        const int t = on ? t_of(step) : 0;
        const bool padding = t >= p.Tmin && (in.pat & 0xFFu) == 0;
        const StepIn now = in;
        // A operand: lane = 16 * gate + 4 * (four source cells) + sequence; the sums come out as lane = 16 * gate + cell
        // with one sequence per register: the gates' shares meet in the lane of their sequence
        f32x4 x = solo_product<2, K>(wreg, &ds[parity][lane & 3][lane >> 4][lane & 12], [&]() __attribute__((always_inline)) {
            store_done();  // the step before's results leave while the LDS reads are under way
            request(step + kSoloAhead, in);
        });
        // everything that does not depend on the recursion; beyond the last step the cell state reads as zero, which is
        // what makes the forget gate's last delta zero
        const float tc = tanh_act(now.c);
        const float k_og = logistic_deriv(now.og) * tc, k_ce = now.og * tanh_deriv(tc), k_ni = now.ig * tanh_deriv(now.ni);
        const float k_fg = logistic_deriv(now.fg) * next.c, k_ig = logistic_deriv(now.ig) * now.ni;
        const float fg = now.fg, dog_old = now.dog_old;
        float e = now.e;
        {
            float x0 = x[0], x1 = x[1], x2 = x[2], x3 = x[3];
            swap_halves(x0, x2); swap_halves(x1, x3);
            float even = x0 + x2, odd = x1 + x3;
            swap_rows(even, odd);
            e += even + odd;
        }
        const float d_og = k_og * e + dog_old;
        float ce = k_ce * e + p_og * d_og;
        ce += (fg_later * cerr_later + p_ig * dig_later + p_fg * dfg_later);
        float s_ni = clip1(k_ni * ce), s_ig = clip1(k_ig * ce), s_fg = clip1(k_fg * ce), s_og = clip1(d_og);
        s_ni = padding ? 0.0f : s_ni; s_ig = padding ? 0.0f : s_ig; s_fg = padding ? 0.0f : s_fg; s_og = padding ? 0.0f : s_og;
        ce = padding ? 0.0f : ce;
        float (*d)[PITCH] = ds[parity ^ 1][j];
        d[0][cell] = s_ni; d[1][cell] = s_ig; d[2][cell] = s_fg; d[3][cell] = s_og;
        fg_later = fg; cerr_later = ce; dig_later = s_ig; dfg_later = s_fg;
        done = StepOut{s_ni, s_ig, s_fg, s_og, ce, e, on ? off : kSoloNowhere, t};
        lds_barrier();
    };
    StepIn in[kSoloAhead];
#pragma unroll
    for (int i = 0; i < kSoloAhead; ++i) {
        store_done();
        request(sb + i, in[i]);
        __builtin_amdgcn_sched_barrier(0);
    }
    __syncthreads();
    for (int step = sb; step < se; step += kSoloAhead) {
#pragma unroll
        for (int i = 0; i < kSoloAhead; ++i) run(step + i, i & 1, in[i], in[(i + 1) % kSoloAhead]);
    }
    store_done();
}
