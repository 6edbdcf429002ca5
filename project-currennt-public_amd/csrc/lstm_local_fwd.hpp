// XCD-local forward recursion (included by lstm.hip inside its anonymous namespace, after lstm_local.hpp).
//
// Same cut as the backward recursion: jobs = (direction, at most four sequences), a team of G = H/JB workgroups per
// job on one XCD, roles handed out at run time (local_claim_role).  The forward step is a GATHER -- every workgroup
// needs h[t-1] of all H cells -- and a team whose members all poll the same lines of one L2 waits 1.6-2.5 rounds per
// step for them.  Here every receiver has its own copy: a workgroup writes the h values of its JB cells G times, once
// into the private block of every member of the team (the same 4*JB*G words per step a backward workgroup
// publishes), so polls of different workgroups never meet on a line.
//
// Mailbox of a job: plain 4-byte words [slot][receiver][source cell / 4][sequence][source cell % 4], kEmpty = not
// written yet, four slots; a receiver hands the words of a slot back as empty in the step after it has read them.
//
// Waves and roles, one LDS-only barrier per step, every LDS buffer twice (step parity):
//   gather waves (H/64)  each takes 64 source cells for all of the workgroup's (cell, gate) rows: polls its quarter of
//                        the block, one 16-byte vector per lane, which is the A operand of the step's recurrent product as
//                        it stands (lane = 4 * source cells / 4 + sequence; local_product broadcasts the blocks), leaves
//                        its share of the recurrent sums in LDS.  They issue no stores.
//   cell waves (CW)      after the barrier: lane = one gate of one (cell, sequence) element.  Pre-activation = input
//                        projection + recurrent sums, first pass of the gate function (the four lanes of an element
//                        evaluate the gates side by side; tanh and logistic differ in constants only), cell state in every
//                        lane, second pass: tanh(c) and the output gate side by side.  The row of sixteen lanes holds four
//                        neighbouring cells of a sequence: h[t] is broadcast inside the row and published to every member's
//                        block as it stands.
//   load wave (1)        input projections of several steps at a time.
//   store wave (1)       gate activations, cell states and outputs of finished steps to the state arrays, 64 lanes' worth at a
//                        time; empties the block that was read.
// What bounds a step: the chain sums -> gates -> c -> h -> LDS -> store -> L2 -> poll -> 4 * JB matrix instructions -> LDS.  With one
// cell wave that computed all gates of an element in one lane (five gate functions, two of them side by side at best, twenty LDS
// reads), gather waves that passed the words through LDS into B operands, messages of four sequences throughout and one wave for all
// loads and stores, a step took, us on MI355X (input products included): 256 cells, 8 jobs of 2-3 sequences 1.34, 2 jobs of one
// 1.29, 16 jobs of four 1.43; 128 cells, 8 jobs of two 1.22; 512 cells, 6 jobs of one 1.97.  Then 0.99, 0.85, 1.18, 0.89 and 1.34;
// now, with a branch of the whole wave out of the poll loop and pauses of a job's own, 0.92, 0.77, 1.14, 0.75 and 1.26.
// Publishing without LDS, by a broadcast inside the row of sixteen lanes, saves a round trip of 0.03 but stores pieces of 16
// bytes: 1.05 instead of 1.00.

// LDS of a job
template <int PW, int JB, int NSQ>
struct ForwardShared {
    using Shape = LocalShape<JB, NSQ>;
    static constexpr int EL = Shape::EL, RING = 2 * Shape::BATCH, ROWS = 4 * JB;
    // element = (group of four cells * NSQ + sequence) * 4 + cell of the group, as in the messages
    __attribute__((aligned(16))) float red[2][PW][ROWS][NSQ];  // recurrent sums of the step, one share per gather wave
    __attribute__((aligned(16))) float pre[RING][EL][4];    // input projections of the step
    int pre_dummy[RING][EL];
    __attribute__((aligned(16))) float res_gate[2][EL][4];     // results of the step
    __attribute__((aligned(16))) float res[2][EL][4];          // cell state, output, not 0: padding slot
    __attribute__((aligned(16))) float hpub[Shape::CW][Shape::VPW][4];
    int wait_failed;
};

// One job by one workgroup of its team.  PW = ceil(cells per direction / 64) gather waves, JB cells per workgroup, a job of up to
// NSQ sequences
template <int PW, int JB, int NSQ, bool CLOCKS>
__device__ __forceinline__ void forward_job(const ChainParams &p, const LocalJob &part, int job, int me, unsigned mail_words, ForwardShared<PW, JB, NSQ> &sh) {
    using Shape = LocalShape<JB, NSQ>;
    const int H = p.H, G = p.team;       // G = ceil(H / JB) workgroups; the last one may own fewer than JB cells
    constexpr int EL = Shape::EL, VEC = Shape::VEC, VPW = Shape::VPW, CW = Shape::CW;
    constexpr int STEPS = Shape::STEPS, BATCH = Shape::BATCH, SETS = Shape::SETS, RING = 2 * BATCH;
    constexpr int TEAM = (64 * PW + JB - 1) / JB;  // G at most
    constexpr int ROWS = 4 * JB;         // (cell, gate) rows of this workgroup: row = cell * 4 + gate
    constexpr int PUB = (TEAM * VPW + 63) / 64;  // publishing stores per lane; the last may lie past the team
    constexpr int NQ = (TEAM * VEC + 63) / 64;  // vectors per lane that hand a block back
    const unsigned RECV = (unsigned)(G * EL);   // words of a receiver's block
    const int vectors = G * VEC;                // 16-byte vectors of a receiver's block
    auto &red = sh.red;
    auto &pre = sh.pre;
    auto &pre_dummy = sh.pre_dummy;
    auto &res_gate = sh.res_gate;
    auto &res = sh.res;
    auto &hpub = sh.hpub;
    int &wait_failed = sh.wait_failed;

    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    if (wave >= PW + CW + 2) return;  // (of a launch whose largest jobs need more waves)
    const int nseq = part.nseq, begin_step = part.begin, end_step = part.end;
    int dir = part.dir;
    asm volatile("" : "+s"(dir));  // the direction's pointers are read here, not in front of the choice of the kernel's three jobs
    const DirPtrs &D = p.d[dir];
    const int S = p.S, T = p.T;
    const int j0 = me * JB;
    const int n = S * H;
    float *const mailbox = p.flmail + (size_t)job * mail_words;
    const unsigned slot_words = (unsigned)G * RECV;
    const __amdgpu_buffer_rsrc_t mail =
        __builtin_amdgcn_make_buffer_rsrc(mailbox, 0, (int)(local_job_words(G, JB, NSQ) * sizeof(float)), 0x00020000);
    auto slot_of = [&](int step) { return dir ? (T - 1 - step) : step; };
    auto given_up = [&]() { return *(__attribute__((address_space(3))) volatile int *)&wait_failed; };

    // the load and the store wave: lane = (step of an access, sequence, cell)
    const int cs = lane % EL / JB, cj = lane % JB;
    const bool valid = cs < nseq && j0 + cj < H;
    const int ahead = lane / EL;

    if (wave == PW + CW) {
        // ------------------------------------------------------------------ load wave
        struct StepIn { float a[4]; char pat; };
        const int s = part.order[min(cs, nseq - 1)], el = (cj / 4 * NSQ + cs) * 4 + cj % 4;
        auto load_batch = [&](int first, StepIn (&in)[SETS]) {
#pragma unroll
            for (int i = 0; i < SETS; ++i) {
                StepIn &v = in[i];
                v = StepIn{{0, 0, 0, 0}, 1};
                const int step = first + i * STEPS + ahead;
                if (!valid || step >= end_step) continue;
                const int t = slot_of(step);
                const size_t gi = (size_t)t * n + (size_t)s * H + j0 + cj;
                v.a[0] = D.ni[gi]; v.a[1] = D.ig[gi]; v.a[2] = D.fg[gi]; v.a[3] = D.og[gi];
                v.pat = p.pat[t * S + s];
            }
        };
        auto put_batch = [&](int first, const StepIn (&in)[SETS]) {
#pragma unroll
            for (int i = 0; i < SETS; ++i) {
                const int step = first + i * STEPS + ahead;
                if (step >= end_step) continue;
                *reinterpret_cast<f32x4 *>(pre[(unsigned)step % RING][el]) = f32x4{in[i].a[0], in[i].a[1], in[i].a[2], in[i].a[3]};
                pre_dummy[(unsigned)step % RING][el] = slot_of(step) >= p.Tmin && in[i].pat == 0 ? 1 : 0;
            }
        };
        StepIn in[SETS];
        load_batch(begin_step, in);
        wait_all_vmem();
        put_batch(begin_step, in);
        long long busy = 0;
        lds_barrier();  // start of the recursion
        for (int step = begin_step; step < end_step; ++step) {
            lds_barrier();
            if (given_up()) return;
            const long long since = clock_now<CLOCKS>();
            const int phase = (int)((unsigned)(step - begin_step) % BATCH), next = step - phase + BATCH;
            if (phase == 0) {
                for (int d = 0; d < p.mem_delay_fwd; ++d) __builtin_amdgcn_s_sleep(1);
                load_batch(next, in);
            } else if (phase == BATCH / 2) {
                wait_all_vmem();  // requested two steps ago or more
                put_batch(next, in);
            }
            clock_add<CLOCKS>(busy, since);
        }
        if (lane == 0) clock_store<CLOCKS>(p, CLK_LOAD, busy);
        return;
    }

    if (wave == PW + CW + 1) {
        // ------------------------------------------------------------------ store wave
        const int s = part.order[min(cs, nseq - 1)], el = (cj / 4 * NSQ + cs) * 4 + cj % 4;
        f32x4 g = {0, 0, 0, 0}, r = {0, 0, 0, 0};
        long long busy = 0;
        lds_barrier();  // start of the recursion
        lds_barrier();  // the first step's sums
        for (int step = begin_step; step < end_step; ++step) {
            const int b = step & 1, held = (int)((unsigned)(step - begin_step) % STEPS);
            lds_barrier();  // results of this step are in LDS
            if (given_up()) return;
            const long long since = clock_now<CLOCKS>();
            if (ahead == held) {
                g = *reinterpret_cast<const f32x4 *>(res_gate[b][el]);
                r = *reinterpret_cast<const f32x4 *>(res[b][el]);
            }
            wait_all_vmem();  // the stores of the step before are done
            if ((held == STEPS - 1 || step == end_step - 1) && valid && ahead <= held) {
                // An access stores as many steps as it has lanes for.  A padding slot keeps its summed pre-activations, and its
                // cell state unless the direction is the time-reversed one (the reference clears it there).
                const int mine = step - held + ahead, t = slot_of(mine);
                const bool pad = r[2] != 0.0f;
                const size_t gi = (size_t)t * n + (size_t)s * H + j0 + cj;
                if (!pad || mine > 0) {
                    D.ni[gi] = g[0]; D.ig[gi] = g[1]; D.fg[gi] = g[2]; D.og[gi] = g[3];
                }
                if (!pad || dir) D.c[gi] = r[0];
                D.h[gi] = r[1];
                if (p.out) p.out[((size_t)t * S + s) * p.L + dir * H + j0 + cj] = r[1];
            }
            if (step + 1 < end_step) {
                // the words the gather waves have read for the next step are empty again
                const u32x4 empty = {kEmpty, kEmpty, kEmpty, kEmpty};
#pragma unroll
                for (int q = 0; q < NQ; ++q)
                    if (q * 64 + lane < vectors)
                        __builtin_amdgcn_raw_buffer_store_b128(empty, mail, (int)((unsigned)step % kMailSlots * slot_words * 4u +
                                                               ((unsigned)me * RECV + (unsigned)(q * 64 + lane) * 4u) * 4u), 0, 0);
            }
            clock_add<CLOCKS>(busy, since);
        }
        if (lane == 0) clock_store<CLOCKS>(p, CLK_STORE, busy);
        return;
    }

    if (wave >= PW) {
        // ------------------------------------------------------------------ cell waves
        const int cw = wave - PW;
        const int row = lane >> 4, q = cw * VPW + row % VPW;  // vector of the message: four cells of a sequence
        const int el = 4 * q + (lane >> 2 & 3), gate = lane & 3;
        const int cell = q / NSQ * 4 + (lane >> 2 & 3), seq = q % NSQ;
        const bool cell_valid = seq < nseq && j0 + cell < H;
        float bias = 0, peep = 0, p_og = 0;
        if (cell_valid) {
            bias = p.bias * D.b[gate][j0 + cell];
            if (gate == 1 || gate == 2) peep = D.peep[gate - 1][j0 + cell];
            p_og = D.peep[2][j0 + cell];
        }
        const bool peeps = gate == 1 || gate == 2, is_tanh = gate == 0;
        // tanh_quick for the lanes of the cell input, logistic_quick for the others
        const float lo = is_tanh ? -43.65f : -87.3f, hi = is_tanh ? 44.361415f : 88.72283f;
        const float log2e = is_tanh ? 2.88539008177792681f : 1.44269504088896341f;
        const float log2e_rest = is_tanh ? 3.85192606e-8f : 1.92596303e-8f;
        const float times = is_tanh ? 2.0f : 1.0f, plus = is_tanh ? -1.0f : 0.0f;
        auto gate_fn = [&](float x) __attribute__((always_inline)) {
            return __builtin_fmaf(times, logistic_of_negative<false>(__builtin_amdgcn_fmed3f(-x, lo, hi), log2e, log2e_rest), plus);
        };
        auto of_gate = [](float v, auto g) __attribute__((always_inline)) {
            constexpr int k = decltype(g)::value;
            return __builtin_bit_cast(float, __builtin_amdgcn_update_dpp(0, __builtin_bit_cast(int, v), k * 0x55, 0xF, 0xF, true));
        };
        const std::integral_constant<int, 0> c0; const std::integral_constant<int, 1> c1;
        const std::integral_constant<int, 2> c2; const std::integral_constant<int, 3> c3;
        // publishing role: vector lane % VPW of the wave's goes into the blocks of the receivers lane / VPW + 64 / VPW * i
        const int first_receiver = lane / VPW;
        const unsigned pub_off = ((unsigned)first_receiver * RECV + (unsigned)me * EL + (unsigned)(cw * VPW + lane % VPW) * 4u) * 4u;
        const unsigned pub_stride = (unsigned)(64 / VPW) * RECV * 4u;
        float *const my_h = &hpub[cw][row % VPW][lane >> 2 & 3];
        const float *const sent = hpub[cw][lane % VPW];
        const float *const my_red = &red[0][0][cell * 4 + gate][seq];
        float c_prev = 0.0f, start = bias;
        // the first step has no recurrent sums
        for (int i = 64 * cw + lane; i < PW * ROWS * NSQ; i += 64 * CW) (&red[begin_step & 1][0][0][0])[i] = 0.0f;
        long long busy = 0;
        const bool records = CLOCKS && cw == 0 && lane == 0;
        wait_all_vmem();
        lds_barrier();  // start of the recursion
        for (int step = begin_step; step < end_step; ++step) {
            const int b = step & 1;
            lds_barrier();
            const long long since = clock_now<CLOCKS>();
            if (records) clock_point<CLOCKS>(p, step - begin_step, 3);
            // (looked at at the end of the step: what a step that failed publishes no longer matters)
            const int failed = given_up();
            float a = pre[(unsigned)step % RING][el][gate];
            int padding = pre_dummy[(unsigned)step % RING][el];
            float share[PW];
#pragma unroll
            for (int w = 0; w < PW; ++w) share[w] = my_red[(size_t)(b * PW + w) * ROWS * NSQ];
#pragma unroll
            for (int w = 0; w + 1 < PW; w += 2) share[w / 2] = share[w] + share[w + 1];
            if (PW % 2) share[PW / 2] = share[PW - 1];
#pragma unroll
            for (int w = 0; w < (PW + 1) / 2; ++w) a += share[w];
            asm volatile("" : "+v"(padding));  // read above, with the sums: the compiler would read it between the gates and wait there
            const bool dummy = padding != 0;
            const float x0 = a + start, v1 = gate_fn(x0);
            float c = of_gate(v1, c0) * of_gate(v1, c1) + c_prev * of_gate(v1, c2);
            // second pass: tanh(c) in the lanes of the cell input, the output gate in its own
            const float v2 = gate_fn(is_tanh ? c : x0 + c * p_og);
            float hval = of_gate(v2, c0) * of_gate(v2, c3);
            hval = dummy || !cell_valid ? 0.0f : hval;
            // the publication of the previous step is complete before this step publishes
            wait_all_vmem();
            if (step + 1 < end_step) {
                // through LDS, so that neighbouring lanes hold what goes into one receiver's block
                *my_h = __builtin_bit_cast(float, publishable(hval));
                __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
                __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
                const u32x4 v = *reinterpret_cast<const u32x4 *>(sent);
#pragma unroll
                for (int i = 0; i < PUB; ++i)
                    if (first_receiver + 64 / VPW * i < G)
                        __builtin_amdgcn_raw_buffer_store_b128(v, mail, (int)((unsigned)step % kMailSlots * slot_words * 4u + pub_off + (unsigned)i * pub_stride), 0, 0);
            }
            c = dummy ? 0.0f : c;
            if (row < VPW) {
                // on a padding slot the reference leaves the summed pre-activations in place, clears the cell only in the
                // time-reversed direction and emits a zero output
                res_gate[b][el][gate] = dummy ? a : gate == 3 ? v2 : v1;
                if (gate < 3) res[b][el][gate] = gate == 0 ? c : gate == 1 ? hval : dummy ? 1.0f : 0.0f;
            }
            c_prev = dummy && !dir ? c_prev : c;
            start = peeps ? bias + c_prev * peep : bias;
            clock_add<CLOCKS>(busy, since);
            if (records) clock_point<CLOCKS>(p, step - begin_step, 4);
            if (failed) return;
        }
        lds_barrier();  // results of the last step are in LDS
        if (records) clock_store<CLOCKS>(p, CLK_OTHER, busy);
        return;
    }

    // ---------------------------------------------------------------------- gather waves
    // Wave pw takes the source cells 64*pw .. 64*pw + 63 for ALL of the workgroup's rows; with 32 rows each half of the wave
    // takes 32 of them, and the two halves' sums meet at the end.
    const int pw = wave;
    constexpr int HALVES = 64 / ROWS;    // parts of the wave with source cells of their own
    constexpr int BLOCKS = 16 / HALVES;  // blocks of the A operand (four source cells each) of a part
    float wreg[4 * BLOCKS];
    {
        const int o = lane % ROWS, g = o % 4, jj = o / 4;
        const bool has_row = j0 + jj < H;
        const float *wg = D.w_int + (size_t)g * p.L * H + (size_t)(has_row ? j0 + jj : 0) * H;
        const int from = 64 * pw + 4 * BLOCKS * (lane / ROWS);
        if constexpr (JB == 16) {
            load_weight_row(wg, has_row, from, H, wreg);
        } else {
#pragma unroll
            for (int i = 0; i < 4 * BLOCKS; ++i) wreg[i] = from + i < H && has_row ? wg[from + i] : 0.0f;
        }
    }
    // a lane past the end of the block polls the block's first vector instead and multiplies zeros
    const int my_vec = (16 * pw + (lane >> 2)) * NSQ + (lane & 3) % NSQ;
    const bool inside = my_vec < vectors;
    const int pause = min(p.poll_limit_fwd, p.poll_delay_fwd >= 0 ? p.poll_delay_fwd : forward_pause(EL));
    const unsigned poll_off = ((unsigned)me * RECV + (unsigned)(inside ? my_vec : 0) * 4u) * 4u;
    long long waited = 0, rest = 0, barrier = 0, rounds = 0;
    const bool records = CLOCKS && tid == 0;
    wait_all_vmem();
    lds_barrier();  // start of the recursion
    const long long begin = clock_now<CLOCKS>();
    lds_barrier();  // the first step has nothing to gather

    for (int step = begin_step + 1; step < end_step; ++step) {
        const long long since = clock_now<CLOCKS>();
        if (records) clock_point<CLOCKS>(p, step - begin_step, 0);
        const float *slot = mailbox + (size_t)((unsigned)(step - 1) % kMailSlots) * slot_words;
        u32x4 w[1];
        unsigned spins = 0;
        for (int d = 0; d < pause; ++d) __builtin_amdgcn_s_sleep(1);
        for (;;) {
            poll_load<1>(slot, poll_off, 0u, poll_off, w);
            if constexpr (CLOCKS) ++rounds;
            const unsigned worst = max(max(w[0].x, w[0].y), max(w[0].z, w[0].w));
            if (__builtin_amdgcn_ballot_w64(worst == kEmpty) == 0) break;
            if (poll_gives_up(p, ++spins)) { wait_failed = 1; break; }
            for (int d = 0; d < p.poll_gap; ++d) __builtin_amdgcn_s_sleep(1);
        }
        clock_add<CLOCKS>(waited, since);
        if (records) clock_point<CLOCKS>(p, step - begin_step, 1);
        if (!inside) w[0] = u32x4{0, 0, 0, 0};
        f32x4 sum = local_product<JB == 8 ? 3 : 4, 4 * BLOCKS>(__builtin_bit_cast(f32x4, w[0]), wreg, std::make_integer_sequence<int, BLOCKS>{});
        // register = sequence; where the wave's halves meet, the lower one ends up with the first half of the sequences
        float *const out = &red[step & 1][pw][lane % ROWS][0];
        if constexpr (HALVES == 1) {
#pragma unroll
            for (int r = 0; r < NSQ; ++r) out[r] = sum[r];
        } else if constexpr (NSQ == 4) {
            const float lower = sum_halves(sum[0], sum[2]), upper = sum_halves(sum[1], sum[3]);
            out[lane / ROWS * 2] = lower; out[lane / ROWS * 2 + 1] = upper;
        } else if constexpr (NSQ == 2) {
            out[lane / ROWS] = sum_halves(sum[0], sum[1]);
        } else {
            out[0] = sum_halves(sum[0], sum[0]);
        }
        if (records) clock_point<CLOCKS>(p, step - begin_step, 2);
        const long long at_barrier = clock_now<CLOCKS>();
        lds_barrier();
        clock_add<CLOCKS>(barrier, at_barrier);
        clock_add<CLOCKS>(rest, since);  // the whole step: what was waited is taken off below
        if (given_up()) {
            if (tid == 0) raise_abort(p);
            return;
        }
    }
    lds_barrier();  // results of the last step
    if (records) {
        clock_store<CLOCKS>(p, CLK_WAIT, waited);
        clock_store<CLOCKS>(p, CLK_REST, rest - waited - barrier);
        clock_store<CLOCKS>(p, CLK_BARRIER, barrier);
        clock_store<CLOCKS>(p, CLK_ROUNDS, rounds);
        clock_store<CLOCKS>(p, CLK_STEPS, end_step - begin_step);
        clock_store<CLOCKS>(p, CLK_LOOP, clock_now<CLOCKS>() - begin);
        clock_where<CLOCKS>(p, job, me);
    }
}

template <int PW, int JB, int MOST, bool CLOCKS>
__global__ __launch_bounds__(local_threads(PW, JB, MOST)) void lstm_forward_local(const ChainParams p) {
    __shared__ LocalPlan plan;
    __shared__ union Shared { ForwardShared<PW, JB, 1> one; ForwardShared<PW, JB, MOST < 2 ? 1 : 2> two; ForwardShared<PW, JB, MOST> most; } sh;
    int job = 0, me = 0;
    const LocalJob part = local_setup<MOST, true>(p, plan, job, me);
    if (part.nseq == 0) return;
    fill_padding<JB, true>(p, part, me);
    if (part.begin >= part.end) return;
    const unsigned mail_words = (unsigned)local_job_words(p.team, JB, MOST);
    if (threadIdx.x == 0) (part.nseq == 1 ? sh.one.wait_failed : part.nseq == 2 ? sh.two.wait_failed : sh.most.wait_failed) = 0;
    if (MOST == 1 || part.nseq == 1) forward_job<PW, JB, 1, CLOCKS>(p, part, job, me, mail_words, sh.one);
    else if (part.nseq == 2) forward_job<PW, JB, MOST < 2 ? 1 : 2, CLOCKS>(p, part, job, me, mail_words, sh.two);
    else forward_job<PW, JB, MOST, CLOCKS>(p, part, job, me, mail_words, sh.most);
}
