// XCD-local BPTT error recursion (included by lstm.hip inside its anonymous namespace).
//
// The parallel sequences of a fraction are independent chains, and so are the two directions of a bidirectional
// layer.  The recursion is therefore cut into JOBS = (direction, group of at most four sequences), and
// every job is run by a TEAM of G = ceil(H/JB) workgroups that sit on ONE XCD: the all-to-all exchange of a step then
// stays inside that XCD's L2 (plain stores, loads that only bypass the per-CU cache), which takes about half as
// long as a hop through the memory side, and a step moves G*G*4*JB words per job instead of G*G*S*JB per direction.
//
// Placement.  Nothing guarantees which XCD a workgroup lands on, so roles are handed out at run time: more
// workgroups are launched than needed, each reads the id of its XCD and takes a ticket there; G consecutive
// tickets of one XCD form a team, and a complete team claims the next unclaimed job.  Teams beyond an XCD's first
// give the other XCDs' first teams a head start, so that with an even spread every XCD runs one job on its own
// compute units, while any other spread still finds a team for every job: with W launched workgroups at least
// (W - 8*(G-1)) / G teams complete, whatever the spread, and the launch uses W = njobs*G + 8*(G-1).  Workgroups
// without a job end at once.  A launch never holds more jobs than complete teams fit the compute units at once (the
// host cuts the jobs into launches): a team whose members could only become resident after another team has ended is not
// waited for -- with 19-workgroup teams, one workgroup per compute unit and a second team left half resident, the
// remaining workgroups were never dispatched and the launch gave up.
//
// A job moves and multiplies NSQ sequences (1, 2 or 4: the smallest that holds its own), so one of one or two sequences
// exchanges a quarter or half of the words.  Which sequences share a job, and which steps it leaves out: local_setup.
//
// Per workgroup (cells j0 .. j0+JB-1 of the job's direction, all T steps): the recurrent weights that read this
// workgroup's gate deltas, W[h][k] for every cell h of the direction and k = (own cell, gate), live in registers
// as B operands of v_mfma_f32_4x4x1 (sixteen independent 4 x 4 outer products per instruction).  The step's deltas are the
// A operand, read from LDS ONCE per lane for the whole step -- lane = 4 * own cell + sequence holds the four gates --, and
// the instruction's operand broadcast (2^CBSZ neighbouring blocks take block I of the operand) hands them to every block.
// Waves and roles, ONE LDS-only barrier per step (every LDS buffer exists twice, by step parity):
//   product waves      after the barrier: multiply the fresh deltas with the weight slice (lane = receiving cell, register
//   (PW = ceil(H/64))  = sequence) and publish.  They never wait for a load.
//   cell waves (CW)    each polls four (or two) of the 16-byte vectors every sender addresses to this workgroup, side by
//                      side for all senders, and sums them by lane swaps that leave a register less at every level, so
//                      that the sums end up one element per lane without a select, four copies of it in the row of sixteen
//                      lanes: one per gate.  A lane computes one gate's delta.  The step's coefficients were fetched from
//                      LDS while the poll was in flight.  These waves issue no stores.
//   load wave (1)      loads the inputs of the cell update for several steps at a time, folds what does not depend on the
//                      recursion into coefficients.
//   store wave (1)     writes the results of finished steps to the state arrays, 64 lanes' worth at a time, hands the consumed
//                      words back as empty.
// What bounds a step: the chain sum -> delta -> LDS -> 4 * JB matrix instructions -> store -> L2 -> poll.  A lone wave issues a
// dependent vector instruction every 8 to 12 clocks and a matrix instruction of this size every 8, so instructions on that
// chain are what counts.  With one cell wave, all gates of an element in one lane, a sum of 32 lane swaps, a product whose B
// operand was read from LDS once per four instructions, messages of four sequences throughout and one wave for all loads and
// stores (whose pause then set the step's length) a step took, us on MI355X: 256 cells, 8 jobs of 2-3 sequences 1.25, 2 jobs of
// one 1.24, 16 jobs of four 1.73; 128 cells, 8 jobs of two 1.24; 512 cells, 6 jobs of one 1.85.  Then 0.87, 0.78, 1.15, 0.83 and
// 1.22; now, with a branch of the whole wave out of the poll loop and what does not wait for the poll worked out in front of it,
// 0.81, 0.69, 1.05, 0.69 and 1.11.  (A hop inside an XCD with nothing but a
// poll and a store at its ends takes 0.25, one of a 4 KB message 0.45.)
//
// Mailbox of a job: plain 4-byte words [slot][receiver][sender][cell of the receiver][sequence], kEmpty = not
// written yet, four slots, the receiver hands its words back as empty after use.  A store is acknowledged once the XCD's L2 holds it, which is where the team's
// polls read.

constexpr int kLocalSeqs = 4;     // sequences of a job at most
constexpr int kLocalXcds = 8;
// control words (zero before every launch): jobs claimed; per XCD its tickets, and per team arrivals and job.  What one XCD counts lies
// on cache lines of its own: with all tickets on one line the eight L2s passed it around.  Teams are counted up to
// ChainParams::ctl_teams per XCD, which the launch makes large enough for all of its workgroups on one XCD
constexpr int kCtlLine = 32;
constexpr int ctl_xcd_words(int teams) { return kCtlLine + (2 * teams + kCtlLine - 1) / kCtlLine * kCtlLine; }
constexpr int ctl_words(int teams) { return kCtlLine + kLocalXcds * ctl_xcd_words(teams); }
constexpr unsigned kNoJob = 0xFFFFFFFFu;

// Elements (cell, sequence) of a workgroup of JB cells with NSQ sequences = words of a (receiver, sender) pair, the 16-byte
// vectors they make, vectors of a cell wave, cell waves
template <int JB, int NSQ>
struct LocalShape {
    static constexpr int EL = JB * NSQ, VEC = EL / 4, VPW = VEC < 4 ? VEC : 4, CW = VEC / VPW;
    static_assert((JB == 8 || JB == 16) && (NSQ == 1 || NSQ == 2 || NSQ == 4), "local recursion geometry");
    // Time steps whose inputs the load wave requests together, and how many of them an access of 64 lanes covers.  A compute
    // unit returns its vector loads in order over all of its waves, so a request that goes to memory holds back the polls
    // issued behind it: once in BATCH steps instead of in every one.
    static constexpr int STEPS = 64 / EL, BATCH = STEPS > 4 ? STEPS : 4, SETS = BATCH / STEPS;
};
constexpr int local_threads(int PW, int JB, int NSQ) { return (PW + (JB * NSQ + 15) / 16 + 2) * 64; }
constexpr size_t local_job_words(int G, int JB, int NSQ) { return (size_t)kMailSlots * G * G * NSQ * JB; }

// What a job does: its direction, its sequences (order[0 .. nseq)), and the launch's steps that it has to take,
// [begin, end) -- on the others all its sequences are padding (fill_padding).
struct LocalJob {
    int dir, nseq;
    const int *order;
    int first, last, begin, end;  // first and last: of the pass, which may lie outside the launch's range
};

// The placement counters carry nothing but their own values (everything else a workgroup reads was written by earlier
// launches), so every access to them is a relaxed device-scope atomic: acquire or release at that scope would write
// back and invalidate the XCD's L2 at every access, also under the launches that run beside this one.
__device__ __forceinline__ unsigned ctl_load(const unsigned *p) {
    return __hip_atomic_load(p, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}

// Rounds of a wait for the team's job in which the thread also looks whether all jobs are taken: every fourth, and the one before it gives up,
// so that a team that stays incomplete is no failure, however small the limit.
__host__ __device__ constexpr bool looks_at_claims(unsigned spins, unsigned spin_limit) { return (spins & 3u) == 3u || spins >= spin_limit; }
static_assert(looks_at_claims(0, 0) && looks_at_claims(1, 1) && looks_at_claims(2, 2) && looks_at_claims(3, 100) && !looks_at_claims(4, 5) &&
              looks_at_claims(5, 5), "the last round before giving up looks");

// Role of this workgroup: job * 64 + member (a team has at most 32 workgroups), or -1.  Called by one thread.
__device__ int local_claim_role(const ChainParams &p, int G) {
    const unsigned xcd = __builtin_amdgcn_s_getreg((3 << 11) | (0 << 6) | 20) & 15u;  // XCC_ID, bits 3:0
    if (xcd >= 8u) return -1;
    unsigned *const claimed = p.ctl, *const own = p.ctl + kCtlLine + xcd * (unsigned)ctl_xcd_words(p.ctl_teams);
    // (A workgroup that finds all jobs taken ends at once.  Those the compute units had no room for come when the recursion is over, and
    // the launch lasts until they are gone.)
    const unsigned taken = ctl_load(claimed);
    const unsigned ticket = __hip_atomic_fetch_add(own, 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    if (taken >= (unsigned)p.njobs) return -1;
    const unsigned team = ticket / (unsigned)G, member = ticket % (unsigned)G;
    if (team >= (unsigned)p.ctl_teams) return -1;
    unsigned *const arrived = own + kCtlLine + 2 * team, *const team_job = arrived + 1;
    const unsigned before = __hip_atomic_fetch_add(arrived, 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    unsigned job = 0;  // 0: undecided, j + 1: job j, kNoJob: none
    if (before == (unsigned)G - 1u) {
        // this arrival completes the team
        if (team > 0) {
            // head start for the earlier teams of the other XCDs: about 20 us, or until they can all have taken a job
            const long long t0 = wall_clock64();
            const unsigned enough = min((unsigned)p.njobs, team * (unsigned)kLocalXcds);
            while (ctl_load(claimed) < enough && wall_clock64() - t0 < 2000) __builtin_amdgcn_s_sleep(8);
        }
        const unsigned c = __hip_atomic_fetch_add(claimed, 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        job = c < (unsigned)p.njobs ? c + 1u : kNoJob;
        __hip_atomic_store(team_job, job, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    } else {
        unsigned spins = 0;
        for (;;) {
            job = ctl_load(team_job);
            if (job != 0u) break;
            // every job is taken and this team is still incomplete: whoever completes it will find none left
            if (looks_at_claims(spins, p.spin_limit) && ctl_load(claimed) >= (unsigned)p.njobs && ctl_load(arrived) < (unsigned)G) { job = kNoJob; break; }
            if (++spins > p.spin_limit || ((spins & 15u) == 0u && __hip_atomic_load(p.abort_flag, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) != 0)) {
                raise_abort(p);
                job = kNoJob;
                break;
            }
            __builtin_amdgcn_s_sleep(2);
        }
    }
    if (job == kNoJob) return -1;
    return (int)((p.job0 + job - 1u) * 64u + member);
}

// How the sequences of a direction are dealt to its groups.  A recursion lasts as long as its longest job, and a step of a job is
// shorter the fewer sequences it has (step_cost), so the longest sequences get jobs of their own and the shortest ones share:
// sorted by length, cut so that the largest product of a job's longest sequence and its step is smallest (greedily for a
// bound, the bound by bisection).  A job then leaves out the steps on which all of its sequences are padding.  The lengths come
// from the pattern types, so every launch of a pass, and every workgroup of a launch, finds the same cut.  The acoustic model's
// pass (ten sequences of 300 to 600 steps, two layers of 256 cells in two directions) 2930 us dealt evenly and in order, 2750 so;
// 150 and 200 cells with twenty sequences of 211 to 500 steps 2455 and 2305.
// Step of a job of 1 to 4 sequences, of 128.  Measured, us per step, forward / backward: 256 cells, 8 per workgroup, 0.72 / 0.63, 0.75 /
// 0.67, 0.82 / 0.71, 0.84 / 0.73, which is 110 / 110, 114 / 117, 125 / 124 and 128; 150 cells, 8 per workgroup, 0.69 / 0.65, 0.72 / 0.67,
// 0.77 / 0.71, 0.77 / 0.72.  With 16 cells per workgroup small jobs are cheaper than this says: 512 cells 1.06 / 0.97, 1.15 / 1.08, 1.31 /
// 1.31, 1.40 / 1.35 (97 / 92, 105 / 102, 120 / 124), 300 cells 1.01 / 0.95, 1.02 / 1.02, 1.11 / 1.09, 1.14 / 1.22; one table for all
// sizes all the same.
template <bool FWD>
__host__ __device__ constexpr int step_cost(int sequences) {
    constexpr int cost[5] = {0, FWD ? 111 : 114, FWD ? 117 : 123, FWD ? 126 : 127, 128};
    return cost[sequences];
}
// in 64 bits: 2^24 steps and more of 128 are no 32-bit number
template <bool FWD>
__host__ __device__ constexpr long long job_cost(int steps, int sequences) { return (long long)steps * step_cost<FWD>(sequences); }
static_assert(job_cost<true>(0x7FFFFFFF, 4) == 0x7FFFFFFFLL * 128 && job_cost<false>(0x7FFFFFFF, 1) > 0x7FFFFFFFLL, "no wrap at any length");
constexpr int kPlannedSeqs = 64;  // more parallel sequences are dealt evenly and in order, and take every step
constexpr int kRoleOpen = -2;  // not decided yet (-1: none)
struct LocalPlan {
    int role;
    int gathered;              // waves that have looked at their share of the pattern types
    int length[kPlannedSeqs];  // steps until the last one that is no padding; then the same, longest first
    int order[kPlannedSeqs];
    int start[kPlannedSeqs + 1];  // first position in `order` of every group
};

// Called by all threads.  The role and the plan do not depend on each other and take some 5 us each, mostly trips to memory and a chain
// of scalar steps: one wave claims the role while the others look at the pattern types and the last one, when they have, sorts and cuts.
// One after the other, and with all XCDs' tickets on one line, the recursion began 12.5 us after the first workgroup (4 sequences of 150 to 200
// steps) or 16 to 20 (10 of 300 to 600), 5.5 of it the role and 1 to 4 the plan.  One lstm layer 359 -> 350 us per pass, one utterance 1234 -> 1216, 150
// and 200 cells with twenty sequences 2094 -> 2073, 32 sequences 2247 -> 2229, the acoustic model 2482 -> 2471.
template <int MOST, bool FWD>
__device__ __forceinline__ LocalJob local_setup(const ChainParams &p, LocalPlan &plan, int &job, int &me) {
    const int tid = threadIdx.x, lane = tid & 63, S = p.S, T = p.T, Tmin = min(p.Tmin, T);
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6), claims = (int)blockDim.x / 64 - 2;
    const bool planned = S <= kPlannedSeqs;
    if (tid < kPlannedSeqs) plan.length[tid] = Tmin;
    if (tid == 0) { plan.gathered = 0; plan.role = kRoleOpen; }
    __syncthreads();
    if (wave == claims) {
        if (lane == 0) __hip_atomic_store(&plan.role, local_claim_role(p, p.team), __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
    } else if (wave < claims) {
        if (planned && Tmin < T) {
            const int rows = 64 * claims / S, s = tid % S, row = tid / S;
            if (row < rows) {
                int length = 0;
#pragma unroll 8
                for (int t = Tmin + row; t < T; t += rows) length = p.pat[(size_t)t * S + s] != 0 ? t + 1 : length;
                atomicMax(&plan.length[s], length);
            }
        }
        __builtin_amdgcn_fence(__ATOMIC_RELEASE, "workgroup", "local");
        if (lane == 0) atomicAdd(&plan.gathered, 1);
    } else if (planned) {
        while (__hip_atomic_load(&plan.gathered, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP) < claims) __builtin_amdgcn_s_sleep(1);
        __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "workgroup", "local");
        const bool needed = __hip_atomic_load(&plan.role, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP) != -1;
        const int mine = lane < S ? plan.length[lane] : -1;
        int rank = 0;
        for (int s = 0; s < S && needed; ++s) {
            const int other = __builtin_amdgcn_readlane(mine, s);
            rank += other > mine || (other == mine && s < lane) ? 1 : 0;
        }
        if (lane < S) { plan.order[rank] = lane; plan.length[rank] = mine; }
        __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
        __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
        const int sorted = lane < S ? plan.length[lane] : 0;
        long long cost[MOST];  // of a job of this lane's sequence and the q behind it
#pragma unroll
        for (int q = 0; q < MOST; ++q) cost[q] = job_cost<FWD>(sorted, q + 1);
        auto most_within = [&](long long bound) {  // sequences of a job that starts with this lane's
            int n = 0;
#pragma unroll
            for (int q = 0; q < MOST; ++q) n = cost[q] <= bound ? q + 1 : n;
            return n;
        };
        auto cut = [&](long long bound, bool keep) {
            const int n = most_within(bound);
            int at = 0, g = 0;
            for (; at < S && g < p.groups; ++g) {
                const int take = __builtin_amdgcn_readlane(n, at);
                if (take == 0) break;
                if (keep && lane == 0) plan.start[g] = at;
                at = min(at + take, S);
            }
            if (keep)
                for (; g <= p.groups; ++g)
                    if (lane == 0) plan.start[g] = S;
            return at >= S;
        };
        const int top = __builtin_amdgcn_readlane(sorted, 0);
        long long low = job_cost<FWD>(top, 1) - 1, high = job_cost<FWD>(top, MOST);  // `high` always suffices
        // (four in every job: nothing to choose)
        for (int q = 0; q < 10 && needed && high - low > 1 && p.groups * MOST > S; ++q) {
            const long long mid = (low + high) / 2;
            if (cut(mid, false)) high = mid;
            else low = mid;
        }
        if (needed) cut(high, true);
    }
    __syncthreads();
    LocalJob part = {0, 0, plan.order, 0, 0, 0, 0};
    if (plan.role < 0) return part;
    const int role = __builtin_amdgcn_readfirstlane(plan.role);
    job = role >> 6; me = role & 63;
    part.dir = job / p.groups;
    const int group = job % p.groups;
    int longest = T;
    if (!planned) {
        const int each = S / p.groups, more = S % p.groups;
        part.nseq = each + (group < more ? 1 : 0);
        // (jobs of more than kPlannedSeqs sequences in all still hold at most MOST each)
        if (tid < part.nseq) plan.order[tid] = group * each + min(group, more) + tid;
    } else {
        const int from = __builtin_amdgcn_readfirstlane(plan.start[group]);
        part.nseq = __builtin_amdgcn_readfirstlane(plan.start[group + 1]) - from;
        part.order = plan.order + from;
        longest = part.nseq > 0 ? max(__builtin_amdgcn_readfirstlane(plan.length[from]), 1) : 0;
    }
    __syncthreads();
    // Steps of the pass: those on which a sequence is no padding, and where time runs forward one more, the first slot behind the
    // sequences, which still sees what the last one hands on.
    const bool forward_in_time = FWD ? part.dir == 0 : part.dir != 0;
    part.first = forward_in_time ? 0 : T - longest;
    part.last = (forward_in_time ? min(T, longest + 1) : T) - 1;
    part.begin = max(part.first, p.step_begin);
    part.end = min(part.last + 1, p.step_end);
    return part;
}

// The launch's steps that the job leaves out: what a padding slot gets there.  me = the workgroup's place in its team.
template <int JB, bool FWD>
__device__ __forceinline__ void fill_padding(const ChainParams &p, const LocalJob &part, int me) {
    const DirPtrs &D = p.d[part.dir];
    const int H = p.H, S = p.S, j0 = me * JB, per_step = part.nseq * JB;
    // before the job's steps or behind them
    const int b0 = p.step_begin, e0 = min(p.step_end, max(part.begin, b0)), b1 = max(part.end, e0), e1 = max(p.step_end, b1);
    const int before = e0 - b0, steps = before + (e1 - b1);
    const bool forward_in_time = FWD ? part.dir == 0 : part.dir != 0;
    // as many steps side by side as the workgroup has threads for
    const int rows = (int)blockDim.x / per_step, r = (int)threadIdx.x % per_step, c = j0 + r % JB, first = (int)threadIdx.x / per_step;
    if (first >= rows || c >= H) return;
    for (int q = first; q < steps; q += rows) {
        const int step = q < before ? b0 + q : b1 + q - before, t = forward_in_time ? step : p.T - 1 - step;
        const size_t slot = (size_t)t * S + part.order[r / JB], gi = slot * H + c, oi = slot * p.L + part.dir * H + c;
        if (FWD) {
            if (part.dir) D.c[gi] = 0.0f;
            D.h[gi] = 0.0f;
            if (p.out) p.out[oi] = 0.0f;
        } else {
            D.dni[gi] = 0.0f; D.dig[gi] = 0.0f; D.dfg[gi] = 0.0f; D.dog[gi] = 0.0f; D.cerr[gi] = 0.0f;
            // (a layer of one direction keeps the summed errors where the output errors stand: nothing is added here)
            if (!p.herr_out) D.herr[gi] = p.outerr[oi];
        }
    }
}

// v + (v rotated by N lanes within its row of sixteen).  Rotations by 8, 4, ... in this order add up what the lanes of a row
// that are N apart hold, with the same rounding in every one of them (each pair adds the same two values).
template <int N>
__device__ __forceinline__ float add_rotated(float v) {
    return v + __builtin_bit_cast(float, __builtin_amdgcn_update_dpp(0, __builtin_bit_cast(int, v), 0x120 + N, 0xF, 0xF, true));
}
// the sums of a and b over lanes 32 apart: a's in the lower half of the wave, b's in the upper one
__device__ __forceinline__ float sum_halves(float a, float b) {
    const auto r = __builtin_amdgcn_permlane32_swap(__builtin_bit_cast(unsigned, a), __builtin_bit_cast(unsigned, b), false, false);
    return __builtin_bit_cast(float, (unsigned)r[0]) + __builtin_bit_cast(float, (unsigned)r[1]);
}
// the sums of a and b over neighbouring rows of sixteen lanes: a's in the even rows, b's in the odd ones
__device__ __forceinline__ float sum_rows(float a, float b) {
    const auto r = __builtin_amdgcn_permlane16_swap(__builtin_bit_cast(unsigned, a), __builtin_bit_cast(unsigned, b), false, false);
    return __builtin_bit_cast(float, (unsigned)r[0]) + __builtin_bit_cast(float, (unsigned)r[1]);
}
// what is published may hold every value but the empty marker: a NaN that happens to look like it is sent as the NaN beside it
__device__ __forceinline__ unsigned publishable(float v) { return min(__builtin_bit_cast(unsigned, v), kEmpty - 1u); }
__device__ __forceinline__ void mail_store(const u32x4 &v, __amdgpu_buffer_rsrc_t mail, unsigned off, std::integral_constant<int, 4>) {
    __builtin_amdgcn_raw_buffer_store_b128(v, mail, (int)off, 0, 0);
}
__device__ __forceinline__ void mail_store(const u32x4 &v, __amdgpu_buffer_rsrc_t mail, unsigned off, std::integral_constant<int, 2>) {
    typedef unsigned u32x2 __attribute__((ext_vector_type(2)));
    __builtin_amdgcn_raw_buffer_store_b64(u32x2{v.x, v.y}, mail, (int)off, 0, 0);
}
__device__ __forceinline__ void mail_store(const u32x4 &v, __amdgpu_buffer_rsrc_t mail, unsigned off, std::integral_constant<int, 1>) {
    __builtin_amdgcn_raw_buffer_store_b32(v.x, mail, (int)off, 0, 0);
}
// The recurrent product of a wave: lane = 4 * block + row holds four neighbouring source values in `a`, and wreg[4 * I + r] is the
// weight of the r-th value of the I-th block of the lane's group of 2^CBSZ blocks.  Two accumulator chains: an instruction issues
// every 8 clocks and its result is there after 12.
template <int CBSZ, int K, int... I>
__device__ __forceinline__ f32x4 local_product(const f32x4 &a, const float (&wreg)[K], std::integer_sequence<int, I...>) {
    f32x4 acc0 = {0, 0, 0, 0}, acc1 = {0, 0, 0, 0};
    auto one = [&](auto block) __attribute__((always_inline)) {
        constexpr int b = decltype(block)::value;
        acc0 = __builtin_amdgcn_mfma_f32_4x4x1f32(a[0], wreg[4 * b + 0], acc0, CBSZ, b, 0);
        acc1 = __builtin_amdgcn_mfma_f32_4x4x1f32(a[1], wreg[4 * b + 1], acc1, CBSZ, b, 0);
        acc0 = __builtin_amdgcn_mfma_f32_4x4x1f32(a[2], wreg[4 * b + 2], acc0, CBSZ, b, 0);
        acc1 = __builtin_amdgcn_mfma_f32_4x4x1f32(a[3], wreg[4 * b + 3], acc1, CBSZ, b, 0);
    };
    (one(std::integral_constant<int, I>{}), ...);
    return acc0 + acc1;
}

// Diagnostic clocks (CNT_LSTM_TIMING, CNT_LSTM_TRACE): every kernel of the two recursions exists a second time, with CLOCKS, in
// which the workgroups add up what their waves spend in the parts of a step and, for some steps of the job, counted from its first, note when
// they pass five points of it, on the 100 MHz clock that all compute units share.  The kernels without are free of all of
// it: a branch on the chain of a step costs some of what it would measure.
constexpr unsigned kClockBlocks = 512;  // workgroups that record
enum { CLK_WAIT, CLK_REST, CLK_BARRIER, CLK_LOOP, CLK_ROUNDS, CLK_LOAD, CLK_STORE, CLK_OTHER, CLK_STEPS, kClockCounts };
constexpr int kTraceFirst = 64, kTraceSteps = 4, kTracePoints = 5, kTraceWords = 4 + kTraceSteps * kTracePoints;
constexpr size_t kClockWords = (size_t)kClockBlocks * (kClockCounts + kTraceWords);  // of one direction of time
template <bool CLOCKS>
__device__ __forceinline__ long long clock_now() {
    if constexpr (CLOCKS) return wall_clock64();
    return 0;
}
template <bool CLOCKS>
__device__ __forceinline__ void clock_add(long long &sum, long long since) {
    if constexpr (CLOCKS) sum += wall_clock64() - since;
}
// by one lane of the wave that counted
template <bool CLOCKS>
__device__ __forceinline__ void clock_store(const ChainParams &p, int what, long long v) {
    if constexpr (CLOCKS)
        if (blockIdx.x < kClockBlocks) p.clocks[(size_t)blockIdx.x * kClockCounts + what] = v;
}
template <bool CLOCKS>
__device__ __forceinline__ long long *clock_trace(const ChainParams &p) {
    if constexpr (CLOCKS)
        if (blockIdx.x < kClockBlocks) return p.clocks + (size_t)kClockBlocks * kClockCounts + (size_t)blockIdx.x * kTraceWords;
    return nullptr;
}
template <bool CLOCKS>
__device__ __forceinline__ void clock_point(const ChainParams &p, int step, int point) {
    if constexpr (CLOCKS) {
        long long *const trace = clock_trace<true>(p);
        if (trace && step >= kTraceFirst && step < kTraceFirst + kTraceSteps)
            trace[4 + kTracePoints * (step - kTraceFirst) + point] = wall_clock64();
    }
}
template <bool CLOCKS>
__device__ __forceinline__ void clock_where(const ChainParams &p, int job, int member) {
    if constexpr (CLOCKS)
        if (long long *const trace = clock_trace<true>(p)) {
            trace[0] = job; trace[1] = member;
            trace[2] = __builtin_amdgcn_s_getreg((3 << 11) | (0 << 6) | 20) & 15u;  // XCC_ID, bits 3:0
        }
}

// LDS of a job
template <int JB, int NSQ>
struct BackwardShared {
    using Shape = LocalShape<JB, NSQ>;
    static constexpr int EL = Shape::EL, RING = 2 * Shape::BATCH;
    static constexpr int DP = 4 * JB + 16;  // pitch of a sequence's deltas: the four sequences' rows on different banks
    __attribute__((aligned(16))) float dl[2][NSQ][DP];      // [sequence][cell][gate]
    // element = cell * NSQ + sequence, as in the messages
    __attribute__((aligned(16))) float coef[RING][EL][4];      // of e in d_og and in the cell error, stored d_og, e
    __attribute__((aligned(16))) float coef_own[RING][EL][4];  // of the cell error in d_ni, d_ig, d_fg; the cell state
    __attribute__((aligned(16))) float coef_fg[RING][EL][2];   // forget gate activation, 1: padding slot
    __attribute__((aligned(16))) float res[2][EL][2];       // summed output error, cell error
    int wait_failed;
};

// One job by one workgroup of its team.  PW = ceil(cells per direction / 64) product waves, JB cells per workgroup, a job of up to
// NSQ sequences
template <int PW, int JB, int NSQ, bool CLOCKS>
__device__ __forceinline__ void backward_job(const ChainParams &p, const LocalJob &part, int job, int me, unsigned mail_words, BackwardShared<JB, NSQ> &sh) {
    using Shape = LocalShape<JB, NSQ>;
    const int H = p.H, G = p.team;    // G = ceil(H / JB) workgroups; the last one may own fewer than JB cells
    constexpr int EL = Shape::EL, VEC = Shape::VEC, VPW = Shape::VPW, CW = Shape::CW;
    constexpr int STEPS = Shape::STEPS, BATCH = Shape::BATCH, SETS = Shape::SETS, RING = 2 * BATCH;
    constexpr int TEAM = (64 * PW + JB - 1) / JB;  // G at most
    constexpr int SPW = 64 / VPW;     // senders side by side in a polling wave
    constexpr int NL = (TEAM + SPW - 1) / SPW;  // 16-byte loads per polling lane; the last one may lie past the last sender
    constexpr int KW = 4 * JB;        // k extent of the product: (own cell, gate)
    constexpr int DP = BackwardShared<JB, NSQ>::DP;
    constexpr int NQ = (TEAM * VEC + 63) / 64;  // vectors per lane that hand a step's words back
    const unsigned RECV = (unsigned)(G * EL);   // words one receiver gets per step
    auto &dl = sh.dl;
    auto &coef = sh.coef;
    auto &coef_own = sh.coef_own;
    auto &coef_fg = sh.coef_fg;
    auto &res = sh.res;
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
    float *const mailbox = p.lmail + (size_t)job * mail_words;
    const unsigned slot_words = (unsigned)G * RECV;
    const __amdgpu_buffer_rsrc_t mail =
        __builtin_amdgcn_make_buffer_rsrc(mailbox, 0, (int)(local_job_words(G, JB, NSQ) * sizeof(float)), 0x00020000);
    const int last_step = part.last;  // of the pass: its partial errors go nowhere
    auto slot_of = [&](int step) { return dir ? step : (T - 1 - step); };
    // read through the LDS address space: a volatile read through a generic pointer becomes a flat load, which takes the
    // vector-memory path
    auto given_up = [&]() { return *(__attribute__((address_space(3))) volatile int *)&wait_failed; };

    // the load and the store wave: lane = (step of an access, sequence, cell)
    const int ej = lane % EL / JB, ec = lane % JB;  // the job's sequence ej, cell j0 + ec
    const bool valid = ej < nseq && j0 + ec < H;
    const int ahead = lane / EL;

    if (wave == PW + CW) {
        // ------------------------------------------------------------------ load wave
        struct StepIn { float e, ni, ig, fg, og, dog_old, c, c_earlier; char pat; };
        const int s = part.order[min(ej, nseq - 1)], el = ec * NSQ + ej;
        auto load_batch = [&](int first, StepIn (&in)[SETS]) {
#pragma unroll
            for (int i = 0; i < SETS; ++i) {
                StepIn &v = in[i];
                v = StepIn{0, 0, 0, 0, 0, 0, 0, 0, 1};
                const int step = first + i * STEPS + ahead;
                if (!valid || step >= end_step) continue;
                const int t = slot_of(step);
                const size_t gi = (size_t)t * n + (size_t)s * H + j0 + ec;
                v.e = p.outerr[((size_t)t * S + s) * p.L + dir * H + j0 + ec];
                v.ni = D.ni[gi]; v.ig = D.ig[gi]; v.fg = D.fg[gi]; v.og = D.og[gi];
                v.dog_old = D.dog[gi];
                v.c = D.c[gi];
                if (step + 1 < T) v.c_earlier = D.c[(size_t)slot_of(step + 1) * n + (size_t)s * H + j0 + ec];
                v.pat = p.pat[t * S + s];
            }
        };
        auto put_batch = [&](int first, const StepIn (&in)[SETS]) {
#pragma unroll
            for (int i = 0; i < SETS; ++i) {
                const StepIn &x = in[i];
                const int step = first + i * STEPS + ahead;
                if (step >= end_step) continue;
                const int t = slot_of(step), b = (int)((unsigned)(step - begin_step) % RING);
                const float tc = tanh_act(x.c);
                // d_og = first * e + stored d_og, cell error = second * e + ...
                *reinterpret_cast<f32x4 *>(coef[b][el]) = f32x4{logistic_deriv(x.og) * tc, x.og * tanh_deriv(tc), x.dog_old, x.e};
                *reinterpret_cast<f32x4 *>(coef_own[b][el]) = f32x4{x.ig * tanh_deriv(x.ni), logistic_deriv(x.ig) * x.ni,
                                                                    logistic_deriv(x.fg) * x.c_earlier, x.c};
                coef_fg[b][el][0] = x.fg;
                coef_fg[b][el][1] = ((t >= p.Tmin) && (x.pat == 0)) ? 1.0f : 0.0f;
            }
        };
        StepIn in[SETS];
        const int sb = begin_step;
        load_batch(sb, in);
        wait_all_vmem();
        put_batch(sb, in);
        long long busy = 0;
        lds_barrier();  // start of the recursion
        for (int step = sb; step < end_step; ++step) {
            lds_barrier();
            if (given_up()) return;
            const long long since = clock_now<CLOCKS>();
            const int phase = (int)((unsigned)(step - sb) % BATCH), next = step - phase + BATCH;
            if (phase == 0) {
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
        const int s = part.order[min(ej, nseq - 1)], el = ec * NSQ + ej;
        f32x4 d = {0, 0, 0, 0};
        float e = 0, ce = 0, c = 0, c_earlier = 0;
        double sums[kSmallSums] = {};  // over this lane's steps
        long long busy = 0;
        lds_barrier();  // start of the recursion
        for (int step = begin_step; step < end_step; ++step) {
            const int b = step & 1, held = (int)((unsigned)(step - begin_step) % STEPS);
            lds_barrier();  // results of this step are in LDS
            if (given_up()) return;
            const long long since = clock_now<CLOCKS>();
            if (ahead == held) {
                d = *reinterpret_cast<const f32x4 *>(&dl[b][ej][4 * ec]);
                e = res[b][el][0]; ce = res[b][el][1];
                if (p.sum_bias) {
                    // the next step's coefficients have been there since before this step's barrier; behind a job's last step the
                    // cell state is that of a padding slot or of none, whose delta is zero
                    c = coef_own[(unsigned)(step - begin_step) % RING][el][3];
                    c_earlier = step + 1 < end_step ? coef_own[(unsigned)(step + 1 - begin_step) % RING][el][3] : 0.0f;
                }
            }
            for (int i = 0; i < p.mem_delay; ++i) __builtin_amdgcn_s_sleep(1);
            wait_all_vmem();  // the stores of the step before are done
            if ((held == STEPS - 1 || step == end_step - 1) && valid && ahead <= held) {
                // an access stores as many steps as it has lanes for
                const size_t gi = (size_t)slot_of(step - held + ahead) * n + (size_t)s * H + j0 + ec;
                D.dni[gi] = d[0]; D.dig[gi] = d[1]; D.dfg[gi] = d[2]; D.dog[gi] = d[3];
                D.cerr[gi] = ce;
                if (p.herr_out) p.herr_out[gi] = e;
                else D.herr[gi] = e;
                if (p.sum_bias) {
                    const double c64 = c, earlier64 = c_earlier, d_ig = d[1], d_fg = d[2], d_og = d[3];
                    sums[0] += (double)d[0]; sums[1] += d_ig; sums[2] += d_fg; sums[3] += d_og;
                    sums[6] += c64 * d_og;
                    // (a job's last step has no earlier state: a zero in its place would be NaN with a delta that is not finite)
                    if (step - held + ahead + 1 < end_step) { sums[4] += earlier64 * d_ig; sums[5] += earlier64 * d_fg; }
                }
            }
            if (step > part.first) {
                // The words the cell waves consumed in this step (before the barrier) are empty again.  The slot is used
                // again three steps from now, so this hand-back can wait for this wave's turn instead of sitting in
                // front of the next poll in the compute unit's queue.
                const u32x4 empty = {kEmpty, kEmpty, kEmpty, kEmpty};
#pragma unroll
                for (int q = 0; q < NQ; ++q)
                    if (q * 64 + lane < G * VEC)
                        __builtin_amdgcn_raw_buffer_store_b128(empty, mail, (int)((unsigned)(step - 1) % kMailSlots * slot_words * 4u +
                                                               ((unsigned)me * RECV + (unsigned)(q * 64 + lane) * 4u) * 4u), 0, 0);
            }
            clock_add<CLOCKS>(busy, since);
        }
        if (p.sum_bias) {
            // a cell's sums of the steps and sequences of an access, JB lanes apart
#pragma unroll
            for (int k = 0; k < kSmallSums; ++k) {
                float v = (float)sums[k];
#pragma unroll
                for (int o = JB; o < 64; o *= 2) v += __shfl_xor(v, o);
                if (lane < JB && j0 + ec < H) put_sum(p, dir, job % p.groups, k, j0 + ec, v);
            }
        }
        if (lane == 0) clock_store<CLOCKS>(p, CLK_STORE, busy);
        return;
    }

    if (wave < PW) {
        // ------------------------------------------------------------------ product waves
        const int h = 64 * wave + lane;  // receiving cell of this lane (column of the B operand and of the accumulator)
        float wreg[KW];
#pragma unroll
        for (int k = 0; k < KW; ++k) {
            const int g = k % 4, jj = k / 4;
            wreg[k] = h < H && j0 + jj < H ? D.w_int[(size_t)g * p.L * H + (size_t)(j0 + jj) * H + h] : 0.0f;
        }
        // with eight cells the two halves of the wave hold the same eight blocks of the A operand
        const float *const mine = &dl[0][(lane & 3) % NSQ][4 * ((lane >> 2) % JB)];
        const unsigned pub_off = ((unsigned)(h / JB) * RECV + (unsigned)me * EL + (unsigned)(h % JB) * NSQ) * 4u;
        const bool publishes = h < G * JB;
        long long busy = 0;
        wait_all_vmem();
        lds_barrier();  // start of the recursion
        for (int step = begin_step; step < end_step; ++step) {
            lds_barrier();  // the deltas of this step are in LDS
            const long long since = clock_now<CLOCKS>();
            if (tid == 0) clock_point<CLOCKS>(p, step - begin_step, 3);
            // looked at only at the end of the step: the read is in flight behind the barrier together with the
            // deltas', and what a failed step publishes no longer matters
            const f32x4 a = *reinterpret_cast<const f32x4 *>(mine + (step & 1) * NSQ * DP);
            const int failed = given_up();
            // everything this wave stored in the previous step has reached the L2 before it publishes again
            wait_all_vmem();
            if (step < last_step) {
                const f32x4 sum = local_product<JB == 8 ? 3 : 4, KW>(a, wreg, std::make_integer_sequence<int, JB>{});
                const u32x4 v = {publishable(sum[0]), publishable(sum[1]), publishable(sum[2]), publishable(sum[3])};
                if (publishes)
                    mail_store(v, mail, (unsigned)step % kMailSlots * slot_words * 4u + pub_off, std::integral_constant<int, NSQ>{});
            }
            clock_add<CLOCKS>(busy, since);
            if (tid == 0) clock_point<CLOCKS>(p, step - begin_step, 4);
            if (failed) return;
        }
        if (tid == 0) clock_store<CLOCKS>(p, CLK_OTHER, busy);
        return;
    }

    // ---------------------------------------------------------------------- cell waves
    // polling role: lane l reads vector l % VPW of the wave's VPW of the senders l / VPW + SPW * i
    const int cw = wave - PW;
    const int vec = cw * VPW + lane % VPW;
    const unsigned poll_off = ((unsigned)me * RECV + (unsigned)((lane / VPW) * EL + vec * 4)) * 4u;
    constexpr unsigned poll_stride = (unsigned)SPW * EL * 4u;
    // lanes past the last sender poll their first vector once more and leave it out of the sum
    const bool last_counts = lane / VPW + SPW * (NL - 1) < G;
    const int pause = min(p.poll_limit, p.poll_delay >= 0 ? p.poll_delay : backward_pause(EL));
    const unsigned poll_off_last = last_counts ? poll_off + (unsigned)(NL - 1) * poll_stride
                                               : ((unsigned)me * RECV + (unsigned)(vec * 4)) * 4u;
    // cell-update role: after the sum a lane holds word lane / 16 of its vector; of the copies in the row each takes a gate
    const int el = vec * 4 + (lane >> 4), cc = el / NSQ, cj = el % NSQ, gate = lane / VPW % 4;
    const bool real_cell = j0 + cc < H;
    float p_og = 0, p_own = 0;
    if (real_cell) {
        p_og = D.peep[2][j0 + cc];
        if (gate == 1 || gate == 2) p_own = D.peep[gate - 1][j0 + cc];
    }
    const bool peeps = gate == 1 || gate == 2;
    float fg_later = 0, cerr_later = 0, own_later = 0;
    if (begin_step > part.first && real_cell && cj < nseq) {
        // a launch that starts in the middle: what the step before carried over stands in the state arrays
        const size_t gi = (size_t)slot_of(begin_step - 1) * n + (size_t)part.order[cj] * H + j0 + cc;
        fg_later = D.fg[gi]; cerr_later = D.cerr[gi];
        if (peeps) own_later = gate == 1 ? D.dig[gi] : D.dfg[gi];
    }
    long long waited = 0, rest = 0, barrier = 0, rounds = 0;
    const bool records = CLOCKS && cw == 0 && lane == 0;
    wait_all_vmem();  // peepholes are in registers before the recursion starts
    lds_barrier();    // start of the recursion: coefficients of steps 0 and 1 are in LDS
    const long long begin = clock_now<CLOCKS>();

    for (int step = begin_step; step < end_step; ++step) {
        const bool first = (step == part.first), last = (step == T - 1);
        const int b = step & 1, r = (int)((unsigned)(step - begin_step) % RING);
        const long long since = clock_now<CLOCKS>();
        if (records) clock_point<CLOCKS>(p, step - begin_step, 0);
        // this step's coefficients: in LDS since before the previous barrier, fetched while the poll is in flight
        const f32x4 k = *reinterpret_cast<const f32x4 *>(coef[r][el]);
        const float k_own = coef_own[r][el][gate], fg = coef_fg[r][el][0], dummy = coef_fg[r][el][1];
        float carry = peeps ? p_own * own_later : 0.0f;
        if (VPW == 4) carry = add_rotated<4>(add_rotated<8>(carry));
        else carry = add_rotated<2>(add_rotated<4>(carry));
        carry = first ? 0.0f : fg_later * cerr_later + carry;
        const bool no_delta = dummy != 0.0f || (last && gate == 2);
        float e = k[3];
        // what does not wait for the poll is worked out while it is in flight (the compiler would move it behind)
        unsigned to_dl = (unsigned)((b * NSQ + cj) * DP + 4 * cc + gate), to_res = (unsigned)((b * EL + el) * 2 + gate);
        asm volatile("" : "+v"(carry), "+v"(to_dl), "+v"(to_res));
        if (!first) {
            const float *slot = mailbox + (size_t)((unsigned)(step - 1) % kMailSlots) * slot_words;
            u32x4 w[NL];
            unsigned spins = 0;
            for (int d = 0; d < pause; ++d) __builtin_amdgcn_s_sleep(1);
            for (;;) {
                poll_load<NL>(slot, poll_off, poll_stride, poll_off_last, w);
                if constexpr (CLOCKS) ++rounds;
                unsigned worst = 0;
#pragma unroll
                for (int i = 0; i < NL; ++i) worst = max(max(worst, w[i].x), max(max(w[i].y, w[i].z), w[i].w));
                if (__builtin_amdgcn_ballot_w64(worst == kEmpty) == 0) break;
                if (poll_gives_up(p, ++spins)) {
                    wait_failed = 1;
                    if (lane == 0) raise_abort(p);
                    break;
                }
                for (int d = 0; d < p.poll_gap; ++d) __builtin_amdgcn_s_sleep(1);
            }
            clock_add<CLOCKS>(waited, since);
            if (records) clock_point<CLOCKS>(p, step - begin_step, 1);
            f32x4 sum = __builtin_bit_cast(f32x4, w[NL - 1]);
#pragma unroll
            for (int r = 0; r < 4; ++r) sum[r] = last_counts ? sum[r] : 0.0f;
#pragma unroll
            for (int i = 0; i + 1 < NL; ++i) sum += __builtin_bit_cast(f32x4, w[i]);
            const float even = sum_halves(sum[0], sum[2]), odd = sum_halves(sum[1], sum[3]);
            float total = add_rotated<4>(add_rotated<8>(sum_rows(even, odd)));
            if (VPW == 2) total = add_rotated<2>(total);
            e += total;
        }
        const float d_og = k[0] * e + k[2];
        float ce = k[1] * e + p_og * d_og;
        ce += carry;
        float own = gate == 3 ? d_og : k_own * ce;
        const float clipped = __builtin_amdgcn_fmed3f(own, -1.0f, 1.0f);  // clip1, with the test for NaN beside it
        own = no_delta ? 0.0f : own == own ? clipped : own;
        ce = dummy != 0.0f ? 0.0f : ce;
        (&dl[0][0][0])[to_dl] = own;
        if (gate < 2) (&res[0][0][0])[to_res] = gate ? ce : e;
        fg_later = fg; cerr_later = ce; own_later = own;
        if (records) clock_point<CLOCKS>(p, step - begin_step, 2);
        const long long at_barrier = clock_now<CLOCKS>();
        lds_barrier();
        clock_add<CLOCKS>(barrier, at_barrier);
        clock_add<CLOCKS>(rest, since);  // the whole step: what was waited is taken off below
        if (given_up()) return;
    }
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

// the sums of a job that takes no step
template <int JB>
__device__ __forceinline__ void no_sums(const ChainParams &p, int dir, int job, int me) {
    const int u = me * JB + (int)threadIdx.x;
    if (p.sum_bias && threadIdx.x < JB && u < p.H)
        for (int k = 0; k < kSmallSums; ++k) put_sum(p, dir, job % p.groups, k, u, 0.0f);
}

template <int PW, int JB, int MOST, bool CLOCKS>
__global__ __launch_bounds__(local_threads(PW, JB, MOST)) void lstm_backward_local(const ChainParams p) {
    __shared__ LocalPlan plan;
    __shared__ union Shared { BackwardShared<JB, 1> one; BackwardShared<JB, MOST < 2 ? 1 : 2> two; BackwardShared<JB, MOST> most; } sh;
    int job = -1, me = 0;
    const LocalJob part = local_setup<MOST, false>(p, plan, job, me);
    if (part.nseq == 0) {  // no job (-1), or a group that no sequence was left for
        if (job >= 0) no_sums<JB>(p, part.dir, job, me);
        return;
    }
    fill_padding<JB, false>(p, part, me);
    if (part.begin >= part.end) {
        no_sums<JB>(p, part.dir, job, me);
        return;
    }
    const unsigned mail_words = (unsigned)local_job_words(p.team, JB, MOST);
    if (threadIdx.x == 0) (part.nseq == 1 ? sh.one.wait_failed : part.nseq == 2 ? sh.two.wait_failed : sh.most.wait_failed) = 0;
    if (MOST == 1 || part.nseq == 1) backward_job<PW, JB, 1, CLOCKS>(p, part, job, me, mail_words, sh.one);
    else if (part.nseq == 2) backward_job<PW, JB, MOST < 2 ? 1 : 2, CLOCKS>(p, part, job, me, mail_words, sh.two);
    else backward_job<PW, JB, MOST, CLOCKS>(p, part, job, me, mail_words, sh.most);
}
