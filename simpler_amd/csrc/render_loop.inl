// render_loop.inl -- the path kernels' loop: runs until the launch's photons, or
// the group's (GROUPS), are taken and the wave's lanes and stack are empty.
// The text of a function body, included where FIELD, MODE, BATCH, JLDS, MM, GA,
// SPLAT, STEPS, GROUPS, STACK, SPLIT, the arguments S0 and A0, the shared arrays, group
// and wave_steps are declared.  As a function that takes the arguments by
// reference, or by value, it made the 2^17-photon spline render 13 % slower
// (136 -> 154 ms: the compiler keeps other scene scalars in registers).
    Hot h;
    h.steps = 0;
    h.state = ST_NEED;
    h.dead = false;
    PendSplat ps;
    ps.valid = false;
    Tan tan;
    SplineCell scell;
    scell.key = -1;
    int cfg = 0;        // batch: the lane's configuration
    bool left = true;   // photons left in the launch's queue (uniform)
    while (true) {
        // The event code reads the scene, the arguments and its addresses
        // anew on every turn: held across the march loop (about 200 scalars
        // and a few vectors) they would fill the registers and be spilled.
        const DevScene &S = kernel_arg<DevScene>(0);
        const RenderArgs &A = kernel_arg<RenderArgs>(kArgsOffset);
        int tid = (int)threadIdx.x;
        asm volatile("" : "+v"(tid));
        Var vsingle = var_from(S, A);
        if (JLDS && !BATCH) vsingle.f.jtab = jlds;
        // batch: the lane's configuration, read from global memory (L1/L2
        // resident), replaced when the lane takes a photon of another one
        const bool first = !SPLIT || (tid & (S.src_lanes - 1)) == 0;
        Lane L{h, cold[tid], BATCH ? const_cast<Var *>(A.cfgs) + cfg : &vsingle, S, A, first ? cnt : uncounted, nullptr,
               &mcache[tid], SPLAT ? &ps : nullptr, MODE == M_JVP ? &tan : nullptr};
        const int lane = __lane_id();
        if (STACK) {
            const int wave = __builtin_amdgcn_readfirstlane((int)((blockIdx.x * blockDim.x + tid) >> 6));
            L.qn = &nheld[tid >> 6];
            L.qcap = wave < A.nq_waves ? A.nq_cap : 0;
            L.q = A.nq + (size_t)wave * A.nq_cap * job_vec(MODE);
            L.cfg = cfg;
        }
        // fetch: first the wave's next-event stack, then new photons, one
        // atomic per wave for all lanes that take one
        unsigned long long need = __ballot(h.state == ST_NEED);
        if (STACK && need) {
            const uint32_t held = __builtin_amdgcn_readfirstlane(wave_get(L.qn));
            if (held) {
                const uint32_t want = (uint32_t)__popcll(need);
                const uint32_t rank = (uint32_t)__popcll(need & ((1ull << lane) - 1ull));
                if (lane == 0) wave_set(L.qn, held - min(held, want));
                __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
                if (h.state == ST_NEED && rank < held) {
                    nee_pop<FIELD, MODE, BATCH>(L, held - 1u - rank);
                }
                // lanes that found no entry take a photon
                need = __ballot(h.state == ST_NEED && rank >= held);
            }
        }
        const int share = GROUPS ? A.g_photons[group] : A.wave_photons;
        if (STACK && need && left && share < 64) {  // fewer photons than lanes: spread over the waves
            const int mains = __popcll(__ballot(h.state != ST_NEED && L.c.phase != PH_JOB));
            const int room = max(share - mains, 0);
            while (__popcll(need) > room) need &= need - 1ull;
        }
        if (need && left) {
            // the lanes that take: of a ray's lanes the first one
            const unsigned long long take = SPLIT ? __ballot(h.state == ST_NEED && first) : need;
            const unsigned long long base = wave_take(GROUPS ? A.work + group : A.work, take);
            const uint64_t n = GROUPS ? A.g_count[group] : A.n;
            left = base + __popcll(take) < n;
            if ((need >> lane) & 1ull) {
                const int taker = SPLIT ? lane & ~(S.src_lanes - 1) : lane;
                const unsigned long long rank = __popcll(take & ((1ull << taker) - 1ull));
                const unsigned long long idx = base + rank;
                if (idx < n) {
                    uint64_t pid = A.offset + idx;
                    if (BATCH) {
                        // index over all configurations
                        int lo;
                        pid = batch_photon(A, (GROUPS ? A.g_start[group] : A.offset) + idx, lo);
                        L.v = const_cast<Var *>(A.cfgs + lo);  // its image pointer is set per launch
                        L.cfg = lo;
                    }
                    L.c.pid_lo = (uint32_t)pid;
                    L.c.pid_hi = (uint32_t)(pid >> 32);
                    h.state = ST_INIT;
                }
            }
        }
        if (h.state == ST_INIT) photon_init<FIELD, MODE>(L);
        if (h.state == ST_SEG_END) seg_end<FIELD, MODE>(L);
        if (SPLAT) wave_splat(ps, A);
        if (__ballot(h.state == ST_MARCH) == 0ull) {
            if (__ballot(h.state != ST_NEED) == 0ull && !left && (!STACK || __builtin_amdgcn_readfirstlane(wave_get(L.qn)) == 0u)) break;
            continue;
        }
        if (BATCH) cfg = L.cfg;
        FieldP F = BATCH ? L.v->f : field_params(S0);
        if (JLDS) F.jtab = BATCH ? jlds + (F.jtab - A.jtab_base) : jlds;
        float Lcut = BATCH ? L.v->Lcut : S0.Lcut;
        // held in a vector register through the march loop: the kernel's
        // scalar registers are full, and a scalar copy is reloaded from its
        // spill lanes on every step
        asm volatile("" : "+v"(Lcut));
        bool m = h.state == ST_MARCH;
        uint32_t sl = h.steps_left;
        if constexpr (MODE == M_JVP) {
            for (int k = 0; k < A0.spc; ++k) {
                wave_steps += __popcll(__ballot(m));  // one ER step per marching lane
                if (m) m = !march_step_jvp<FIELD>(h, tan, sl, S0, F, Lcut, A0.theta_dot);
            }
        } else if constexpr (STEPS) {
            for (int k = 0; k < A0.spc; ++k) {
                wave_steps += __popcll(__ballot(m));
                if (m) m = !march_step<FIELD, false, MM, false, GA>(h, sl, S0, F, Lcut);
            }
        } else {
            march_chunk<FIELD, false, MM, GA, FIELD == kSpline>(h, sl, m, A0.spc, S0, F, Lcut, &scell, wave_steps);
        }
        h.steps_left = sl;
        if (h.state == ST_MARCH && !m) h.state = ST_SEG_END;
    }
