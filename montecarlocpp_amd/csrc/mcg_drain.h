// mcg_drain.h -- the drain of the general kernel's wavefronts (included by
// mcg_kernels.hip after mcg_box.h, whose box_drain is the same scheme for
// scenes of one box and says what bounds it).
//
// A wavefront left with at most kDrainLanes bundles and no id to claim gives
// its idle lanes the work that does not depend on the bundles' paths: the
// draws of their next events, and the tallies of their flights.
// It is a function of its own, called at most once by a wavefront: inlined, its
// values took registers from the step loop, which spilled 18 to 322 vector
// registers in FP32 and 54 to 317 in FP64 and now spills none and at most 16.
// It publishes the wavefront's statistics (a second round of atomics on the
// same counters cost 40 us a launch).
// Measured, without a drain / inlined / called, same box: tee with 6 x 6 maps
// 1e6 bundles FP32 18.0 / 18.0 / 16.1 ms, FP64 23.2 / 26.0 / 16.8; with 6 x 6 x 2
// maps FP64 24.3 / 49.8 / 18.1; octet truss of finer struts 1e6 FP64 7.8 / 14.5 /
// 6.0; octet 1e6 FP32 2.39 / 2.03 / 1.92; porous film, CumTemp 3e6 FP64 15.6 /
// 23.2 / 15.5; two boxes 1e5 FP32 0.24 / 0.19 / 0.16.
#pragma once

// The kernel's parameters and its LDS as plain numbers, to hand to the drain.
__device__ __forceinline__ uint64_t kernarg_address() {
    return (uint64_t)__builtin_amdgcn_kernarg_segment_ptr();
}
__device__ __forceinline__ uint32_t lds_offset(unsigned char* lds) {
    return (uint32_t)(uintptr_t)(__attribute__((address_space(3))) unsigned char*)lds;
}

// What an event may draw, for any kind of cell.
template <typename F>
struct EventDraws {
    dev::V3<F> iso, lam;     // isotropic; Lambertian about z
    F path;
    uint32_t mode, spec;
};

template <typename F>
__device__ __forceinline__ EventDraws<F> event_draws(const KParams<F>& K, const View<F>& V, uint32_t event,
                                                     int64_t id) {
    const dev::Event ev{K.k0, K.k1, event, uint32_t(id), uint32_t(uint64_t(id) >> 32)};
    const uint4 b0 = ev.block(0), b1 = low_block<F>(ev, 1);
    EventDraws<F> D;
    D.spec = spec_word<F>(ev, b1);
    const F r = dev::Real<F>::uniform(b0.x, b1.x) * F(2) + F(-1);
    const F ar = r < F(0) ? -r : r;
    const F si = dev::Real<F>::sqrt_(F(1) - r * r), sl = dev::Real<F>::sqrt_(ar);
    const F q = dev::Real<F>::uniform(b0.y, b1.y) * F(2) + F(-1);
    F sq, cq;
    dev::Real<F>::sincos_pi(q, sq, cq);
    D.iso = dev::V3<F>{si * cq, si * sq, r};
    D.lam = dev::V3<F>{sl * cq, sl * sq, dev::Real<F>::sqrt_(F(1) - ar)};
    D.mode = dev::alias_draw(V.scat, uint32_t(K.nmodes), b0.w);
    D.path = draw_path<F>(ev, b0, b1, V.mfp[D.mode]);
    return D;
}

// The collision of collide_step with the event's draws given.
template <typename F>
__device__ __forceinline__ void collide_drawn(const KParams<F>& K, const View<F>& V, int hit, Lane<F>& L,
                                              const EventDraws<F>& D, uint32_t& fate, int32_t pbeg, int32_t pore) {
    const bool intr = hit == -1, wall = hit == -3;
    const DevPlane<F>& P = V.planes[hit >= 0 ? hit : pbeg];
    int kind = intr ? -1 : (wall ? V.pores[wall ? pore : 0].kind : P.kind);
    if (kind == MCG_PARTIAL) kind = D.spec < (wall ? V.pores[wall ? pore : 0].spec_thr : P.spec_thr) ? MCG_SPEC : MCG_DIFF;
    L.nscat += intr || kind == MCG_DIFF ? 1u : 0u;
    L.nbdry += intr ? 0u : 1u;
    if (intr) {
        L.dir = dev::normalized(D.iso);
        L.mode = D.mode;
        L.scat_next = D.path;
    } else if (kind == MCG_DIFF || kind == MCG_SPEC) {
        F m[9];
        if (wall) {
            const dev::V3<F> n = wall_normal(V.pores[pore], L.pos);
            if (kind == MCG_SPEC) reflection_off(n, m);
            else rotation_to_wall(n, m);
        } else {
            const F* M = kind == MCG_SPEC ? P.refl : P.rot;
#pragma unroll
            for (int i = 0; i < 9; ++i) m[i] = M[i];
        }
        L.dir = dev::normalized(dev::matvec(m, kind == MCG_DIFF ? D.lam : L.dir));
    } else if (kind == MCG_PERI) {
        const dev::V3<F> p = dev::matvec(P.prot, L.pos);
        L.pos = dev::V3<F>{p.x + P.pt[0], p.y + P.pt[1], p.z + P.pt[2]};
        L.dir = dev::normalized(dev::matvec(P.prot, L.dir));
        L.sdom = P.target;
    } else if (kind == MCG_ISOT) {
        fate = MCG_ABSORBED;
    } else {
        const int target = inter_target<F>(K, V, P, L.pos);
        if (target < 0) fate = MCG_ESCAPED;
        else L.sdom = target;
    }
    if (fate == kAlive) {
        if (int64_t(L.nscat) >= K.maxscat) fate = MCG_MAXSCAT;
        else if (L.nstep >= K.maxloop) fate = MCG_MAXLOOP;
    }
}

template <typename F, bool kLdsTables, bool kLdsTally, int kDefer>
__device__ __attribute__((noinline)) void general_drain(uint64_t params, uint32_t lds_at, int lane, Lane<F> L,
                                                        bool active, LaneStats st) {
    // arguments arrive in vector registers: the parameters' and LDS addresses
    // are the same in all lanes
    const uint64_t at_params = (uint64_t(uint32_t(__builtin_amdgcn_readfirstlane(int(params >> 32)))) << 32) |
                               uint32_t(__builtin_amdgcn_readfirstlane(int(uint32_t(params))));
    const KParams<F>& K = *(const KParams<F>*)(ParamPtr<F>)at_params;
    unsigned char* const lds = (unsigned char*)(__attribute__((address_space(3))) unsigned char*)(uintptr_t)
        __builtin_amdgcn_readfirstlane(int(lds_at));
    const View<F> V = view_of<F, kLdsTables, kLdsTally>(K, lds);
    const Sink sink{V.direct, V.diff, K.cols};
    const uint64_t lt_mask = (lane == 0) ? 0ull : (~0ull >> (kWave - lane));
    int span = 2 * kDrainLanes, shift = 0;
    int at = 0, ahead = 0, slot = 0;
    EventDraws<F> D;
    dev::V3<F> fpre, fpos;                 // this lane's flight to tally
    F fdmin = F(0);
    uint32_t fmode = 0, fnscat = 0;
    int32_t fcell = 0;                     // 2 cell + (sign < 0)
    bool pending = false;
    for (;;) {
        const uint64_t live = __ballot(active);
        if (live == 0ull || slot + span > kWave) {
            WalkOf<F, kDefer> W;
            bool walking = false;
            if (pending)
                walking = tally_step<F, kDefer>(K, V.sdoms[fcell >> 1], sink, fpre, fpos, fdmin, V.vel[fmode],
                                                fcell & 1 ? -1 : 1, fnscat, W);
            if constexpr (kDefer != 0)
                while (__ballot(walking) != 0ull) walk_some<kWalkUnroll>(W, walking, sink);
            pending = false;
            slot = 0;
        }
        if (live == 0ull) break;
        const int n = popc(live);
        if (2 * n <= span) {
            const int to = active ? popc(live & lt_mask) : n + popc(~live & lt_mask);
            const int from = 4 * __builtin_amdgcn_ds_permute(4 * to, lane);
            L.pos = lane_pull(from, L.pos);
            L.dir = lane_pull(from, L.dir);
            L.scat_next = lane_pull(from, L.scat_next);
            L.mode = lane_pull(from, L.mode);
            L.sdom = lane_pull(from, L.sdom);
            L.sign = lane_pull(from, L.sign);
            L.nscat = lane_pull(from, L.nscat);
            L.nbdry = lane_pull(from, L.nbdry);
            L.nstep = lane_pull(from, L.nstep);
            L.id = lane_pull(from, L.id);
            active = lane < n;
            span = 1;
            shift = 6;
            while (span < n) {
                span *= 2;
                --shift;
            }
            ahead = at = 0;
        }
        if (at == ahead) {
            const int of = 4 * (lane >> shift);
            const int64_t id = lane_pull(of, L.id);
            const uint32_t event = lane_pull(of, L.nstep) + 1u + uint32_t(lane & ((1 << shift) - 1));
            D = event_draws<F>(K, V, event, id);
            at = 0;
            ahead = 1 << shift;
        }
        EventDraws<F> E;
        const int src = 4 * (((lane << shift) + at) & (kWave - 1));
        E.iso = lane_pull(src, D.iso);
        E.lam = lane_pull(src, D.lam);
        E.path = lane_pull(src, D.path);
        E.mode = lane_pull(src, D.mode);
        E.spec = lane_pull(src, D.spec);
        ++at;
        dev::V3<F> pre = L.pos;
        F dmin = F(0);
        uint32_t fate = kAlive;
        int hit = -1;
        int32_t pbeg = 0, pore = -1;
        if (active) hit = advect_step<F>(V, L, fate, dmin, pre, pbeg, pore);
        const bool flown = active && fate == kAlive;
        const uint64_t flights = __ballot(flown);
        const int give = lane - slot;
        const int giver = 4 * (give & (kWave - 1));
        const dev::V3<F> gpre = lane_pull(giver, pre), gpos = lane_pull(giver, L.pos);
        const F gdmin = lane_pull(giver, dmin);
        const uint32_t gmode = lane_pull(giver, L.mode), gnscat = lane_pull(giver, L.nscat);
        const int32_t gcell = lane_pull(giver, 2 * L.sdom + (L.sign < 0 ? 1 : 0));
        if (uint32_t(give) < uint32_t(span) && (flights >> (give & (kWave - 1)) & 1ull)) {
            fpre = gpre;
            fpos = gpos;
            fdmin = gdmin;
            fmode = gmode;
            fnscat = gnscat;
            fcell = gcell;
            pending = true;
        }
        slot += span;
        if (flown) collide_drawn<F>(K, V, hit, L, E, fate, pbeg, pore);
        if (active && fate != kAlive) {
            if (K.c_nscat) {
                const int64_t k = L.id - K.first;
                K.c_nscat[k] = L.nscat;
                K.c_nbdry[k] = L.nbdry;
                K.c_nstep[k] = L.nstep;
                K.c_fate[k] = fate;
            }
            st.add(fate, L.nstep);
            active = false;
        }
    }
    st.publish(K.counters, lane);
}
