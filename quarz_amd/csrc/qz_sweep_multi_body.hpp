// Body of the persistent gfx950 kernel of one quasi-static sweep (the slice loop of Simulation::step_fields,
// src/Simulation.cpp:727-783) run by G cooperating workgroups.  It serves runs that one workgroup cannot hold:
// more than 4096 plasma particles per slice, or grids whose solve sets do not fit one compute unit's LDS (the
// m = 0 + 1 long-box workload: 32768 particles, 1025 nodes).
//
// Workgroup g owns the particles [g P, (g + 1) P) of the run (P = 512 x PT) for the whole sweep.  Per slice:
//   1. geometry of the owned particles (registers) and a stable counting sort by cell in LDS;
//   2. the per-cell counts of every workgroup meet in global memory (grid barrier); each workgroup reads them
//      all and forms the global cell starts and its own offsets, so that every contribution gets its position in
//      its node's list in global particle-index order: workgroups hold consecutive index ranges, so the particles
//      of earlier workgroups come first, and within a workgroup the local sort gives the order;
//   3. the contributions to every deposit array go to these global lists, an entry holding all arrays side by side
//      (grid barrier); a lane sums one or three arrays of a node's list sequentially -- the serial atomic_add order --
//      and adds the background and beam sources (combine_sources) (grid barrier);
//   4. the solves: the psi / E_z / B_z systems of L0, those of L1D (m = 1) and the chi-dependent Thomas factors
//      of the B+ operators are three jobs for three workgroups, each staging its operators in its own LDS and
//      running its chains in one wave (qz_chain.hpp) (grid barrier);
//   5. every workgroup forms W+ from psi and stages W+, E_z, B_z in LDS; the owned particles gather them, keep the
//      gathered values in the workspace for the push and write their S+ contributions (grid barrier); the node sums
//      of S+ as in 3 (grid barrier);
//   6. the Picard iterations of B+: the systems of each operator pair are one job per workgroup, reading the
//      previous iterate of the coupled modes from global memory and writing the next one to the other of two
//      buffers (one grid barrier per iteration);
//   7. the field store (node ranges per workgroup) and the Adams-Bashforth push of the owned particles.
// The grid barrier is a counter in the run's workspace that only grows during a launch: barrier n of the launch
// completes when it reaches n G; the last workgroup to leave the launch puts it back to zero.  Every wait is bounded in
// time: a barrier not reached within two seconds marks the run's error flag and ends the launch in every workgroup, and
// the host reports it.  Whatever crosses a barrier is stored through to memory (share).  A launch is refused unless all its
// workgroups (and those of the launches the caller keeps in flight beside it) fit the device together, one per
// compute unit, so every workgroup is resident.  Arithmetic per term is that of the one-workgroup kernel
// (qz_sweep.hip), so the result is the serial oracle's bit for bit.
#pragma once

#include <hip/hip_runtime.h>

#include <algorithm>
#include <vector>

#include "qz_device.hpp"
#include "qz_internal.hpp"
#include "qz_sweep_common.hpp"

namespace qz {

namespace {
constexpr int mBS = 512;              // threads per workgroup
constexpr int mNW = mBS / 64;         // waves per workgroup
constexpr int mLds = 160 * 1024;      // LDS bytes per workgroup
constexpr unsigned long long kBarrierTicks = 200000000ull;   // 2 s of the 100 MHz wall clock

// layout of the multi-workgroup workspace of a run (doubles): misc | counts | lists | Picard second buffer | the fields
// every particle gathered for S+ (W+ x, y, E_z, B_z), which its push takes again.  These last are their own workgroup's
// and stay in its L2, so a cache line lies between them and what the workgroups share, and after them.
constexpr int kLineDoubles = 16;
constexpr int kEntrySlots = 24;   // doubles of a list entry in m = 1 (8 in m = 0)
// bw0 of the chi factors: lines away from the counters, which atomics change in place, and from the counts
constexpr int kBw0 = 2 * kLineDoubles;
struct MwsLayout {
    size_t misc = 0, cnt, lists, bpalt, gath, total;
    __host__ __device__ MwsLayout(int M, int N, int np, int G, bool m1) {
        cnt = 64;   // words 0 barrier, 1 exit count, 2 error; doubles [kBw0, kBw0 + 4) bw0
        lists = cnt + (static_cast<size_t>(G) * (N + 1) + 1) / 2 + 1;     // G x N ints
        lists = (lists + kLineDoubles - 1) / kLineDoubles * kLineDoubles;
        bpalt = lists + static_cast<size_t>(kEntrySlots) * 2 * (np > 1 ? np : 1);
        gath = bpalt + static_cast<size_t>(m1 ? 6 : 2) * M + kLineDoubles;
        total = gath + 4 * static_cast<size_t>(np) + kLineDoubles;
    }
};

// LDS carve-up (bytes): r | 1/h | 1/V | local cell starts | global cell starts | own offsets | misc (flags, counts, the
// deposit array list) | region (Mp-double slots).  The sort's wave counters and sorted slots lie at the start of the
// region: nothing else is in it while the particles are sorted.
struct MLds {
    int Mp, wcnt, cs, gcs, goff, sidx, misc, region, sort;
    __host__ __device__ MLds(int N, int pt) {
        const int M = N + 1;
        Mp = (M + 1) & ~1;
        cs = 3 * Mp * 8;
        gcs = cs + ((((N + 3) * 4) + 15) & ~15);
        goff = gcs + ((((N + 3) * 4) + 15) & ~15);
        misc = goff + ((((N + 2) * 4) + 15) & ~15);
        region = misc + 256;
        wcnt = region;
        sidx = wcnt + (((mNW * N * 2) + 15) & ~15);
        sort = sidx + (((mBS * pt * 2) + 15) & ~15) - region;   // bytes of the sort's arrays
    }
};

// region slots (Mp doubles each)
template <bool M1> struct MSlots {
    // fields staged for the S+ gather and the push: W+ (r1 i1 r0 i0 r2 i2), E_z modes, B_z modes
    static constexpr int W = 0, EZ = M1 ? 6 : 2, BZ = EZ + (M1 ? 3 : 1), NFIELD = BZ + (M1 ? 3 : 1);
    // the largest job: m = 1 the chi factors (three operators and chi0), m = 0 the Picard pair (two a, two factor
    // pairs, two right-hand sides)
    static constexpr int NJOB = M1 ? 10 : 8;
    static constexpr int NREGION = NFIELD > NJOB ? NFIELD : NJOB;
    // doubles of a list entry: every deposit array of one particle and node side by side, in the order of entry_comp
    static constexpr int ENTRY = M1 ? kEntrySlots : 8;
    // and of S+ (r1 i1 r0 i0 r2 i2), and the doubles its entry takes
    static constexpr int NS = M1 ? 6 : 2, SENTRY = M1 ? 8 : 2;
};
__device__ constexpr int entry_comp(int slot) {
    constexpr int order[kEntrySlots] = {W_CHI0, W_RHOT0, W_DRHO0, W_JZ0, W_NE0, W_NI0, W_JPR1, W_JPI1,
                                        W_CHI1R, W_CHI1I, W_RHOT1R, W_RHOT1I, W_DRHO1R, W_DRHO1I, W_JZ1R, W_JZ1I,
                                        W_NE1R, W_NE1I, W_NI1R, W_NI1I, W_JPR0, W_JPI0, W_JPR2, W_JPI2};
    return order[slot];
}
// What becomes of a slot's node sum (combine_sources, Simulation.cpp:408-457): kind | destination << 4 (a WsArr or a
// DiagComp) | beam source << 12 | background << 20 (in units of M); kKindNone for a species sign the run does not have
enum SumKind : int { kKindChi = 0, kKindBeam, kKindBackground, kKindDxi, kKindDiag, kKindIons, kKindNone = -1 };
__device__ __forceinline__ int entry_code(int slot, bool has_neg, bool has_pos) {
    const int comp = entry_comp(slot);
    auto code = [](int kind, int dst, int beam = 0, int bg = 0) { return kind | dst << 4 | beam << 12 | bg << 20; };
    switch (comp) {
        case W_RHOT0: return code(kKindBackground, comp, B_RT0, 0);
        case W_RHOT1R: return code(kKindBackground, comp, B_RT1R, 1);
        case W_RHOT1I: return code(kKindBackground, comp, B_RT1I, 2);
        case W_DRHO0: return code(kKindDxi, comp, B_RT0);
        case W_DRHO1R: return code(kKindDxi, comp, B_RT1R);
        case W_DRHO1I: return code(kKindDxi, comp, B_RT1I);
        case W_JZ0: return code(kKindBeam, comp, B_JZ0);
        case W_JZ1R: return code(kKindBeam, comp, B_JZ1R);
        case W_JZ1I: return code(kKindBeam, comp, B_JZ1I);
        case W_JPR1: return code(kKindBeam, comp, B_JP1R);
        case W_JPI1: return code(kKindBeam, comp, B_JP1I);
        case W_JPR0: return code(kKindBeam, comp, B_JP0R);
        case W_JPI0: return code(kKindBeam, comp, B_JP0I);
        case W_JPR2: return code(kKindBeam, comp, B_JP2R);
        case W_JPI2: return code(kKindBeam, comp, B_JP2I);
        case W_NE0: return has_neg ? code(kKindDiag, D_NE0) : kKindNone;
        case W_NE1R: return has_neg ? code(kKindDiag, D_NE1R) : kKindNone;
        case W_NE1I: return has_neg ? code(kKindDiag, D_NE1I) : kKindNone;
        case W_NI0: return has_pos ? code(kKindIons, D_NI0, 0, 3) : kKindNone;
        case W_NI1R: return has_pos ? code(kKindDiag, D_NI1R) : kKindNone;
        case W_NI1I: return has_pos ? code(kKindDiag, D_NI1I) : kKindNone;
        default: return code(kKindChi, comp);
    }
}
}  // namespace

// What one workgroup stores and another reads, and every other value of the arrays that hold such values, goes to memory
// with an agent-scope store: it is written through this die's L2, so no line of these arrays is ever dirty there.  A
// reader's acquire then drops its die's copies, and nothing depends on what a write-back of an L2 reaches while the
// workgroups of other launches use it too.  The arrays are reached through pointers to const, so that a plain store to
// them does not compile.
template <class T> __device__ __forceinline__ void share(const T* p, T v) {
    __hip_atomic_store(const_cast<T*>(p), v, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}

// two doubles `off` bytes into such an array, described by `buf`: a store of 16 bytes at agent scope (sc1).  A
// written-through store costs its request, so what a lane stores side by side goes in as few as it can.
typedef unsigned int Word4 __attribute__((ext_vector_type(4)));
typedef double Pair16 __attribute__((ext_vector_type(2)));
constexpr int kAgentScope = 16;   // the sc1 bit of a buffer instruction's cache policy
__device__ __forceinline__ void share_pair(__amdgpu_buffer_rsrc_t buf, unsigned int off, Real x, Real y) {
    const Pair16 v = {x, y};
    __builtin_amdgcn_raw_buffer_store_b128(__builtin_bit_cast(Word4, v), buf, off, 0, kAgentScope);
}
// The four lanes of a quad hold 64 bytes of a list entry each (p: four pairs of doubles), which belong at `off`: they exchange
// them so that every store writes one lane's 64 bytes, side by side, in one request.  Called by all lanes of a wave; a lane
// without an entry gives kNoEntry.  A workgroup's requests leave at one per four cycles or so, whatever their size: the
// entries of 4096 particles (m = 1, 8 workgroups) and the wait for them take 53 us a slice, 175 us as 16 bytes per lane.
constexpr unsigned int kNoEntry = ~0u;   // past every buffer's end
template <int ctrl> __device__ __forceinline__ Word4 quad_move(Word4 v) {
    Word4 r;
#pragma unroll
    for (int i = 0; i < 4; ++i) r[i] = __builtin_amdgcn_mov_dpp(static_cast<int>(v[i]), ctrl, 0xF, 0xF, true);
    return r;
}
__device__ __forceinline__ void share_entry(__amdgpu_buffer_rsrc_t buf, unsigned int off, const Real (&p)[8]) {
    const int l = threadIdx.x & 3;
    Word4 a[4];
#pragma unroll
    for (int i = 0; i < 4; ++i) a[i] = __builtin_bit_cast(Word4, Pair16{p[2 * i], p[2 * i + 1]});
    // a 4 x 4 transposition: with the lane beside (quad_perm 1 0 3 2), then with the lane two over (2 3 0 1)
#pragma unroll
    for (int i = 0; i < 4; i += 2) {
        const Word4 y = quad_move<0xB1>(l & 1 ? a[i] : a[i + 1]);
        a[i] = l & 1 ? y : a[i];
        a[i + 1] = l & 1 ? a[i + 1] : y;
    }
#pragma unroll
    for (int i = 0; i < 2; ++i) {
        const Word4 y = quad_move<0x4E>(l & 2 ? a[i] : a[i + 2]);
        a[i] = l & 2 ? y : a[i];
        a[i + 2] = l & 2 ? a[i + 2] : y;
    }
    auto put = [&](Word4 v, int first) {   // piece l of the entry of the quad's lane whose offset is `first`
        if (first != static_cast<int>(kNoEntry))
            __builtin_amdgcn_raw_buffer_store_b128(v, buf, static_cast<unsigned int>(first) + 16 * l, 0, kAgentScope);
    };
    put(a[0], __builtin_amdgcn_mov_dpp(static_cast<int>(off), 0x00, 0xF, 0xF, true));
    put(a[1], __builtin_amdgcn_mov_dpp(static_cast<int>(off), 0x55, 0xF, 0xF, true));
    put(a[2], __builtin_amdgcn_mov_dpp(static_cast<int>(off), 0xAA, 0xF, 0xF, true));
    put(a[3], __builtin_amdgcn_mov_dpp(static_cast<int>(off), 0xFF, 0xF, 0xF, true));
}
__device__ __forceinline__ __amdgpu_buffer_rsrc_t shared_buffer(const Real* p, size_t doubles) {
    return __builtin_amdgcn_make_buffer_rsrc(const_cast<Real*>(p), 0, static_cast<int>(doubles * sizeof(Real)), 0x00020000);
}

// Grid barrier of the G workgroups of a run.  `target` counts this workgroup's barriers; the shared counter only
// grows, so barrier n completes when it reaches n G.  Returns false (and sets the run's error flag) when the
// others do not arrive in time, or when another workgroup has already given up.
// Every wave waits until its own stores are complete (a workgroup's barrier does not wait for that, and the release fence
// of one wave waits for that wave's stores alone); then one release fence before the arrival and one acquire fence after
// the wait, with the counter itself relaxed (fence-to-fence synchronisation through the counter's release sequence).  An
// agent-scope release writes back the die's whole L2 and an acquire invalidates it, operations every other kernel on the
// die waits behind, so the barrier issues one of each and none per poll.
__device__ __forceinline__ bool grid_sync(unsigned int* __restrict__ ctr, unsigned int* __restrict__ err, int G,
                                          unsigned int& target, int* s_ok) {
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
    __syncthreads();
    target += 1;
    if (threadIdx.x == 0) {
        int ok = 1;
        __builtin_amdgcn_fence(__ATOMIC_RELEASE, "agent");   // this workgroup's writes before the arrival
        __hip_atomic_fetch_add(ctr, 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        const unsigned int want = target * static_cast<unsigned int>(G);
        const unsigned long long t0 = wall_clock64();
        while (__hip_atomic_load(ctr, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) < want) {
            if (__hip_atomic_load(err, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) != 0u ||
                wall_clock64() - t0 > kBarrierTicks) {
                __hip_atomic_store(err, 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
                ok = 0;
                break;
            }
            __builtin_amdgcn_s_sleep(2);
        }
        __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "agent");   // the other workgroups' writes after it
        *s_ok = ok;
    }
    __syncthreads();
    return *s_ok != 0;
}

// The sweep of workgroup `block` of a launch: block_map[2 block] is its run, block_map[2 block + 1] its index in the
// run's G workgroups.
template <bool M1, int PT>
__device__ __forceinline__ void sweep_multi_run(const qz_sweep_args* __restrict__ runs,
                                                const int* __restrict__ block_map, int block) {
    using SL = MSlots<M1>;
    const int run = block_map[2 * block], grp = block_map[2 * block + 1];
    const qz_sweep_args& A = runs[run];
    const int G = A.groups;
    extern __shared__ double smem_d[];
    char* smem = reinterpret_cast<char*>(smem_d);

    const int N = A.grid.N, M = N + 1;
    const Real R = A.grid.R;
    const Real* ws = A.ws;   // written through share()
    auto WS = [&](int arr) -> const Real* { return ws + static_cast<size_t>(arr) * M; };
    const int K = A.nslices;
    const int kb = A.k_begin, ke = A.k_end > 0 ? A.k_end : K;
    const Real dxi = A.dxi;
    const Real idxi = Real(1) / dxi;
    const Stencil stn{A.grad_m, A.grad_0, A.grad_p, A.inv_r, N};

    // species, as the one-workgroup kernel: particle gi of the run is slot gi of species 0, then species 1
    const int nsp = A.nspecies;
    const int np0 = nsp > 0 ? A.sp[0].np : 0, np1 = nsp > 1 ? A.sp[1].np : 0;
    const int NP = np0 + np1;
    const Real q0 = nsp > 0 ? A.sp[0].q : Real(0), q1 = nsp > 1 ? A.sp[1].q : Real(0);
    const Real qm0 = nsp > 0 ? A.sp[0].q / A.sp[0].m : Real(0), qm1 = nsp > 1 ? A.sp[1].q / A.sp[1].m : Real(0);
    const bool has_neg = (nsp > 0 && q0 < 0) || (nsp > 1 && q1 < 0);
    const bool has_pos = (nsp > 0 && !(q0 < 0)) || (nsp > 1 && !(q1 < 0));
    const int own0 = grp * mBS * PT;   // first particle of this workgroup

    // the run's multi-workgroup workspace
    const MwsLayout mw(M, N, NP, G, M1);
    Real* mws = A.mws;
    unsigned int* bar = reinterpret_cast<unsigned int*>(mws);
    unsigned int* err = bar + 2;
    const Real* g_bw0 = mws + kBw0;
    const int* g_cnt = reinterpret_cast<const int*>(mws + mw.cnt);
    const Real* g_list = mws + mw.lists;
    const __amdgpu_buffer_rsrc_t list_buf = shared_buffer(g_list, mw.bpalt - mw.lists);
    const __amdgpu_buffer_rsrc_t fac_buf = shared_buffer(WS(W_FAC0), 8 * static_cast<size_t>(M));
    Real* __restrict__ g_gath = mws + mw.gath;
    const Real* bpbuf[2] = {WS(W_BPR1), mws + mw.bpalt};   // Picard iterates: W_BPR1.. of ws, then the second buffer
    unsigned int nbar = 0;

    // LDS
    const MLds plan(N, PT);
    const int Mp = plan.Mp;
    Real* s_r = smem_d;
    Real* s_ih = s_r + Mp;
    Real* s_iv = s_ih + Mp;
    unsigned short* s_wcnt = reinterpret_cast<unsigned short*>(smem + plan.wcnt);
    int* s_cs = reinterpret_cast<int*>(smem + plan.cs);
    int* s_gcs = reinterpret_cast<int*>(smem + plan.gcs);
    int* s_goff = reinterpret_cast<int*>(smem + plan.goff);
    unsigned short* s_sidx = reinterpret_cast<unsigned short*>(smem + plan.sidx);
    int* s_misc = reinterpret_cast<int*>(smem + plan.misc);   // [0] barrier verdict [1] live [2] last cell count
    int* s_code = s_misc + 8;                                  // entry_code of every slot
    int& s_ok = s_misc[0];
    int& s_live = s_misc[1];
    Real* B = reinterpret_cast<Real*>(smem + plan.region);
    auto BA = [&](int slot) -> Real* { return B + static_cast<size_t>(slot) * Mp; };

    const int tid = threadIdx.x;
    const int w = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int gthreads = G * mBS;
    for (int j = tid; j < M; j += mBS) {
        s_r[j] = A.grid.r[j];
        s_iv[j] = A.grid.inv_V[j];
        if (j < N) s_ih[j] = A.grid.inv_h[j];
    }
    if (kb == 0)   // B+ := 0 at the head (Simulation.cpp:705-708); every workgroup its share of the nodes
        for (int j = grp * mBS + tid; j < M; j += gthreads)
            for (int a = 0; a < (M1 ? 6 : 2); ++a) share(WS(W_BPR1 + a) + j, Real(0));
    for (int i = tid; i < SL::ENTRY; i += mBS) s_code[i] = entry_code(i, has_neg, has_pos);
    const Real dmin = A.delta_min, qsamax = A.max_qsa;
    const int ord = A.ab_order;
    const int niter = M1 ? A.picard : 1;
    __syncthreads();
    if (kb == 0 && A.load) {   // this workgroup's particles of the plasma at the head of the box
        const int own1 = own0 + mBS * PT;
        if (nsp > 0) load_rings(A.rings[0], A.sp[0], ord, s_r, own0 + tid, min(own1, np0), mBS);
        if (nsp > 1) load_rings(A.rings[1], A.sp[1], ord, s_r, max(own0, np0) - np0 + tid, min(own1 - np0, np1), mBS);
        __syncthreads();
    }

    int cj[PT], lrank[PT], cpos[PT];   // cell; rank; positions in this workgroup's own lists, left | right << 16
    // rows per lane of the chains, as the one-workgroup kernel (here 8 rows beside 8 particles take no longer)
    constexpr int kRows = PT <= 4 ? kChainR : 4;
    constexpr bool kMom = PT <= 2;                 // momenta, Delta and weight in registers for the slice
    constexpr int PM = kMom ? PT : 1, PB = PT <= 4 ? PT : 2;
    Real cpx[PM], cpy[PM], cdl[PM], cw[PM];
    Real ct[PT], cc[PT], cs[PT], cir[PT], cinvd[PT], cgam[PT];
    auto species_of = [&](int gi, int& li) -> const qz_species_state& {
        const bool s1 = gi >= np0;
        li = s1 ? gi - np0 : gi;
        return s1 ? A.sp[1] : A.sp[0];
    };

#pragma unroll
    for (int pp = 0; pp < PT; ++pp) cj[pp] = 0;
    bool alive = true;
    for (int k = kb; k < ke && alive; ++k) {
        // every per-thread value (addresses, lane roles) is formed inside the slice, not kept live across it
        int tid_k = threadIdx.x;
        asm volatile("" : "+v"(tid_k));
        const int tid = tid_k;
        const int lane = tid & 63;
        const int gtid = grp * mBS + tid;
        auto slot_of = [&](int pp) { return w * (PT * 64) + pp * 64 + lane; };   // local slot; particle own0 + slot
        // ================================================================ 1. geometry and the local sort
#pragma unroll
        for (int pp = 0; pp < PT; ++pp) {
            const int gi = own0 + slot_of(pp);
            const int near = max(cj[pp], 0);   // the last slice's cell
            cj[pp] = -1;
            if (gi < NP) {
                int li;
                const qz_species_state& st = species_of(gi, li);
                const Real wi = st.w[li];
                if (wi != Real(0)) {
                    const Real X = st.x[li], Y = st.y[li];
                    const Real PX = st.px[li], PY = st.py[li], D = st.dl[li];
                    const Real r = dsqrt(X * X + Y * Y);
                    Real c, s_;
                    if (r > Real(0)) { c = X / r; s_ = Y / r; } else { c = Real(1); s_ = Real(0); }
                    int j; Real t;
                    grid_weights_near(s_r, s_ih, N, R, r, near, j, t);
                    cj[pp] = j; ct[pp] = t; cc[pp] = c; cs[pp] = s_;
                    cir[pp] = r > Real(0) ? Real(1) / r : Real(0);
                    cgam[pp] = (Real(1) + PX * PX + PY * PY + D * D) / (Real(2) * D);
                    cinvd[pp] = Real(1) / D;
                    if constexpr (kMom) { cpx[pp] = PX; cpy[pp] = PY; cdl[pp] = D; cw[pp] = wi; }
                }
            }
        }
        for (int i = tid; i < mNW * N; i += mBS) s_wcnt[i] = 0;
        if (tid == 0) s_live = 0;
        __syncthreads();
        {
            const unsigned long long lt_mask = (1ull << lane) - 1ull;
            int nbits = 1;
            while ((1 << nbits) < N) ++nbits;
            int live = 0;
#pragma unroll
            for (int pp = 0; pp < PT; ++pp) {
                const int key = cj[pp];
                unsigned long long mask = __ballot(key >= 0);
                for (int b = 0; b < nbits; ++b) {
                    const bool bit = key >= 0 && ((key >> b) & 1);
                    const unsigned long long bb = __ballot(bit);
                    mask &= bit ? bb : ~bb;
                }
                int old = 0;
                if (key >= 0) old = s_wcnt[w * N + key];
                const int rk = __popcll(mask & lt_mask);
                lrank[pp] = old + rk;
                live += key >= 0 ? 1 : 0;
                __builtin_amdgcn_wave_barrier();
                if (key >= 0 && rk == 0) s_wcnt[w * N + key] = static_cast<unsigned short>(old + __popcll(mask));
                __builtin_amdgcn_wave_barrier();
            }
            for (int d = 32; d >= 1; d >>= 1) live += __shfl_xor(live, d, 64);
            if (lane == 0) atomicAdd(&s_live, live);
        }
        __syncthreads();
        for (int c = tid; c < N; c += mBS) {   // per-cell prefix over the waves; cell totals to global memory
            int run_ = 0;
            for (int ww = 0; ww < mNW; ++ww) {
                const int v = s_wcnt[ww * N + c];
                s_wcnt[ww * N + c] = static_cast<unsigned short>(run_);
                run_ += v;
            }
            s_cs[c + 1] = run_;
            share(g_cnt + static_cast<size_t>(grp) * N + c, run_);
        }
        __syncthreads();
        const int Lloc = s_live;
        if (w == 0) wave_exclusive_scan(s_cs + 1, N, lane);
        if (tid == 0) { s_cs[0] = 0; s_cs[N + 1] = Lloc; s_cs[N + 2] = Lloc; }
        __syncthreads();
#pragma unroll
        for (int pp = 0; pp < PT; ++pp) {
            const int j = cj[pp];
            if (j >= 0) {
                const int pos = s_cs[j + 1] + s_wcnt[w * N + j] + lrank[pp];
                s_sidx[pos] = static_cast<unsigned short>(slot_of(pp));
                lrank[pp] = pos - s_cs[j + 1];   // rank within the cell, index order
            }
        }
        if (!(alive = grid_sync(bar, err, G, nbar, &s_ok))) break;

        // ================================================================ 2. global cell starts, own offsets
        // s_gcs[c + 1] = start of cell c over all workgroups; s_goff[c + 1] = particles of cell c in the
        // workgroups before this one (s_goff[0] = s_goff[N + 1] = 0: no cells beyond the grid)
        for (int c = tid; c < N; c += mBS) {
            int before = 0, total = 0;
            for (int g = 0; g < G; ++g) {
                const int v = g_cnt[static_cast<size_t>(g) * N + c];
                before += g < grp ? v : 0;
                total += v;
            }
            s_goff[c + 1] = before;
            s_gcs[c + 1] = total;
            if (c == N - 1) s_misc[2] = total;
        }
        __syncthreads();
        if (w == 0) wave_exclusive_scan(s_gcs + 1, N, lane);
        __syncthreads();
        const int Ltot = s_gcs[N] + s_misc[2];   // start of the last cell and its particles
        if (tid == 0) {
            s_gcs[0] = 0; s_gcs[N + 1] = Ltot; s_gcs[N + 2] = Ltot;
            s_goff[0] = 0; s_goff[N + 1] = 0;
            if (grp == 0 && A.stats) atomicAdd(A.stats, static_cast<unsigned long long>(Ltot));
        }
        __syncthreads();
        // The two contributions of every owned particle get their positions in the run's node lists: node n holds cell
        // n-1 (right entries) and cell n (left entries), merged in particle-index order, and this workgroup's entries are
        // one run of it after those of the earlier workgroups.  Of the position only that among the workgroup's own
        // entries is kept, in 16 bits a side; the offset of the run follows from the cell.
#pragma unroll
        for (int pp = 0; pp < PT; ++pp) {
            const int j = cj[pp];
            cpos[pp] = 0;
            if (j >= 0) {
                const int sl = slot_of(pp);
                const int less_m = count_less(s_sidx, s_cs[j], s_cs[j + 1], sl);
                const int less_p = count_less(s_sidx, s_cs[j + 2], s_cs[j + 3], sl);
                const int pl = (s_cs[j] + s_cs[j + 1]) + lrank[pp] + less_m;
                const int pr = (s_cs[j + 1] + s_cs[j + 2]) + lrank[pp] + less_p;
                cpos[pp] = pl | (pr << 16);
            }
        }
        auto shift = [&](int n) {   // own run of node n: from its place in the own lists to that in the run's
            return (s_gcs[n] + s_gcs[n + 1]) + s_goff[n] + s_goff[n + 1] - (s_cs[n] + s_cs[n + 1]);
        };
        __syncthreads();   // the sorted slots are read: staged fields may take their place
        // momenta, Delta and weight of PB consecutive particles from p0, all loads issued before any is used
        auto load_batch = [&](int p0, Real (&PX)[PB], Real (&PY)[PB], Real (&D)[PB], Real (&wi)[PB]) {
#pragma unroll
            for (int u = 0; u < PB; ++u) {
                if constexpr (kMom) {
                    PX[u] = cpx[p0 + u]; PY[u] = cpy[p0 + u]; D[u] = cdl[p0 + u]; wi[u] = cw[p0 + u];
                } else {
                    PX[u] = PY[u] = D[u] = wi[u] = Real(0);
                    if (cj[p0 + u] >= 0) {
                        int gi = own0 + slot_of(p0 + u), li;
                        asm volatile("" : "+v"(gi));
                        const qz_species_state& st = species_of(gi, li);
                        PX[u] = st.px[li]; PY[u] = st.py[li]; D[u] = st.dl[li]; wi[u] = st.w[li];
                    }
                }
            }
        };
        auto fence_cache = [&]() {
            fence_regs(cj); fence_regs(cpos); fence_regs(ct); fence_regs(cc); fence_regs(cs); fence_regs(cir);
            fence_regs(cinvd); fence_regs(cgam);
        };

        // ================================================================ 3. deposit: contributions, node sums
        {
            fence_cache();
#pragma unroll
            for (int p0 = 0; p0 < PT; p0 += PB) {
                Real PXb[PB], PYb[PB], Db[PB], wb[PB];
                load_batch(p0, PXb, PYb, Db, wb);
#pragma unroll
                for (int u = 0; u < PB; ++u) {
                    const int pp = p0 + u;
                    const bool live = cj[pp] >= 0;
                    const int j = max(cj[pp], 0);   // lanes without a particle take part in the exchanges
                    const Real PX = PXb[u], PY = PYb[u], D = Db[u], wi = wb[u];
                    const bool s1 = own0 + slot_of(pp) >= np0;
                    const Real q = s1 ? q1 : q0, qm = s1 ? qm1 : qm0;
                    const Real ih = s_ih[j];
                    const Real pz = cgam[pp] - D;
#pragma unroll
                    for (int side = 0; side < 2; ++side) {
                        const int at = (side == 0 ? (cpos[pp] & 0xffff) : (cpos[pp] >> 16)) + shift(j + side);
                        const unsigned int off = static_cast<unsigned int>(at) * (SL::ENTRY * 8);
                        const Real iv = s_iv[j + side];
                        auto pass = [&](auto first) {   // eight of the entry's arrays, from entry_comp(first)
                            constexpr int S = decltype(first)::value;
                            Real v[8];
                            for_each_batch<8>([&](auto i) {
                                v[i] = dep_value(entry_comp(S + i), side, j, ct[pp], cc[pp], cs[pp], cir[pp], cinvd[pp], cgam[pp],
                                                 PX, PY, pz, wi, q, qm, iv, ih);
                            });
                            share_entry(list_buf, live ? off + S * 8 : kNoEntry, v);
                        };
                        pass(IC<0>{});
                        if constexpr (M1) {
                            pass(IC<8>{});
                            pass(IC<16>{});
                        }
                    }
                }
            }
        }
        if (!(alive = grid_sync(bar, err, G, nbar, &s_ok))) break;
        {
            Real* __restrict__ Dg = A.diag + static_cast<size_t>(k) * M * A.ncd;
            const int ncd = A.ncd, ncb = A.ncb;
            const Real* __restrict__ bs = A.bsrc;
            const Real* __restrict__ bg = A.bg;
            const bool ngp = A.ngp != 0;
            // combine_sources' xi derivative of a beam source: half (row hi - row lo) / dxi, row -1 zero
            const int hi = ngp || k == K - 1 ? k : k + 1, lo = ngp || k > 0 ? k - 1 : 0;
            const Real half = ngp || k == 0 || k == K - 1 ? Real(1) : Real(0.5);
            const bool flat = !ngp && K == 1;
            // a wave sums the lists of eight nodes: eight lanes read 64 bytes of an entry side by side, a lane the same double
            // of each such part, and the sums of eight nodes are stored side by side.  Bound by the trips to memory: 29 us
            // a slice (m = 1, 1025 nodes, 64 entries a node, 8 workgroups), 42 us with the sources read after the sums,
            // 9 and 18 us with 513 nodes and 16 entries.  11 entries in flight beside eight particles per thread, where
            // two registers spill (four with 12, 34 with 16).
            constexpr int P = SL::ENTRY / 8;
            for (int tile = grp * mNW + w; tile < (M + 7) / 8; tile += G * mNW) {
                const int n = 8 * tile + (lane >> 3);
                if (n >= M) continue;
                const int e0 = s_gcs[n] + s_gcs[n + 1], e1 = s_gcs[n + 1] + s_gcs[n + 2];
                // the sources are on their way while the lists are summed
                int code[P];
                Real u[P], v[P], sums[P];
#pragma unroll
                for (int part = 0; part < P; ++part) {
                    code[part] = s_code[8 * part + (lane & 7)];
                    const int c = max(code[part], 0), kind = c & 15, beam = c >> 12 & 255;
                    const bool from_bg = kind == kKindBackground || kind == kKindIons, dxi_b = kind == kKindDxi;
                    u[part] = *(from_bg ? bg + (c >> 20) * M + n
                                        : bs + (static_cast<size_t>(dxi_b ? hi : k) * M + n) * ncb + beam);
                    v[part] = bs[(static_cast<size_t>(dxi_b ? max(lo, 0) : k) * M + n) * ncb + beam];
                }
                sum_rows<SL::ENTRY, P, (P == 1 || PT <= 4 ? 16 : 11)>(g_list + (lane & 7), e0, e1, sums);
#pragma unroll
                for (int part = 0; part < P; ++part) {
                    const int kind = code[part] & 15, dst = code[part] >> 4 & 255;
                    Real acc = sums[part];
                    if (code[part] < 0) continue;
                    if (kind == kKindBackground) acc = acc + (u[part] + v[part]);
                    if (kind == kKindBeam) acc = acc + u[part];
                    if (kind == kKindDxi)
                        acc = acc + (flat ? Real(0) : half * (u[part] - (lo < 0 ? Real(0) : v[part])) * idxi);
                    if (kind == kKindIons && u[part] > Real(0)) acc = acc + u[part];   // Simulation.cpp:441
                    if (kind >= kKindDiag) Dg[static_cast<size_t>(n) * ncd + dst] = acc;
                    else share(WS(dst) + n, acc);
                }
            }
            // densities of absent species are zero, plus the positive background for n_i
            for (int n = gtid; n < M; n += gthreads) {
                Real* Dn = Dg + static_cast<size_t>(n) * ncd;
                if (!has_neg) {
                    Dn[D_NE0] = Real(0);
                    if (M1) { Dn[D_NE1R] = Real(0); Dn[D_NE1I] = Real(0); }
                }
                if (!has_pos) {
                    const Real bgr0 = bg[3 * M + n];
                    Dn[D_NI0] = bgr0 > Real(0) ? Real(0) + bgr0 : Real(0);
                    if (M1) { Dn[D_NI1R] = Real(0); Dn[D_NI1I] = Real(0); }
                }
            }
        }
        if (!(alive = grid_sync(bar, err, G, nbar, &s_ok))) break;

        // ================================================================ 4. the solves (three jobs)
        // job 0: psi0, E_z0, B_z0 with L0;  job 1 (m = 1): psi1, E_z1, B_z1 (r, i) with L1D;  job 2: this
        // slice's Thomas factors of (L - chi0) for L1D, L1F (and L0, L2D in m = 1).  Job j runs on workgroup j % G.
        for (int job = grp; job < 3; job += G) {
            if (job == 1 && !M1) continue;
            if (job < 2) {
                const bool l0 = job == 0;
                const int op = l0 ? OP_L0 : OP_L1D;
                Real* a = BA(0);
                Real* m = BA(1);
                Real* cp = BA(2);
                const int nsys = l0 ? 3 : 6;
                for (int j = tid; j < M; j += mBS) {
                    a[j] = A.op_a[op][j];
                    m[j] = l0 ? A.fac_l0_m[j] : A.fac_l1_m[j];
                    cp[j] = l0 ? A.fac_l0_cp[j] : A.fac_l1_cp[j];
                    if (l0) {
                        BA(3)[j] = WS(W_RHOT0)[j];
                        BA(4)[j] = WS(W_DRHO0)[j];
                        // B_z right-hand side (compute_bz, Simulation.cpp:506-526)
                        const Real t1 = stn.grad_odd(WS(W_JPI1), j), t2 = stn.over_r(WS(W_JPI1), j);
                        BA(5)[j] = -(t1 + t2);
                    } else {
                        BA(3)[j] = WS(W_RHOT1R)[j];
                        BA(4)[j] = WS(W_RHOT1I)[j];
                        BA(5)[j] = WS(W_DRHO1R)[j];
                        BA(6)[j] = WS(W_DRHO1I)[j];
                        const Real gr0 = stn.grad_odd(WS(W_JPR2), j), gi0 = stn.over_r(WS(W_JPR2), j);
                        const Real gr1 = stn.grad_odd(WS(W_JPI2), j), gi1 = stn.over_r(WS(W_JPI2), j);
                        const Real gr2 = stn.grad(WS(W_JPR0), j), gi2 = stn.grad(WS(W_JPI0), j);
                        const Real D1r = gr0 + Real(2) * gi0, D1i = gr1 + Real(2) * gi1;
                        const Real Dmr = gr2, Dmi = gi2;
                        BA(7)[j] = -Real(0.5) * (D1i + Dmi);
                        BA(8)[j] = Real(0.5) * (D1r - Dmr);
                    }
                }
                __syncthreads();
                if (w < nsys / 3) {   // a DPP row per system, three per wave
                    // psi and E_z: -rhs; B_z: +rhs (FieldSolver::solve scale); L0 keeps the axis row regular
                    const int sys = 3 * w + min(lane >> 4, 2);
                    const bool bz = l0 ? sys == 2 : sys >= 4;
                    thomas_wave<kRows>(a, m, cp, A.op_b[op][0], BA(3 + sys), BA(3 + sys), bz ? Real(1) : Real(-1), !l0, true,
                                false, Real(0), M);
                }
                __syncthreads();
                // results: psi over its right-hand side in ws, E_z and B_z to their arrays
                for (int j = tid; j < M; j += mBS) {
                    if (l0) {
                        share(WS(W_RHOT0) + j, BA(3)[j]);
                        share(WS(W_EZ0) + j, BA(4)[j]);
                        share(WS(W_BZ0) + j, BA(5)[j]);
                    } else {
                        share(WS(W_RHOT1R) + j, BA(3)[j]);
                        share(WS(W_RHOT1I) + j, BA(4)[j]);
                        share(WS(W_EZ1R) + j, BA(5)[j]);
                        share(WS(W_EZ1I) + j, BA(6)[j]);
                        share(WS(W_BZ1R) + j, BA(7)[j]);
                        share(WS(W_BZ1I) + j, BA(8)[j]);
                    }
                }
                __syncthreads();
            } else {
                // rows of L1 (shared by L1D and L1F up to the last row), L0 and L2D, and chi0
                for (int j = tid; j < M; j += mBS) {
                    BA(0)[j] = A.op_a[OP_L1D][j]; BA(1)[j] = A.op_b[OP_L1D][j]; BA(2)[j] = A.op_c[OP_L1D][j];
                    BA(3)[j] = WS(W_CHI0)[j];
                    if (A.chi_out) A.chi_out[static_cast<size_t>(k) * M + j] = WS(W_CHI0)[j];   // for the laser march
                    if (M1) {
                        BA(4)[j] = A.op_a[OP_L0][j]; BA(5)[j] = A.op_b[OP_L0][j]; BA(6)[j] = A.op_c[OP_L0][j];
                        BA(7)[j] = A.op_a[OP_L2D][j]; BA(8)[j] = A.op_b[OP_L2D][j]; BA(9)[j] = A.op_c[OP_L2D][j];
                    }
                }
                __syncthreads();
                if (w == 0) {
                    const int f = min(lane >> 4, M1 ? 3 : 1);
                    const int base = f < 2 ? 0 : (f == 2 ? 4 : 7);
                    const int op = f == 0 ? OP_L1D : f == 1 ? OP_L1F : f == 2 ? OP_L0 : OP_L2D;
                    const Real aN = A.op_a[op][N], bN = A.op_b[op][N];
                    const bool dir0 = op != OP_L0, dirN = op != OP_L1F;
                    // m and c' of a row side by side, operator after operator
                    share(g_bw0 + f,
                          thomas_factor_wave<kRows>(BA(base), BA(base + 1), BA(base + 2), BA(3), aN, bN, dir0, dirN, M,
                                                    [&](int i, Real m, Real cp) {
                                                        share_pair(fac_buf, (static_cast<unsigned int>(f) * M + i) * 16, m, cp);
                                                    }));
                }
                __syncthreads();
            }
        }
        if (!(alive = grid_sync(bar, err, G, nbar, &s_ok))) break;

        // ================================================================ 5. W+, field outputs, S+ deposit
        {
            Real* __restrict__ F = A.fld + static_cast<size_t>(k) * M * A.ncf;
            Real* __restrict__ Dg = A.diag + static_cast<size_t>(k) * M * A.ncd;
            const int ncf = A.ncf, ncd = A.ncd;
            const Real* psi0 = WS(W_RHOT0);
            const Real* psr = WS(W_RHOT1R);
            const Real* psi_ = WS(W_RHOT1I);
            for (int j = tid; j < M; j += mBS) {   // compute_wplus (Simulation.cpp:477-498) into LDS
                const Real t1 = stn.grad(psi0, j);
                BA(SL::W + 0)[j] = -t1;
                BA(SL::W + 1)[j] = Real(0);
                BA(SL::EZ)[j] = WS(W_EZ0)[j];
                BA(SL::BZ)[j] = WS(W_BZ0)[j];
                if (M1) {
                    const Real t2 = stn.grad_odd(psr, j), t3 = stn.over_r(psr, j);
                    const Real t4 = stn.grad_odd(psi_, j), rh = stn.over_r(psi_, j);
                    BA(SL::W + 4)[j] = -(t2 - t3);
                    BA(SL::W + 5)[j] = -(t4 - rh);
                    BA(SL::W + 2)[j] = -(t2 + t3);
                    BA(SL::W + 3)[j] = (t4 + rh);
                    BA(SL::EZ + 1)[j] = WS(W_EZ1R)[j]; BA(SL::EZ + 2)[j] = WS(W_EZ1I)[j];
                    BA(SL::BZ + 1)[j] = WS(W_BZ1R)[j]; BA(SL::BZ + 2)[j] = WS(W_BZ1I)[j];
                }
            }
            __syncthreads();
            // this workgroup's share of the nodes: psi, E_z, B_z to the stores, W+ to ws for the field store
            for (int j = gtid; j < M; j += gthreads) {
                Real* Fj = F + static_cast<size_t>(j) * ncf;
                Real* Dj = Dg + static_cast<size_t>(j) * ncd;
                Dj[D_PSI0] = psi0[j];
                Fj[F_EZ0] = BA(SL::EZ)[j];
                Fj[F_BZ0] = BA(SL::BZ)[j];
                for (int a = 0; a < (M1 ? 6 : 2); ++a) share(WS(W_WPR1 + a) + j, BA(SL::W + a)[j]);
                if (M1) {
                    Dj[D_PSI1R] = psr[j]; Dj[D_PSI1I] = psi_[j];
                    Fj[F_EZ1R] = BA(SL::EZ + 1)[j]; Fj[F_EZ1I] = BA(SL::EZ + 2)[j];
                    Fj[F_BZ1R] = BA(SL::BZ + 1)[j]; Fj[F_BZ1I] = BA(SL::BZ + 2)[j];
                }
            }
            // S+ contributions of the owned particles (PlasmaSpecies::deposit_S, PlasmaSpecies.cpp:516-558): the gather of
            // W+, E_z, B_z and the particle's a_x, a_y, and from these its entries of every component
            fence_cache();
#pragma unroll
            for (int p0 = 0; p0 < PT; p0 += PB) {
                Real PXb[PB], PYb[PB], Db[PB], wb[PB];
                load_batch(p0, PXb, PYb, Db, wb);
#pragma unroll
                for (int u = 0; u < PB; ++u) {
                    const int pp = p0 + u;
                    const bool live = cj[pp] >= 0;
                    const int j = max(cj[pp], 0);
                    const Real PX = PXb[u], PY = PYb[u], wi = wb[u];
                    const bool s1 = own0 + slot_of(pp) >= np0;
                    const Real qq = s1 ? q1 : q0, qm = s1 ? qm1 : qm0;
                    const Real t = ct[pp], c = cc[pp], sn = cs[pp];
                    const Real invd = cinvd[pp];
                    Real Wx, Wy;
                    if (M1)
                        eval_vector(lin(BA(SL::W + 2), j, t), lin(BA(SL::W + 3), j, t), lin(BA(SL::W + 0), j, t),
                                    lin(BA(SL::W + 1), j, t), lin(BA(SL::W + 4), j, t), lin(BA(SL::W + 5), j, t), c, sn, true,
                                    Wx, Wy);
                    else
                        eval_vector(Real(0), Real(0), lin(BA(SL::W + 0), j, t), lin(BA(SL::W + 1), j, t), Real(0), Real(0), c,
                                    sn, false, Wx, Wy);
                    const Real Ez = eval_scalar(lin(BA(SL::EZ), j, t), M1 ? lin(BA(SL::EZ + 1), j, t) : Real(0),
                                                M1 ? lin(BA(SL::EZ + 2), j, t) : Real(0), c, sn, M1);
                    const Real Bz = eval_scalar(lin(BA(SL::BZ), j, t), M1 ? lin(BA(SL::BZ + 1), j, t) : Real(0),
                                                M1 ? lin(BA(SL::BZ + 2), j, t) : Real(0), c, sn, M1);
                    if (live) {
                        Real* gt = g_gath + own0 + slot_of(pp);
                        gt[0] = Wx;
                        gt[static_cast<size_t>(NP)] = Wy;
                        gt[2 * static_cast<size_t>(NP)] = Ez;
                        gt[3 * static_cast<size_t>(NP)] = Bz;
                    }
                    const Real dA = Real(0);
                    const Real gam = cgam[pp];
                    const Real fp = -Real(0.5) * qm * qm * dA * invd;
                    const Real dD = qm * ((PX * Wx + PY * Wy) * invd - Ez);
                    const Real ax = (qm * (gam * Wx + PY * Bz) * invd + fp * c) * invd - PX * dD * invd * invd;
                    const Real ay = (qm * (gam * Wy - PX * Bz) * invd + fp * sn) * invd - PY * dD * invd * invd;
                    const Real ux = PX * invd, uy = PY * invd;
                    const Real ur = c * ux + sn * uy, uth = c * uy - sn * ux;
                    const Real wq = wi * qq;
                    const Real ih = s_ih[j];
#pragma unroll
                    for (int side = 0; side < 2; ++side) {
                        const int at = (side == 0 ? (cpos[pp] & 0xffff) : (cpos[pp] >> 16)) + shift(j + side);
                        const unsigned int off = static_cast<unsigned int>(at) * (SL::SENTRY * 8);
                        const Real iv = s_iv[j + side] * wq;
                        const Real W = side == 0 ? Real(1) - t : t;
                        const Real dW = side == 0 ? -ih : ih;
                        Real v[8] = {};
                        auto s_pass = [&](auto cst, int slot) {   // the real and imaginary components of one mode
                            constexpr int mode = decltype(cst)::value;
                            const Real ck = mode == 1 ? c : (mode == 0 ? Real(1) : c * c - sn * sn);
                            const Real sk = mode == 1 ? sn : (mode == 0 ? Real(0) : Real(2) * c * sn);
                            Real Ar = ax * W + ux * ur * dW;
                            Real Ai = ay * W + uy * ur * dW;
                            if (mode != 0) {
                                const Real Wor = (j == 0) ? (side == 0 ? Real(0) : ih) : W * cir[pp];
                                const Real f2 = mode * uth * Wor;
                                Ar += f2 * uy;
                                Ai -= f2 * ux;
                            }
                            v[slot] = iv * (Ar * ck + Ai * sk);
                            v[slot + 1] = iv * (Ai * ck - Ar * sk);
                        };
                        s_pass(IC<1>{}, 0);
                        if constexpr (M1) {
                            s_pass(IC<0>{}, 2);
                            s_pass(IC<2>{}, 4);
                            share_entry(list_buf, live ? off : kNoEntry, v);
                        } else if (live) {
                            share_pair(list_buf, off, v[0], v[1]);
                        }
                    }
                }
            }
        }
        if (!(alive = grid_sync(bar, err, G, nbar, &s_ok))) break;
        {
            constexpr int nodes = 64 / SL::NS;   // of a wave
            const int tiles = (M + nodes - 1) / nodes;
            for (int tile = grp * mNW + w; tile < tiles; tile += G * mNW) {
                const int u = lane / SL::NS, sc = lane - u * SL::NS, n = tile * nodes + u;
                if (u >= nodes || n >= M) continue;
                const int e0 = s_gcs[n] + s_gcs[n + 1], e1 = s_gcs[n + 1] + s_gcs[n + 2];
                Real acc[1];
                sum_rows<SL::SENTRY, 1, 16>(g_list + sc, e0, e1, acc);
                share(WS(W_SR1 + sc) + n, acc[0]);
            }
        }
        if (!(alive = grid_sync(bar, err, G, nbar, &s_ok))) break;

        // ================================================================ 6. Picard iterations of B+ (Simulation.cpp:535-591)
        // jobs: 0 (B_r1 with L1D, B_i1 with L1F), m = 1: 1 (B_r0, B_i0 with L0), 2 (B_r2, B_i2 with L2D).  The
        // iterate `it` reads buffer it % 2 (buffer 0 is ws' B+: the warm start) and writes buffer (it + 1) % 2.
        {
            const int njob = M1 ? 3 : 1;
            const Real fcw = A.flux_coef * WS(W_JZ0)[N];
            for (int it = 0; it < niter; ++it) {
                const Real* bp = bpbuf[it & 1];
                const Real* bn = bpbuf[(it + 1) & 1];
                auto BP = [&](int f, int j) { return bp[static_cast<size_t>(f) * M + j]; };
                for (int job = grp; job < njob; job += G) {
                    // slots: 0 a (first system), 1 a (second), 2,3 factors of the first, 4,5 of the second,
                    // 6,7 right-hand sides, then solutions in place
                    const int sys0 = 2 * job;   // B+ arrays: 0 r1, 1 i1, 2 r0, 3 i0, 4 r2, 5 i2
                    const int fa = job == 0 ? 0 : (job == 1 ? 2 : 3);                      // factor set: L1D L1F L0 L2D
                    const int fb = job == 0 ? 1 : fa;
                    const int opa = job == 0 ? OP_L1D : (job == 1 ? OP_L0 : OP_L2D);
                    const int opb = job == 0 ? OP_L1F : opa;
                    // a workgroup with one job keeps its operators, factors and gz (slots 8, 9) over the iterations
                    const bool staged = it > 0 && G >= njob;
                    for (int j = tid; j < M; j += mBS) {
                        Real gr, gi;
                        if (staged) {
                            gr = BA(8)[j];
                            gi = BA(9)[j];
                        } else {
                            BA(0)[j] = A.op_a[opa][j];
                            BA(1)[j] = A.op_a[opb][j];
                            const Real *fca = WS(W_FAC0 + 2 * fa) + 2 * j, *fcb = WS(W_FAC0 + 2 * fb) + 2 * j;
                            BA(2)[j] = fca[0]; BA(3)[j] = fca[1];
                            BA(4)[j] = fcb[0]; BA(5)[j] = fcb[1];
                            // gz: ((d_x + i d_y) J_z)_k + S_k, and the chi_1 coupling with the previous iterate
                            if (job == 0) {
                                const Real t1 = stn.grad(WS(W_JZ0), j);
                                gr = t1 + WS(W_SR1)[j];
                                gi = WS(W_SI1)[j];
                            } else {
                                const Real* fr = WS(W_JZ1R);
                                const Real* fi = WS(W_JZ1I);
                                const Real t2 = stn.grad_odd(fr, j), t3 = stn.over_r(fr, j);
                                const Real t4 = stn.grad_odd(fi, j), rh = stn.over_r(fi, j);
                                if (job == 1) {
                                    gr = (t2 + t3) + WS(W_SR0)[j];
                                    gi = -(t4 + rh) + WS(W_SI0)[j];
                                } else {
                                    gr = (t2 - t3) + WS(W_SR2)[j];
                                    gi = (t4 - rh) + WS(W_SI2)[j];
                                }
                            }
                            if (M1) {
                                BA(8)[j] = gr;
                                BA(9)[j] = gi;
                            }
                        }
                        Real rr = -gi, ri = gr;
                        if (M1) {
                            const Real cr = WS(W_CHI1R)[j], ci = WS(W_CHI1I)[j];
                            const Real b1r = BP(0, j), b1i = BP(1, j), b0r = BP(2, j), b0i = BP(3, j);
                            const Real b2r = BP(4, j), b2i = BP(5, j);
                            if (job == 0) {
                                rr += cr * b0r - ci * b0i + cr * b2r + ci * b2i;
                                ri += cr * b0i + ci * b0r + cr * b2i - ci * b2r;
                            } else if (job == 1) {
                                rr += cr * b1r + ci * b1i; ri += cr * b1i - ci * b1r;
                            } else {
                                rr += cr * b1r - ci * b1i; ri += cr * b1i + ci * b1r;
                            }
                        }
                        BA(6)[j] = rr;
                        BA(7)[j] = ri;
                    }
                    __syncthreads();
                    if (w == 0) {
                        const int sys = min(lane >> 4, 1);
                        const int f = sys == 0 ? fa : fb;
                        const bool flux = f == 1;
                        thomas_wave<kRows>(BA(sys), BA(2 + 2 * sys), BA(3 + 2 * sys), g_bw0[f], BA(6 + sys), BA(6 + sys),
                                    Real(1), f != 2, !flux, flux, flux ? fcw : Real(0), M);
                    }
                    __syncthreads();
                    for (int j = tid; j < M; j += mBS) {
                        share(bn + static_cast<size_t>(sys0) * M + j, BA(6)[j]);
                        share(bn + static_cast<size_t>(sys0 + 1) * M + j, BA(7)[j]);
                    }
                    __syncthreads();
                }
                if (!(alive = grid_sync(bar, err, G, nbar, &s_ok))) break;
            }
            if (!alive) break;
        }

        // ================================================================ 7. store (Simulation.cpp:594-633) and push
        {
            const Real* bfin = bpbuf[niter & 1];
            auto BF = [&](int f, int j) { return bfin[static_cast<size_t>(f) * M + j]; };
            Real* __restrict__ F = A.fld + static_cast<size_t>(k) * M * A.ncf;
            const int ncf = A.ncf;
            for (int j = gtid; j < M; j += gthreads) {
                Real* Fj = F + static_cast<size_t>(j) * ncf;
                const Real b1r = BF(0, j), b1i = BF(1, j);
                Fj[F_EP1R] = WS(W_WPR1)[j] + b1i;
                Fj[F_EP1I] = WS(W_WPI1)[j] - b1r;
                Fj[F_BP1R] = b1r;
                Fj[F_BP1I] = b1i;
                if (M1) {
                    const Real b0r = BF(2, j), b0i = BF(3, j), b2r = BF(4, j), b2i = BF(5, j);
                    Fj[F_EP0R] = WS(W_WPR0)[j] + b0i;
                    Fj[F_EP0I] = WS(W_WPI0)[j] - b0r;
                    Fj[F_EP2R] = WS(W_WPR2)[j] + b2i;
                    Fj[F_EP2I] = WS(W_WPI2)[j] - b2r;
                    Fj[F_BP0R] = b0r; Fj[F_BP0I] = b0i; Fj[F_BP2R] = b2r; Fj[F_BP2I] = b2i;
                }
                if (niter & 1)   // the warm start of the next slice goes back to ws
                    for (int f = 0; f < (M1 ? 6 : 2); ++f) share(WS(W_BPR1 + f) + j, BF(f, j));
            }
            if (k < K - 1) {
                // ---- Adams-Bashforth push (PlasmaSpecies::push, src/PlasmaSpecies.cpp:600-667); B+ staged in LDS
                const int slot = k % ord;
                const bool first = (k == 0);
                const int older = first ? 0 : ord;   // slots of the history to read, this one's included
                for (int j = tid; j < M; j += mBS)
                    for (int f = 0; f < (M1 ? 6 : 2); ++f) BA(f)[j] = BF(f, j);
                __syncthreads();
                fence_cache();
                constexpr int PP = PT == 2 ? 2 : 1;   // particles whose state and history are loaded together
                for_each_batch<PT / PP>([&](auto batch) {
                constexpr int p0 = decltype(batch)::value * PP;
                Real Xb[PP], Yb[PP], Db[PP], PXb[PP], PYb[PP], Gb[PP][4], Hb[PP][4][5];
#pragma unroll
                for (int u = 0; u < PP; ++u) {
                    Xb[u] = Yb[u] = Db[u] = PXb[u] = PYb[u] = Real(0);
                    Gb[u][0] = Gb[u][1] = Gb[u][2] = Gb[u][3] = Real(0);
                    if (cj[p0 + u] >= 0) {
                        int li;
                        const int gi = own0 + slot_of(p0 + u);
                        const qz_species_state& st = species_of(gi, li);
                        Xb[u] = st.x[li]; Yb[u] = st.y[li];
                        if constexpr (!kMom) { Db[u] = st.dl[li]; PXb[u] = st.px[li]; PYb[u] = st.py[li]; }
#pragma unroll
                        for (int v = 0; v < 4; ++v) Gb[u][v] = g_gath[static_cast<size_t>(v) * NP + gi];
                        const Real* h = st.hist + li;
#pragma unroll
                        for (int mm = 1; mm < 5; ++mm)
                            if (mm < older) {
                                const int sl = slot - mm + (slot < mm ? ord : 0);
#pragma unroll
                                for (int v = 0; v < 5; ++v) Hb[u][mm - 1][v] = h[static_cast<size_t>(sl * 5 + v) * st.cap];
                            }
                    }
                }
#pragma unroll
                for (int u = 0; u < PP; ++u) {
                    const int pp = p0 + u;
                    const int j = cj[pp];
                    if (j < 0) continue;
                    int li;
                    const int gi = own0 + slot_of(pp);
                    const bool s1 = gi >= np0;
                    const qz_species_state& st = species_of(gi, li);
                    const int cap = st.cap;
                    Real* __restrict__ hist = st.hist;
                    const Real X = Xb[u], Y = Yb[u];
                    Real D, PX, PY;
                    if constexpr (kMom) { D = cdl[pp]; PX = cpx[pp]; PY = cpy[pp]; }
                    else { D = Db[u]; PX = PXb[u]; PY = PYb[u]; }
                    const Real qm = s1 ? qm1 : qm0;
                    const Real t = ct[pp], c = cc[pp], sn = cs[pp];
                    const Real Wx = Gb[u][0], Wy = Gb[u][1], Ez = Gb[u][2], Bz = Gb[u][3];
                    Real Bx, By;
                    if (M1)
                        eval_vector(lin(BA(2), j, t), lin(BA(3), j, t), lin(BA(0), j, t), lin(BA(1), j, t), lin(BA(4), j, t),
                                    lin(BA(5), j, t), c, sn, true, Bx, By);
                    else
                        eval_vector(Real(0), Real(0), lin(BA(0), j, t), lin(BA(1), j, t), Real(0), Real(0), c, sn, false, Bx,
                                    By);
                    const Real dA = Real(0);
                    const Real gam = cgam[pp];
                    const Real invd = cinvd[pp];
                    const Real fp = -Real(0.5) * qm * qm * dA * invd;
                    const Real f0 = PX * invd;
                    const Real f1 = PY * invd;
                    const Real f2 = qm * (gam * Wx * invd + By + PY * Bz * invd) + fp * c;
                    const Real f3 = qm * (gam * Wy * invd - Bx - PX * Bz * invd) + fp * sn;
                    const Real f4 = qm * ((PX * Wx + PY * Wy) * invd - Ez);
                    auto H = [&](int sl, int v) -> Real& { return hist[(static_cast<size_t>(sl) * 5 + v) * cap + li]; };
                    Real s0 = 0, sm1 = 0, sm2 = 0, sm3 = 0, sm4 = 0;
                    if (first) {
                        for (int sl = 0; sl < ord; ++sl) {
                            H(sl, 0) = f0; H(sl, 1) = f1; H(sl, 2) = f2; H(sl, 3) = f3; H(sl, 4) = f4;
                        }
                        for (int mm = 0; mm < ord; ++mm) {
                            const Real cm = A.ab_c[mm];
                            s0 += cm * f0; sm1 += cm * f1; sm2 += cm * f2; sm3 += cm * f3; sm4 += cm * f4;
                        }
                    } else {
                        H(slot, 0) = f0; H(slot, 1) = f1; H(slot, 2) = f2; H(slot, 3) = f3; H(slot, 4) = f4;
#pragma unroll
                        for (int mm = 0; mm < 5; ++mm) {
                            if (mm >= ord) continue;
                            const Real cm = A.ab_c[mm];
                            if (mm == 0) {
                                s0 += cm * f0; sm1 += cm * f1; sm2 += cm * f2; sm3 += cm * f3; sm4 += cm * f4;
                            } else {
                                const Real* h = Hb[u][mm - 1];
                                s0 += cm * h[0]; sm1 += cm * h[1]; sm2 += cm * h[2]; sm3 += cm * h[3]; sm4 += cm * h[4];
                            }
                        }
                    }
                    Real xn = X + dxi * s0, yn = Y + dxi * sm1;
                    Real pxn = PX + dxi * sm2, pyn = PY + dxi * sm3;
                    const Real dn = D + dxi * sm4;
                    const Real gn = (Real(1) + pxn * pxn + pyn * pyn + dn * dn) / (Real(2) * dn);
                    if (!(dn > dmin) || gn > qsamax * dn) {
                        st.w[li] = Real(0);
                        atomicAdd(&A.lost[s1 ? 1 : 0], 1);
                        continue;
                    }
                    const Real rn = dsqrt(xn * xn + yn * yn);
                    if (rn > R) {
                        const Real nx = xn / rn, ny = yn / rn;
                        const Real rr = Real(2) * R - rn;
                        if (rr < Real(0)) {
                            st.w[li] = Real(0);
                            atomicAdd(&A.lost[s1 ? 1 : 0], 1);
                            continue;
                        }
                        xn = nx * rr; yn = ny * rr;
                        const Real pn = pxn * nx + pyn * ny;
                        pxn -= Real(2) * pn * nx; pyn -= Real(2) * pn * ny;
                        for (int sl = 0; sl < ord; ++sl) {
                            const Real aa = H(sl, 0) * nx + H(sl, 1) * ny;
                            H(sl, 0) -= Real(2) * aa * nx; H(sl, 1) -= Real(2) * aa * ny;
                            const Real bb2 = H(sl, 2) * nx + H(sl, 3) * ny;
                            H(sl, 2) -= Real(2) * bb2 * nx; H(sl, 3) -= Real(2) * bb2 * ny;
                        }
                    }
                    st.x[li] = xn; st.y[li] = yn; st.px[li] = pxn; st.py[li] = pyn; st.dl[li] = dn;
                }
                });
            }
        }
        __syncthreads();
    }
    // every workgroup has passed its last barrier: the last one out puts the barrier counter (word 0) and the
    // exit counter (word 1) back to zero, so the next launch on this workspace needs no reset of its own (the
    // error flag, word 2, stays)
    if (threadIdx.x == 0) {
        const unsigned int out = __hip_atomic_fetch_add(bar + 1, 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        if (out + 1 == static_cast<unsigned int>(G)) {
            __hip_atomic_store(bar, 0u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
            __hip_atomic_store(bar + 1, 0u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        }
    }
}

}  // namespace qz
