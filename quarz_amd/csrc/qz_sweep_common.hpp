// Device helpers of the quasi-static sweep kernels (one workgroup per run, qz_sweep.hip; several per run,
// qz_sweep_multi.hip): the workspace layout of a run, the deposit terms, the Thomas recurrences, the sequential
// node sums and the radial stencils.  Every expression keeps the reference's operation order (file:line at
// each function), so both kernels reproduce a serial CPU build bit for bit.
#pragma once

#include <hip/hip_runtime.h>

#include <type_traits>

#include "qz_chain.hpp"
#include "qz_device.hpp"
#include "../../include/quarz_amd.h"

namespace qz {

// workspace arrays (M doubles each)
enum WsArr : int {
    // node sums of the plasma deposit (the first 24 ids are also the deposit component ids)
    W_RHOT0 = 0, W_DRHO0, W_JZ0, W_CHI0, W_NE0, W_NI0, W_JPR1, W_JPI1,
    W_RHOT1R, W_RHOT1I, W_DRHO1R, W_DRHO1I, W_JZ1R, W_JZ1I, W_CHI1R, W_CHI1I, W_NE1R, W_NE1I, W_NI1R, W_NI1I,
    W_JPR0, W_JPI0, W_JPR2, W_JPI2,
    // S+ node sums, order r1 i1 r0 i0 r2 i2
    W_SR1, W_SI1, W_SR0, W_SI0, W_SR2, W_SI2,
    // fields of the slice
    W_EZ0, W_EZ1R, W_EZ1I, W_BZ0, W_BZ1R, W_BZ1I,
    W_WPR1, W_WPI1, W_WPR0, W_WPI0, W_WPR2, W_WPI2,
    W_BPR1, W_BPI1, W_BPR0, W_BPI0, W_BPR2, W_BPI2,
    // Thomas factors (m, c') of this slice's chi-dependent operators, in the order L1D, L1F, L0, L2D
    W_FAC0,
    W_NARR = W_FAC0 + 8
};

enum OpId : int { OP_L0 = 0, OP_L1D = 1, OP_L1F = 2, OP_L2D = 3 };

template <int V> using IC = std::integral_constant<int, V>;

// value of deposit component `comp` for the node on side cc (0: j, 1: j+1) of one particle
// (PlasmaSpecies::deposit, src/PlasmaSpecies.cpp:420-477; rho is not read on this path and not formed)
__device__ __forceinline__ Real dep_value(int comp, int cc, int j, Real t, Real c, Real sn, Real ir, Real invd,
                                          Real gam, Real PX, Real PY, Real pz, Real wi, Real q, Real qm, Real iv,
                                          Real ih) {
    const Real W = cc == 0 ? Real(1) - t : t;
    const Real dW = cc == 0 ? -ih : ih;
    const Real ux = PX * invd, uy = PY * invd;
    const Real ur = c * ux + sn * uy, uth = c * uy - sn * ux;
    const Real wq = wi * q;
    const Real chif = Real(1);
    const Real a = wq * W * iv;
    switch (comp) {
        case W_RHOT0: return a;
        case W_DRHO0: return wq * ur * dW * iv;
        case W_JZ0: return a * pz * invd;
        case W_CHI0: return chif * a * qm * invd;
        case W_NE0: return q < 0 ? wi * W * iv * gam * invd : Real(0);
        case W_NI0: return q < 0 ? Real(0) : wi * W * iv * gam * invd;
        case W_JPR1: return a * ur;
        case W_JPI1: return a * uth;
        case W_RHOT1R: return a * c;
        case W_RHOT1I: return -a * sn;
        case W_DRHO1R:
        case W_DRHO1I: {
            const Real dr = wq * ur * dW * iv;
            const Real Wor = (j == 0) ? (cc == 0 ? Real(0) : ih) : W * ir;
            const Real th = wq * uth * Wor * iv;
            return comp == W_DRHO1R ? dr * c - th * sn : -dr * sn - th * c;
        }
        case W_JZ1R: return a * pz * invd * c;
        case W_JZ1I: return -(a * pz * invd) * sn;
        case W_CHI1R: return chif * a * qm * invd * c;
        case W_CHI1I: return -(chif * a * qm * invd) * sn;
        case W_NE1R: return q < 0 ? wi * W * iv * gam * invd * c : Real(0);
        case W_NE1I: return q < 0 ? -(wi * W * iv * gam * invd) * sn : Real(0);
        case W_NI1R: return q < 0 ? Real(0) : wi * W * iv * gam * invd * c;
        case W_NI1I: return q < 0 ? Real(0) : -(wi * W * iv * gam * invd) * sn;
        case W_JPR0: return a * ux;
        case W_JPI0: return a * uy;
        case W_JPR2: {
            const Real c2 = c * c - sn * sn, s2 = Real(2) * c * sn;
            return a * (ux * c2 + uy * s2);
        }
        case W_JPI2: {
            const Real c2 = c * c - sn * sn, s2 = Real(2) * c * sn;
            return a * (uy * c2 - ux * s2);
        }
        default: return Real(0);
    }
}

// exclusive scan of n ints in place by one wave
__device__ __forceinline__ void wave_exclusive_scan(int* __restrict__ v, int n, int lane) {
    const int per = (n + 63) / 64;
    const int lo = lane * per, hi = min(lo + per, n);
    int s = 0;
    for (int i = lo; i < hi; ++i) s += v[i];
    int incl = s;
    for (int d = 1; d < 64; d <<= 1) {
        const int o = __shfl_up(incl, d, 64);
        if (lane >= d) incl += o;
    }
    int run = incl - s;
    for (int i = lo; i < hi; ++i) {
        const int t = v[i];
        v[i] = run;
        run += t;
    }
}

// ((0 + v[e0]) + v[e0+1]) + ... + v[e1-1]: the sequential sum of one node list.  Lists are long where the
// plasma is compressed (hundreds of entries in a blowout sheath), so the loads run one batch of eight ahead of
// the dependent adds: a long list costs about one add latency per entry.
struct Batch8 {
    Real a0, a1, a2, a3, a4, a5, a6, a7;
    __device__ __forceinline__ void load(const Real* v) {
        a0 = v[0]; a1 = v[1]; a2 = v[2]; a3 = v[3]; a4 = v[4]; a5 = v[5]; a6 = v[6]; a7 = v[7];
    }
    __device__ __forceinline__ void add_to(Real& acc) const {
        acc += a0; acc += a1; acc += a2; acc += a3; acc += a4; acc += a5; acc += a6; acc += a7;
    }
};

// the same sums of a list of rows of S doubles in global memory: of the row's doubles 0, 8, 16 ... (P of them), side by
// side.  U P loads in flight, each a trip to another die's data.
template <int S, int P, int U> __device__ __forceinline__ void sum_rows(const Real* v, int e0, int e1, Real (&acc)[P]) {
    int e = e0;
#pragma unroll
    for (int c = 0; c < P; ++c) acc[c] = Real(0);
    auto take = [&](auto count) {
        constexpr int n = decltype(count)::value;
        Real p[n][P];
        const Real* q = v + static_cast<size_t>(e) * S;
#pragma unroll
        for (int u = 0; u < n; ++u)
#pragma unroll
            for (int c = 0; c < P; ++c) p[u][c] = q[u * S + 8 * c];
#pragma unroll
        for (int u = 0; u < n; ++u)
#pragma unroll
            for (int c = 0; c < P; ++c) acc[c] += p[u][c];
        e += n;
    };
    while (e + U <= e1) take(IC<U>{});
    if (e + 8 <= e1) take(IC<8>{});
    if (e + 4 <= e1) take(IC<4>{});
    while (e < e1) take(IC<1>{});
}

// the same sums of two lists of one range, the second `off` doubles after the first (off = 0: the first again); kDeep: 16
// entries of each in flight (64 registers), else 8
template <bool kDeep>
__device__ __forceinline__ void sum_lists(const Real* v, int off, int e0, int e1, Real& x, Real& y) {
    Real ax = Real(0), ay = Real(0);
    int e = e0;
    const Real* w = v + off;
    if constexpr (kDeep)
        for (; e + 16 <= e1; e += 16) {
            Batch8 a, b, c, d;
            a.load(v + e); b.load(w + e); c.load(v + e + 8); d.load(w + e + 8);
            a.add_to(ax); b.add_to(ay); c.add_to(ax); d.add_to(ay);
        }
    for (; e + 8 <= e1; e += 8) {
        Batch8 a, b;
        a.load(v + e); b.load(w + e);
        a.add_to(ax); b.add_to(ay);
    }
    if (e + 4 <= e1) {
        const Real a0 = v[e], a1 = v[e + 1], a2 = v[e + 2], a3 = v[e + 3];
        const Real b0 = w[e], b1 = w[e + 1], b2 = w[e + 2], b3 = w[e + 3];
        ax += a0; ax += a1; ax += a2; ax += a3;
        ay += b0; ay += b1; ay += b2; ay += b3;
        e += 4;
    }
    for (; e < e1; ++e) {
        const Real a0 = v[e], b0 = w[e];
        ax += a0;
        ay += b0;
    }
    x = ax;
    y = ay;
}

// entries < key in the index-sorted range idx[lo, hi)
__device__ __forceinline__ int count_less(const unsigned short* __restrict__ idx, int lo, int hi, int key) {
    int a = lo, b = hi;
    while (a < b) {
        const int mid = (a + b) >> 1;
        if (static_cast<int>(idx[mid]) < key) a = mid + 1; else b = mid;
    }
    return a - lo;
}

// Opaque register fence: the compiler must assume the values changed here, so nothing derived from them is
// hoisted out of the enclosing loop (per-particle live ranges stay at the cache itself).
template <class T, int PT> __device__ __forceinline__ void fence_regs(T (&a)[PT]) {
#pragma unroll
    for (int i = 0; i < PT; ++i) asm volatile("" : "+v"(a[i]));
}

// f(IC<0>) ... f(IC<n - 1>)
template <int n, int i = 0, class F> __device__ __forceinline__ void for_each_batch(F&& f) {
    if constexpr (i < n) {
        f(IC<i>{});
        for_each_batch<n, i + 1>(f);
    }
}

// grid_weights with the cell searched from `near`: a particle moves by a cell or less in most slices, and the cell and
// its neighbours' four nodes cost one LDS round trip where the bisection costs one per level
__device__ __forceinline__ void grid_weights_near(const Real* __restrict__ r, const Real* __restrict__ inv_h, int N, Real R,
                                                  Real x, int near, int& j, Real& t) {
    const Real a = r[max(near - 1, 0)], b = r[near], c = r[near + 1], d = r[min(near + 2, N)];
    if (x > Real(0) && x < R && a <= x && x < d) j = x < b ? near - 1 : (x < c ? near : near + 1);
    else j = grid_locate(r, N, R, x);
    t = (x - r[j]) * inv_h[j];
    t = t < Real(0) ? Real(0) : (t > Real(1) ? Real(1) : t);
}

__device__ __forceinline__ Real lin(const Real* f, int j, Real t) { return (Real(1) - t) * f[j] + t * f[j + 1]; }

// 3-point gradients and f/r (FieldSolver::gradient / gradient_odd / over_r, src/FieldSolver.cpp:263-289)
struct Stencil {
    const Real *gm, *g0, *gp, *ir;
    int N;
    __device__ __forceinline__ Real grad(const Real* f, int j) const {
        if (j == 0) return Real(0);
        if (j == N) return g0[N] * f[N] + gm[N] * f[N - 1] + gp[N] * f[N - 2];
        return gm[j] * f[j - 1] + g0[j] * f[j] + gp[j] * f[j + 1];
    }
    __device__ __forceinline__ Real grad_odd(const Real* f, int j) const {
        if (j == 0) return f[1] * ir[0];
        if (j == N) return g0[N] * f[N] + gm[N] * f[N - 1] + gp[N] * f[N - 2];
        return gm[j] * f[j - 1] + g0[j] * f[j] + gp[j] * f[j + 1];
    }
    __device__ __forceinline__ Real over_r(const Real* f, int j) const { return (j == 0 ? f[1] : f[j]) * ir[j]; }
};

// The cold rings of one species at the head of the box (PlasmaSpecies::load, src/PlasmaSpecies.cpp:202-295, with
// the host load's expression order): particles [i0, i1) of `st`, node radii r (LDS), and a fresh AB history.
__device__ __forceinline__ void load_rings(const qz_plasma_rings& rg, const qz_species_state& st, int ord,
                                           const Real* r, int i0, int i1, int stride) {
    constexpr Real PI = 3.14159265358979323846;
    const int nt = rg.ntheta, ppc = rg.ppc;
    for (int i = i0; i < i1; i += stride) {
        const int ring = i / nt, l = i - ring * nt;
        const int j = ring / ppc, sub = ring - j * ppc;
        const Real hc = r[j + 1] - r[j];
        const Real ra = r[j] + Real(sub) * hc / Real(ppc), rb = r[j] + Real(sub + 1) * hc / Real(ppc);
        const Real rc = (Real(2.0) / Real(3.0)) * (rb * rb * rb - ra * ra * ra) / (rb * rb - ra * ra);
        const Real volume = (Real(1.0) * rg.density) * PI * (rb * rb - ra * ra);
        const int a = (ring % 2) * nt + l;
        st.x[i] = nt == 1 ? rc : rc * rg.cs[a];
        st.y[i] = nt == 1 ? Real(0) : rc * rg.cs[2 * nt + a];
        st.px[i] = Real(0);
        st.py[i] = Real(0);
        st.dl[i] = Real(1);   // gamma - p_z of a particle at rest
        st.w[i] = Real(1.0) * volume / Real(nt);
        for (int v = 0; v < 5 * ord; ++v) st.hist[static_cast<size_t>(v) * st.cap + i] = Real(0);
    }
}

}  // namespace qz
