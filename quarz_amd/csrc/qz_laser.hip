// Laser envelope of the quasi-static step on the device (src/Laser.hpp, src/Laser.cpp): the complex envelope
// a^ of one box, K slices x M nodes x (Re, Im) doubles in HBM, slice 0 at the head of the box, advanced by one
// time step per call.
//
//   - laser_pond_kernel (Laser::prepare_slice, src/Laser.cpp:292-315): <a^2>, d<a^2>/dr and d<a^2>/dxi of every
//     (slice, node) at time level n.  Each depends only on a^n, so all slices run at once: one thread per
//     (slice, node), HBM-bound (reads 48 B of envelope around the node, writes 24 B).
//   - laser_factor_kernel and laser_march_kernel (Laser::advance_slice, :317-419): the Crank-Nicolson step in t of
//     every slice, marched from the head of the box.  Slice k needs X = a^(n+1) - a^n of slices k-1 and k-2, so
//     the march is serial in xi and runs in one workgroup: per slice the workgroup forms the right-hand sides of
//     all nodes in LDS, one wave runs the right-hand side's Thomas recurrence and the back substitution (serial
//     chains, as in the reference), and the workgroup forms the carry and a^(n+1).  The pivots and c' of the
//     recurrence depend only on the slice's susceptibility, so the factor kernel forms them beforehand for all
//     slices at once, one thread per slice, and the march's serial chain holds one complex quotient per node
//     instead of two: a product with a reciprocal, corrected, checked against the division, and divided where that
//     differs (march_box).  The carry stays in registers and the right-hand sides in LDS.
//
// The arithmetic of each node follows the reference's expressions in the same order (no contraction), so the
// result equals the serial CPU restatement bit for bit.  Scope: laser.l = 0 (no vortex), no ionization losses,
// one rank that owns the whole box (the guard rows of the head of the box are zero).
#include "qz_internal.hpp"
#include "host/simulation.hpp"

#include <cmath>
#include <cstring>
#include <memory>
#include <stdexcept>

namespace {

using qz::Real;

struct Cx { double re, im; };
// src/Laser.cpp:13-21
__device__ __forceinline__ Cx cadd(Cx a, Cx b) { return {a.re + b.re, a.im + b.im}; }
__device__ __forceinline__ Cx csub(Cx a, Cx b) { return {a.re - b.re, a.im - b.im}; }
__device__ __forceinline__ Cx cmul(Cx a, Cx b) { return {a.re * b.re - a.im * b.im, a.re * b.im + a.im * b.re}; }
__device__ __forceinline__ Cx cscale(double s, Cx a) { return {s * a.re, s * a.im}; }
__device__ __forceinline__ Cx cdiv(Cx a, Cx b) {
    const double d = b.re * b.re + b.im * b.im;
    return {(a.re * b.re + a.im * b.im) / d, (a.im * b.re - a.re * b.im) / d};
}

constexpr int kPondThreads = 256;
constexpr int kFactorThreads = 64;
constexpr int kMarchThreads = 512;
constexpr long kMaxLds = 160 * 1024;
constexpr int kMaxNodes = 1861;   // 11 doubles per node in 160 KB (MarchLds)
static_assert(kMaxNodes <= 4 * kMarchThreads, "a thread of the march owns at most four nodes");

// the diagonal's constant part, cd 2/(dt dxi) - 4 i k0 / dt (src/Laser.cpp:352-361)
__device__ __forceinline__ Cx march_alpha(double dxi, double dt, double k0, int scheme) {
    const double cd = scheme == 0 ? 4.0 : (scheme == 1 ? 3.0 : 2.0);
    const double s0 = 2.0 / (dt * dxi);
    const double s1 = cd * s0, s2 = 4.0 / dt;
    return Cx{s1, -s2 * k0};
}

__device__ __forceinline__ void pond_node(long i, const double* __restrict__ a, double* __restrict__ pond,
                                          const double* __restrict__ gm, const double* __restrict__ g0,
                                          const double* __restrict__ gp, int M, double fac, double idxi) {
    const int k = static_cast<int>(i / M), j = static_cast<int>(i - static_cast<long>(k) * M);
    const int N = M - 1;
    auto mag = [&](int l, int jj) {   // <a^2> / fac at (slice l, node jj)
        const double* p = a + (static_cast<long>(l) * M + jj) * 2;
        return p[0] * p[0] + p[1] * p[1];
    };
    const double m0 = fac * mag(k, j);
    const double m1 = k >= 1 ? fac * mag(k - 1, j) : 0.0;
    const double m2 = k >= 2 ? fac * mag(k - 2, j) : 0.0;
    // FieldSolver::gradient of <a^2> (src/FieldSolver.cpp:193-201): one-sided at the wall, zero on the axis
    double d;
    if (j == 0) d = 0.0;
    else if (j == N) d = g0[N] * m0 + gm[N] * (fac * mag(k, N - 1)) + gp[N] * (fac * mag(k, N - 2));
    else d = gm[j] * (fac * mag(k, j - 1)) + g0[j] * m0 + gp[j] * (fac * mag(k, j + 1));
    double* q = pond + i * 3;
    q[0] = m0;
    q[1] = d;
    q[2] = (3.0 * m0 - 4.0 * m1 + m2) * 0.5 * idxi;
}

// The coefficient half of each slice's Thomas recurrence, for every slice at once (one thread per slice): the
// pivots m_j = diag_j + a_j c'_{j-1} and c'_j = -c_j / m_j of src/Laser.cpp:385-393 depend on the slice's
// susceptibility and the operator, not on the carry, so only the right-hand side's recurrence stays in the
// march.  fac: (K, N, 4) doubles, m.re, m.im, c'.re, c'.im of (slice k, node j): slice-major, so that the march's
// workgroup reads a slice's rows with neighbouring addresses.
__device__ __forceinline__ void factor_slice(int k, const double* __restrict__ chi, const double* __restrict__ la,
                                             const double* __restrict__ lb, const double* __restrict__ lc,
                                             double* __restrict__ fac, int M, double dxi, double dt, double k0,
                                             int scheme) {
    const int N = M - 1;
    const Cx alpha = march_alpha(dxi, dt, k0, scheme);
    const double* ch = chi ? chi + static_cast<long>(k) * M : nullptr;
    Cx cprev{0.0, 0.0};
    for (int j = 0; j < N; ++j) {
        const double aj = j > 0 ? la[j] : 0.0, bj = lb[j], cj = lc[j];
        const Cx hd{bj - (ch ? ch[j] : 0.0), 0.0};
        const Cx diag = csub(alpha, hd);
        const double lo = -aj, up = -cj;
        const Cx m = csub(diag, cscale(lo, cprev));
        const Cx cpj = cdiv(Cx{up, 0.0}, m);
        double* f = fac + (static_cast<long>(k) * N + j) * 4;
        f[0] = m.re; f[1] = m.im; f[2] = cpj.re; f[3] = cpj.im;
        cprev = cpj;
    }
}

// the other lane's value within each pair of lanes (0 with 1): the real and imaginary parts of one complex number
__device__ __forceinline__ double pair_swap(double x) {
    const int lo = __builtin_amdgcn_mov_dpp(__double2loint(x), 0xB1, 0xF, 0xF, true);   // quad_perm [1, 0, 3, 2]
    const int hi = __builtin_amdgcn_mov_dpp(__double2hiint(x), 0xB1, 0xF, 0xF, true);
    return __hiloint2double(hi, lo);
}
// `src` of the pair of lanes before (after) this one among the 16 of a DPP row; the first (last) pair keeps `edge`
__device__ __forceinline__ double pair_prev(double edge, double src) {
    const int lo = __builtin_amdgcn_update_dpp(__double2loint(edge), __double2loint(src), 0x112, 0xF, 0xF, false);
    const int hi = __builtin_amdgcn_update_dpp(__double2hiint(edge), __double2hiint(src), 0x112, 0xF, 0xF, false);
    return __hiloint2double(hi, lo);
}
__device__ __forceinline__ double pair_next(double edge, double src) {
    const int lo = __builtin_amdgcn_update_dpp(__double2loint(edge), __double2loint(src), 0x102, 0xF, 0xF, false);
    const int hi = __builtin_amdgcn_update_dpp(__double2hiint(edge), __double2hiint(src), 0x102, 0xF, 0xF, false);
    return __hiloint2double(hi, lo);
}
// the last pair's value to the first (the first's to the last), by a rotation of the DPP row
__device__ __forceinline__ double pair_ror(double x) {
    const int lo = __builtin_amdgcn_mov_dpp(__double2loint(x), 0x122, 0xF, 0xF, true);
    const int hi = __builtin_amdgcn_mov_dpp(__double2hiint(x), 0x122, 0xF, 0xF, true);
    return __hiloint2double(hi, lo);
}
__device__ __forceinline__ double pair_rol(double x) {
    const int lo = __builtin_amdgcn_mov_dpp(__double2loint(x), 0x12E, 0xF, 0xF, true);
    const int hi = __builtin_amdgcn_mov_dpp(__double2hiint(x), 0x12E, 0xF, 0xF, true);
    return __hiloint2double(hi, lo);
}
constexpr int kMarchR = 8;                  // nodes per pair of lanes in the chain
constexpr int kMarchBlock = 8 * kMarchR;
__device__ __forceinline__ double sign_flip(double x, int signbit) {
    return __hiloint2double(__double2hiint(x) ^ signbit, __double2loint(x));
}
__device__ __forceinline__ bool same_bits(double a, double b) {
    return __double_as_longlong(a) == __double_as_longlong(b);
}

// LDS of a march, in doubles: per node of 0 .. N-1 the pivot (re, im), its |m|^2 and 1 / |m|^2, c' and -a_j; per node
// of 0 .. N the right-hand side (then d') and X, real and imaginary parts in arrays of their own; a flag
struct MarchLds {
    int Ne, Me, mm, dy, cp, low, dre, xre, flag, total;
    __host__ __device__ explicit MarchLds(int M) {
        Ne = M & ~1;   // N = M - 1 rounded up to even
        Me = (M + 1) & ~1;
        mm = 0;
        dy = mm + 2 * Ne;
        cp = dy + 2 * Ne;
        low = cp + 2 * Ne;
        dre = low + Ne;
        xre = dre + 2 * Me;
        flag = xre + 2 * Me;
        total = flag + 1;
    }
};

// One workgroup marches the K slices of one box; thread tid owns nodes tid + u kMarchThreads, u < NPT.  The
// serial chain of a slice (d'_j = (rhs_j + a_j d'_{j-1}) / m_j, then the back substitution) bounds the march: it runs
// in one wave, which issues an instruction every four cycles at best, so its instruction count is its time.  A pair
// of lanes forms a node's real and imaginary parts.  As in qz_chain.hpp, 8 pairs hold 8 consecutive nodes each in
// registers and repeat their nodes on the value that the pair before them had after the last step: after 8 steps it has
// passed through 64 nodes, which cost one set of LDS accesses (an LDS read costs the wave 9 to 14 cycles, a write 13 to
// 27; one pair walking the nodes through LDS took 186 cycles per node).  A quotient n / |m|^2 in the chain is n y corrected once by its exact
// residual, y = 1 / |m|^2 formed beforehand: three dependent operations against about twelve of a division.  The
// correction gives the correctly rounded quotient but for operands at the ends of the exponent range, so every node's
// numerator is divided again with the IEEE division and the bits compared: waves 1 to 7 do so while wave 0 runs the back
// substitution, wave 0 for its own nodes after it.  A slice with any difference has its chain run again with that
// division.  The next slice's rows and envelope are loaded beside the chain, and the carry stays in its owner's registers.
// The three forms are one kernel, which takes all 256 registers and spills beside them (alone, NPT = 1 takes 230 and
// spills none, 2 and 4 spill 40 and about 290); a compute unit so holds one march: 256 boxes of 513 nodes x 101 slices
// 3.4 ms, 512 boxes 6.8 and 768 10.3, where the form of 66 registers, three to a unit, took 16.8, 21.6 and 25.4.
// Measured on 401 slices x 321 nodes (bdf2): 6.8 ms a step, 41e3 cycles per slice, where one lane dividing in the
// chain took 30.8 ms.
// Every barrier is reached by all threads in every slice.
template <int NPT>
__device__ __forceinline__ void march_box(const double* __restrict__ a, const double* __restrict__ chi,
                                          double* __restrict__ an, const double* __restrict__ la,
                                          const double* __restrict__ lb, const double* __restrict__ lc,
                                          const double* __restrict__ fac, int K, int M, double dxi, double dt,
                                          double k0, int scheme) {
    extern __shared__ double lds[];
    const MarchLds P(M);
    double2* const ml = reinterpret_cast<double2*>(lds + P.mm);
    double2* const dyl = reinterpret_cast<double2*>(lds + P.dy);   // |m|^2, 1 / |m|^2
    double2* const cpl = reinterpret_cast<double2*>(lds + P.cp);
    double* const low = lds + P.low;
    double* const dre = lds + P.dre;
    double* const dim = dre + P.Me;
    double* const xre = lds + P.xre;
    double* const xim = xre + P.Me;
    int* const bad = reinterpret_cast<int*>(lds + P.flag);
    const int tid = threadIdx.x, N = M - 1;
    // src/Laser.cpp:352-361
    const double c1 = scheme == 0 ? 4.0 : (scheme == 1 ? 4.0 : 2.0);
    const double c2 = scheme == 1 ? -1.0 : 0.0;
    const double s0 = 2.0 / (dt * dxi);
    const double s2 = 4.0 / dt;
    // owned nodes: operator rows, carry (X of the previous slice; G of it (trapezoid) or X two slices back), and the
    // coming slice's envelope around the node, rows and susceptibility
    double aj[NPT], bj[NPT], cj[NPT], hc[NPT];
    Cx car0[NPT], car1[NPT], am[NPT], a0[NPT], ap[NPT], fm[NPT], fc[NPT];
    auto load = [&](int k) {
        const double* ak = a + static_cast<long>(k) * M * 2;
        const double* fk = fac + static_cast<long>(k) * N * 4;
#pragma unroll
        for (int u = 0; u < NPT; ++u) {
            // nodes past the wall repeat it: every load is issued before the first is waited for
            const int j = min(tid + u * kMarchThreads, N), jl = max(j - 1, 0), jr = min(j + 1, N), jn = min(j, N - 1);
            a0[u] = Cx{ak[2 * j], ak[2 * j + 1]};
            am[u] = Cx{ak[2 * jl], ak[2 * jl + 1]};
            ap[u] = Cx{ak[2 * jr], ak[2 * jr + 1]};
            const double* f = fk + static_cast<long>(jn) * 4;
            fm[u] = Cx{f[0], f[1]};
            fc[u] = Cx{f[2], f[3]};
            hc[u] = chi ? chi[static_cast<long>(k) * M + j] : 0.0;
        }
    };
#pragma unroll
    for (int u = 0; u < NPT; ++u) {
        const int j = tid + u * kMarchThreads;
        aj[u] = bj[u] = cj[u] = 0.0;
        car0[u] = car1[u] = Cx{0.0, 0.0};
        if (j < N) {
            aj[u] = j > 0 ? la[j] : 0.0;
            bj[u] = lb[j];
            cj[u] = lc[j];
            low[j] = -aj[u];
        }
    }
    if (tid == 0) *bad = 0;
    load(0);
    for (int k = 0; k < K; ++k) {
        double* ank = an + static_cast<long>(k) * M * 2;
        Cx r[NPT], A0[NPT], Am[NPT], Ap[NPT];   // this slice's right-hand side and envelope
        double hdr[NPT];
        // the right-hand side: hist + 2 H a^n (src/Laser.cpp:371-384); the slice's pivots and c' into LDS
#pragma unroll
        for (int u = 0; u < NPT; ++u) {
            const int j = tid + u * kMarchThreads;
            A0[u] = a0[u]; Am[u] = am[u]; Ap[u] = ap[u];
            hdr[u] = bj[u] - hc[u];
            r[u] = Cx{0.0, 0.0};
            if (j >= N) continue;
            const Cx m = fm[u];
            const double d = m.re * m.re + m.im * m.im;
            ml[j] = make_double2(m.re, m.im);
            dyl[j] = make_double2(d, 1.0 / d);
            cpl[j] = make_double2(fc[u].re, fc[u].im);
            const Cx hd{hdr[u], 0.0};
            Cx Ha = cmul(hd, A0[u]);
            if (j > 0) Ha = cadd(Ha, cscale(aj[u], Am[u]));
            Ha = cadd(Ha, cscale(cj[u], Ap[u]));
            const Cx xp = car0[u], gp = car1[u];
            const Cx hist = scheme == 0 ? cadd(cscale(c1 * s0, xp), cscale(s2, gp))
                                        : cadd(cscale(c1 * s0, xp), cscale(c2 * s0, gp));
            r[u] = cadd(hist, cscale(2.0, Ha));
            dre[j] = r[u].re;
            dim[j] = r[u].im;
        }
        __syncthreads();
        if (k + 1 < K) load(k + 1);
        const int p = tid & 1, g = (tid >> 1) & 7;
        const int neg_im = p ? static_cast<int>(0x80000000u) : 0, neg_re = p ? 0 : static_cast<int>(0x80000000u);
        if (tid < 16) {   // d' from the axis outwards
            double* const D = p ? dim : dre;
            double carry = 0.0;
            for (int b0 = 0; b0 < N; b0 += kMarchBlock) {
                const int i0 = b0 + g * kMarchR, last = P.Ne - 2;
                double mre[kMarchR], mim[kMarchR], dd[kMarchR], yy[kMarchR], lo[kMarchR], rr[kMarchR], dv[kMarchR];
#pragma unroll
                for (int t = 0; t < kMarchR; t += 2) {
                    const int i = min(i0 + t, last);
                    const double2 l2 = *reinterpret_cast<const double2*>(low + i);
                    const double2 r2 = *reinterpret_cast<const double2*>(D + i);
                    lo[t] = l2.x; lo[t + 1] = l2.y;
                    rr[t] = r2.x; rr[t + 1] = r2.y;
#pragma unroll
                    for (int v = 0; v < 2; ++v) {
                        const double2 m2 = ml[i + v], d2 = dyl[i + v];
                        mre[t + v] = m2.x;
                        mim[t + v] = sign_flip(m2.y, neg_im);
                        dd[t + v] = d2.x;
                        yy[t + v] = d2.y;
                    }
                }
                if (b0 + kMarchBlock > N) {   // no nodes from N on: d' = 0
#pragma unroll
                    for (int t = 0; t < kMarchR; ++t)
                        if (i0 + t >= N) {
                            lo[t] = rr[t] = mim[t] = 0.0;
                            mre[t] = dd[t] = yy[t] = 1.0;
                        }
                }
                const int steps = min(8, (N - b0 + kMarchR - 1) / kMarchR);
                double q = carry;
                dv[kMarchR - 1] = 0.0;
#pragma unroll 1
                for (int st = 0; st < steps; ++st) {
                    q = pair_prev(q, dv[kMarchR - 1]);
                    double dp = q;
#pragma unroll
                    for (int t = 0; t < kMarchR; ++t) {
                        const double sv = rr[t] - lo[t] * dp;
                        const double num = sv * mre[t] + pair_swap(sv) * mim[t];
                        const double q0 = num * yy[t];
                        dp = __builtin_fma(__builtin_fma(-dd[t], q0, num), yy[t], q0);
                        dv[t] = dp;
                    }
                }
#pragma unroll
                for (int t = 0; t < kMarchR; t += 2)
                    if (i0 + t < N) *reinterpret_cast<double2*>(D + i0 + t) = make_double2(dv[t], dv[t + 1]);
                carry = pair_ror(dv[kMarchR - 1]);
            }
        }
        __syncthreads();
        if (tid < 16) {   // back substitution (src/Laser.cpp:394-399), X_N = 0
            const double* const D = p ? dim : dre;
            double* const X = p ? xim : xre;
            double carry = 0.0;
            for (int b0 = (N - 1) / kMarchBlock * kMarchBlock; b0 >= 0; b0 -= kMarchBlock) {
                const int i0 = b0 + g * kMarchR, last = P.Ne - 2;
                double cre[kMarchR], cim[kMarchR], dv[kMarchR], xv[kMarchR];
#pragma unroll
                for (int t = 0; t < kMarchR; t += 2) {
                    const int i = min(i0 + t, last);
                    const double2 d2 = *reinterpret_cast<const double2*>(D + i);
                    dv[t] = d2.x; dv[t + 1] = d2.y;
#pragma unroll
                    for (int v = 0; v < 2; ++v) {
                        const double2 c2 = cpl[i + v];
                        cre[t + v] = c2.x;
                        cim[t + v] = sign_flip(c2.y, neg_re);
                    }
                }
                if (b0 + kMarchBlock > N) {   // X = 0 from N on
#pragma unroll
                    for (int t = 0; t < kMarchR; ++t)
                        if (i0 + t >= N) cre[t] = cim[t] = dv[t] = 0.0;
                }
                const int steps = min(8, (N - b0 + kMarchR - 1) / kMarchR);
                double q = carry;
                xv[0] = 0.0;
#pragma unroll 1
                for (int st = 0; st < steps; ++st) {
                    q = pair_next(q, xv[0]);
                    double x = q;
#pragma unroll
                    for (int t = kMarchR - 1; t >= 0; --t) {
                        x = dv[t] - (cre[t] * x + cim[t] * pair_swap(x));
                        xv[t] = x;
                    }
                }
#pragma unroll
                for (int t = 0; t < kMarchR; t += 2)
                    if (i0 + t < M) *reinterpret_cast<double2*>(X + i0 + t) = make_double2(xv[t], xv[t + 1]);
                carry = pair_rol(xv[0]);
            }
            if (g == 0) X[N] = 0.0;
        }
        // every d' against the IEEE division
        auto quotient = [&](Cx rr, double lo, Cx dprev, Cx m) { return cdiv(csub(rr, cscale(lo, dprev)), m); };
#pragma unroll
        for (int u = 0; u < NPT; ++u) {
            const int j = tid + u * kMarchThreads;
            if (j >= N) continue;
            const Cx dprev = j > 0 ? Cx{dre[j - 1], dim[j - 1]} : Cx{0.0, 0.0};
            const Cx q = quotient(r[u], -aj[u], dprev, Cx{ml[j].x, ml[j].y});
            if (!same_bits(q.re, dre[j]) || !same_bits(q.im, dim[j])) *bad = 1;
        }
        __syncthreads();
        if (*bad) {   // uniform: the slice's chain again, divided (operands at the ends of the exponent range)
#pragma unroll
            for (int u = 0; u < NPT; ++u) {
                const int j = tid + u * kMarchThreads;
                if (j < N) {
                    dre[j] = r[u].re;
                    dim[j] = r[u].im;
                }
            }
            __syncthreads();
            if (tid == 0) {
                *bad = 0;
                Cx dp{0.0, 0.0}, x{0.0, 0.0};
                for (int j = 0; j < N; ++j) {
                    dp = quotient(Cx{dre[j], dim[j]}, low[j], dp, Cx{ml[j].x, ml[j].y});
                    dre[j] = dp.re;
                    dim[j] = dp.im;
                }
                for (int j = N - 1; j >= 0; --j) {
                    x = csub(Cx{dre[j], dim[j]}, cmul(Cx{cpl[j].x, cpl[j].y}, x));
                    xre[j] = x.re;
                    xim[j] = x.im;
                }
            }
            __syncthreads();
        }
        // the carry for the next slice and a^(n+1) = a^n + X (src/Laser.cpp:400-418).  The next slice's first phase
        // writes the pivots and right-hand sides, which nothing reads any more; X is written after its barrier.
#pragma unroll
        for (int u = 0; u < NPT; ++u) {
            const int j = tid + u * kMarchThreads;
            if (j > N) continue;
            const Cx X{xre[j], xim[j]};
            if (scheme != 0) {
                car1[u] = car0[u];
                car0[u] = X;
            } else {
                Cx G{0.0, 0.0};
                if (j < N) {
                    auto Y = [&](Cx av, int jj) { return Cx{xre[jj] + 2.0 * av.re, xim[jj] + 2.0 * av.im}; };
                    const Cx hd{hdr[u], 0.0};
                    Cx HY = cmul(hd, Y(A0[u], j));
                    if (j > 0) HY = cadd(HY, cscale(aj[u], Y(Am[u], j - 1)));
                    HY = cadd(HY, cscale(cj[u], Y(Ap[u], j + 1)));
                    G = cadd(cmul(Cx{0.0, k0}, X), cscale(0.25 * dt, HY));
                }
                car0[u] = X;
                car1[u] = G;
            }
            ank[2 * j] = X.re + A0[u].re;
            ank[2 * j + 1] = X.im + A0[u].im;
        }
    }
}

// One box of a step, the kernels' argument: its arrays, operator rows and constants.  active = 0: a box whose
// envelope is not advanced (dt <= 0); only its ponderomotive arrays are formed.
struct LaserBox {
    const double* a;
    const double* chi;
    double *an, *pond, *fac;
    const double *la, *lb, *lc, *gm, *g0, *gp;
    int K, M, scheme, active;
    double dxi, dt, k0, fac2, idxi;   // fac2: <a^2> / |a^|^2 (1 circular, 1/2 linear); idxi = 1 / dxi
};

// kBatch = false: one box, passed by value; true: box blockIdx.y (pond, factor) or blockIdx.x (march) of `many`
template <bool kBatch>
__global__ __launch_bounds__(kPondThreads) void laser_pond_kernel(LaserBox one, const LaserBox* __restrict__ many) {
    const LaserBox B = kBatch ? many[blockIdx.y] : one;
    const long i = static_cast<long>(blockIdx.x) * kPondThreads + threadIdx.x;
    if (i >= static_cast<long>(B.K) * B.M) return;
    pond_node(i, B.a, B.pond, B.gm, B.g0, B.gp, B.M, B.fac2, B.idxi);
}

template <bool kBatch>
__global__ __launch_bounds__(kFactorThreads) void laser_factor_kernel(LaserBox one,
                                                                      const LaserBox* __restrict__ many) {
    const LaserBox B = kBatch ? many[blockIdx.y] : one;
    const int k = blockIdx.x * kFactorThreads + threadIdx.x;
    if (!B.active || k >= B.K) return;
    factor_slice(k, B.chi, B.la, B.lb, B.lc, B.fac, B.M, B.dxi, B.dt, B.k0, B.scheme);
}

template <bool kBatch>
__global__ __launch_bounds__(kMarchThreads) void laser_march_kernel(LaserBox one, const LaserBox* __restrict__ many) {
    const LaserBox B = kBatch ? many[blockIdx.x] : one;
    if (!B.active) return;   // the whole workgroup, before any barrier
    // nodes per thread: a box of at most 512 nodes keeps one node's rows in registers
    if (B.M <= kMarchThreads)
        march_box<1>(B.a, B.chi, B.an, B.la, B.lb, B.lc, B.fac, B.K, B.M, B.dxi, B.dt, B.k0, B.scheme);
    else if (B.M <= 2 * kMarchThreads)
        march_box<2>(B.a, B.chi, B.an, B.la, B.lb, B.lc, B.fac, B.K, B.M, B.dxi, B.dt, B.k0, B.scheme);
    else
        march_box<4>(B.a, B.chi, B.an, B.la, B.lb, B.lc, B.fac, B.K, B.M, B.dxi, B.dt, B.k0, B.scheme);
}

long march_lds(int M) { return static_cast<long>(MarchLds(M).total) * static_cast<long>(sizeof(double)); }

// glibc exp / cos / sin called through pointers, so that no compiler folds or replaces them: the pulse is
// formed from the C library's values at run time, as the CPU restatement forms it
double (*volatile host_exp)(double) = ::exp;
double (*volatile host_cos)(double) = ::cos;
double (*volatile host_sin)(double) = ::sin;

}  // namespace

struct qz_laser {
    qz::RadialGrid grid;
    qz::FieldSolver solver;
    int K = 0, M = 0, scheme = 1;
    bool circular = false;
    double xi_min = 0, dxi = 0, dt = 0, k0 = 0;
    qz::DevBuf<Real> a, an, pond, fac;
    hipStream_t own = nullptr;
    // a batched step led by this handle: the boxes' descriptors (kept until the next such step) and their copy
    std::vector<LaserBox> boxes;
    qz::DevBuf<char> dboxes;
    ~qz_laser() {
        if (own) (void)hipStreamDestroy(own);
    }
};

#define QZ_LASER_TRY(...)                                   \
    try {                                                   \
        __VA_ARGS__;                                        \
        return QZ_OK;                                       \
    } catch (const std::exception& e) {                     \
        return qz_fail(QZ_EINVAL, e.what());                \
    }

static void laser_check(hipError_t e, const char* what) {
    if (e != hipSuccess) throw std::runtime_error(std::string(what) + ": " + hipGetErrorString(e));
}

extern "C" int qz_laser_create(const double* nodes, int M, int K, double xi_min, double dxi, double dt, double k0,
                               int scheme, int circular, qz_laser** out) {
    if (!nodes || !out) return qz_fail(QZ_EINVAL, "qz_laser_create: null argument");
    if (M < 3 || K < 1) return qz_fail(QZ_EINVAL, "qz_laser_create: need M >= 3 nodes and K >= 1 slices");
    if (scheme < 0 || scheme > 2)
        return qz_fail(QZ_EINVAL, "qz_laser_create: scheme 0 (trapezoid), 1 (bdf2) or 2 (euler)");
    if (!(dxi > 0)) return qz_fail(QZ_EINVAL, "qz_laser_create: dxi must be positive");
    if (!(k0 > 1)) return qz_fail(QZ_EINVAL, "qz_laser_create: k0 = omega0/omega_p must be > 1 (underdense plasma)");
    if (M > kMaxNodes || march_lds(M) > kMaxLds)
        return qz_fail(QZ_ERANGE, "qz_laser_create: the march holds at most 1861 nodes in LDS");
    QZ_LASER_TRY({
        auto L = std::make_unique<qz_laser>();
        laser_check(hipStreamCreateWithFlags(&L->own, hipStreamNonBlocking), "hipStreamCreate");
        L->grid.finalize(std::vector<Real>(nodes, nodes + M), L->own);
        L->solver.init(L->grid, L->own);
        L->K = K; L->M = M; L->scheme = scheme; L->circular = circular != 0;
        L->xi_min = xi_min; L->dxi = dxi; L->dt = dt; L->k0 = k0;
        const size_t n = static_cast<size_t>(K) * M;
        L->a.alloc(2 * n); L->an.alloc(2 * n); L->pond.alloc(3 * n);
        if (dt > 0) L->fac.alloc(4 * static_cast<size_t>(K) * (M - 1));
        laser_check(hipMemsetAsync(L->a.p, 0, sizeof(Real) * 2 * n, L->own), "hipMemsetAsync");
        laser_check(hipMemsetAsync(L->an.p, 0, sizeof(Real) * 2 * n, L->own), "hipMemsetAsync");
        laser_check(hipMemsetAsync(L->pond.p, 0, sizeof(Real) * 3 * n, L->own), "hipMemsetAsync");
        laser_check(hipStreamSynchronize(L->own), "hipStreamSynchronize");
        *out = L.release();
    })
}

extern "C" void qz_laser_destroy(qz_laser* L) { delete L; }

// Laser::Laser's Gaussian pulse (src/Laser.cpp:195-236), laser.l = 0: a^ = a0 / (1 + i s)
// exp(-r^2 / (w0^2 (1 + i s))) exp(-(xi - xi0)^2 / L0^2), s = -focus / Z_R, Z_R = k0 w0^2 / 2, zero at the wall
extern "C" int qz_laser_gaussian(qz_laser* L, double a0, double w0, double L0, double xi0, double focus) {
    if (!L) return qz_fail(QZ_EINVAL, "qz_laser_gaussian: null argument");
    if (!(w0 > 0) || !(L0 > 0)) return qz_fail(QZ_EINVAL, "qz_laser_gaussian: w0 and L0 must be positive");
    QZ_LASER_TRY({
        const int K = L->K, M = L->M;
        std::vector<Real> h(static_cast<size_t>(K) * M * 2);
        const Real zR = 0.5 * L->k0 * w0 * w0;
        const Real s = -focus / zR;
        for (int kl = 0; kl < K; ++kl) {
            const Real xi = L->xi_min + kl * L->dxi;
            const Real lon = host_exp(-(xi - xi0) * (xi - xi0) / (L0 * L0));
            for (int j = 0; j < M; ++j) {
                const Real r = L->grid.r[j];
                const Real den = 1 + s * s;
                const Real pre_re = 1 / den, pre_im = -s / den;
                const Real ex = host_exp(-r * r / (w0 * w0 * den)), ph = r * r * s / (w0 * w0 * den);
                const Real e_re = ex * host_cos(ph), e_im = ex * host_sin(ph);
                const Real amp = (j == M - 1) ? 0.0 : a0 * lon;
                Real* p = h.data() + (static_cast<size_t>(kl) * M + j) * 2;
                p[0] = amp * (pre_re * e_re - pre_im * e_im);
                p[1] = amp * (pre_re * e_im + pre_im * e_re);
            }
        }
        L->a.upload(h, L->own);
        laser_check(hipStreamSynchronize(L->own), "hipStreamSynchronize");
    })
}

extern "C" int qz_laser_set_envelope(qz_laser* L, const double* a_host) {
    if (!L || !a_host) return qz_fail(QZ_EINVAL, "qz_laser_set_envelope: null argument");
    QZ_LASER_TRY({
        laser_check(hipMemcpyAsync(L->a.p, a_host, sizeof(Real) * L->a.n, hipMemcpyHostToDevice, L->own),
                    "hipMemcpyAsync");
        laser_check(hipStreamSynchronize(L->own), "hipStreamSynchronize");
    })
}

extern "C" int qz_laser_get(qz_laser* L, int what, double* out_host) {
    if (!L || !out_host) return qz_fail(QZ_EINVAL, "qz_laser_get: null argument");
    if (what != 0 && what != 1) return qz_fail(QZ_EINVAL, "qz_laser_get: what is 0 (envelope) or 1 (ponderomotive)");
    const qz::DevBuf<Real>& b = what == 0 ? L->a : L->pond;
    QZ_LASER_TRY({
        laser_check(hipMemcpyAsync(out_host, b.p, sizeof(Real) * b.n, hipMemcpyDeviceToHost, L->own),
                    "hipMemcpyAsync");
        laser_check(hipStreamSynchronize(L->own), "hipStreamSynchronize");
    })
}

extern "C" int qz_laser_device(qz_laser* L, int what, double** ptr) {
    if (!L || !ptr) return qz_fail(QZ_EINVAL, "qz_laser_device: null argument");
    if (what != 0 && what != 1) return qz_fail(QZ_EINVAL, "qz_laser_device: what is 0 (envelope) or 1 (ponderomotive)");
    *ptr = what == 0 ? L->a.p : L->pond.p;
    return QZ_OK;
}

static LaserBox box_of(qz_laser* L, const double* chi) {
    LaserBox B{};
    B.a = L->a.p; B.chi = chi; B.an = L->an.p; B.pond = L->pond.p; B.fac = L->fac.p;
    B.la = L->solver.d_a[qz::FieldSolver::L0].p;
    B.lb = L->solver.d_b[qz::FieldSolver::L0].p;
    B.lc = L->solver.d_c[qz::FieldSolver::L0].p;
    B.gm = L->solver.d_gm.p; B.g0 = L->solver.d_g0.p; B.gp = L->solver.d_gp.p;
    B.K = L->K; B.M = L->M; B.scheme = L->scheme; B.active = L->dt > 0 ? 1 : 0;
    B.dxi = L->dxi; B.dt = L->dt; B.k0 = L->k0;
    B.fac2 = L->circular ? 1.0 : 0.5;
    B.idxi = 1.0 / L->dxi;
    return B;
}

static int set_march_lds(long lds) {
    QZ_HIP(hipFuncSetAttribute(reinterpret_cast<const void*>(laser_march_kernel<false>),
                               hipFuncAttributeMaxDynamicSharedMemorySize, static_cast<int>(lds)));
    QZ_HIP(hipFuncSetAttribute(reinterpret_cast<const void*>(laser_march_kernel<true>),
                               hipFuncAttributeMaxDynamicSharedMemorySize, static_cast<int>(lds)));
    return QZ_OK;
}

// One time step of the envelope: prepare_slice of every slice (the ponderomotive arrays at level n), then the
// march of advance_slice from the head of the box; the advanced envelope becomes the current one
// (Laser::begin_step of the next step, src/Laser.cpp:258-262).  chi: (K, M) device array, or null for vacuum.
extern "C" int qz_laser_step(qz_laser* L, const double* chi, void* stream) {
    if (!L) return qz_fail(QZ_EINVAL, "qz_laser_step: null argument");
    hipStream_t st = stream ? static_cast<hipStream_t>(stream) : L->own;
    const LaserBox B = box_of(L, chi);
    const long n = static_cast<long>(B.K) * B.M;
    hipLaunchKernelGGL(laser_pond_kernel<false>, dim3(static_cast<unsigned>((n + kPondThreads - 1) / kPondThreads)),
                       dim3(kPondThreads), 0, st, B, nullptr);
    QZ_HIP(hipGetLastError());
    if (B.active) {
        const int rc = set_march_lds(march_lds(B.M));
        if (rc != QZ_OK) return rc;
        hipLaunchKernelGGL(laser_factor_kernel<false>, dim3((B.K + kFactorThreads - 1) / kFactorThreads),
                           dim3(kFactorThreads), 0, st, B, nullptr);
        QZ_HIP(hipGetLastError());
        hipLaunchKernelGGL(laser_march_kernel<false>, dim3(1), dim3(kMarchThreads), march_lds(B.M), st, B, nullptr);
        QZ_HIP(hipGetLastError());
        std::swap(L->a, L->an);
    }
    if (!stream) QZ_HIP(hipStreamSynchronize(st));
    return QZ_OK;
}

// Many boxes, one step each, in one launch per kernel: every box's march is one workgroup, so the boxes march
// at once.  Each box's results are those of qz_laser_step.
extern "C" int qz_laser_step_batched(qz_laser* const* Ls, int n, const double* const* chis, void* stream) {
    if (!Ls || n < 1) return qz_fail(QZ_EINVAL, "qz_laser_step_batched: no boxes");
    if (n > 65535) return qz_fail(QZ_ERANGE, "qz_laser_step_batched: at most 65535 boxes per call");
    for (int i = 0; i < n; ++i) {
        if (!Ls[i]) return qz_fail(QZ_EINVAL, "qz_laser_step_batched: null box");
        for (int j = 0; j < i; ++j)
            if (Ls[j] == Ls[i]) return qz_fail(QZ_EINVAL, "qz_laser_step_batched: a box appears twice");
    }
    qz_laser* L0 = Ls[0];
    hipStream_t st = stream ? static_cast<hipStream_t>(stream) : L0->own;
    QZ_LASER_TRY({
        // the descriptors of an earlier batched step on this stream may still be read: wait for it
        laser_check(hipStreamSynchronize(st), "hipStreamSynchronize");
        L0->boxes.resize(static_cast<size_t>(n));
        long maxn = 1, lds = 0;
        int maxk = 1;
        for (int i = 0; i < n; ++i) {
            L0->boxes[i] = box_of(Ls[i], chis ? chis[i] : nullptr);
            const LaserBox& B = L0->boxes[i];
            maxn = std::max(maxn, static_cast<long>(B.K) * B.M);
            maxk = std::max(maxk, B.K);
            if (B.active) lds = std::max(lds, march_lds(B.M));
        }
        const size_t bytes = sizeof(LaserBox) * static_cast<size_t>(n);
        if (L0->dboxes.n < bytes) L0->dboxes.alloc(bytes);
        laser_check(hipMemcpyAsync(L0->dboxes.p, L0->boxes.data(), bytes, hipMemcpyHostToDevice, st), "hipMemcpyAsync");
        const LaserBox* dev = reinterpret_cast<const LaserBox*>(L0->dboxes.p);
        hipLaunchKernelGGL(laser_pond_kernel<true>,
                           dim3(static_cast<unsigned>((maxn + kPondThreads - 1) / kPondThreads), n),
                           dim3(kPondThreads), 0, st, LaserBox{}, dev);
        laser_check(hipGetLastError(), "laser_pond_kernel");
        if (lds > 0) {
            if (set_march_lds(lds) != QZ_OK) throw std::runtime_error(qz_last_error());
            hipLaunchKernelGGL(laser_factor_kernel<true>, dim3((maxk + kFactorThreads - 1) / kFactorThreads, n),
                               dim3(kFactorThreads), 0, st, LaserBox{}, dev);
            laser_check(hipGetLastError(), "laser_factor_kernel");
            hipLaunchKernelGGL(laser_march_kernel<true>, dim3(n), dim3(kMarchThreads), lds, st, LaserBox{}, dev);
            laser_check(hipGetLastError(), "laser_march_kernel");
            for (int i = 0; i < n; ++i)
                if (L0->boxes[i].active) std::swap(Ls[i]->a, Ls[i]->an);
        }
        if (!stream) laser_check(hipStreamSynchronize(st), "hipStreamSynchronize");
    })
}

// Laser::sums (src/Laser.cpp:421-438) of the current envelope, on the host in slice and node order:
// {sum |a|^2 dV, sum |a|^2 xi dV (the user's xi), sum |a|^2 r^2 dV, max |a|, sum |a|^2 xi^2 dV}
extern "C" int qz_laser_sums(qz_laser* L, double* out5) {
    if (!L || !out5) return qz_fail(QZ_EINVAL, "qz_laser_sums: null argument");
    QZ_LASER_TRY({
        std::vector<Real> h;
        L->a.download(h, L->own);
        const int K = L->K, M = L->M;
        double S[5] = {0, 0, 0, 0, 0};
        for (int kl = 0; kl < K; ++kl) {
            const Real xi = L->xi_min + kl * L->dxi;
            for (int j = 0; j < M; ++j) {
                const Real* p = h.data() + (static_cast<size_t>(kl) * M + j) * 2;
                const Real m2 = p[0] * p[0] + p[1] * p[1];
                const Real dv = L->grid.V[j] * L->dxi;
                S[0] += m2 * dv;
                S[1] += m2 * (Real(0) - xi) * dv;
                S[2] += m2 * L->grid.r[j] * L->grid.r[j] * dv;
                S[3] = std::max(S[3], std::sqrt(m2));
                S[4] += m2 * xi * xi * dv;
            }
        }
        std::memcpy(out5, S, sizeof(S));
    })
}
