// Serial recurrences over the radial rows (Thomas solves and factors) run by one wave, in the serial order and with
// the serial operations of every row.
//
// A lone wave issues one instruction per four cycles at best (five to six in these loops, 35 more per taken branch), and
// an FP64 add, multiply or fma depends on the one before it at no extra cost; an LDS read costs it 9 to 14 cycles
// and a write 13 to 27 (measured).  One lane walking the rows
// through LDS therefore spends most of its time on the reads and writes: 118 cycles per row of a solve.  Here the
// 16 lanes of a DPP row hold R consecutive rows each in registers, and every step all lanes run their R rows on the
// value that the lane before them had after the last step (row_shr / row_shl): after 16 steps the value has passed
// through all 16 R rows, each row formed from its true predecessor, and 16 R rows cost one set of LDS accesses.  A
// step costs 4 + 3 R instructions forward and 4 + 2 R backward, so the recurrence itself is nearly all of it.  The
// four DPP rows of the wave hold four systems.
#pragma once

#include <hip/hip_runtime.h>

#include "qz_device.hpp"

namespace qz {

constexpr int kChainR = 8;                  // rows per lane
constexpr int kChainBlock = 16 * kChainR;   // rows of one block of steps

// `src` of the lane before (after) this one in its DPP row; the row's first (last) lane keeps `edge`
__device__ __forceinline__ Real dpp_prev(Real edge, Real src) {
    const int lo = __builtin_amdgcn_update_dpp(__double2loint(edge), __double2loint(src), 0x111, 0xF, 0xF, false);
    const int hi = __builtin_amdgcn_update_dpp(__double2hiint(edge), __double2hiint(src), 0x111, 0xF, 0xF, false);
    return __hiloint2double(hi, lo);
}
__device__ __forceinline__ Real dpp_next(Real edge, Real src) {
    const int lo = __builtin_amdgcn_update_dpp(__double2loint(edge), __double2loint(src), 0x101, 0xF, 0xF, false);
    const int hi = __builtin_amdgcn_update_dpp(__double2hiint(edge), __double2hiint(src), 0x101, 0xF, 0xF, false);
    return __hiloint2double(hi, lo);
}
// rotate right (left) by one lane within a DPP row: the last lane's value to the first (the first's to the last)
__device__ __forceinline__ Real dpp_ror(Real src) {
    const int lo = __builtin_amdgcn_mov_dpp(__double2loint(src), 0x121, 0xF, 0xF, true);
    const int hi = __builtin_amdgcn_mov_dpp(__double2hiint(src), 0x121, 0xF, 0xF, true);
    return __hiloint2double(hi, lo);
}
__device__ __forceinline__ Real dpp_rol(Real src) {
    const int lo = __builtin_amdgcn_mov_dpp(__double2loint(src), 0x12F, 0xF, 0xF, true);
    const int hi = __builtin_amdgcn_mov_dpp(__double2hiint(src), 0x12F, 0xF, 0xF, true);
    return __hiloint2double(hi, lo);
}

// 1 / d by the hardware's estimate (a relative error of at most 2^-24) and one third-order step: the correctly rounded
// value but for about one operand in 2^19, and at the ends of the exponent range.  Its users compare every result with
// the division.
__device__ __forceinline__ Real chain_recip(Real d) {
    const Real y = __builtin_amdgcn_rcp(d);
    const Real e = __builtin_fma(-d, y, Real(1));
    return __builtin_fma(__builtin_fma(e, e, e), y, y);
}

// rows i .. i + R - 1 (i even) of an LDS array of M values padded to an even count and aligned to 16 bytes; rows from
// M on repeat the array's last pair
template <int R> __device__ __forceinline__ void chain_load(const Real* p, int i, int M, Real (&v)[R]) {
    const int last = (M - 1) & ~1;
#pragma unroll
    for (int r = 0; r < R; r += 2) {
        const double2 t = *reinterpret_cast<const double2*>(p + min(i + r, last));
        v[r] = t.x;
        v[r + 1] = t.y;
    }
}
// the same rows to such an array (its padding may be written)
template <int R> __device__ __forceinline__ void chain_store(Real* p, int i, int M, const Real (&v)[R]) {
#pragma unroll
    for (int r = 0; r < R; r += 2)
        if (i + r < M) *reinterpret_cast<double2*>(p + i + r) = make_double2(v[r], v[r + 1]);
}

// Thomas solve with factors formed beforehand, every array in LDS (Tridiag.cpp:114-125 with c', m precomputed):
//   dp_0 = d_0 / b_0,  dp_i = (d_i - a_i dp_{i-1}) m_i,  x_{M-1} = dp_{M-1},  x_i = dp_i - c'_i x_{i+1}
// d_i is the prepared right-hand side of FieldSolver::solve (src/FieldSolver.cpp:253-259): 0 on Dirichlet
// rows, scale * rhs otherwise, minus fcw on the flux row.  w holds rhs on entry and dp afterwards; the solution goes
// to x (which may be w).  Called by all 64 lanes of a wave, every DPP row with its own system's arguments (a row
// without one repeats another's, and writes the same values).
// Measured (both directions, one wave alone): 513 rows 9.0 us, 257 rows 5.1 us, 65 rows 1.9 us, where one lane per
// system walking the rows through LDS took 23, 12.6 and 3.8 us.  More rows per lane (16) took no less.
template <int R = kChainR>
__device__ __forceinline__ void thomas_wave(const Real* a, const Real* m, const Real* cp, Real b0, Real* w, Real* x,
                                            Real scale, bool dir0, bool dirN, bool fluxN, Real fcw, int M) {
    constexpr int kBlock = 16 * R;
    const int N = M - 1, l = threadIdx.x & 15;
    const int nb = (M + kBlock - 1) / kBlock;
    Real carry = Real(0);   // dp of the row before the block, in its first lane
    for (int b = 0; b < nb; ++b) {
        const int i0 = b * kBlock + l * R;
        Real d[R], av[R], mv[R], pv[R];
        chain_load<R>(w, i0, M, d);
        chain_load<R>(a, i0, M, av);
        chain_load<R>(m, i0, M, mv);
#pragma unroll
        for (int r = 0; r < R; ++r) d[r] = scale * d[r];
        if (i0 == 0) {   // row 0 as (dp_0 - 0 * 0) * 1
            d[0] = (dir0 ? Real(0) : d[0]) / b0;
            av[0] = Real(0);
            mv[0] = Real(1);
        }
        if (b == nb - 1) {   // the wall row, and no rows after it
#pragma unroll
            for (int r = 0; r < R; ++r) {
                if (i0 + r == N) {
                    if (dirN) d[r] = Real(0);
                    else if (fluxN) d[r] -= fcw;
                }
                if (i0 + r > N) d[r] = av[r] = mv[r] = Real(0);
            }
        }
        const int steps = min(16, (M - b * kBlock + R - 1) / R);
        Real q = carry;
        pv[R - 1] = Real(0);
        for (int s = 0; s < steps; s += 4) {
#pragma unroll
            for (int v = 0; v < 4; ++v) {
                q = dpp_prev(q, pv[R - 1]);
                Real p = q;
#pragma unroll
                for (int r = 0; r < R; ++r) {
                    p = (d[r] - av[r] * p) * mv[r];
                    pv[r] = p;
                }
            }
        }
        chain_store<R>(w, i0, M, pv);
        carry = dpp_ror(pv[R - 1]);
    }
    carry = Real(0);   // x of the row after the block, in its last lane
    for (int b = nb - 1; b >= 0; --b) {
        const int i0 = b * kBlock + l * R;
        Real pv[R], cv[R], xv[R];
        chain_load<R>(w, i0, M, pv);
        chain_load<R>(cp, i0, M, cv);
        if (b == nb - 1) {   // x_N = dp_N - 0 * 0; rows after it zero
#pragma unroll
            for (int r = 0; r < R; ++r) {
                if (i0 + r >= N) cv[r] = Real(0);
                if (i0 + r > N) pv[r] = Real(0);
            }
        }
        // the rows' values reach the last block's used lanes from lanes that hold zeros
        Real q = carry;
        xv[0] = Real(0);
        const int steps = min(16, (M - b * kBlock + R - 1) / R);
        for (int s = 0; s < steps; s += 4) {
#pragma unroll
            for (int v = 0; v < 4; ++v) {
                q = dpp_next(q, xv[0]);
                Real p = q;
#pragma unroll
                for (int r = R - 1; r >= 0; --r) {
                    p = pv[r] - cv[r] * p;
                    xv[r] = p;
                }
            }
        }
        chain_store<R>(x, i0, M, xv);
        carry = dpp_rol(xv[0]);
    }
}

// Thomas factors of (L - chi) with the Dirichlet rows of FieldSolver::solve (src/FieldSolver.cpp:253-256):
//   bw_i = b_i (Dirichlet row) or b_i - chi_i;  c'_0 = c_0 / bw_0;  m_i = 1 / (bw_i - a_i c'_{i-1});  c'_i = c_i m_i
// Rows 0 .. N-1 from a, b, c (LDS); the last row's a_N, b_N given (the flux and Dirichlet variants of L_1
// share every other row).  put(i, m_i, c'_i) takes every row, from the lane that holds it.  Returns bw_0.  Called as
// thomas_wave.
// The reciprocal in the chain is chain_recip; after its steps a block is divided once more with the IEEE division, all
// its rows at once, and one with any difference is run again with that division in the chain.
// Measured: 513 rows 16.8 us, 257 rows 9.1 us, where one lane per system dividing in the chain took 48 and 23 us.
template <int R = kChainR, class Put>
__device__ __forceinline__ Real thomas_factor_wave(const Real* a, const Real* b, const Real* c, const Real* chi, Real aN,
                                                   Real bN, bool dir0, bool dirN, int M, Put put) {
    constexpr int kBlock = 16 * R;
    const int N = M - 1, l = threadIdx.x & 15;
    const int nb = (M + kBlock - 1) / kBlock;
    const Real bw0 = dir0 ? b[0] : b[0] - chi[0];
    Real carry = Real(0);
    for (int k = 0; k < nb; ++k) {
        const int i0 = k * kBlock + l * R;
        Real w[R], av[R], cv[R], mv[R], pv[R];
        chain_load<R>(b, i0, M, w);
        chain_load<R>(chi, i0, M, av);
#pragma unroll
        for (int r = 0; r < R; ++r) w[r] = w[r] - av[r];
        chain_load<R>(a, i0, M, av);
        chain_load<R>(c, i0, M, cv);
        if (i0 == 0) {   // row 0 as c'_0 * (1 / (1 - 0 * 0))
            w[0] = Real(1);
            av[0] = Real(0);
            cv[0] = cv[0] / bw0;
        }
        if (k == nb - 1) {
#pragma unroll
            for (int r = 0; r < R; ++r) {
                if (i0 + r == N) {
                    w[r] = dirN ? bN : bN - chi[N];
                    av[r] = aN;
                }
                if (i0 + r > N) {
                    w[r] = Real(1);
                    av[r] = cv[r] = Real(0);
                }
            }
        }
        const int steps = min(16, (M - k * kBlock + R - 1) / R);
        auto rows = [&](Real p, auto recip) {
#pragma unroll
            for (int r = 0; r < R; ++r) {
                mv[r] = recip(w[r] - av[r] * p);
                p = cv[r] * mv[r];
                pv[r] = p;
            }
        };
        auto newton = [](Real d) { return chain_recip(d); };
        auto divide = [](Real d) { return Real(1) / d; };
        Real q = carry;
        pv[R - 1] = Real(0);
        for (int s = 0; s < steps; s += 2) {
#pragma unroll
            for (int v = 0; v < 2; ++v) {
                q = dpp_prev(q, pv[R - 1]);
                rows(q, newton);
            }
        }
        bool bad = false;
        {
            Real p = q;
#pragma unroll
            for (int r = 0; r < R; ++r) {
                const Real t = divide(w[r] - av[r] * p);
                bad = bad || __double_as_longlong(t) != __double_as_longlong(mv[r]);
                p = pv[r];
            }
        }
        if (__ballot(bad ? 1 : 0)) {
            q = carry;
            pv[R - 1] = Real(0);
            for (int s = 0; s < steps; ++s) {
                q = dpp_prev(q, pv[R - 1]);
                rows(q, divide);
            }
        }
#pragma unroll
        for (int r = 0; r < R; ++r)
            if (i0 + r < M) put(i0 + r, i0 + r == 0 ? Real(0) : mv[r], pv[r]);
        carry = dpp_ror(pv[R - 1]);
    }
    return bw0;
}

}  // namespace qz
