// The r-tridiagonal solves of the mode systems on a group of G lanes of a
// wavefront (64/G systems per wavefront), two right-hand sides per system.
//
// The lane at position p of a group owns rows [R p, R p + R).  Rows 0..R-2 are eliminated
// inside the lane from both ends towards the middle row (two independent
// chains of R/2 - 1 reciprocals instead of one of R - 1), with the two
// neighbouring interface unknowns kept symbolic; the interface rows R-1 of the
// G lanes are then solved by parallel cyclic reduction over the group.
//
// What bounds it: the VALU issue of binary64 operations and the latency of
// the chain.  One solve is about 230 binary64 operations per wavefront at
// R = 8, G = 32.  Two things keep the rest small:
//   - the interface rows travel scaled by their diagonal (4 values instead of
//     5 with the reciprocal beside them), and the last reduction step, where
//     every row has one partner only, exchanges 3 values once;
//   - no row is selected at a group's edge: the coefficient that would
//     multiply a row from outside the group is exactly zero there (AM of the
//     first row and CM of the last are zero, and every reduction step keeps
//     them so), and what it multiplies is another finite row.
#pragma once

#include <hip/hip_runtime.h>

#include "lanes.h"

namespace chy {

// 1/x to binary64 accuracy: the hardware estimate (28 bits) and one
// third-order step r (1 + e + e^2), e = 1 - x r.
__device__ __forceinline__ double rcp_full(double x)
{
    const double r = __builtin_amdgcn_rcp(x);
    const double e = __builtin_fma(-x, r, 1.0);
    return __builtin_fma(r, __builtin_fma(e, e, e), r);
}

// Where the lanes of a group stand along r.  Up to 16 lanes: in lane order,
// inside one row of 16 lanes.  32 and 64 lanes: row b of a group's 2 or 4
// rows holds the positions b modulo the number of rows, so that after one or
// two reduction steps the rows are independent systems and every later step
// is a DPP move within a row (no LDS crossbar: at 32 lanes its 54 accesses
// per solve kept the wavefronts waiting 40% of the time).
template <int G>
struct Group {
    static constexpr int ROWS = G <= 16 ? 1 : G / 16;
    static __device__ __forceinline__ int pos(int gl) { return ROWS == 1 ? gl : ROWS * (gl & 15) + (gl >> 4); }
    static __device__ __forceinline__ int lane(int p) { return ROWS == 1 ? p : (p % ROWS) * 16 + p / ROWS; }
};

// Values of the positions p - 1 (lo) and p + 1 (hi) of a group; any finite
// value past its ends.  at: the crossbar addresses of both (64 lanes).
struct Neigh {
    int lo, hi;
};

template <int G>
__device__ __forceinline__ Neigh neighbours(int lane)
{
    if constexpr (G < 64) {
        return Neigh{0, 0};
    } else {
        const int p = Group<64>::pos(lane);
        return Neigh{4 * Group<64>::lane((p + 63) & 63), 4 * Group<64>::lane((p + 1) & 63)};
    }
}

// Even and odd halves S lanes apart, position p of the even half between
// p - 1 and p of the odd one: each half's neighbours lie in the other, one of
// them at the same lane of the row.
template <int S>
__device__ __forceinline__ int half_lo(int v)
{
    int e, o;
    half_pair<S>(v, e, o);
    return __builtin_amdgcn_update_dpp(e, o, kDppRowShr + 1, S == 16 ? 0x5 : 0x3, 0xF, false);
}

template <int S>
__device__ __forceinline__ int half_hi(int v)
{
    int e, o;
    half_pair<S>(v, e, o);
    return __builtin_amdgcn_update_dpp(o, e, kDppRowShl + 1, S == 16 ? 0xA : 0xC, 0xF, false);
}

template <int G>
__device__ __forceinline__ double pos_prev(double x, Neigh at)
{
    if constexpr (G <= 16) return row_move<kDppRowShr + 1>(x);
    else if constexpr (G == 32) return by_word(x, [](int v) { return half_lo<16>(v); });
    else return by_word(x, [&](int v) { return crossbar_word(v, at.lo); });
}

template <int G>
__device__ __forceinline__ double pos_next(double x, Neigh at)
{
    if constexpr (G <= 16) return row_move<kDppRowShl + 1>(x);
    else if constexpr (G == 32) return by_word(x, [](int v) { return half_hi<16>(v); });
    else return by_word(x, [&](int v) { return crossbar_word(v, at.hi); });
}

// values S positions down and up
template <int S, int G>
__device__ __forceinline__ double step_lo(double x, Neigh at)
{
    if constexpr (S == 1) return pos_prev<G>(x, at);
    else if constexpr (G == 64 && S == 2) return by_word(x, [](int v) { return half_lo<32>(v); });
    else return row_move<kDppRowShr + S / Group<G>::ROWS>(x);
}

template <int S, int G>
__device__ __forceinline__ double step_hi(double x, Neigh at)
{
    if constexpr (S == 1) return pos_next<G>(x, at);
    else if constexpr (G == 64 && S == 2) return by_word(x, [](int v) { return half_hi<32>(v); });
    else return row_move<kDppRowShl + S / Group<G>::ROWS>(x);
}

// One row of the interface system, scaled to diagonal 1:
// al x_{i-s} + x_i + ga x_{i+s} = d
struct Iface {
    double al, ga, d0, d1;
};

// False when no row of the wavefront is coupled to another any more: a row's
// couplings (relative to its diagonal) square with every step, and below
// kUncoupled a partner changes nothing within binary64.  The larger a system's
// root, the sooner: on a grid alike in r and z the roots of a column need 2.9
// of the 5 steps of 32 lanes on average.
constexpr double kUncoupled = 1e-20;
__device__ __forceinline__ bool coupled(const Iface &r)
{
    return __any(fmax(fabs(r.al), fabs(r.ga)) > kUncoupled);
}

// The steps of distance S, 2S, .. < G/2; false once uncoupled.  A right-hand
// side with an infinity or NaN takes every step (all: found at the first
// check), so that it reaches every row of its system as the reference's
// sweeps carry it.
template <int S, int G>
__device__ __forceinline__ bool pcr_steps(Iface &r, Neigh at, bool all = false)
{
    if constexpr (S == 4) all = __any(!__builtin_isfinite(fabs(r.d0) + fabs(r.d1)));
    if constexpr (S >= 4)
        if (!all && !coupled(r)) return false;
    if constexpr (2 * S < G) {
        const double lal = step_lo<S, G>(r.al, at), lga = step_lo<S, G>(r.ga, at);
        const double ld0 = step_lo<S, G>(r.d0, at), ld1 = step_lo<S, G>(r.d1, at);
        const double hal = step_hi<S, G>(r.al, at), hga = step_hi<S, G>(r.ga, at);
        const double hd0 = step_hi<S, G>(r.d0, at), hd1 = step_hi<S, G>(r.d1, at);
        const double be = __builtin_fma(-r.ga, hal, __builtin_fma(-r.al, lga, 1.0));
        const double inv = rcp_full(be);
        const double t0 = __builtin_fma(-r.ga, hd0, __builtin_fma(-r.al, ld0, r.d0));
        const double t1 = __builtin_fma(-r.ga, hd1, __builtin_fma(-r.al, ld1, r.d1));
        r.al = -(r.al * lal) * inv;
        r.ga = -(r.ga * hga) * inv;
        r.d0 = t0 * inv;
        r.d1 = t1 * inv;
        return pcr_steps<2 * S, G>(r, at, all);
    }
    return true;
}

// LDS vectors of R*G values: element j = R p + r (position p) at
// r (G + 2) + lane(p), so that the lanes of a solve read consecutive words and
// 16 consecutive j (a matrix operand) fall in 16 different 8-byte banks
template <int R, int G>
struct Vec {
    static constexpr int PITCH = G + 2, SIZE = R * PITCH;
    static __device__ __forceinline__ int at(int j) { return (j % R) * PITCH + Group<G>::lane(j / R); }
};

// (T - rt) x = d in place in d0, d1.  tri: this lane's rows of T in LDS (Vec
// layout; sub-diagonal, diagonal, super-diagonal one after the other), rows
// past the system with zero off-diagonals, a large diagonal and d = 0 (their x
// is 0).  The rows are read here, where they are used, and not kept in
// registers: 48 registers less at R = 8 let a third wavefront run per SIMD.
template <int R, int G>
__device__ __forceinline__ void rtri_solve(const double *tri, double rt, Neigh at, double (&d0)[R], double (&d1)[R])
{
    static_assert(G >= 8, "group");
    typedef Vec<R, G> V;
    double ca[R], cb[R], cc[R];
#pragma unroll
    for (int r = 0; r < R; ++r) {
        ca[r] = tri[r * V::PITCH];
        cb[r] = tri[V::SIZE + r * V::PITCH];
        cc[r] = tri[2 * V::SIZE + r * V::PITCH];
    }
    constexpr int MID = R / 2 - 1, LAST = R - 2;
    // x_i = d_i + P_i XL + Q_i XR for i < R-1 (XL, XR: the last rows of the
    // previous lane and of this one); before the inner substitution Q_i of the
    // rows above the middle holds the factor of x_{i+1}, P_i below it that of x_{i-1}
    double P[R], Q[R];
    Iface f;
    double be = cb[R - 1] - rt;
    if constexpr (R == 1) {
        f.al = ca[0];
        f.ga = cc[0];
    } else {
#pragma unroll
        for (int i = 0; i < MID; ++i) {
            double den = cb[i] - rt;
            if (i > 0) den = __builtin_fma(-ca[i], Q[i - 1], den);
            const double inv = rcp_full(den), t = ca[i] * inv;
            d0[i] *= inv;
            d1[i] *= inv;
            if (i > 0) {
                d0[i] = __builtin_fma(-t, d0[i - 1], d0[i]);
                d1[i] = __builtin_fma(-t, d1[i - 1], d1[i]);
                P[i] = -t * P[i - 1];
            } else {
                P[0] = -t;
            }
            Q[i] = cc[i] * inv;
        }
#pragma unroll
        for (int i = LAST; i > MID; --i) {
            double den = cb[i] - rt;
            if (i < LAST) den = __builtin_fma(-cc[i], P[i + 1], den);
            const double inv = rcp_full(den), t = cc[i] * inv;
            d0[i] *= inv;
            d1[i] *= inv;
            if (i < LAST) {
                d0[i] = __builtin_fma(-t, d0[i + 1], d0[i]);
                d1[i] = __builtin_fma(-t, d1[i + 1], d1[i]);
                Q[i] = -t * Q[i + 1];
            } else {
                Q[LAST] = -t;
            }
            P[i] = ca[i] * inv;
        }
        {
            double den = cb[MID] - rt;
            if constexpr (MID > 0) den = __builtin_fma(-ca[MID], Q[MID - 1], den);
            if constexpr (MID < LAST) den = __builtin_fma(-cc[MID], P[MID + 1], den);
            const double inv = rcp_full(den), ta = ca[MID] * inv, tc = cc[MID] * inv;
            d0[MID] *= inv;
            d1[MID] *= inv;
            if constexpr (MID > 0) {
                d0[MID] = __builtin_fma(-ta, d0[MID - 1], d0[MID]);
                d1[MID] = __builtin_fma(-ta, d1[MID - 1], d1[MID]);
                P[MID] = -ta * P[MID - 1];
            } else {
                P[MID] = -ta;
            }
            if constexpr (MID < LAST) {
                d0[MID] = __builtin_fma(-tc, d0[MID + 1], d0[MID]);
                d1[MID] = __builtin_fma(-tc, d1[MID + 1], d1[MID]);
                Q[MID] = -tc * Q[MID + 1];
            } else {
                Q[MID] = -tc;
            }
        }
#pragma unroll
        for (int i = MID - 1; i >= 0; --i) {
            d0[i] = __builtin_fma(-Q[i], d0[i + 1], d0[i]);
            d1[i] = __builtin_fma(-Q[i], d1[i + 1], d1[i]);
            P[i] = __builtin_fma(-Q[i], P[i + 1], P[i]);
            Q[i] = -Q[i] * Q[i + 1];
        }
#pragma unroll
        for (int i = MID + 1; i <= LAST; ++i) {
            d0[i] = __builtin_fma(-P[i], d0[i - 1], d0[i]);
            d1[i] = __builtin_fma(-P[i], d1[i - 1], d1[i]);
            Q[i] = __builtin_fma(-P[i], Q[i - 1], Q[i]);
            P[i] = -P[i] * P[i - 1];
        }
        // interface row: the next lane's first row enters through its D, P, Q
        const double nP = pos_next<G>(P[0], at), nQ = pos_next<G>(Q[0], at);
        const double n0 = pos_next<G>(d0[0], at), n1 = pos_next<G>(d1[0], at);
        const double a = ca[R - 1], c = cc[R - 1];
        f.al = a * P[LAST];
        be = __builtin_fma(c, nP, __builtin_fma(a, Q[LAST], be));
        f.ga = c * nQ;
        d0[R - 1] = __builtin_fma(-c, n0, __builtin_fma(-a, d0[LAST], d0[R - 1]));
        d1[R - 1] = __builtin_fma(-c, n1, __builtin_fma(-a, d1[LAST], d1[R - 1]));
    }
    {
        const double inv = rcp_full(be);
        f.al *= inv;
        f.ga *= inv;
        f.d0 = d0[R - 1] * inv;
        f.d1 = d1[R - 1] * inv;
    }
    const bool more = pcr_steps<1, G>(f, at);
    d0[R - 1] = f.d0;
    d1[R - 1] = f.d1;
    if (more) {
        // last step: a row's one partner lies G/2 positions away (al is zero
        // in the lower half of the group, ga in the upper)
        constexpr int H = G < 16 ? G / 2 : 8;  // in lanes of a row
        const double c = f.al + f.ga;
        const double pc = row_swap<H>(c), p0 = row_swap<H>(f.d0), p1 = row_swap<H>(f.d1);
        const double inv = rcp_full(__builtin_fma(-c, pc, 1.0));
        d0[R - 1] = __builtin_fma(-c, p0, f.d0) * inv;
        d1[R - 1] = __builtin_fma(-c, p1, f.d1) * inv;
    }
    if constexpr (R > 1) {
        // XL: at a group's first position any finite value (its P is zero)
        const double xl0 = pos_prev<G>(d0[R - 1], at), xl1 = pos_prev<G>(d1[R - 1], at);
#pragma unroll
        for (int i = 0; i <= LAST; ++i) {
            d0[i] = __builtin_fma(P[i], xl0, __builtin_fma(Q[i], d0[R - 1], d0[i]));
            d1[i] = __builtin_fma(P[i], xl1, __builtin_fma(Q[i], d1[R - 1], d1[i]));
        }
    }
}

// The rows of T_m (am, cm, bm of the grid, padded to R G rows) into LDS for
// rtri_solve by a block of nt threads, rows >= M made inert.
constexpr double kInertDiag = 1e150;
template <int R, int G>
__device__ __forceinline__ void rtri_load(double *tri, const double *am, const double *cm, const double *bm, int M,
                                          int nt)
{
    typedef Vec<R, G> V;
    for (int j = threadIdx.x; j < R * G; j += nt) {
        tri[V::at(j)] = am[j];
        tri[V::SIZE + V::at(j)] = j < M ? bm[j] : kInertDiag;
        tri[2 * V::SIZE + V::at(j)] = cm[j];
    }
}

}  // namespace chy
