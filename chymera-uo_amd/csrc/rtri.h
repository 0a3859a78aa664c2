// The r-tridiagonal solves of the mode systems on a group of G lanes of a
// wavefront (64/G systems per wavefront), two right-hand sides per system.
//
// Lane gl of a group owns rows [R gl, R gl + R).  Rows 0..R-2 are eliminated
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

// x of lane i - S / i + S of a group of G lanes (any finite value past the
// group's edges): DPP moves where the group lies in a row of 16 lanes, the
// LDS crossbar otherwise; distance 1 by DPP for every group
template <int S, int G>
__device__ __forceinline__ double lane_lo(double x, int lane4)
{
    if constexpr (S == 1) {
        return lane_prev(x);
    } else if constexpr (G <= 16) {
        return dpp_move<kDppRowShr + S>(x);
    } else {
        return crossbar(x, lane4 - 4 * S);
    }
}

template <int S, int G>
__device__ __forceinline__ double lane_hi(double x, int lane4)
{
    if constexpr (S == 1) {
        return lane_next(x);
    } else if constexpr (G <= 16) {
        return dpp_move<kDppRowShl + S>(x);
    } else {
        return crossbar(x, lane4 + 4 * S);
    }
}

// One row of the interface system, scaled to diagonal 1:
// al x_{i-s} + x_i + ga x_{i+s} = d
struct Iface {
    double al, ga, d0, d1;
};

template <int S, int G>
__device__ __forceinline__ void pcr_steps(Iface &r, int lane4)
{
    if constexpr (2 * S < G) {
        const double lal = lane_lo<S, G>(r.al, lane4), lga = lane_lo<S, G>(r.ga, lane4);
        const double ld0 = lane_lo<S, G>(r.d0, lane4), ld1 = lane_lo<S, G>(r.d1, lane4);
        const double hal = lane_hi<S, G>(r.al, lane4), hga = lane_hi<S, G>(r.ga, lane4);
        const double hd0 = lane_hi<S, G>(r.d0, lane4), hd1 = lane_hi<S, G>(r.d1, lane4);
        const double be = __builtin_fma(-r.ga, hal, __builtin_fma(-r.al, lga, 1.0));
        const double inv = rcp_full(be);
        const double t0 = __builtin_fma(-r.ga, hd0, __builtin_fma(-r.al, ld0, r.d0));
        const double t1 = __builtin_fma(-r.ga, hd1, __builtin_fma(-r.al, ld1, r.d1));
        r.al = -(r.al * lal) * inv;
        r.ga = -(r.ga * hga) * inv;
        r.d0 = t0 * inv;
        r.d1 = t1 * inv;
        pcr_steps<2 * S, G>(r, lane4);
    }
}

// (T - rt) x = d in place in d0, d1.  ca, cb, cc: the lane's rows of T (sub,
// diagonal, super), rows past the system with ca = cc = 0, a large cb and
// d = 0 (their x is 0); lane4: 4 * lane (byte address in the crossbar).
template <int R, int G>
__device__ __forceinline__ void rtri_solve(const double (&ca)[R], const double (&cb)[R], const double (&cc)[R],
                                           double rt, int lane4, double (&d0)[R], double (&d1)[R])
{
    static_assert(G >= 2, "group");
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
        const double nP = lane_next(P[0]), nQ = lane_next(Q[0]);
        const double n0 = lane_next(d0[0]), n1 = lane_next(d1[0]);
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
    pcr_steps<1, G>(f, lane4);
    // last step: a row's one partner lies G/2 lanes away (al is zero in the
    // lower half of the group, ga in the upper)
    {
        const double c = f.al + f.ga;
        const double pc = lane_swap<G / 2>(c, lane4), p0 = lane_swap<G / 2>(f.d0, lane4);
        const double p1 = lane_swap<G / 2>(f.d1, lane4);
        const double inv = rcp_full(__builtin_fma(-c, pc, 1.0));
        d0[R - 1] = __builtin_fma(-c, p0, f.d0) * inv;
        d1[R - 1] = __builtin_fma(-c, p1, f.d1) * inv;
    }
    if constexpr (R > 1) {
        // XL: for a group's first lane any finite value (its P is zero)
        const double xl0 = lane_prev(d0[R - 1]), xl1 = lane_prev(d1[R - 1]);
#pragma unroll
        for (int i = 0; i <= LAST; ++i) {
            d0[i] = __builtin_fma(P[i], xl0, __builtin_fma(Q[i], d0[R - 1], d0[i]));
            d1[i] = __builtin_fma(P[i], xl1, __builtin_fma(Q[i], d1[R - 1], d1[i]));
        }
    }
}

// The rows of T_m one lane owns (am, cm, bm of the grid, padded to whole
// groups), rows >= M made inert.
constexpr double kInertDiag = 1e150;
template <int R>
__device__ __forceinline__ void rtri_rows(const double *am, const double *cm, const double *bm, int f, int M,
                                          double (&ca)[R], double (&cb)[R], double (&cc)[R])
{
#pragma unroll
    for (int r = 0; r < R; ++r) {
        ca[r] = am[f + r];
        cc[r] = cm[f + r];
        cb[r] = f + r < M ? bm[f + r] : kInertDiag;
    }
}

}  // namespace chy
