// Host-side plan of the per-mode cyclic reduction (pot/blktri.f): the root
// tables BLKTRI's initialisation computes (COMPB, pot/blktri.f:264-344, with
// the eigenvalues of TQLRAT, :348-423) and the weights with which the
// reduction's products (PRDCT, :177-260) become sums of independent r solves.
//
// The z rows form a tree.  Row i = odd * h has a block of the 2h - 1 rows
// i-h+1 .. i+h-1; with P(a..b) = det(T + Z(a..b)) = prod (T - root) over the
// block's roots (negated eigenvalues of the z sub-matrix), l and r the roots
// of the block's halves (rows before and after i) and b_p those of the block,
// the block's Green's function gives
//   from (i, i):      P(l) P(r) / P                        = sum a_p  / (T - b_p)
//   to the row i + h: (-1)^h prod AN(i+1 .. i+h) P(l) / P  = sum wR_p / (T - b_p)
//   to the row i - h: (-1)^h prod CN(i-h .. i-1) P(r) / P  = sum wL_p / (T - b_p)
//   from X(i - h):    (-1)^h prod AN(i-h+1 .. i) P(r) / P  = sum cL_p / (T - b_p)
//   from X(i + h):    (-1)^h prod CN(i .. i+h-1) P(l) / P  = sum cR_p / (T - b_p)
// which are BLKTRI's products with its root tables in each P: its chains
// divide by the half blocks' roots that the product before them multiplied by.
// Every weight is formed in long double, numerator and denominator factors in
// pairs so that no partial product overflows.
//
// The roots are formed with the reference's own arithmetic and convergence
// rule.  That matters for parity: the reference's FP64 result differs from the
// exact solution of the discrete system by up to a few 1e-12 (256x128x256),
// and that difference comes from these root values, not from the rounding of
// the r solves (any elimination order with the same roots reproduces it to
// ~1e-14).  It comes from the large blocks, whose smallest roots lie furthest
// below the convergence rule's scale.  Blocks of up to 31 rows can be solved
// at once, with their exact eigenvectors and BLKTRI's roots, and stay within
// 7e-14 of the reference's result; at 63 rows the roots' errors no longer fit
// those of the blocks inside and around them (4e-12; KMAX = 32..512).  The
// leaves have at most 15 rows (cr.hip), and fewer than half of the column:
// solved as one leaf, a whole column on a grid much finer in r than in z
// (512x16) lands 9e-13 away, with one node above the leaves 1.5e-13.
#include <algorithm>
#include <cmath>
#include <numeric>
#include <vector>

#include "chypot_impl.h"

namespace chy {

namespace {

// 100 x the first power of ten below binary64 resolution, formed by repeated
// division as pot/blktri.f:271-277 forms its EPSLON.
double cr_machep()
{
    volatile double e = 1.0, one_plus;
    do {
        e = e / 10.0;
        one_plus = 1.0 + e;
    } while (one_plus > 1.0);
    return 100.0 * e;
}

// Eigenvalues of the symmetric tridiagonal with diagonal d[0..n-1] and
// squared couplings e2[0..n-2] (e2[i] couples rows i and i+1): Reinsch's
// rational QL iteration (EISPACK TQLRAT), with the convergence test and
// ordering of pot/blktri.f:348-423: the result is sorted by increasing
// magnitude.  Returns 0, or the 1-based row that failed to converge.
int rational_ql(int n, double *d, double *e2, double machep)
{
    if (n == 1) return 0;
    e2[n - 1] = 0.0;
    double f = 0.0, b = 0.0, c = 0.0;
    for (int l = 0; l < n; ++l) {
        double h = machep * (std::fabs(d[l]) + std::sqrt(e2[l]));
        if (!(b > h)) {
            b = h;
            c = b * b;
        }
        int m = l;
        while (!(e2[m] <= c)) ++m;
        if (m != l) {
            for (int it = 0;; ++it) {
                if (it == 30) return l + 1;
                double s = std::sqrt(e2[l]), g = d[l];
                double p = (d[l + 1] - g) / (2.0 * s);
                double r = std::sqrt(p * p + 1.0);
                d[l] = s / (p + std::copysign(r, p));
                h = g - d[l];
                for (int i = l + 1; i < n; ++i) d[i] = d[i] - h;
                f = f + h;
                g = d[m];
                if (g == 0.0) g = b;
                h = g;
                s = 0.0;
                for (int i = m - 1; i >= l; --i) {
                    p = g * h;
                    r = p + e2[i];
                    e2[i + 1] = s * r;
                    s = e2[i] / r;
                    d[i + 1] = h + s * (h + d[i]);
                    g = d[i] - e2[i] / g;
                    if (g == 0.0) g = b;
                    h = g * p / r;
                }
                e2[l] = s * g;
                d[l] = h;
                if (h == 0.0) break;
                if (std::fabs(e2[l]) <= std::fabs(c / h)) break;
                e2[l] = h * e2[l];
                if (e2[l] == 0.0) break;
            }
        }
        double p = d[l] + f;
        int i = l;
        while (i > 0 && !(std::fabs(p) >= std::fabs(d[i - 1]))) {
            d[i] = d[i - 1];
            --i;
        }
        d[i] = p;
    }
    return 0;
}

// out_p = prod(num(p, f)) / prod_{k != p} (b_p - b_k): num fills f with the
// numerator's factors and returns their number; they are paired with the
// denominator's
template <typename Num>
void pole_weights(int nd, const double *b, std::vector<long double> &f, Num num, double *out, size_t stride)
{
    for (int p = 0; p < nd; ++p) {
        const int nf = num(p, f.data());
        const long double bp = b[p];
        long double v = 1.0L;
        int k = 0;
        for (int i = 0; i < nf; ++i, ++k) {
            if (k == p) ++k;
            v *= k < nd ? f[i] / (bp - (long double)b[k]) : f[i];
        }
        for (; k < nd; ++k)
            if (k != p) v /= bp - (long double)b[k];
        out[(size_t)p * stride] = (double)v;
    }
}

// the tables of the leaf whose first row is r0 (0-based): the block's
// eigenvectors in 80-bit arithmetic, rounded once, each with BLKTRI's root
int leaf_table(double *t, int r0, int rows, int n, const double *an, const double *bn, const double *cn,
               const double *roots)
{
    std::vector<long double> d(rows), e(rows + 1, 0.0L), q, sc(rows, 1.0L);
    for (int k = 0; k < rows; ++k) {
        d[k] = bn[r0 + k];
        if (k == 0) continue;
        sc[k] = sc[k - 1] * std::sqrt((long double)cn[r0 + k - 1] / (long double)an[r0 + k]);
        e[k] = std::sqrt((long double)an[r0 + k] * (long double)cn[r0 + k - 1]);
    }
    const int rc = symmetric_tridiag_eigen(rows, d, e, q);
    if (rc != CHY_OK) return rc;
    // eigenvector order[p] belongs to the p-th root by value
    std::vector<int> order(rows);
    std::iota(order.begin(), order.end(), 0);
    std::sort(order.begin(), order.end(), [&](int a, int b) { return -d[a] < -d[b]; });
    std::vector<double> rt(roots, roots + rows);
    std::sort(rt.begin(), rt.end());
    const bool left = r0 > 0, right = r0 + rows < n;
    for (int p = 0; p < rows; ++p) {
        auto u = [&](int k) { return sc[k] * q[(size_t)k * rows + order[p]]; };
        auto v = [&](int k) { return q[(size_t)k * rows + order[p]] / sc[k]; };
        for (int k = 0; k < rows; ++k) {
            t[kLeafU + p * (kLeafSpan + 4) + k] = (double)u(k);
            t[kLeafV + k * kLeafSpan + p] = (double)v(k);
        }
        if (left) {
            t[kLeafU + p * (kLeafSpan + 4) + kLeafSpan] = (double)(-(long double)an[r0] * u(0));
            t[kLeafLeft + p] = (double)(-(long double)cn[r0 - 1] * v(0));
        }
        if (right) {
            t[kLeafU + p * (kLeafSpan + 4) + kLeafSpan + 1] = (double)(-(long double)cn[r0 + rows - 1] * u(rows - 1));
            t[kLeafRight + p] = (double)(-(long double)an[r0 + rows] * v(rows - 1));
        }
        t[kLeafRoot + p] = rt[p];
    }
    for (int p = rows; p < kLeafSpan; ++p) t[kLeafRoot + p] = rt[rows - 1];
    return CHY_OK;
}

}  // namespace

int build_cr_plan(CrPlan &plan, int n, const double *an, const double *bn, const double *cn)
{
    int kx = 0;
    while ((1 << kx) - 1 < n) ++kx;
    if ((1 << kx) - 1 != n || kx < 2) return CHY_EUNSUPPORTED;
    // squared symmetrised couplings, formed as the reference forms them:
    // the square of sqrt(AN(i) CN(i-1)) (pot/blktri.f:283-293, :360-362)
    std::vector<double> cpl2(n, 0.0);
    for (int i = 1; i < n; ++i) {
        double arg = an[i] * cn[i - 1];
        if (arg < 0.0) return CHY_ENUMERIC;
        double e = std::sqrt(arg);
        cpl2[i] = e * e;
    }
    // lev[lv][b * (2^(lv+1)-1) + i]: roots of block b of level lv (rows
    // 1 + b 2^lv .. b 2^lv + 2^(lv+1) - 1), negated eigenvalues of the z
    // sub-tridiagonal, by increasing magnitude
    const double machep = cr_machep();
    std::vector<std::vector<double>> lev(kx);
    lev[0].resize(n);
    for (int i = 0; i < n; ++i) lev[0][i] = -bn[i];
    for (int lv = 1; lv < kx; ++lv) {
        const int step = 1 << lv, size = 2 * step - 1, nblk = (1 << (kx - lv)) - 1;
        lev[lv].resize((size_t)size * nblk);
        std::vector<double> d(size), e2(size);
        for (int b = 0; b < nblk; ++b) {
            const int r0 = b * step;
            for (int i = 0; i < size; ++i) d[i] = bn[r0 + i];
            for (int i = 0; i + 1 < size; ++i) e2[i] = cpl2[r0 + i + 1];
            if (rational_ql(size, d.data(), e2.data(), machep) != 0) return CHY_ENUMERIC;
            for (int i = 0; i < size; ++i) lev[lv][(size_t)b * size + i] = -d[i];
        }
    }
    auto block = [&](int lv, int b) { return lev[lv].data() + (size_t)b * ((2 << lv) - 1); };

    plan.kx = kx;
    plan.phases.clear();
    const int lv0 = std::min(kx - 1, 4);  // the lowest nodes' level: leaves of 2^lv0 - 1 rows
    plan.rows = (1 << lv0) - 1;
    plan.nleaf = (n + 1) >> lv0;
    plan.leaf.assign((size_t)plan.nleaf * kLeafStride, 0.0);
    for (int b = 0; b < plan.nleaf; ++b) {
        const int rc = leaf_table(&plan.leaf[(size_t)b * kLeafStride], b << lv0, plan.rows, n, an, bn, cn,
                                  block(lv0 - 1, 2 * b));
        if (rc != CHY_OK) return rc;
    }
    plan.nsolve = 2L * plan.nleaf * plan.rows;
    // the nodes' records, level by level (h = 2^lv is even, so (-1)^h = 1)
    std::vector<int> rec0(kx, 0);
    std::vector<long double> factors(n + 1);
    plan.node.clear();
    for (int lv = lv0; lv < kx; ++lv) {
        const int h = 1 << lv, nd = 2 * h - 1, nnode = (n + 1) / (2 * h), np = node_roots(h);
        rec0[lv] = (int)(plan.node.size() / kNodeRec);
        plan.node.resize(plan.node.size() + (size_t)nnode * np * kNodeRec, 0.0);
        for (int t = 0; t < nnode; ++t) {
            const int i = (2 * t + 1) * h;  // 1-based row
            const double *b = block(lv, 2 * t), *l = block(lv - 1, 4 * t), *r = block(lv - 1, 4 * t + 2);
            double *rec = &plan.node[((size_t)rec0[lv] + (size_t)t * np) * kNodeRec];
            for (int p = 0; p < np; ++p) rec[p * kNodeRec] = b[std::min(p, nd - 1)];
            // half: a half block's roots; c: h couplings, c[0] the first (1-based row first)
            auto weights = [&](int slot, const double *half, const double *half2, const double *c, int first) {
                pole_weights(nd, b, factors, [&](int p, long double *f) {
                    const long double bp = b[p];
                    int nf = 0;
                    for (int j = 0; j < h - 1; ++j) {
                        f[nf++] = bp - (long double)half[j];
                        f[nf++] = half2 ? bp - (long double)half2[j] : (long double)c[first - 1 + j];
                    }
                    if (!half2) f[nf++] = c[first - 1 + h - 1];
                    return nf;
                }, rec + slot, kNodeRec);
            };
            weights(3, l, r, nullptr, 0);
            if (i + h <= n) {
                weights(1, l, nullptr, an, i + 1);
                weights(5, l, nullptr, cn, i);
            }
            if (i - h >= 1) {
                weights(2, r, nullptr, cn, i - h);
                weights(4, r, nullptr, an, i - h + 1);
            }
        }
        plan.nsolve += (long)nnode * nd * (lv < kx - 1 ? 2 : 1);
    }
    auto nodes = [&](int kind, int lv) {
        plan.phases.push_back(CrPhase{kind, 1 << lv, (n + 1) / (2 << lv), rec0[lv]});
    };
    plan.phases.push_back(CrPhase{CR_LEAF_UP, 0, 0, 0});
    for (int lv = lv0; lv < kx - 1; ++lv) nodes(CR_NODE_UP, lv);
    for (int lv = kx - 1; lv >= lv0; --lv) nodes(CR_NODE_DOWN, lv);
    plan.phases.push_back(CrPhase{CR_LEAF_DOWN, 0, 0, 0});
    return CHY_OK;
}

}  // namespace chy
