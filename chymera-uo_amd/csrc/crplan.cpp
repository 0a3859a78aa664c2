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
// That is for evenly spaced rows.  Where the spacing varies, the roots of small
// blocks miss the exact ones by more and leaves of 15 rows put the result 7e-13
// (cells growing by 3% a row, KMAX 32 and 128), 1e-12 (10%, 64) and 7e-11 (30%,
// 32) from BLKTRI's, leaves of 3 rows nowhere more than 5e-14 (64 rows along r;
// growths of -30% to 60% a row, random heights, KMAX 16..256): so 3 rows
// there (one solve at 256x128x256, cells growing by 1%: 404 us, with 15 rows
// 234, level by level 766).  Spacings that vary by up to 1%, from rounding to noise, stay within
// 5e-13 with 15 rows (KMAX 16..256).
#include <algorithm>
#include <array>
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
void pole_weights(int nd, const double *b, std::vector<long double> &f, Num num, double *out)
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
        out[p] = (double)v;
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

// A block's roots b_p and the weights of its three functions sum w_p / (t + b_p)
// of t, the negated eigenvalues of T (t >= 0): of the node's right-hand side
// and of the solved rows to its left and right (zero where there is none).
struct Poles {
    std::vector<double> b, w[3];
};

double dot(const double *x, const double *y, int n)
{
    double s[4] = {0.0, 0.0, 0.0, 0.0};  // four chains: an addition takes four cycles
    int i = 0;
    for (; i + 4 <= n; i += 4)
        for (int k = 0; k < 4; ++k) s[k] += x[i + k] * y[i + k];
    for (; i < n; ++i) s[0] += x[i] * y[i];
    return (s[0] + s[1]) + (s[2] + s[3]);
}

double dot(const std::vector<double> &x, const std::vector<double> &y)
{
    return dot(x.data(), y.data(), (int)x.size());
}

void add_to(std::vector<double> &x, double f, const std::vector<double> &y)
{
    for (size_t i = 0; i < x.size(); ++i) x[i] += f * y[i];
}

// Eigenvectors (rows of v, n x n) of the symmetric positive a (destroyed) by
// cyclic Jacobi rotations, to 10 digits.
void jacobi_eigenvectors(int n, std::vector<double> &a, std::vector<double> &v)
{
    v.assign((size_t)n * n, 0.0);
    for (int i = 0; i < n; ++i) v[(size_t)i * n + i] = 1.0;
    bool done = false;
    for (int sweep = 0; sweep < 30 && !done; ++sweep) {
        done = true;
        for (int i = 0; i < n - 1; ++i)
            for (int j = i + 1; j < n; ++j) {
                double *ri = &a[(size_t)i * n], *rj = &a[(size_t)j * n];
                const double x = ri[j], aii = ri[i], ajj = rj[j];
                if (!(x * x > 1e-20 * aii * ajj)) continue;
                done = false;
                const double th = (ajj - aii) / (2.0 * x);
                const double t = std::copysign(1.0 / (std::fabs(th) + std::sqrt(1.0 + th * th)), th);
                const double c = 1.0 / std::sqrt(1.0 + t * t), s = t * c;
                auto rotate = [&](double *p, double *q) {
                    for (int k = 0; k < n; ++k) {
                        const double u = p[k], w = q[k];
                        p[k] = c * u - s * w;
                        q[k] = s * u + c * w;
                    }
                };
                rotate(ri, rj);
                ri[i] = aii - t * x;
                rj[j] = ajj + t * x;
                ri[j] = rj[i] = 0.0;
                for (int k = 0; k < n; ++k) {
                    a[(size_t)k * n + i] = ri[k];
                    a[(size_t)k * n + j] = rj[k];
                }
                rotate(&v[(size_t)i * n], &v[(size_t)j * n]);
            }
    }
}

// Least squares for the weights of n roots on nt points: inv[i n + p] =
// 1 / (t_i + b_p), errors counted times scale[i].  The corrections are held small
// (kHold) where the points cannot tell roots apart.
struct WeightFit {
    int n, nt;
    const std::vector<double> &b;
    const std::vector<long double> &inv, &scale;
    std::vector<std::vector<double>> q, r;  // modified Gram-Schmidt; column p's rows below nt + p are zero

    double qdot(int p, const std::vector<double> &x) const { return dot(q[p].data(), x.data(), nt + p + 1); }
    void qsub(int p, double d, std::vector<double> &x) const
    {
        for (int i = 0; i <= nt + p; ++i) x[i] -= d * q[p][i];
    }
    WeightFit(const std::vector<double> &roots, int points, const std::vector<long double> &inverses,
              const std::vector<long double> &scales)
        : n((int)roots.size()), nt(points), b(roots), inv(inverses), scale(scales)
    {
        constexpr double kHold = 1e-11;
        q.assign(n, std::vector<double>(nt + n, 0.0));
        r.assign(n, std::vector<double>(n, 0.0));
        for (int p = 0; p < n; ++p) {
            for (int i = 0; i < nt; ++i) q[p][i] = (double)(scale[i] * b[p] * inv[(size_t)i * n + p]);
            q[p][nt + p] = kHold;
        }
        for (int p = 0; p < n; ++p) {
            r[p][p] = std::sqrt(qdot(p, q[p]));
            for (int i = 0; i <= nt + p; ++i) q[p][i] /= r[p][p];
            for (int k = p + 1; k < n; ++k) {
                r[p][k] = qdot(p, q[k]);
                qsub(p, r[p][k], q[k]);
            }
        }
    }
    // Weights w (a start on entry) so that sum w_p / (t + b_p) is f: three
    // corrections from errors in 80-bit arithmetic.  Returns the largest error left.
    double operator()(const std::vector<long double> &f, std::vector<double> &w) const
    {
        std::vector<double> e(nt + n), y(n);
        for (int round = 0;; ++round) {
            double worst = 0.0;
            std::fill(e.begin(), e.end(), 0.0);
            for (int i = 0; i < nt; ++i) {
                long double d = f[i];
                for (int p = 0; p < n; ++p) d -= w[p] * inv[(size_t)i * n + p];
                e[i] = (double)(d * scale[i]);
                worst = std::max(worst, std::fabs(e[i]));
            }
            if (round == 3) return worst;
            for (int p = 0; p < n; ++p) {
                y[p] = qdot(p, e);
                qsub(p, y[p], e);
            }
            for (int p = n - 1; p >= 0; --p) {
                for (int k = p + 1; k < n; ++k) y[p] -= r[p][k] * y[k];
                y[p] /= r[p][p];
                w[p] += y[p] * b[p];
            }
        }
    }
};

// The same three functions with fewer roots.  They are smooth: a block of nd
// rows has about 5 digits of t between its smallest and largest root, and a
// function sum g_p^2 / (t + b_p) is known to rounding from about one root per
// factor 1.6 of t in that range (two and a half with the functions of the
// separators).  The roots are those of the block's z matrix on the few vectors
// that the solutions (Z + t)^-1 (node, left, right) of all t span: with g, l,
// r the three in the eigenvectors (w = g g, g l, g r) their samples over t are
// orthogonalised, the largest first, until nothing above kNegligible is left;
// an error e of that space changes the functions by e^2.  The new weights fit
// the functions of the old roots, errors of BLKTRI's roots included, on
// points closer than the samples (at every second of them a fit through 40
// roots was off by up to 1e-12 in between).
// Accepted where every function is met to kSame (relative for the first one; of
// the separators' values for the others) or, where the roots of a symmetric
// block's odd eigenvectors, whose weights are the roots' errors, add more than
// that, to a thousandth of theirs, and where the weights have not grown (what
// their alternating signs cost in rounding).  False: nothing gained or not met.
bool fewer_roots(const Poles &in, Poles &out)
{
    constexpr double kNegligible = 5e-9, kSame = 1e-15;
    const int nd = (int)in.b.size();
    const double wmax = *std::max_element(in.w[0].begin(), in.w[0].end());
    const double bmin = *std::min_element(in.b.begin(), in.b.end());
    const double bmax = *std::max_element(in.b.begin(), in.b.end());
    if (!(bmin > 0.0) || !std::isfinite(bmax) || !(wmax > 0.0) || !std::isfinite(wmax)) return false;

    std::vector<double> s, v[3];
    double odd[3] = {0.0, 0.0, 0.0};
    for (int p = 0; p < nd; ++p) {
        const bool on = in.w[0][p] > 1e-20 * wmax;
        const double g = on ? std::sqrt(in.w[0][p]) : 0.0;
        if (on) s.push_back(in.b[p]);
        for (int c = 0; c < 3; ++c) {
            if (on) v[c].push_back(in.w[c][p] / g);
            else odd[c] += std::fabs(in.w[c][p]) / in.b[p];
        }
    }
    const int m = (int)s.size();

    std::vector<std::vector<double>> x{v[0]};  // the samples; t -> infinity
    auto sample = [&](double t) {
        double f0 = 0.0;
        for (int p = 0; p < m; ++p) f0 += v[0][p] * v[0][p] / (t + s[p]);
        for (int c = 0; c < 3; ++c) {
            const double sc = std::sqrt((t + bmin) * (c ? f0 : 1.0 / f0));
            std::vector<double> y(m);
            for (int p = 0; p < m; ++p) y[p] = sc * v[c][p] / (t + s[p]);
            if (dot(y, y) > 0.0) x.push_back(std::move(y));
        }
    };
    sample(0.0);
    for (double t = 0.25 * bmin; t < 4.0 * bmax; t *= 1.6) sample(t);

    std::vector<long double> t{0.0L};
    for (long double u = bmin / 64; u < 1e6L * bmax; u *= u < 16 * bmax ? 1.25L : 8.0L) t.push_back(u);
    std::vector<long double> f[3], scale(t.size(), 1.0L);
    for (int c = 0; c < 3; ++c) f[c].assign(t.size(), 0.0L);
    for (size_t i = 0; i < t.size(); ++i)
        for (int p = 0; p < nd; ++p) {
            const long double u = 1.0L / (t[i] + in.b[p]);
            for (int c = 0; c < 3; ++c)
                if (in.w[c][p] != 0.0) f[c][i] += in.w[c][p] * u;
        }
    std::vector<long double> relative(t.size());
    for (size_t i = 0; i < t.size(); ++i) relative[i] = 1.0L / f[0][i];

    std::vector<std::vector<double>> q;  // the orthonormal vectors
    std::vector<double> size;            // the samples' squared lengths outside them
    for (const auto &y : x) size.push_back(dot(y, y));
    double stop = 0.0;
    for (int attempt = 0; attempt < 4; ++attempt) {
        for (int added = 0;; ++added) {
            const size_t at = std::max_element(size.begin(), size.end()) - size.begin();
            const double most = size[at];
            if (q.empty()) stop = kNegligible * kNegligible * most;
            if ((int)q.size() == m || !(most > 0.0) || (attempt == 0 ? most <= stop : added == 2)) break;
            std::vector<double> y = x[at];
            for (int pass = 0; pass < 2; ++pass) {
                for (const auto &u : q) add_to(y, -dot(u, y), u);
                const double k = 1.0 / std::sqrt(dot(y, y));
                for (double &e : y) e *= k;
            }
            for (size_t i = 0; i < x.size(); ++i) {
                if (size[i] <= 1e-4 * stop) continue;
                add_to(x[i], -dot(y, x[i]), y);
                size[i] = dot(x[i], x[i]);
            }
            q.push_back(std::move(y));
        }
        const int n = (int)q.size();
        if (4 * n > 3 * nd) return false;
        std::vector<double> z((size_t)n * n), e;
        for (int i = 0; i < n; ++i) {
            std::vector<double> sq(m);
            for (int p = 0; p < m; ++p) sq[p] = s[p] * q[i][p];
            for (int j = 0; j <= i; ++j) z[(size_t)i * n + j] = z[(size_t)j * n + i] = dot(sq, q[j]);
        }
        jacobi_eigenvectors(n, z, e);
        // a root from its vector's quotient, whose error is the vector's squared
        out.b.assign(n, 0.0);
        for (int c = 0; c < 3; ++c) out.w[c].assign(n, 0.0);
        for (int i = 0; i < n; ++i) {
            std::vector<double> y(m, 0.0);
            for (int k = 0; k < n; ++k) add_to(y, e[(size_t)i * n + k], q[k]);
            long double yy = 0.0L, ys = 0.0L;
            for (int p = 0; p < m; ++p) {
                yy += (long double)y[p] * y[p];
                ys += (long double)y[p] * y[p] * s[p];
            }
            out.b[i] = (double)(ys / yy);
            for (int c = 0; c < 3; ++c) out.w[c][i] = dot(y, v[0]) * dot(y, v[c]);
        }
        const int nt = (int)t.size();
        std::vector<long double> inv((size_t)nt * n);
        for (int i = 0; i < nt; ++i)
            for (int p = 0; p < n; ++p) inv[(size_t)i * n + p] = 1.0L / (t[i] + out.b[p]);
        const WeightFit fit0(out.b, nt, inv, relative), fit1(out.b, nt, inv, scale);
        bool same = true;
        for (int c = 0; c < 3 && same; ++c) {
            if (f[c][0] == 0.0L) continue;
            same = (c ? fit1 : fit0)(f[c], out.w[c]) <= std::max(kSame, 1e-3 * odd[c]);
            double sum = 0.0, had = 0.0;
            for (int p = 0; p < n; ++p) sum += std::fabs(out.w[c][p]) / out.b[p];
            for (int p = 0; p < nd; ++p) had += std::fabs(in.w[c][p]) / in.b[p];
            same = same && sum <= 1.5 * had;
        }
        if (same) return true;
    }
    return false;
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
    // the lowest nodes' level: leaves of 2^lv0 - 1 rows, up to 15 on columns spaced
    // evenly (to 1%: couplings within 4%), up to 3 on others (see above)
    double least = cn[0], greatest = cn[0];
    for (int i = 1; i < n; ++i) {
        least = std::min({least, an[i], i + 1 < n ? cn[i] : an[i]});
        greatest = std::max({greatest, an[i], i + 1 < n ? cn[i] : an[i]});
    }
    plan.even = greatest <= 1.04 * least;
    const int lv0 = std::min(kx - 1, plan.even ? 4 : 2);
    const double machep = cr_machep();
    std::vector<std::vector<double>> lev(kx);
    lev[0].resize(n);
    for (int i = 0; i < n; ++i) lev[0][i] = -bn[i];
    for (int lv = std::max(1, lv0 - 1); lv < kx; ++lv) {
        const int step = 1 << lv, size = 2 * step - 1, nblk = (1 << (kx - lv)) - 1;
        lev[lv].resize((size_t)size * nblk);
        std::vector<double> d(size), e2(size);
        for (int b = 0; b < nblk; b += 2) {  // the others lie across the tree's blocks
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
    std::vector<CrPhase> levels(kx);
    std::vector<long double> factors(n + 1);
    plan.node.clear();
    for (int lv = lv0; lv < kx; ++lv) {
        const int h = 1 << lv, nd = 2 * h - 1, nnode = (n + 1) / (2 * h);
        std::vector<Poles> level(nnode);
        // the weights of the messages to the right and left over those of the rows there
        std::vector<std::array<double, 2>> message(nnode, {0.0, 0.0});
        int most = 0;
        for (int t = 0; t < nnode; ++t) {
            const int i = (2 * t + 1) * h;  // 1-based row
            const double *b = block(lv, 2 * t), *l = block(lv - 1, 4 * t), *r = block(lv - 1, 4 * t + 2);
            Poles full;
            full.b.assign(b, b + nd);
            for (auto &w : full.w) w.assign(nd, 0.0);
            // half: a half block's roots; c: h couplings, c[0] the first (1-based row first)
            auto weights = [&](std::vector<double> &out, const double *half, const double *half2, const double *c,
                               int first) {
                pole_weights(nd, b, factors, [&](int p, long double *f) {
                    const long double bp = b[p];
                    int nf = 0;
                    for (int j = 0; j < h - 1; ++j) {
                        f[nf++] = bp - (long double)half[j];
                        f[nf++] = half2 ? bp - (long double)half2[j] : (long double)c[first - 1 + j];
                    }
                    if (!half2) f[nf++] = c[first - 1 + h - 1];
                    return nf;
                }, out.data());
            };
            weights(full.w[0], l, r, nullptr, 0);
            if (i - h >= 1) weights(full.w[1], r, nullptr, an, i - h + 1);
            if (i + h <= n) weights(full.w[2], l, nullptr, cn, i);
            long double right = 1.0L, left = 1.0L;
            for (int j = 0; j < h; ++j) {
                if (i + h <= n) right *= (long double)an[i + j] / (long double)cn[i - 1 + j];
                if (i - h >= 1) left *= (long double)cn[i - h - 1 + j] / (long double)an[i - h + j];
            }
            message[t] = {(double)right, (double)left};
            if (!fewer_roots(full, level[t])) level[t] = std::move(full);
            most = std::max(most, (int)level[t].b.size());
            plan.nsolve += (long)level[t].b.size() * (lv < kx - 1 ? 2 : 1);
        }
        const int np = (most + kNodePad - 1) / kNodePad * kNodePad;
        const size_t rec0 = plan.node.size() / kNodeRec;
        levels[lv] = CrPhase{0, h, nnode, (int)rec0, np};
        plan.node.resize((rec0 + (size_t)nnode * (1 + np)) * kNodeRec, 0.0);
        for (int t = 0; t < nnode; ++t) {
            const Poles &f = level[t];
            const int nf = (int)f.b.size();
            double *rec = &plan.node[(rec0 + (size_t)t * (1 + np)) * kNodeRec];
            rec[0] = nf;
            for (int p = 0; p < np; ++p) {
                rec += kNodeRec;
                rec[0] = f.b[std::min(p, nf - 1)];
                if (p >= nf) continue;
                rec[1] = f.w[2][p] * message[t][0];
                rec[2] = f.w[1][p] * message[t][1];
                for (int c = 0; c < 3; ++c) rec[3 + c] = f.w[c][p];
            }
        }
    }
    auto nodes = [&](int kind, int lv) {
        plan.phases.push_back(levels[lv]);
        plan.phases.back().kind = kind;
    };
    plan.phases.push_back(CrPhase{CR_LEAF_UP, 0, 0, 0, 0});
    for (int lv = lv0; lv < kx - 1; ++lv) nodes(CR_NODE_UP, lv);
    for (int lv = kx - 1; lv >= lv0; --lv) nodes(CR_NODE_DOWN, lv);
    plan.phases.push_back(CrPhase{CR_LEAF_DOWN, 0, 0, 0, 0});
    return CHY_OK;
}

}  // namespace chy
