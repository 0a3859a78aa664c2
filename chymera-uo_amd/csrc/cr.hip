// Per-mode solves on the GPU with BLKTRI's root tables: the systems POT3 hands
// to BLKTRI for every azimuthal mode (pot/blktri.f:60-260, called at
// pot/pot3.f:233-239).
//
// A mode's unknowns are X(j, i): j = 1..M along r (JMAX-1 rows), i = 1..N
// along z (KMAX-1 = 2^k - 1 rows).  BLKTRI eliminates the rows level by level,
// applying products of r-tridiagonal solves (T_m - rt)^-1.  The same
// elimination is a tree here (crplan.cpp): leaves of 15 z rows, then one node
// per row i = odd * h, h = 16, 32, .., whose block of 2h - 1 rows has its
// roots in BLKTRI's table.  Up the tree every block sends what its right-hand
// side adds to the two rows beside it; down the tree every block is solved
// from its own right-hand side and the solved rows beside it.  BLKTRI's
// product of a block (all its roots below the line, the roots of its halves
// above) and the chain that follows it (the roots of one half below the line)
// cancel root by root, so each message and each solution is one sum of
// independent solves with the block's own roots:
//   up    Y(i +- h) += sum_p b_p (T - r_p)^-1 Y(i)
//   down  X(i)       = sum_p (T - r_p)^-1 (a_p Y(i) + cL_p X(i-h) + cR_p X(i+h))
// and no intermediate vectors, chains or extra launches remain: 867 r solves
// per mode in 7 launches at KMAX = 128, where level by level it is 2215 in 19
// (11.0 ms per 32 fields at 256x128x256).  The weights alternate in sign; the
// terms stay as small as the block's own Green's function, so the sums round
// as one more elimination order does (1-2e-14 from BLKTRI's result at KMAX up
// to 512 on grids alike in r and z, 3-5e-14 with the leaves, whose rows are
// solved together in their eigenvectors).
//
// One block of a launch is one tree node (or leaf) of one order m: the cosine
// and sine parts share T_m, so every solve has two right-hand sides; solves
// run on groups of G lanes (rtri.h), 64/G roots per wavefront at a time.  The
// leaves' changes of basis (16 roots x 15..17 rows) run on the FP64 matrix
// cores through LDS.  The spectrum spec[q][k][j] (J contiguous) is the mode
// right-hand side on entry (with POT3's boundary terms applied) and the mode
// solution on exit.  What a block adds to the row on its left goes to the
// grid's second workspace buffer (yh), what it adds to the row on its right
// into the spectrum itself, so every row has one writer per launch and the
// order of every sum is fixed.
#include <hip/hip_runtime.h>

#include "chypot_impl.h"
#include "rtri.h"

namespace chy {

namespace {

struct CrArgs {
    const double *am, *cm, *bm;  // r operator: [JP], [JP], [(N+1)][JP]
    const double *leaf;          // leaf tables (kLeafStride doubles each)
    const double *node;          // node tables (kNodeRec doubles per root)
    int J, K, M, N, PP, JP;
    int nleaf, rows;             // leaves, rows per leaf
};

typedef double dx4 __attribute__((ext_vector_type(4)));

// the order and field of a block, its two modes' planes
template <int R, int G>
struct Plane {
    double *sc, *ss, *pc, *ps;  // spectrum and second-buffer planes of the cosine and sine parts
    bool two;
    __device__ Plane(const CrArgs &a, const Fields &F, int m)
    {
        double *spec = static_cast<double *>(F.spec[blockIdx.y]);
        double *pv = static_cast<double *>(F.yh[blockIdx.y]);
        two = m >= 1 && m <= a.N - 1;
        const size_t qc = (size_t)m, qs = two ? (size_t)(a.N + m) : qc;
        sc = spec + qc * a.K * a.J;
        ss = spec + qs * a.K * a.J;
        pc = pv + qc * a.PP * a.JP;
        ps = pv + qs * a.PP * a.JP;
    }
};

// LDS vectors of R*G values: element j = R g + r at r (G + 2) + g, so that
// the lanes of a solve read consecutive words and 16 consecutive j (a matrix
// operand) fall in 16 different 8-byte banks
template <int R, int G>
struct Vec {
    static constexpr int PITCH = G + 2, SIZE = R * PITCH;
    static __device__ __forceinline__ int at(int j) { return (j % R) * PITCH + j / R; }
};

// The two sums (to the right neighbour, to the left one) of a block's W
// wavefronts, each lane holding its part for its root's group: added over the
// wavefront's groups, then over the wavefronts in order, and handed to
// out(sum, part, j, value) for j < M.
template <int R, int G, int W, int NSUM, typename Out>
__device__ __forceinline__ void block_sums(double (&s)[NSUM][2][R], double *lds, int M, Out out)
{
    typedef Vec<R, G> V;
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6, gl = lane % G;
    const int lane4 = 4 * lane;
#pragma unroll
    for (int n = 0; n < NSUM; ++n)
#pragma unroll
        for (int h = 0; h < 2; ++h)
#pragma unroll
            for (int r = 0; r < R; ++r) {
                if constexpr (G <= 8) s[n][h][r] += lane_swap<8>(s[n][h][r], lane4);
                if constexpr (G <= 16) s[n][h][r] += lane_swap<16>(s[n][h][r], lane4);
                if constexpr (G <= 32) s[n][h][r] += lane_swap<32>(s[n][h][r], lane4);
            }
    __syncthreads();  // every wavefront is done with what lds held
    if (lane < G) {
#pragma unroll
        for (int n = 0; n < NSUM; ++n)
#pragma unroll
            for (int h = 0; h < 2; ++h)
#pragma unroll
                for (int r = 0; r < R; ++r)
                    lds[((wave * NSUM + n) * 2 + h) * V::SIZE + r * V::PITCH + gl] = s[n][h][r];
    }
    __syncthreads();
    for (int e = threadIdx.x; e < NSUM * 2 * R * G; e += 64 * W) {
        const int j = e % (R * G), nh = e / (R * G);
        double v = lds[nh * V::SIZE + V::at(j)];
#pragma unroll
        for (int w = 1; w < W; ++w) v += lds[(w * NSUM * 2 + nh) * V::SIZE + V::at(j)];
        if (j < M) out(nh / 2, nh % 2, j, v);
    }
}

// A leaf: rows i0 .. i0 + rows - 1 (0-based, i0 = (rows + 1) b), the separating rows
// i0 - 1 and i0 + rows beside it.  Up: the leaf's messages to the separators.
// Down: its rows from the solved separators.  16 roots (zero-padded).
//   gather   D[p][j] = sum_k U[p][k] Y[k][j]   (down: k = 16, 17 the separators)
//   solves   one root per group of lanes
//   scatter  X[k][j] = sum_p V[k][p] D[p][j]   (down)
// V_MFMA_F64_16X16X4F64: A lane l holds A[l%16][l/16], B lane l B[l/16][l%16],
// the result D[l/16 + 4v][l%16].  LDS holds the 16 x 2 vectors: 70 KB at
// JMAX <= 256 (two blocks per CU), 135 KB at 512.
template <int R, int G, int W, bool DOWN>
__global__ __launch_bounds__(64 * W, 2) void k_cr_leaf(CrArgs a, const Fields F)
{
    typedef Vec<R, G> V;
    constexpr int SPW = 64 / G, JP = R * G, CT = JP / 16, KS = DOWN ? 5 : 4;
    __shared__ double lds[16 * 2 * V::SIZE];
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    const int gl = lane % G, sub = lane / G, lr = lane & 15, lk = lane >> 4, lane4 = 4 * lane;
    const int m = (int)blockIdx.x / a.nleaf, b = (int)blockIdx.x % a.nleaf;
    const int M = a.M, nr = a.rows, i0 = b * (nr + 1);
    const double *tab = a.leaf + (size_t)b * kLeafStride;
    const Plane<R, G> q(a, F, m);

    double av[KS];
#pragma unroll
    for (int ks = 0; ks < KS; ++ks) av[ks] = tab[kLeafU + lr * 20 + 4 * ks + lk];
    int row[KS];  // the z row this lane loads for each k-step (any valid row where U is zero)
#pragma unroll
    for (int ks = 0; ks < KS; ++ks) {
        const int k = 4 * ks + lk;
        if (k < 16) row[ks] = i0 + (k < nr ? k : nr - 1);
        else row[ks] = k == 16 ? (i0 > 0 ? i0 - 1 : 0) : i0 + nr;
    }
#pragma unroll 4
    for (int t = wave; t < 2 * CT; t += W) {
        const int h = t / CT, j = (t % CT) * 16 + lr, jc = j < M ? j : M - 1;
        dx4 acc = dx4{0.0, 0.0, 0.0, 0.0};
        if (h == 0 || q.two) {
            const double *src = (h ? q.ss : q.sc) + jc;
            double y[KS];
#pragma unroll
            for (int ks = 0; ks < KS; ++ks) y[ks] = src[(size_t)row[ks] * a.J];
#pragma unroll
            for (int ks = 0; ks < KS; ++ks)
                acc = __builtin_amdgcn_mfma_f64_16x16x4f64(av[ks], j < M ? y[ks] : 0.0, acc, 0, 0, 0);
        }
#pragma unroll
        for (int v = 0; v < 4; ++v) lds[((lk + 4 * v) * 2 + h) * V::SIZE + V::at(j)] = acc[v];
    }
    double ca[R], cb[R], cc[R];
    rtri_rows<R>(a.am, a.cm, a.bm + (size_t)m * a.JP, gl * R, M, ca, cb, cc);
    __syncthreads();

    double s[2][2][R];
    if constexpr (!DOWN) {
#pragma unroll
        for (int r = 0; r < R; ++r) s[0][0][r] = s[0][1][r] = s[1][0][r] = s[1][1][r] = 0.0;
    }
#pragma unroll 1
    for (int p0 = wave * SPW; p0 < nr; p0 += W * SPW) {
        const int p = p0 + sub;
        const double rt = tab[kLeafRoot + p];
        double d0[R], d1[R];
        double *v0 = lds + (size_t)(p * 2) * V::SIZE + gl, *v1 = v0 + V::SIZE;
#pragma unroll
        for (int r = 0; r < R; ++r) {
            d0[r] = v0[r * V::PITCH];
            d1[r] = v1[r * V::PITCH];
        }
        rtri_solve<R, G>(ca, cb, cc, rt, lane4, d0, d1);
        if constexpr (DOWN) {
#pragma unroll
            for (int r = 0; r < R; ++r) {
                v0[r * V::PITCH] = d0[r];
                v1[r * V::PITCH] = d1[r];
            }
        } else {
            const double wr = tab[kLeafRight + p], wl = tab[kLeafLeft + p];
#pragma unroll
            for (int r = 0; r < R; ++r) {
                s[0][0][r] = __builtin_fma(wr, d0[r], s[0][0][r]);
                s[0][1][r] = __builtin_fma(wr, d1[r], s[0][1][r]);
                s[1][0][r] = __builtin_fma(wl, d0[r], s[1][0][r]);
                s[1][1][r] = __builtin_fma(wl, d1[r], s[1][1][r]);
            }
        }
    }

    if constexpr (!DOWN) {
        block_sums<R, G, W, 2>(s, lds, M, [&](int n, int h, int j, double v) {
            if (h == 1 && !q.two) return;
            if (n == 0) {
                if (b + 1 < a.nleaf) (h ? q.ss : q.sc)[(size_t)(i0 + nr) * a.J + j] += v;
            } else if (b > 0) {
                (h ? q.ps : q.pc)[(size_t)(i0 - 1) * a.JP + j] = v;
            }
        });
    } else {
        double vv[4];
#pragma unroll
        for (int ks = 0; ks < 4; ++ks) vv[ks] = tab[kLeafV + lr * 16 + 4 * ks + lk];
        __syncthreads();
#pragma unroll 4
        for (int t = wave; t < 2 * CT; t += W) {
            const int h = t / CT, j = (t % CT) * 16 + lr;
            if (h == 1 && !q.two) break;  // the same for the wavefront, and for every later t
            dx4 acc = dx4{0.0, 0.0, 0.0, 0.0};
#pragma unroll
            for (int ks = 0; ks < 4; ++ks)
                acc = __builtin_amdgcn_mfma_f64_16x16x4f64(
                    vv[ks], lds[((4 * ks + lk) * 2 + h) * V::SIZE + V::at(j)], acc, 0, 0, 0);
            double *dst = (h ? q.ss : q.sc) + (size_t)i0 * a.J + j;
#pragma unroll
            for (int v = 0; v < 4; ++v) {
                const int k = lk + 4 * v;
                if (k < nr && j < M) dst[(size_t)k * a.J] = acc[v];
            }
        }
    }
}

// A node of the tree: row i = (2 n + 1) h (1-based) with its block of 2h - 1
// rows; the roots are dealt to the block's W wavefronts in turn.  Its
// right-hand side is the spectrum's row plus the second buffer's.
template <int R, int G, int W, bool DOWN>
__global__ __launch_bounds__(64 * W, 2) void k_cr_node(CrArgs a, const Fields F, CrPhase ph)
{
    typedef Vec<R, G> V;
    constexpr int SPW = 64 / G, JP = R * G, NIN = DOWN ? 3 : 1, NSUM = DOWN ? 1 : 2;
    constexpr int NV = NIN * 2 > W * NSUM * 2 ? NIN * 2 : W * NSUM * 2;
    __shared__ double lds[NV * V::SIZE];
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    const int gl = lane % G, sub = lane / G, lane4 = 4 * lane;
    const int m = (int)blockIdx.x / ph.nnode, n = (int)blockIdx.x % ph.nnode;
    const int h = ph.h, M = a.M;
    const int i = (2 * n + 1) * h - 1;          // this row, 0-based
    const bool left = n > 0, right = n + 1 < ph.nnode;
    const Plane<R, G> q(a, F, m);

    // the node's right-hand side and (down) the solved rows beside it
    for (int e = threadIdx.x; e < NIN * 2 * JP; e += 64 * W) {
        const int j = e % JP, c = (e / JP) % 2, w = e / (2 * JP);
        double v = 0.0;
        if (j < M && (c == 0 || q.two)) {
            const double *S = (c ? q.ss : q.sc) + j, *Pv = (c ? q.ps : q.pc) + j;
            if (w == 0) v = S[(size_t)i * a.J] + Pv[(size_t)i * a.JP];
            else if (w == 1 ? left : right) v = S[(size_t)(w == 1 ? i - h : i + h) * a.J];
        }
        lds[(w * 2 + c) * V::SIZE + V::at(j)] = v;
    }
    double ca[R], cb[R], cc[R];
    rtri_rows<R>(a.am, a.cm, a.bm + (size_t)m * a.JP, gl * R, M, ca, cb, cc);
    __syncthreads();

    double s[NSUM][2][R], x0[R], x1[R];
#pragma unroll
    for (int r = 0; r < R; ++r) {
#pragma unroll
        for (int t = 0; t < NSUM; ++t) s[t][0][r] = s[t][1][r] = 0.0;
        if constexpr (!DOWN) {
            x0[r] = lds[r * V::PITCH + gl];
            x1[r] = lds[V::SIZE + r * V::PITCH + gl];
        }
    }
    const double *rec = a.node + ((size_t)ph.rec0 + (size_t)n * node_roots(h) + sub) * kNodeRec;
    double rt = rec[(size_t)wave * SPW * kNodeRec];
#pragma unroll 1
    for (int p = wave * SPW; p < 2 * h; p += W * SPW) {
        const double *rp = rec + (size_t)p * kNodeRec;
        const double w0 = rp[DOWN ? 3 : 1], w1 = rp[DOWN ? 4 : 2], w2 = DOWN ? rp[5] : 0.0;
        const int pn = p + W * SPW < 2 * h ? p + W * SPW : p;
        const double rt_next = rec[(size_t)pn * kNodeRec];
        double d0[R], d1[R];
#pragma unroll
        for (int r = 0; r < R; ++r) {
            if constexpr (DOWN) {
                const double *l = lds + r * V::PITCH + gl;
                d0[r] = __builtin_fma(w2, l[4 * V::SIZE], __builtin_fma(w1, l[2 * V::SIZE], w0 * l[0]));
                d1[r] = __builtin_fma(w2, l[5 * V::SIZE], __builtin_fma(w1, l[3 * V::SIZE], w0 * l[V::SIZE]));
            } else {
                d0[r] = x0[r];
                d1[r] = x1[r];
            }
        }
        rtri_solve<R, G>(ca, cb, cc, rt, lane4, d0, d1);
#pragma unroll
        for (int r = 0; r < R; ++r) {
            if constexpr (DOWN) {
                s[0][0][r] += d0[r];
                s[0][1][r] += d1[r];
            } else {
                s[0][0][r] = __builtin_fma(w0, d0[r], s[0][0][r]);
                s[0][1][r] = __builtin_fma(w0, d1[r], s[0][1][r]);
                s[1][0][r] = __builtin_fma(w1, d0[r], s[1][0][r]);
                s[1][1][r] = __builtin_fma(w1, d1[r], s[1][1][r]);
            }
        }
        rt = rt_next;
    }
    block_sums<R, G, W, NSUM>(s, lds, M, [&](int t, int c, int j, double v) {
        if (c == 1 && !q.two) return;
        if constexpr (DOWN) {
            (c ? q.ss : q.sc)[(size_t)i * a.J + j] = v;
        } else if (t == 0) {
            if (right) (c ? q.ss : q.sc)[(size_t)(i + h) * a.J + j] += v;
        } else if (left) {
            (c ? q.ps : q.pc)[(size_t)(i - h) * a.JP + j] += v;
        }
    });
}

template <int R, int G, int W>
void launch_node(const CrPhase &ph, const CrArgs &a, const Fields &F, hipStream_t s)
{
    const dim3 grid((unsigned)((a.N + 1) * ph.nnode), F.nf);
    if (ph.kind == CR_NODE_DOWN)
        hipLaunchKernelGGL((k_cr_node<R, G, W, true>), grid, dim3(64 * W), 0, s, a, F, ph);
    else
        hipLaunchKernelGGL((k_cr_node<R, G, W, false>), grid, dim3(64 * W), 0, s, a, F, ph);
}

// One launch per phase.  Wavefronts per node: four rounds of 64/G roots each,
// at most 8, so that a single field's launch of any level holds about one
// wavefront per SIMD (N+1 orders x nodes x W).
template <int R, int G>
int launch_phases(const chy_grid *g, const CrArgs &a, const Fields &F, hipStream_t s)
{
    constexpr int SPW = 64 / G;
    constexpr int WL = G == 64 ? 8 : (G == 8 ? 2 : 4);
    const dim3 leaves((unsigned)((g->N + 1) * a.nleaf), F.nf);
    for (const CrPhase &ph : g->cr.phases) {
        if (ph.kind == CR_LEAF_UP) {
            hipLaunchKernelGGL((k_cr_leaf<R, G, WL, false>), leaves, dim3(64 * WL), 0, s, a, F);
        } else if (ph.kind == CR_LEAF_DOWN) {
            hipLaunchKernelGGL((k_cr_leaf<R, G, WL, true>), leaves, dim3(64 * WL), 0, s, a, F);
        } else {
            switch (2 * ph.h / (4 * SPW)) {
            case 0:
            case 1: launch_node<R, G, 1>(ph, a, F, s); break;
            case 2: launch_node<R, G, 2>(ph, a, F, s); break;
            case 4: launch_node<R, G, 4>(ph, a, F, s); break;
            default: launch_node<R, G, 8>(ph, a, F, s); break;
            }
        }
    }
    return (int)hipGetLastError();
}

}  // namespace

bool cr_supported(const chy_grid *g)
{
    const int r = g->JP / 64;
    return g->cr.kx >= 2 && (r == 1 || r == 2 || r == 4 || r == 8);
}

// 64: one system per wavefront, JP/64 rows per lane.  32: the packed form, 8
// rows per lane and JP/8 lanes per system, where that is at most 32 lanes.
bool cr_lanes_ok(const chy_grid *g, int lanes)
{
    if (lanes == 64) return cr_supported(g);
    if (lanes == 32) return cr_supported(g) && g->JP / 32 <= 8;
    return false;
}

int launch_cr_solve_f(const chy_grid *g, const Fields &F, hipStream_t s)
{
    CrArgs a{};
    a.am = g->d.am;
    a.cm = g->d.cm;
    a.bm = g->d.bm;
    a.leaf = g->d.cr_leaf;
    a.node = g->d.cr_node;
    a.J = g->J; a.K = g->K; a.M = g->M; a.N = g->N; a.PP = g->PP; a.JP = g->JP;
    a.nleaf = g->cr.nleaf;
    a.rows = g->cr.rows;
    if (g->cr_lanes == 32) {
        switch (g->JP) {
        case 64: return launch_phases<8, 8>(g, a, F, s);
        case 128: return launch_phases<8, 16>(g, a, F, s);
        case 256: return launch_phases<8, 32>(g, a, F, s);
        default: break;
        }
    }
    switch (g->JP) {
    case 64: return launch_phases<1, 64>(g, a, F, s);
    case 128: return launch_phases<2, 64>(g, a, F, s);
    case 256: return launch_phases<4, 64>(g, a, F, s);
    case 512: return launch_phases<8, 64>(g, a, F, s);
    default: return (int)hipErrorInvalidValue;
    }
}

}  // namespace chy
