// Per-mode solves on the GPU with BLKTRI's root tables: the systems POT3 hands
// to BLKTRI for every azimuthal mode (pot/blktri.f:60-260, called at
// pot/pot3.f:233-239).
//
// A mode's unknowns are X(j, i): j = 1..M along r (JMAX-1 rows), i = 1..N
// along z (KMAX-1 = 2^k - 1 rows).  BLKTRI eliminates the rows level by level,
// applying products of r-tridiagonal solves (T_m - rt)^-1.  The same
// elimination is a tree here (crplan.cpp): leaves of 15 z rows (3 where their
// spacing varies), then one node per row i = odd * h, h = 16, 32, .. (4, 8, ..),
// whose block of 2h - 1 rows has its roots in BLKTRI's table.  Up the tree every
// block sends what its right-hand side adds to the two rows beside it; down the
// tree every block is solved from its own right-hand side and the solved rows
// beside it.  BLKTRI's
// product of a block (all its roots below the line, the roots of its halves
// above) and the chain that follows it (the roots of one half below the line)
// cancel root by root, so each message and each solution is one sum of
// independent solves with the block's own roots:
//   up    Y(i +- h) += sum_p b_p (T - r_p)^-1 Y(i)
//   down  X(i)       = sum_p (T - r_p)^-1 (a_p Y(i) + cL_p X(i-h) + cR_p X(i+h))
// and no intermediate vectors, chains or extra launches remain.  A node's sums
// run over 15 to 35 roots that give the same functions of T as the block's
// 31 to 511 (crplan.cpp): 505 r solves per mode in 7 launches at KMAX = 128 (867
// with every root of the nodes' blocks, a solve of 32 fields at 256x128x256
// 5.66 ms against 4.97; level by level it is 2215 in 19, 13.6 ms).  The weights
// alternate in sign; the terms stay as small as the block's own Green's
// function, so the sums round as one more elimination order does (1-2e-14 from
// BLKTRI's result at KMAX up to 512 on grids alike in r and z, 3-5e-14 with the
// leaves, whose rows are solved together in their eigenvectors).
//
// One block of a launch is one tree node (or leaf) of one order m: the cosine
// and sine parts share T_m, so every solve has two right-hand sides; solves
// run on groups of G lanes (rtri.h), 64/G roots per wavefront at a time.  The
// leaves' changes of basis run on the FP64 matrix cores through LDS.  The
// spectrum spec[q][k][j] (J contiguous) is the mode right-hand side on entry
// (with POT3's boundary terms applied) and the mode solution on exit.  What the
// blocks add to a separating row goes to the grid's second workspace buffer
// (yh), from its right side into its own row there and from its left side into
// the row before (unused inside a leaf), so every row has one writer per launch
// and the order of every sum is fixed.
#include <hip/hip_runtime.h>

#include <algorithm>

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

// The sums of a node (one or two, two parts each) by its team of W wavefronts
// (tid: thread of the team): every lane holds its root group's share; the
// W * 64/G shares of one part at a time meet in LDS and are added in order,
// out(sum, part, j, value) for j < M.  (Adding the groups of a wavefront by lane
// exchanges first cost 300 instructions per wavefront, two thirds of a solve.)
template <int R, int G, int W, int NSUM, typename Out>
__device__ __forceinline__ void team_sums(const double (&s)[NSUM][2][R], double *lds, int tid, int M, Out out)
{
    typedef Vec<R, G> V;
    constexpr int SLOTS = W * 64 / G;
    const int slot = tid / G, gl = tid % G;
#pragma unroll
    for (int n = 0; n < NSUM; ++n) {
#pragma unroll
        for (int h = 0; h < 2; ++h) {
            __syncthreads();  // every wavefront is done with what lds held
#pragma unroll
            for (int r = 0; r < R; ++r) lds[slot * V::SIZE + r * V::PITCH + gl] = s[n][h][r];
            __syncthreads();
            for (int j = tid; j < R * G; j += 64 * W) {
                const double *p = lds + V::at(j);
                double v = p[0];
#pragma unroll
                for (int t = 1; t < SLOTS; ++t) v += p[t * V::SIZE];
                if (j < M) out(n, h, j, v);
            }
        }
    }
}

// Leaves: rows i0 .. i0 + rows - 1 (0-based, i0 = (rows + 1) b), the
// separating rows i0 - 1 and i0 + rows beside them.  Up: a leaf's messages to
// the separators.  Down: its rows from the solved separators.  LS roots
// (zero-padded).
//   gather   D[p][j] = sum_k U[p][k] Y[k][j]   (down: k = LS, LS + 1 the separators)
//   solves   one root per group of lanes
//   scatter  X[k][j] = sum_p V[k][p] D[p][j]   (down)
// V_MFMA_F64_16X16X4F64: A lane l holds A[l%16][l/16], B lane l B[l/16][l%16],
// the result D[l/16 + 4v][l%16].
//
// A block takes `run` leaves (one or two) of one order one after the other.  It
// is bound by HBM (up: the spectrum read once, down: read and written: 0.60 and
// 0.95 ms per 32 fields at 256x128x256, 0.44 and 0.87 at the rate of a copy),
// while its solves keep the VALU busy for about half as long, so the next
// leaf's rows are loaded into registers (a matrix operand each) before the
// current one is solved.  Loads and stores of a wavefront complete in order: nothing the
// solves need is loaded after those rows (the roots and weights wait in LDS),
// and the next leaf's U is loaded before the current one's results are
// stored.  LDS holds the 16 x 2 vectors: 76 KB at JMAX <= 256 (two blocks of 4
// wavefronts per CU), 148 KB at 512 (one of 8).  (Leaves of 31 rows need 146 KB
// at JMAX <= 256 and twice the matrix products per row: one block per CU, its
// phases one after another, 1.45 ms down and 1.2 ms up per 32 fields at
// 256x128x256, more than the saved level of nodes gives.)
template <int R, int G, int W, bool DOWN>
__global__ __launch_bounds__(64 * W, 2) void k_cr_leaf(CrArgs a, const Fields F, int run)
{
    typedef Vec<R, G> V;
    constexpr int LS = kLeafSpan, SPW = 64 / G, JP = R * G, CT = JP / 16, KS = LS / 4 + (DOWN ? 1 : 0);
    constexpr int NT = (2 * CT + W - 1) / W;  // column tiles per wavefront
    __shared__ double lds[LS * 2 * V::SIZE], tri[3 * V::SIZE], wts[3 * LS];
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    const int gl = lane % G, sub = lane / G, lr = lane & 15, lk = lane >> 4;
    const int nrun = (a.nleaf + run - 1) / run;
    const int m = (int)blockIdx.x / nrun, b0 = (int)blockIdx.x % nrun * run, b1 = min(b0 + run, a.nleaf);
    const int M = a.M, nr = a.rows;
    const Plane<R, G> q(a, F, m);

    // this wavefront's column tiles of leaf b: row k of lane l, any valid row
    // where U is zero
    double y[NT][KS];
    auto fetch = [&](int b) {
        const int i0 = b * (nr + 1);
        size_t off[KS];
#pragma unroll
        for (int ks = 0; ks < KS; ++ks) {
            const int k = 4 * ks + lk;
            const int row = k < LS ? i0 + min(k, nr - 1) : (k == LS ? max(i0 - 1, 0) : i0 + nr);
            off[ks] = (size_t)row * a.J;
        }
#pragma unroll
        for (int t = 0; t < NT; ++t) {
            const int tt = min(wave + t * W, 2 * CT - 1), h = tt / CT;  // the same for the wavefront
            const int j = min((tt % CT) * 16 + lr, M - 1);
            const double *src = (h ? q.ss : q.sc) + j;
#pragma unroll
            for (int ks = 0; ks < KS; ++ks) y[t][ks] = src[off[ks]];
        }
    };
    double av[KS], wt;  // U's operands; this thread's root or weight
    auto tables = [&](int b) {
        const double *tab = a.leaf + (size_t)b * kLeafStride;
#pragma unroll
        for (int ks = 0; ks < KS; ++ks) av[ks] = tab[kLeafU + lr * (LS + 4) + 4 * ks + lk];
        wt = tab[kLeafRoot + min((int)threadIdx.x, 3 * LS - 1)];
    };
    fetch(b0);
    tables(b0);
    rtri_load<R, G>(tri, a.am, a.cm, a.bm + (size_t)m * a.JP, M, 64 * W);
    const Neigh at = neighbours<G>(lane);

#pragma unroll 1
    for (int b = b0; b < b1; ++b) {
        const int i0 = b * (nr + 1);
        if (threadIdx.x < 3 * LS) wts[threadIdx.x] = wt;
#pragma unroll
        for (int t = 0; t < NT; ++t) {
            const int tt = wave + t * W, h = tt / CT, j = (tt % CT) * 16 + lr;
            if (tt >= 2 * CT) break;
            const bool on = j < M && (h == 0 || q.two);
            dx4 acc = dx4{0.0, 0.0, 0.0, 0.0};
#pragma unroll
            for (int ks = 0; ks < KS; ++ks)
                acc = __builtin_amdgcn_mfma_f64_16x16x4f64(av[ks], on ? y[t][ks] : 0.0, acc, 0, 0, 0);
#pragma unroll
            for (int v = 0; v < 4; ++v) lds[((lk + 4 * v) * 2 + h) * V::SIZE + V::at(j)] = acc[v];
        }
        __syncthreads();
        if (b + 1 < b1) fetch(b + 1);

#pragma unroll 1
        for (int p0 = wave * SPW; p0 < nr; p0 += W * SPW) {
            const int p = p0 + sub;
            const double rt = wts[p];
            asm volatile("" ::: "memory");  // T's rows are read anew in every round, not kept in registers
            double d0[R], d1[R];
            double *v0 = lds + (size_t)(p * 2) * V::SIZE + gl, *v1 = v0 + V::SIZE;
#pragma unroll
            for (int r = 0; r < R; ++r) {
                d0[r] = v0[r * V::PITCH];
                d1[r] = v1[r * V::PITCH];
            }
            rtri_solve<R, G>(tri + gl, rt, at, d0, d1);
#pragma unroll
            for (int r = 0; r < R; ++r) {
                v0[r * V::PITCH] = d0[r];
                v1[r * V::PITCH] = d1[r];
            }
        }

        if constexpr (!DOWN) {
            if (b + 1 < b1) tables(b + 1);
            __syncthreads();
            // to the right separator through the second buffer's row before
            // it, to the left one through its own
            for (int e = threadIdx.x; e < 2 * JP; e += 64 * W) {
                const int h = e / JP, j = e % JP;
                const double *x = lds + h * V::SIZE + V::at(j);
                double right = 0.0, left = 0.0;
#pragma unroll
                for (int p = 0; p < LS; ++p) {
                    const double v = x[(size_t)(p * 2) * V::SIZE];
                    right = __builtin_fma(wts[LS + p], v, right);
                    left = __builtin_fma(wts[2 * LS + p], v, left);
                }
                if (j >= M || (h == 1 && !q.two)) continue;
                double *out = (h ? q.ps : q.pc) + j;
                if (b + 1 < a.nleaf) out[(size_t)(i0 + nr - 1) * a.JP] = right;
                if (b > 0) out[(size_t)(i0 - 1) * a.JP] = left;
            }
        } else {
            double vv[LS / 4];
            {
                const double *tab = a.leaf + (size_t)b * kLeafStride + kLeafV;
#pragma unroll
                for (int ks = 0; ks < LS / 4; ++ks) vv[ks] = tab[lr * LS + 4 * ks + lk];
            }
            if (b + 1 < b1) tables(b + 1);
            __syncthreads();
#pragma unroll 4
            for (int t = wave; t < 2 * CT; t += W) {
                const int h = t / CT, j = (t % CT) * 16 + lr;
                if (h == 1 && !q.two) break;  // the same for the wavefront, and for every later t
                dx4 acc = dx4{0.0, 0.0, 0.0, 0.0};
#pragma unroll
                for (int ks = 0; ks < LS / 4; ++ks)
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
        __syncthreads();  // lds is free for the next leaf
    }
}

// A node of the tree: row i = (2 n + 1) h (1-based) with its block of 2h - 1
// rows; the roots are dealt to the team's W wavefronts in turn.  Its
// right-hand side is the spectrum's row plus the messages from its right (the
// second buffer's row) and from its left (the row before).  With two or three
// rounds of solves a block's loads, barriers and sums take as long as its
// solves; LDS holds one vector per root in flight (24 KB, six blocks per CU)
// and the sums' parts pass through it one after another (both at once, 41 KB
// and three blocks: 272 instead of 250 us for the lowest level up).
template <int R, int G>
struct Node {
    // wavefronts: 256x128x256's levels of 16-23, 23-29 and 21 roots take 250/265,
    // 144/154 and 71 us up and down per 32 fields with 4 or 2, and alone 14, 12
    // and 10 us with 4 but 20, 19 and 16 with 2; two rounds of roots on fewer
    // wavefronts took 64x128x64 and 128x32x64 from 83.5 and 56.8 to 87.8 and 58.8
    // us alone, and no less per field of a batch.  (8 wavefronts: the top node 8
    // us alone, 105 per 32 fields.  The count does not depend on the number of
    // fields, as it orders the sums.)
    static constexpr int W = G == 8 ? 2 : 4;
    static constexpr int VECTORS(bool down) { return W * 64 / G > (down ? 6 : 2) ? W * 64 / G : down ? 6 : 2; }
};

// (n past the level's nodes: nothing is stored)
template <int R, int G, bool DOWN>
__device__ __forceinline__ void node_run(const CrArgs &a, const Plane<R, G> &q, const CrPhase &ph, double *lds,
                                         const double *tri, int tid, int n)
{
    typedef Vec<R, G> V;
    constexpr int W = Node<R, G>::W, SPW = 64 / G, JP = R * G, NIN = DOWN ? 3 : 1, NSUM = DOWN ? 1 : 2;
    const int lane = tid & 63, wave = tid >> 6;
    const int gl = lane % G, sub = lane / G;
    const bool real = n < ph.nnode;
    const int h = ph.h, M = a.M;
    n = min(n, ph.nnode - 1);
    const int i = (2 * n + 1) * h - 1;          // this row, 0-based
    const bool left = n > 0, right = n + 1 < ph.nnode;
    const double *rec = a.node + ((size_t)ph.rec0 + (size_t)n * (1 + ph.np)) * kNodeRec;
    const int np = real ? (int)rec[0] : 0;
    rec += (1 + sub) * kNodeRec;

    // the node's right-hand side and (down) the solved rows beside it
    for (int e = tid; e < NIN * 2 * JP; e += 64 * W) {
        const int j = e % JP, c = (e / JP) % 2, w = e / (2 * JP);
        double v = 0.0;
        if (j < M && (c == 0 || q.two)) {
            const double *S = (c ? q.ss : q.sc) + j, *Pv = (c ? q.ps : q.pc) + j;
            if (w == 0) v = S[(size_t)i * a.J] + (Pv[(size_t)i * a.JP] + Pv[(size_t)(i - 1) * a.JP]);
            else if (w == 1 ? left : right) v = S[(size_t)(w == 1 ? i - h : i + h) * a.J];
        }
        lds[(w * 2 + c) * V::SIZE + V::at(j)] = v;
    }
    const Neigh at = neighbours<G>(lane);
    __syncthreads();

    double s[NSUM][2][R];
#pragma unroll
    for (int r = 0; r < R; ++r)
#pragma unroll
        for (int t = 0; t < NSUM; ++t) s[t][0][r] = s[t][1][r] = 0.0;
    double rt = rec[(size_t)min(wave * SPW, ph.np - SPW) * kNodeRec];
#pragma unroll 1
    for (int p = wave * SPW; p < np; p += W * SPW) {
        const double *rp = rec + (size_t)p * kNodeRec;
        const double w0 = rp[DOWN ? 3 : 1], w1 = rp[DOWN ? 4 : 2], w2 = DOWN ? rp[5] : 0.0;
        const int pn = p + W * SPW < np ? p + W * SPW : p;
        const double rt_next = rec[(size_t)pn * kNodeRec];
        asm volatile("" ::: "memory");  // the LDS operands are read anew in every round, not kept in registers
        double d0[R], d1[R];
#pragma unroll
        for (int r = 0; r < R; ++r) {
            const double *l = lds + r * V::PITCH + gl;
            if constexpr (DOWN) {
                d0[r] = __builtin_fma(w2, l[4 * V::SIZE], __builtin_fma(w1, l[2 * V::SIZE], w0 * l[0]));
                d1[r] = __builtin_fma(w2, l[5 * V::SIZE], __builtin_fma(w1, l[3 * V::SIZE], w0 * l[V::SIZE]));
            } else {
                d0[r] = l[0];
                d1[r] = l[V::SIZE];
            }
        }
        rtri_solve<R, G>(tri + gl, rt, at, d0, d1);
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
    team_sums<R, G, W, NSUM>(s, lds, tid, M, [&](int t, int c, int j, double v) {
        if (!real || (c == 1 && !q.two)) return;
        if constexpr (DOWN) {
            (c ? q.ss : q.sc)[(size_t)i * a.J + j] = v;
        } else if (t == 0) {
            if (right) (c ? q.ps : q.pc)[(size_t)(i + h - 1) * a.JP + j] += v;
        } else if (left) {
            (c ? q.ps : q.pc)[(size_t)(i - h) * a.JP + j] += v;
        }
    });
}

template <int R, int G, bool DOWN>
__global__ __launch_bounds__((64 * Node<R, G>::W), R == 8 ? 3 : 4) void k_cr_node(CrArgs a, const Fields F, CrPhase ph)
{
    __shared__ double lds[Node<R, G>::VECTORS(DOWN) * Vec<R, G>::SIZE], tri[3 * Vec<R, G>::SIZE];
    const int m = (int)blockIdx.x / ph.nnode;
    const Plane<R, G> q(a, F, m);
    rtri_load<R, G>(tri, a.am, a.cm, a.bm + (size_t)m * a.JP, a.M, 64 * Node<R, G>::W);
    node_run<R, G, DOWN>(a, q, ph, lds, tri, threadIdx.x, (int)blockIdx.x % ph.nnode);
}

// The two highest levels, up, down and down again, by one block per order (two
// teams, one of which the top node leaves idle): one launch instead of three for
// launches too small to fill the chip.  What one phase leaves for the next lies
// in global memory, written and read by the same block across a barrier.  The
// teams are those of k_cr_node: the same results bit for bit.  One field at
// 256x128x256 29.4 us, 33.8 in three launches (the solve 237 -> 232); with orders
// past one per CU it is no faster (two fields 54.8 and 45.3, 32 fields 499 and
// 370).  (The same for the whole tree, leaves and all: 153 us, 129 in its seven
// launches; a CU's 8 wavefronts do not hide the solves' latency.)
template <int R, int G>
__global__ __launch_bounds__((128 * Node<R, G>::W)) void k_cr_top(CrArgs a, const Fields F, CrPhase second, CrPhase top)
{
    typedef Node<R, G> D;
    constexpr int SIZE = D::VECTORS(true) * Vec<R, G>::SIZE;
    __shared__ double lds[2 * SIZE], tri[3 * Vec<R, G>::SIZE];
    const int team = threadIdx.x / (64 * D::W), tid = threadIdx.x % (64 * D::W);
    const Plane<R, G> q(a, F, (int)blockIdx.x);
    rtri_load<R, G>(tri, a.am, a.cm, a.bm + (size_t)blockIdx.x * a.JP, a.M, 128 * D::W);
    node_run<R, G, false>(a, q, second, lds + team * SIZE, tri, tid, team);
    __syncthreads();
    node_run<R, G, true>(a, q, top, lds + team * SIZE, tri, tid, team);
    __syncthreads();
    node_run<R, G, true>(a, q, second, lds + team * SIZE, tri, tid, team);
}

template <int R, int G>
void launch_leaf(const CrPhase &ph, const chy_grid *g, const CrArgs &a, const Fields &F, hipStream_t s)
{
    // wavefronts: all roots in one round of 64/G each for short r systems (at
    // JMAX 64 one round 4.7 + 6.4 us, two rounds 5.8 + 8.8), two rounds at 32 and
    // 64 lanes (twice the wavefronts at 32: 1.08 instead of 1.00 ms down per 32
    // fields at 256x128x256, and no faster alone)
    constexpr int rounds = kLeafSpan * G / 64, W = rounds >= 16 ? 8 : rounds >= 8 ? rounds / 2 : rounds;
    // leaves per block: two hide a part of each other's loads once the chip has
    // its blocks eight times over (8 fields at 256x128x256 279 + 185 us, one leaf
    // 285 + 188, four 293 + 192); below that more blocks are better (one field
    // 40 + 30 us with one, 43 + 33 with two, 49 + 38 with four)
    constexpr int lds = (2 * kLeafSpan + 3) * Vec<R, G>::SIZE * 8;
    const long slots = (long)g->ncu * std::max(1, std::min(160 * 1024 / lds, 8 / W));
    const int run = (long)(g->N + 1) * a.nleaf * F.nf >= 8 * slots ? 2 : 1;
    const dim3 grid((unsigned)((g->N + 1) * ((a.nleaf + run - 1) / run)), F.nf);
    if (ph.kind == CR_LEAF_UP)
        hipLaunchKernelGGL((k_cr_leaf<R, G, W, false>), grid, dim3(64 * W), 0, s, a, F, run);
    else
        hipLaunchKernelGGL((k_cr_leaf<R, G, W, true>), grid, dim3(64 * W), 0, s, a, F, run);
}

// One launch per phase, or one for the three highest.
template <int R, int G>
int launch_phases(const chy_grid *g, const CrArgs &a, const Fields &F, hipStream_t s)
{
    const std::vector<CrPhase> &ph = g->cr.phases;
    // first: the last level up, before the top and the way down from it
    const size_t levels = (ph.size() - 1) / 2, first = levels - 1;
    const bool fuse = levels >= 2 && (long)(g->N + 1) * F.nf <= g->ncu;
    for (size_t i = 0; i < ph.size(); ++i) {
        const dim3 grid((unsigned)((a.N + 1) * ph[i].nnode), F.nf), block(64 * Node<R, G>::W);
        if (ph[i].kind == CR_LEAF_UP || ph[i].kind == CR_LEAF_DOWN) {
            launch_leaf<R, G>(ph[i], g, a, F, s);
        } else if (fuse && i == first) {
            hipLaunchKernelGGL((k_cr_top<R, G>), dim3(g->N + 1, F.nf), dim3(2 * block.x), 0, s, a, F, ph[i], ph[i + 1]);
            i += 2;
        } else if (ph[i].kind == CR_NODE_DOWN) {
            hipLaunchKernelGGL((k_cr_node<R, G, true>), grid, block, 0, s, a, F, ph[i]);
        } else {
            hipLaunchKernelGGL((k_cr_node<R, G, false>), grid, block, 0, s, a, F, ph[i]);
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
