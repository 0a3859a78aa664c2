/*
 * chypot.h -- C-ABI of the MI355X self-gravity potential solve (libchypot.so).
 *
 * Drop-in boundary for CHYMERA's potential solve.  The reference exposes it as
 * three Fortran subroutines that exchange data through COMMON blocks:
 *
 *   SUBROUTINE SETBDY(NCALL,ISYM)          pot/boundary.f:2
 *   SUBROUTINE BDYGEN(MAXTRM,ISYM,REDGE)   pot/boundary.f:88
 *   SUBROUTINE POT3(NPOINT,IPRINT)         pot/pot3.f:15   (calls ZAXPHI, pot/pot3.f:311)
 *
 * with PHI/RHO in /POIS/ (headers/globals.h:55-58), the grid in /GRID/
 * (headers/globals.h:104-109), DTHETA/PI/GRAV in /blok6/ (headers/globals.h:8-10),
 * COEF in /COEFS/ (pot/pot3.f:20) and TMASS/PHICHK/KLOCAT in /INSIDE/
 * (pot/pot3.f:317).  Here the same operations take explicit pointers instead of
 * COMMON storage; the Fortran shims in chymera-uo_amd/fortran/ map the COMMON
 * blocks onto these calls.
 *
 * Array layout is the reference's Fortran layout, unchanged:
 *   phi, rho : PHI(JMAX+2, KMAX+2, LMAX)      J fastest (element (J,K,L) at
 *              (J-1) + (JMAX+2)*((K-1) + (KMAX+2)*(L-1)), 1-based J,K,L)
 *   coef     : COEF(JMAX+2, KMAX+2, LMAX/2, 2)
 *   r, rhf   : length JMAX+2;  z, zhf : length KMAX+2   (host memory)
 *
 * Every entry point returns 0 on success or one of the CHY_E* codes below;
 * chy_strerror() gives the message.  The reference stops the program on the
 * errors it detects (pot/boundary.f:311,901-907; pot/fft.f:625-627) and
 * ignores BLKTRI's IERROR (pot/pot3.f:234-239); here every such condition is a
 * returned error and nothing is computed.
 *
 * Pointers named *_d are device pointers (HIP device memory on the context's
 * device); *_h are host pointers.  Calls on one context are issued on that
 * context's HIP stream in order; the *_d entry points return without waiting
 * for the GPU unless stated.
 */
#ifndef CHYPOT_H
#define CHYPOT_H

#include <stddef.h>

#ifdef __cplusplus
extern "C" {
#endif

enum {
    CHY_OK = 0,
    CHY_EINVAL = 1,       /* bad argument or grid description */
    CHY_EUNSUPPORTED = 2, /* grid the solver cannot take: KMAX not 2^k (BLKTRI's own
                             precondition, pot/blktri.f:29-31), LMAX odd or above
                             1024, LMAX/2 with a prime factor above 23 (FFT's own
                             limit, pot/fft.f:111-126), JMAX above 4096,
                             |ISYM| != 2 */
    CHY_ENOMEM = 3,       /* device or host allocation failed */
    CHY_EDEVICE = 4,      /* HIP runtime error */
    CHY_ESTATE = 5,       /* call out of order (e.g. BDYGEN before SETBDY,
                             pot/boundary.f:311) */
    CHY_ENUMERIC = 6,     /* z operator not symmetrisable (AN(k)*CN(k-1) <= 0) or
                             eigen-solver failed to converge */
    CHY_ELIMIT = 7        /* input larger than the fixed scratch of a
                             no-allocation entry point (chy_last_device_error
                             names the sizes) */
};

/* Grid as the reference holds it in /GRID/ and /blok6/. */
typedef struct {
    int jmax, kmax, lmax;      /* JMAX, KMAX, LMAX (headers/hydroparam.h:16-20) */
    const double *r, *z;       /* R(JMAX+2), Z(KMAX+2)   cell faces   (host) */
    const double *rhf, *zhf;   /* RHF(JMAX+2), ZHF(KMAX+2) cell centres (host) */
    double dtheta, pi, grav;   /* DTHETA, PI, GRAV */
} chy_grid_desc;

/* /INSIDE/ diagnostics written by BDYGEN (TMASS) and ZAXPHI (PHICHK, KLOCAT). */
typedef struct {
    double tmass;   /* total mass of the rings BDYGEN integrated (boundary.f:554) */
    double phichk;  /* largest azimuthal spread of the z-axis potential (pot3.f:389-399) */
    int klocat;     /* K where it occurs; unchanged when every spread is 0 */
} chy_diag;

/* What POT3's COEF output covers (pot3.f:105-132).  The hydro loop reads only
 * the K=2 plane (radhydro/3dhyd-main.f:708,784), so the plane alone saves a
 * full-field write per solve. */
enum { CHY_COEF_NONE = 0, CHY_COEF_K2 = 1, CHY_COEF_FULL = 2 };

typedef struct chy_ctx chy_ctx;
typedef struct chy_grid chy_grid;

/* ---- context (no reference counterpart: the reference runs in-process) ---- */

/* Context on HIP device `device`; owns a stream unless one is set. */
int chy_ctx_create(int device, chy_ctx **out);
int chy_ctx_destroy(chy_ctx *ctx);
/* Issue all later work of this context on `stream` (a hipStream_t; NULL = the
 * context's own stream). */
int chy_ctx_set_stream(chy_ctx *ctx, void *stream);
/* Wait for all work issued on the context's stream. */
int chy_ctx_sync(chy_ctx *ctx);

/* ---- SETBDY (pot/boundary.f:2-82) ----
 * Builds and uploads everything that depends only on the grid: the boundary
 * point list and cos/sin tables of SETBDY, BLKTRI's m-independent z-operator
 * data (here: its eigenbasis), the radial coefficients of pot3.f:158-194, FFT
 * twiddles and the workspace.  ISYM as in SETBDY; only |ISYM|=2 (equatorial
 * symmetry) is supported, the geometry POT3's midplane condition assumes. */
int chy_setbdy(chy_ctx *ctx, const chy_grid_desc *grid, int isym, chy_grid **out);
int chy_grid_destroy(chy_grid *g);
/* Device bytes held by a prepared grid (tables + workspace). */
size_t chy_grid_device_bytes(const chy_grid *g);

/* How POT3's per-mode 2-D solves (pot/pot3.f:233-239) are done on a grid.
 *   CHY_MODES_CR    (default) BLKTRI's generalised cyclic reduction
 *                   (pot/blktri.f:60-260) with BLKTRI's own root tables
 *                   (COMPB/TQLRAT, pot/blktri.f:264-423, the same arithmetic),
 *                   its products as sums of independent solves: the
 *                   reference's results to rounding (2.2e-13 relative at
 *                   256x128x256), and the faster one (32 fields there 4.85
 *                   ms, 5.97 by CHY_MODES_EIGEN).
 *   CHY_MODES_EIGEN the m-independent z operator diagonalised once per grid
 *                   (80-bit arithmetic) and r-tridiagonal solves per z
 *                   eigenvalue, the transforms on FP64 matrix cores: closer to
 *                   the exact solution of the discrete system than BLKTRI
 *                   (whose root tables put it up to a few 1e-12 from it at
 *                   256x128x256, and further where the z spacing varies).
 * CHY_MODES_CR needs JMAX-1 <= 512 (CHY_EUNSUPPORTED otherwise; such grids
 * start with CHY_MODES_EIGEN).  Changing the solver drops the captured batches
 * that use the grid. */
enum { CHY_MODES_CR = 0, CHY_MODES_EIGEN = 1 };
int chy_grid_set_mode_solver(chy_grid *g, int kind);
int chy_grid_mode_solver(const chy_grid *g);

/* Kernel shapes and precision split of a grid (no reference counterpart).
 *   CHY_TUNE_CR_LANES    r systems of the cyclic reduction per wavefront: 64
 *                        (64 lanes, one system) or 32 (8 rows per lane, so 8
 *                        to 32 lanes, up to 8 systems; JMAX-1 <= 256)
 *   CHY_TUNE_REFINE_M64  refined solves in binary32: the r solves of orders
 *                        m <= this value run in binary64 (-1..LMAX/2;
 *                        default 4)
 *   CHY_TUNE_REFINE_FUSED refined solves of 1 or 2 steps launched for at
 *                        most this many fields (0..32; default 0) run all
 *                        mode work of a mode plane in one kernel with the
 *                        binary32 plane in LDS, where it fits (KMAX <= 129,
 *                        JMAX <= 257) instead of the mode solves that
 *                        chy_solve_refined otherwise uses.  Above 0 a refined
 *                        field's result may depend on how many run with it:
 *                        the two forms agree to the steps' accuracy (1e-6 for
 *                        one, 1e-10 for two)
 * Otherwise results do not depend on the shapes beyond rounding.  Changing a value
 * drops the captured batches that use the grid.  CHY_EINVAL for a value the grid
 * cannot take. */
enum { CHY_TUNE_CR_LANES = 0, CHY_TUNE_REFINE_M64 = 1, CHY_TUNE_REFINE_FUSED = 2 };
int chy_grid_set_tune(chy_grid *g, int param, int value);
int chy_grid_tune(const chy_grid *g, int param);

/* ---- BDYGEN (pot/boundary.f:88-908) ----
 * Multipole boundary potential (l <= maxtrm <= 10) from rho_d into the boundary
 * cells of phi_d: K=KMAX+1 for J=2..JMAX+1, J=JMAX+1 for K=2..KMAX, and the
 * ISYM=2 ghosts PHI(JMAX+1,1,L) and PHI(1,KMAX+1,L).  Nothing else in phi_d is
 * written.  redge > 0 skips mass beyond spherical radius redge
 * (boundary.f:379).  diag (host, may be NULL) receives tmass after the call
 * has completed on the GPU (the call then waits). */
int chy_bdygen(chy_grid *g, int maxtrm, int isym, double redge, const double *rho_d,
               double *phi_d, chy_diag *diag);

/* ---- POT3 + ZAXPHI (pot/pot3.f:15-423) ----
 * Solves for phi_d given rho_d and the boundary values BDYGEN left in phi_d.
 * Writes PHI on J=1..JMAX+2 x K=1..KMAX+1 exactly as the reference does (the
 * K=KMAX+2 row and PHI(JMAX+2,1,L) are left as they were), and COEF per
 * coef_mode into coef_d (same full COEF shape; may be NULL for CHY_COEF_NONE;
 * amplitudes are left unchanged in lanes whose mean is exactly 0, as
 * pot3.f:106 does).  npoint is ZAXPHI's NPOINT (1..10; larger is clamped to
 * 10 as pot3.f:328-333 does).  diag (host, may be NULL) receives phichk and
 * klocat; klocat is read from diag first so that it stays unchanged when every
 * spread is 0 (pot3.f:391-398).  When diag is non-NULL the call waits. */
int chy_pot3(chy_grid *g, int npoint, const double *rho_d, double *phi_d, double *coef_d,
             int coef_mode, chy_diag *diag);

/* BDYGEN followed by POT3: one potential solve, device-resident, one stream.
 * Writes the same cells of phi_d as chy_bdygen then chy_pot3 would.  The
 * kernels are launched one after another: replayed as a HIP graph (captured
 * per set of arguments) a solve took 5-8 us longer behind earlier work, for
 * the graph's start and the event that guards its release, and no less
 * alone. */
int chy_solve(chy_grid *g, int maxtrm, int isym, double redge, int npoint, const double *rho_d,
              double *phi_d, double *coef_d, int coef_mode, chy_diag *diag);
/* Enable (default) or disable graph replay of chy_solve_batch on this context. */
int chy_ctx_graphs(chy_ctx *ctx, int enable);

/* ---- batched solves (no reference counterpart: the reference solves one
 * field per call; this serves many independent fields) ----
 * One item per field: chy_solve's arguments.  The items run on the context's
 * worker streams, forked from and joined back to the context's stream, so
 * the call is ordered after earlier work on that stream and later work waits
 * for the whole batch.  Items on one grid object run in order (they share
 * its workspace).  Items on different grid objects prepared from identical
 * descriptions, with the same tunables, maxtrm, isym, redge, npoint and
 * coef_mode, run together, up to 32 per launch of each kernel; other items
 * overlap on the worker streams.  Each item's results are bitwise those of chy_solve on the
 * same arguments.  If any item has a diag pointer the call waits and fills
 * every such diag.  Every item is checked before anything is launched.
 * A batch whose items all run together goes to the context's stream itself.
 * Any other one is captured into one HIP graph (fork, groups, join) the second
 * time it runs (same grids, arrays, arguments, worker count and stream) and
 * replayed as one launch by later calls, unless stage timing is on, graphs are
 * off or the caller is capturing the context's stream; a change to a grid's
 * solver or tuning drops the graphs that use it. */
typedef struct {
    chy_grid *grid;
    const double *rho_d;
    double *phi_d, *coef_d;
    int coef_mode, maxtrm, isym, npoint;
    double redge;
    chy_diag *diag;  /* host, may be NULL */
} chy_solve_item;
#define CHY_MAX_WORKERS 16
int chy_solve_batch(chy_ctx *ctx, const chy_solve_item *items, int n);
/* Number of worker streams chy_solve_batch uses (1..CHY_MAX_WORKERS, default
 * 4).  Streams are made on first use and kept until chy_ctx_destroy; a
 * smaller count leaves the others idle.  Work already issued is not waited
 * for. */
int chy_ctx_workers(chy_ctx *ctx, int n);

/* Host-pointer forms used by the Fortran shims: rho_h/phi_h/coef_h are the
 * COMMON arrays.  They copy to the grid's device buffers, run, copy back and
 * wait.  phi_h is read (boundary values, untouched cells) and written. */
int chy_bdygen_host(chy_grid *g, int maxtrm, int isym, double redge, const double *rho_h,
                    double *phi_h, chy_diag *diag);
int chy_pot3_host(chy_grid *g, int npoint, const double *rho_h, double *phi_h, double *coef_h,
                  int coef_mode, chy_diag *diag);

/* ---- refined solve (no reference counterpart) ----
 * The same results as chy_solve (PHI, COEF, diagnostics) to a stated
 * accuracy: for 2 or more steps within 1e-10 of chy_solve's on evenly spaced
 * columns and of chy_solve's with CHY_MODES_EIGEN on every one.  (Where the z
 * spacing varies BLKTRI's roots, and so CHY_MODES_CR, may be further than that
 * from the exact solution of the mode systems: 1.3e-9 at 64x128x24 with cells
 * growing by 3% a row.)  BDYGEN, COEF, both transforms, POT3's ghost cells and
 * ZAXPHI in binary64 as chy_solve computes them; the mode systems in one of
 * two ways:
 *   - 1 or 2 steps on an evenly spaced column (to 1%) with CHY_MODES_CR,
 *     rel_corr NULL and no one-kernel form in force (CHY_TUNE_REFINE_FUSED): by
 *     that solver's binary64 solves, which are the faster way there and no
 *     further from the exact solution than two steps are;
 *   - otherwise by iterative refinement in the azimuthal spectrum: `steps`
 *     (1..8) mode solves in binary32 (z transforms on the FP32 matrix cores,
 *     r solves in binary32 except the orders m <= CHY_TUNE_REFINE_M64, which
 *     are solved in binary64), the first of the right-hand side, each later
 *     one of the binary64 residual of the mode systems (pot/pot3.f:203-231) at
 *     the binary64 solution so far, rounded to binary32, its solution added
 *     in binary64.  One step puts PHI within ~1e-6 of chy_solve's, two within
 *     ~1e-11 at 256x128x256; three and more reach the exact solution of the
 *     mode systems, as CHY_MODES_EIGEN does (2.4e-12 from CHY_MODES_CR's there).
 * KMAX <= 256 (CHY_EUNSUPPORTED otherwise).  rel_corr (host, may be NULL)
 * receives, per step, the largest correction relative to the largest
 * |solution| after it (1 for the first step).  Waits when diag or rel_corr is
 * non-NULL. */
int chy_solve_refined(chy_grid *g, int maxtrm, int isym, double redge, int npoint, const double *rho_d,
                      double *phi_d, double *coef_d, int coef_mode, int steps, chy_diag *diag,
                      double *rel_corr);
/* chy_solve_batch with every item solved as chy_solve_refined with `steps`
 * correction steps (items grouped and launched together as in
 * chy_solve_batch; each item's results are bitwise those of its own
 * chy_solve_refined, unless CHY_TUNE_REFINE_FUSED says otherwise). */
int chy_solve_batch_refined(chy_ctx *ctx, const chy_solve_item *items, int n, int steps);

/* ---- ZAXPHI alone (pot/pot3.f:311-399) ----
 * The NPOINT-point extrapolation of PHI to the z axis from PHI(J=2..,K,L) and
 * PHI(J=2..,K,L+N): writes PHI(JMAX+2,K,L) and PHI(JMAX+2,K,L+N) for
 * K=2..KMAX+1 and PHAC/PHICHK/KLOCAT as POT3's own call does (POT3 already
 * includes it).  npoint as for chy_pot3; diag as for chy_pot3. */
int chy_zaxphi(chy_grid *g, int npoint, double *phi_d, chy_diag *diag);
int chy_zaxphi_host(chy_grid *g, int npoint, double *phi_h, chy_diag *diag);
/* PHAC(K) for K=2..KMAX+1 (pot3.f:380-387) from the last POT3/ZAXPHI on the
 * grid, n <= KMAX values into phac_h (host); waits for the stream.  For the
 * IPRINT=1 report of pot3.f:402-404. */
int chy_phac(chy_grid *g, double *phac_h, int n);

/* ---- momentum sources that read the potential (radhydro/source.f:41-79) ----
 * The first loop of SOURCE with BINARY=0, which the hydro step runs right
 * after BDYGEN+POT3 (radhydro/3dhyd-main.f:475-477): for K=2..KMAX+1,
 * L=1..LMAX (periodic), S at J=JSTART+1..JMAX+1 and T, A at J=JSTART..JMAX+1
 * get DELT times the centrifugal, gravity (PHI) and pressure terms, in the
 * reference's order of operations (bitwise the reference's results).
 * Device arrays in Fortran order: rho_d, phi_d (POT3JMAX+2, POT3KMAX+2, LMAX)
 * as in /POIS/; omega_d, p_d, s_d, t_d, a_d (JMAX+2, KMAX+2, LMAX) as in /EOM/
 * and /STATES/; r_d is R(1..POT3JMAX+2) of /GRID/.  s_d, t_d and a_d are
 * updated in place; no other cell is written.  Asynchronous on the context's
 * stream.  CHY_EINVAL for null pointers, a hydro grid larger than the
 * potential grid, JSTART outside 2..JMAX+1, or a spacing that is not > 0. */
typedef struct {
    int jmax, kmax, lmax;   /* hydro grid (JMAX, KMAX, LMAX) */
    int pot_jmax, pot_kmax; /* potential grid (POT3JMAX, POT3KMAX) */
    int jstart;             /* max(JMIN, 2) (source.f:31-35) */
    double delt;            /* DELT */
    double dr, dz, dtheta;  /* ROF3N, ZOF3N, DTHETA */
} chy_source_desc;
int chy_source_grav(chy_ctx *ctx, const chy_source_desc *d, const double *r_d, const double *rho_d,
                    const double *omega_d, const double *phi_d, const double *p_d, double *s_d,
                    double *t_d, double *a_d);

/* ---- the central star's potential (pot/ExternalPot.f:1-88) ----
 * ExternalPot as the default build runs it (EXTERNAL_POT=1, INDIRECT=0,
 * BINARY=0), which the hydro step calls after POT3
 * (radhydro/3dhyd-main.f:494-511): with the star at (RPSTAR cos PHI_STAR,
 * RPSTAR sin PHI_STAR), STARPHI(J,K,L) = -(MASS_STAR+TMASSACC)/|x - x*| at
 * (RHF(J), ZHF(K), psi_L = (L-1/2) DTHETA) for J=1..JMAX+2, K=1..KMAX+2,
 * L=1..LMAX, and PHI += STARPHI there (bitwise the reference's arithmetic).
 * phi_d has the potential grid's layout (POT3JMAX+2, POT3KMAX+2, LMAX), starphi_d
 * (/GAP/) the hydro grid's (JMAX+2, KMAX+2, LMAX); rhf_d, zhf_d are RHF, ZHF of
 * /GRID/ (at least JMAX+2 and KMAX+2 values).  The first call for an LMAX and
 * DTHETA builds a small cos/sin table (waits once).  Asynchronous on the
 * context's stream otherwise.  CHY_EINVAL for null pointers, a hydro grid
 * larger than the potential grid, or DTHETA not > 0. */
typedef struct {
    int jmax, kmax, lmax;   /* hydro grid (JMAX, KMAX, LMAX) */
    int pot_jmax, pot_kmax; /* potential grid (POT3JMAX, POT3KMAX) */
    double dtheta;          /* DTHETA */
    double mass_star, tmassacc;
    double rpstar, phi_star; /* the star's position (/movingstar/) */
} chy_extpot_desc;
int chy_external_pot(chy_ctx *ctx, const chy_extpot_desc *d, const double *rhf_d, const double *zhf_d,
                     double *phi_d, double *starphi_d);

/* ---- the disk's pull on the star (pot/wiggle.F:99-135) ----
 * find_force, which wiggle calls every hydro step to move the star: the sum
 * over L=1..LMAX, K=2..KMAX+1, J=JMIN-3..JMAX+1 of the point-mass force of
 * each cell (mass RHO*RHF*DR*DZ*DPHI*2 at (RHF, phi_L = L DPHI - DPHI/2,
 * ZHF), softening GSOFT) on a star at (x, y, 0).  rho_d is read with the
 * leading dimensions (JMAX+2, KMAX+2) find_force declares (wiggle.F:103);
 * rhf_d, zhf_d as for chy_external_pot.  The sum runs in a fixed order (one
 * partial per thread block, added in block order), so results repeat run to
 * run; the reference's OpenMP order differs, so they agree with it to
 * rounding.  Writes (fx, fy) to f_h (host) and waits.  CHY_EINVAL for null
 * pointers, JMIN outside 4..JMAX+1 (find_force reads J=JMIN-3), or
 * spacings not > 0. */
typedef struct {
    int jmax, kmax, lmax, jmin;   /* JMAX, KMAX, LMAX, JMIN */
    double dr, dz, dphi, gsoft;   /* ROF3N, ZOF3N, DTHETA, GSOFT */
} chy_force_desc;
int chy_find_force(chy_ctx *ctx, const chy_force_desc *d, const double *rhf_d, const double *zhf_d,
                   const double *rho_d, double x, double y, double *f_h);

/* find_force without any allocation.  No counterpart in the reference: for
 * callers that cannot allocate device or host memory (code under HIP graph
 * capture, tight serving loops, harnesses that forbid hipMalloc).  The same
 * sum as chy_find_force into f_d (device, 2 doubles: fx, fy), asynchronous on
 * the context's stream (no wait, no host copy).  Its block partials and
 * cos/sin table live in a fixed per-GPU scratch array (1.1 MiB, held until
 * the process ends), so it takes at most 65536 block partials (the partial
 * count is ceil((JMAX-JMIN+5)*KMAX/256) * ceil(LMAX/16)) and LMAX <= 4096,
 * else CHY_ELIMIT.  The cos/sin table is computed on the GPU, so results agree
 * with chy_find_force's to rounding, not bit for bit.  Every call on one GPU
 * shares that scratch: calls that overlap on one GPU (other streams, other
 * contexts, other threads) race. */
int chy_find_force_noalloc(chy_ctx *ctx, const chy_force_desc *d, const double *rhf_d, const double *zhf_d,
                           const double *rho_d, double x, double y, double *f_d);

/* ---- stage timing (no reference counterpart; for benchmarks) ----
 * While enabled, every stage of chy_bdygen/chy_pot3/chy_solve is bracketed by
 * HIP events on the context's stream.  chy_ctx_stage_times() waits for the
 * stream and returns, per stage, the summed milliseconds and the number of
 * launches since profiling was (re)enabled. */
enum {
    CHY_STAGE_BDYGEN = 0, /* radial split sums, boundary evaluation, ghosts */
    CHY_STAGE_FFT_FWD,    /* forward azimuthal RFFT (+ COEF, + BDYGEN ring moments) */
    CHY_STAGE_ZFWD,       /* mode right-hand sides -> z eigen coordinates (refined: every step's) */
    CHY_STAGE_RSOLVE,     /* r-tridiagonal solves (refined: every step's) */
    CHY_STAGE_ZINV,       /* z eigen coordinates -> mode solutions (refined: every step's) */
    CHY_STAGE_FFT_INV,    /* inverse azimuthal RFFT */
    CHY_STAGE_GHOST,      /* ghosts, ZAXPHI, PHICHK */
    CHY_STAGE_FFT_BDY,    /* forward RFFT of the boundary lanes (chy_solve) */
    CHY_STAGE_CR,         /* per-mode cyclic reduction (CHY_MODES_CR) */
    CHY_STAGE_RESID,      /* refined solves: the mode systems' residual in the spectrum */
    CHY_STAGE_PLANES,     /* refined solves: every step's mode work, one kernel per mode plane */
    CHY_NSTAGES
};
int chy_ctx_profile(chy_ctx *ctx, int enable);
int chy_ctx_stage_times(chy_ctx *ctx, double *ms, int *counts, int n);

const char *chy_strerror(int code);
/* Last HIP error text seen by the library (for CHY_EDEVICE). */
const char *chy_last_device_error(void);

#ifdef __cplusplus
}
#endif

#endif /* CHYPOT_H */
