"""The work a user of the potential solve has it do, as measurable cases.

Sizes are those of this repository's tests, tuning table and benchmark: the
64x32x64 torus, the 256x128x256 spiral torus alone and in batches, the serving
mix's 512x256x512 grid, the heterogeneous batch over J in {64,128,256},
K in {32,64,128}, L in {64,128,256}, mixed-radix LMAX and ragged JMAX, and the
hydro step's other gravity calls (SOURCE, ExternalPot, find_force).  Densities
are polytropic tori with logarithmic spiral arms and log-normal noise over a
thin noisy floor, generated on the GPU from the seed alone.

A case is a dict of plain values: `kind` (solve, refined, calls, mix, source,
star), `jmax`, `kmax`, `lmax`, and per kind `fields` (independent fields of one
call), `coef` (what COEF output covers), `redge`, `modes`.
"""
import functools
import math
import pathlib
import random
import sys

import numpy as np
import torch

_PKG = str(pathlib.Path(__file__).resolve().parents[1] / "chymera-uo_amd")
if _PKG not in sys.path:
    sys.path.insert(0, _PKG)

import chypot  # noqa: E402
from chypot import fields as grids  # noqa: E402

F64 = torch.float64
COEF = {"none": chypot.COEF_NONE, "k2": chypot.COEF_K2, "full": chypot.COEF_FULL}
STEPS = 2       # correction steps of a refined solve
NPOINT = 8      # POT3(8, ..), as the hydro step calls it
MAXTRM = 10


def listed():
    return [
        # the CPU-runnable grid, one field: a small run's solve, the shortest call of the range
        _solve("solve_64x32x64", "solve", 64, 32, 64, coef="k2"),
        # the reference's production grid, one field per hydro step (COEF's K=2 plane is what the hydro loop reads)
        _solve("solve_256x128x256", "solve", 256, 128, 256, coef="k2"),
        # many independent fields of that grid in one call: parameter studies, served batches
        _solve("solve_256x128x256_x32", "solve", 256, 128, 256, fields=32),
        # the serving mix's largest grid by the reference's own reduction
        _solve("solve_512x256x512", "solve", 512, 256, 512),
        # SETBDY's two calls as the Fortran caller makes them, COEF written whole by none, REDGE at
        # the grid's edge, a ragged JMAX and a mixed-radix LMAX
        _solve("calls_200x64x192", "calls", 200, 64, 192, redge=0.9),
        # a grid past the cyclic reduction's JMAX: the z eigenbasis (the default there)
        _solve("solve_1000x32x96", "solve", 1000, 32, 96),
        # the refined solve of one field and of a batch
        _solve("refined_256x128x256", "refined", 256, 128, 256, coef="k2"),
        _solve("refined_256x128x256_x32", "refined", 256, 128, 256, fields=32, coef="k2"),
        # the serving mix's largest grid, refined
        _solve("refined_512x256x512", "refined", 512, 256, 512),
        # fields of uneven grids in one call
        {"name": "refined_mix_x16", "kind": "mix", "fields": 16, "mix": 7},
        # the hydro step after the solve: the momentum sources that read PHI
        {"name": "source_256x128x256", "kind": "source", "jmax": 256, "kmax": 128, "lmax": 256},
        # the star: its pull from the disk (waits for the two numbers), then its potential
        {"name": "star_256x128x256", "kind": "star", "jmax": 256, "kmax": 128, "lmax": 256},
    ]


def _solve(name, kind, jmax, kmax, lmax, fields=1, coef="none", redge=0.0, modes="default"):
    return {"name": name, "kind": kind, "jmax": jmax, "kmax": kmax, "lmax": lmax, "fields": fields, "coef": coef,
            "redge": redge, "modes": modes}


def _smooth_l(lo, hi):
    """Even LMAX in [lo, hi] whose half has prime factors up to 23 (the transforms' sizes)."""
    out = []
    for l in range(lo + lo % 2, hi + 1, 2):
        n = l // 2
        for p in (2, 3, 5, 7, 11, 13, 17, 19, 23):
            while n % p == 0:
                n //= p
        if n == 1:
            out.append(l)
    return out


def draw(rng):
    """One more case of the listed ones' ranges."""
    kind = rng.choice(["solve", "solve", "solve", "refined", "refined", "refined", "calls", "mix", "source", "star"])
    if kind == "mix":
        return {"kind": "mix", "fields": rng.randint(3, 24), "mix": rng.randrange(1 << 20)}
    jmax = int(round(math.exp(rng.uniform(math.log(24), math.log(512)))))
    if kind in ("source", "star"):
        kmax = int(round(math.exp(rng.uniform(math.log(16), math.log(160)))))
        lmax = 2 * int(round(math.exp(rng.uniform(math.log(16), math.log(160)))))
        return {"kind": kind, "jmax": jmax, "kmax": kmax, "lmax": lmax}
    kmax = 1 << rng.randint(3, 8)
    if rng.random() < 0.5:
        lmax = 1 << rng.randint(5, 9)
    else:
        choices = _smooth_l(24, 512)
        want = math.exp(rng.uniform(math.log(24), math.log(512)))
        lmax = min(choices, key=lambda l: abs(l - want))
    # a call of several fields stays below the largest listed batch
    most = max(1, min(32, int(24 * 256 * 128 * 256 / (jmax * kmax * lmax))))
    nf = 1 if kind == "calls" or rng.random() < 0.5 else int(round(math.exp(rng.uniform(0.0, math.log(most)))))
    case = _solve("", kind, jmax, kmax, lmax, fields=nf, coef=rng.choice(["none", "k2", "full"]),
                  redge=rng.choice([0.0, 0.0, round(rng.uniform(0.7, 1.1), 3)]),
                  modes="eigen" if kind != "refined" and rng.random() < 0.25 else "default")
    if kind == "calls":
        case["coef"] = "none"
    del case["name"]
    return case


# ---- inputs -----------------------------------------------------------------

def _device():
    return torch.device("cuda" if torch.cuda.is_available() else "cpu")


@functools.lru_cache(maxsize=None)
def _context():
    return chypot.Context(0)


def _shapes(case):
    """[(jmax, kmax, lmax)] of the case's fields."""
    if case["kind"] == "mix":
        rng = random.Random(case["mix"])
        return [(rng.choice((64, 128, 256)), rng.choice((32, 64, 128)), rng.choice((64, 128, 256)))
                for _ in range(case["fields"])]
    return [(case["jmax"], case["kmax"], case["lmax"])] * case.get("fields", 1)


def _density(g, rng, gen, out=None):
    """A torus with spiral arms and noise over a thin noisy floor, (LMAX, KMAX+2, JMAX+2)."""
    dev = _device()
    rc, a, n = rng.uniform(0.35, 0.6), rng.uniform(0.2, 0.35), rng.choice((1.0, 1.5, 2.5))
    turn = rng.uniform(0.0, 2.0 * math.pi)
    r = torch.tensor(g.rhf(), dtype=F64, device=dev)
    z = torch.tensor(g.zhf(), dtype=F64, device=dev)[:, None]
    psi = torch.tensor(g.psi(), dtype=F64, device=dev)[:, None, None]
    base = torch.clamp(1.0 - ((r - rc) ** 2 + z ** 2) / (a * a), min=0.0) ** n
    wind = torch.log(r.abs() / 0.5) / math.tan(math.radians(15.0)) + turn
    arms = 1.0 + 0.1 * sum(torch.cos(m * (psi - wind)) for m in (2, 3, 4))
    f = torch.clamp(base * arms, min=grids.GRIDLIM)
    f *= torch.exp(0.05 * torch.randn(f.shape, generator=gen, dtype=F64, device=dev))
    out = torch.zeros_like(f) if out is None else out
    out[:, 1:g.kmax + 1, 1:g.jmax + 1] = f[:, 1:g.kmax + 1, 1:g.jmax + 1]
    return out


def _seeded(seed):
    gen = torch.Generator(device=_device())
    gen.manual_seed(int(seed))
    return random.Random(int(seed)), gen


def _densities(case, seed):
    """The case's grids and densities; fields of one shape lie in one tensor."""
    rng, gen = _seeded(seed)
    shapes = _shapes(case)
    gs = [grids.unit_grid(*s) for s in shapes]
    if case["kind"] == "mix":
        return gs, [_density(g, rng, gen) for g in gs]
    g = gs[0]
    rho = torch.zeros((len(gs), g.lmax, g.kmax + 2, g.jmax + 2), dtype=F64, device=_device())
    for f in range(len(gs)):
        _density(g, rng, gen, rho[f])
    return gs, rho


def _hydro(case, seed):
    """The hydro step's arrays on one grid: density, potential, pressure, rotation, momenta and the star."""
    rng, gen = _seeded(seed)
    g = grids.unit_grid(case["jmax"], case["kmax"], case["lmax"])
    shape, dev = (g.lmax, g.kmax + 2, g.jmax + 2), _device()
    rho = _density(g, rng, gen)
    r = torch.tensor(g.rhf(), dtype=F64, device=dev).abs()
    z = torch.tensor(g.zhf(), dtype=F64, device=dev)[:, None]

    def noise(scale):
        return 1.0 + scale * torch.randn(shape, generator=gen, dtype=F64, device=dev)

    well = -1.0 / torch.sqrt(r * r + z * z + 0.01)
    return dict(g=g, rho=rho, phi=well * noise(1e-3), p=0.05 * rho.abs() ** (5.0 / 3.0) + 1e-8 * noise(0.1),
                omega=(r + 0.05) ** -1.5 * noise(0.01), s=0.01 * (noise(1.0) - 1.0), t=0.01 * (noise(1.0) - 1.0),
                a=rho * torch.sqrt(r) * noise(0.01), delt=rng.uniform(1e-4, 1e-3),
                mass=rng.uniform(0.5, 2.0), acc=rng.uniform(0.0, 0.01), rp=rng.uniform(0.0, 0.02),
                ang=rng.uniform(0.0, 2.0 * math.pi), x=rng.uniform(-0.01, 0.01), y=rng.uniform(-0.01, 0.01))


def prepare(case, seed):
    ctx = _context()
    kind = case["kind"]
    if kind in ("source", "star"):
        h = _hydro(case, seed)
        g, dev = h["g"], _device()
        h["r"] = torch.tensor(g.r(), dtype=F64, device=dev)
        h["rhf"] = torch.tensor(g.rhf(), dtype=F64, device=dev)
        h["zhf"] = torch.tensor(g.zhf(), dtype=F64, device=dev)
        h["starphi"] = torch.zeros_like(h["phi"])
        h["source"] = chypot.SourceDesc(g.jmax, g.kmax, g.lmax, g.jmax, g.kmax, 2, h["delt"], g.delr, g.delz, g.dtheta)
        h["extpot"] = chypot.ExtPotDesc(g.jmax, g.kmax, g.lmax, g.jmax, g.kmax, g.dtheta, h["mass"], h["acc"], h["rp"],
                                        h["ang"])
        h["force"] = chypot.ForceDesc(g.jmax, g.kmax, g.lmax, 4, g.delr, g.delz, g.dtheta, 0.01)
        return dict(kind=kind, ctx=ctx, h=h)
    gs, rho = _densities(case, seed)
    pgs = [chypot.PreparedGrid(ctx, g) for g in gs]
    if case.get("modes") == "eigen":
        for pg in pgs:
            pg.mode_solver = chypot.MODES_EIGEN
    mode = COEF[case.get("coef", "none")]
    if kind == "mix":
        phi, coef = [torch.zeros_like(x) for x in rho], None
    else:
        phi = torch.zeros_like(rho)
        coef = torch.zeros((len(gs),) + pgs[0].coef_shape, dtype=F64, device=rho.device) if mode else None
    jobs = [dict(grid=pg, rho=rho[f], phi=phi[f], coef=coef[f] if coef is not None else None, coef_mode=mode,
                 maxtrm=MAXTRM, npoint=NPOINT, redge=case.get("redge", 0.0)) for f, pg in enumerate(pgs)]
    return dict(kind=kind, ctx=ctx, jobs=jobs, phi=phi, coef=coef)


def run(state):
    kind, ctx = state["kind"], state["ctx"]
    if kind == "source":
        h = state["h"]
        ctx.source_grav(h["source"], h["r"], h["rho"], h["omega"], h["phi"], h["p"], h["s"], h["t"], h["a"])
        return {"s": h["s"], "t": h["t"], "a": h["a"]}
    if kind == "star":
        h = state["h"]
        pull = ctx.find_force(h["force"], h["rhf"], h["zhf"], h["rho"], h["x"], h["y"])
        ctx.external_pot(h["extpot"], h["rhf"], h["zhf"], h["phi"], h["starphi"])
        return {"pull": list(pull), "phi": h["phi"], "starphi": h["starphi"]}
    jobs = state["jobs"]
    if kind == "calls":
        for j in jobs:
            j["grid"].bdygen(j["rho"], j["phi"], maxtrm=j["maxtrm"], redge=j["redge"])
            j["grid"].pot3(j["rho"], j["phi"], npoint=j["npoint"], coef=j["coef"], coef_mode=j["coef_mode"])
    elif len(jobs) > 1:
        ctx.solve_batch(jobs, refine_steps=0 if kind == "solve" else STEPS)
    else:
        j = jobs[0]
        more = {} if kind == "solve" else {"steps": STEPS}
        call = j["grid"].solve if kind == "solve" else j["grid"].solve_refined
        call(j["rho"], j["phi"], maxtrm=j["maxtrm"], npoint=j["npoint"], coef=j["coef"], coef_mode=j["coef_mode"],
             redge=j["redge"], **more)
    out = {"phi": state["phi"]}
    if state["coef"] is not None:
        out["coef"] = state["coef"]
    return out


def work(case):
    """Each field's density read and potential written once (and COEF where it is asked for); the two real
    transforms along L and a fast direct solver's operations along z and r."""
    if case["kind"] in ("source", "star"):
        cells = case["jmax"] * case["kmax"] * case["lmax"]
        if case["kind"] == "source":
            return {"bytes": 80.0 * cells, "flops": 45.0 * cells}
        return {"bytes": 32.0 * cells, "flops": 45.0 * cells}
    nbytes = flops = 0.0
    for j, k, l in _shapes(case):
        cells = float(j * k * l)
        coef = {"none": 0.0, "k2": 8.0 * j * l, "full": 8.0 * cells}[case.get("coef", "none")]
        nbytes += 16.0 * cells + coef
        flops += cells * (2 * 2.5 * math.log2(l) + 10.0 * math.log2(k) + 10.0)
    return {"bytes": nbytes, "flops": flops}


# ---- 64-bit values ----------------------------------------------------------

def exact(case, seed):
    if case["kind"] == "source":
        return _exact_source(case, seed)
    if case["kind"] == "star":
        return _exact_star(case, seed)
    gs, rho = _densities(case, seed)
    phis, coefs = [], []
    for g, x in zip(gs, rho):
        phi, coef = _exact_solve(g, x, case.get("redge", 0.0), case.get("coef", "none"))
        phis.append(phi)
        coefs.append(coef)
    out = {"phi": phis if case["kind"] == "mix" else torch.stack(phis)}
    if coefs[0] is not None:
        out["coef"] = torch.stack(coefs)
    return out


def _legendre(l, m, c, s):
    """Associated Legendre P_l^m without the Condon-Shortley sign, by the upward recurrence in l."""
    p = np.ones_like(c)
    for i in range(1, m + 1):
        p = p * (2 * i - 1) * s
    if l == m:
        return p
    q = c * (2 * m + 1) * p
    for n in range(m + 2, l + 1):
        p, q = q, ((2 * n - 1) * c * q - (n + m - 1) * p) / (n - m)
    return q


def _boundary_spectrum(g, rho, redge):
    """Packed azimuthal coefficients [LMAX][JMAX+KMAX-1] of BDYGEN's potential on the top row (J=2..JMAX+1) and the
    outer column (K=2..KMAX): multipoles l <= 10, l+m even, of the rings J=2..JMAX, K=2..KMAX."""
    dev, L, N = rho.device, g.lmax, g.lmax // 2
    rhf, zhf, r, z = g.rhf(), g.zhf(), g.r(), g.z()
    rr, zz = np.meshgrid(rhf[1:g.jmax], zhf[1:g.kmax])
    dv = g.dtheta * np.diff(z)[1:g.kmax][:, None] * (np.diff(r ** 2)[1:g.jmax])[None, :]
    rs = np.sqrt(rr * rr + zz * zz).ravel()
    c, s = zz.ravel() / rs, rr.ravel() / rs
    x = rho[:, 1:g.kmax, 1:g.jmax].reshape(L, -1)
    if redge > 0.0:
        x = x * torch.tensor(rs <= redge, dtype=F64, device=dev)
    rb = np.concatenate([rhf[1:g.jmax + 1], np.full(g.kmax - 1, rhf[g.jmax])])
    zb = np.concatenate([np.full(g.jmax, zhf[g.kmax]), zhf[1:g.kmax]])
    rsb = np.sqrt(rb * rb + zb * zb)
    cb, sb = zb / rsb, rb / rsb
    T = functools.partial(torch.tensor, dtype=F64, device=dev)
    order = np.argsort(rs, kind="stable")
    cut = torch.tensor(np.searchsorted(rs[order], rsb, side="right"), device=dev)
    order_d = torch.tensor(order, device=dev)
    psi = T(g.psi())
    spec = torch.zeros((L, rb.size), dtype=F64, device=dev)
    for m in range(MAXTRM + 1):
        if m >= N:
            break
        cm = ((torch.cos(m * psi) @ x) * T(dv.ravel()))[order_d]
        sm = ((torch.sin(m * psi) @ x) * T(dv.ravel()))[order_d]
        C = torch.zeros(rb.size, dtype=F64, device=dev)
        S = torch.zeros_like(C)
        for l in range(m, MAXTRM + 1, 2):
            w = (1.0 if m == 0 else 2.0) * math.factorial(l - m) / math.factorial(l + m)
            p = _legendre(l, m, c, s)
            tin, tout = T((p * rs ** l)[order]), T((p * rs ** -(l + 1))[order])
            pb = w * _legendre(l, m, cb, sb)
            for v, acc in ((cm, C), (sm, S)):
                inside = torch.cat([T([0.0]), torch.cumsum(tin * v, 0)])
                outside = torch.cat([torch.flip(torch.cumsum(torch.flip(tout * v, [0]), 0), [0]), T([0.0])])
                acc += T(pb * rsb ** -(l + 1)) * inside[cut] + T(pb * rsb ** l) * outside[cut]
        # the series in psi_n = (n + 1/2) DTHETA as packed coefficients in n DTHETA
        h = 0.5 * m * g.dtheta
        if m == 0:
            spec[0] = -2.0 * C
        else:
            spec[m] = -(C * math.cos(h) + S * math.sin(h))
            spec[N + m] = -(-C * math.sin(h) + S * math.cos(h))
    return spec


def _exact_solve(g, rho, redge, coef_kind):
    """BDYGEN and POT3 of one field by torch's FFT, the z operator's eigenvectors and elimination along r."""
    J, K, L, N = g.jmax, g.kmax, g.lmax, g.lmax // 2
    dev = rho.device
    T = functools.partial(torch.tensor, dtype=F64, device=dev)
    M, NZ = J - 1, K - 1
    # interior lanes' packed coefficients a_0..a_N, b_1..b_{N-1}
    X = torch.fft.rfft(rho[:, 1:K + 1, 1:J + 1], dim=0).conj()
    spec = torch.zeros((L, K, J), dtype=F64, device=dev)
    spec[:N + 1] = X.real * (2.0 / L)
    spec[N + 1:] = X.imag[1:N] * (2.0 / L)
    del X
    b = _boundary_spectrum(g, rho, redge)
    spec[:, K - 1, :] = b[:, :J]
    spec[:, :K - 1, J - 1] = b[:, J:]
    coef = None
    if coef_kind != "none":
        coef = torch.zeros((2, N, K + 2, J + 2), dtype=F64, device=dev)
        ks = slice(0, 1) if coef_kind == "k2" else slice(0, K)
        a0 = spec[0, ks] * L
        at = coef[:, :, 1:2, 1:J + 1] if coef_kind == "k2" else coef[:, :, 1:K + 1, 1:J + 1]
        A, B = spec[1:N, ks] * L, spec[N + 1:, ks] * L
        at[0, :N - 1] = 2.0 * torch.sqrt(A * A + B * B) / a0.abs()
        ph = torch.where(A != 0.0, torch.atan(B / A) + (A < 0.0).to(F64) * math.pi, torch.sign(B) * (0.5 * math.pi))
        at[1, :N - 1] = torch.where((A == 0.0) & (B == 0.0), T(720.0), ph * 180.0 / math.pi)
        at[0, N - 1] = (spec[N, ks] * L).abs() / a0.abs()
        at[1, N - 1] = a0
        del A, B, ph
    # the 7-point operator's coefficients (cell centres rhf, zhf)
    rhf, zhf = g.rhf(), g.zhf()
    rd, rm = rhf[1:J + 1], 0.5 / rhf[1:J]
    up, dn = 1.0 / (rhf[2:J + 1] - rhf[1:J]), 1.0 / (rhf[1:J] - rhf[0:J - 1])
    den = 1.0 / (rhf[2:J + 1] - rhf[0:J - 1])
    cm, am = 2.0 * (up + rm) * den, 2.0 * (dn - rm) * den
    am[0] = 2.0 * (0.5 / rhf[1] - rm[0]) * den[0]
    cz = 2.0 / (zhf[2:K + 1] - zhf[1:K]) / (zhf[2:K + 1] - zhf[0:K - 1])
    az = 2.0 / (zhf[1:K] - zhf[0:K - 1]) / (zhf[2:K + 1] - zhf[0:K - 1])
    az[0] = 0.5 / zhf[1] * 2.0 / (zhf[2] - zhf[0])
    bz = -cz - az
    bz[0] = -cz[0]
    m = np.concatenate([np.arange(N + 1), np.arange(1, N)])
    bm = np.tile(-cm - am, (N + 1, 1))
    bm += 2.0 * (np.cos(np.arange(N + 1) * g.dtheta) - 1.0)[:, None] / (rd[None, :M] * g.dtheta) ** 2
    bm[:, 0] = (-cm[0] + ((-1.0) ** np.arange(N + 1) - 1.0) * am[0]
                + 2.0 * (np.cos(np.arange(N + 1) * g.dtheta) - 1.0) / (rd[0] * g.dtheta) ** 2)
    # right-hand side with the boundary values moved to it
    Y = spec[:, :NZ, :M] * (4.0 * math.pi)
    Y[:, NZ - 1, :] -= cz[-1] * spec[:, K - 1, :M]
    Y[:, :, M - 1] -= cm[-1] * spec[:, :NZ, J - 1]
    # z eigenvectors of the symmetrised operator
    e = np.sqrt(az[1:] * cz[:-1])
    d = np.concatenate([[1.0], np.cumprod(np.sqrt(cz[:-1] / az[1:]))])
    lam, Q = np.linalg.eigh(np.diag(bz) + np.diag(e, 1) + np.diag(e, -1))
    Wf, Wi = T((Q * d[:, None]).T), T(Q / d[:, None])
    Z = torch.matmul(Wf, Y)                      # [L][p][j]
    del Y
    Z = Z.permute(2, 0, 1).contiguous()          # [j][L][p]
    bmt = T(bm[m].T)[:, :, None] + T(lam)        # [j][L][p]
    amd, cmd = am.tolist(), cm.tolist()
    inv = torch.empty_like(bmt)
    inv[0] = 1.0 / bmt[0]
    Z[0] *= inv[0]
    for j in range(1, M):
        inv[j] = 1.0 / (bmt[j] - amd[j] * cmd[j - 1] * inv[j - 1])
        Z[j] = (Z[j] - amd[j] * Z[j - 1]) * inv[j]
    for j in range(M - 2, -1, -1):
        Z[j] -= cmd[j] * inv[j] * Z[j + 1]
    del bmt, inv
    spec[:, :NZ, :M] = torch.matmul(Wi, Z.permute(1, 2, 0).contiguous())
    del Z
    # back to physical space, POT3's ghost cells, the axis values by extrapolation
    H = torch.zeros((N + 1, K, J), dtype=torch.complex128, device=dev)
    H.real[:] = spec[:N + 1] * (0.5 * L)
    H.imag[1:N] = -spec[N + 1:] * (0.5 * L)
    phi = torch.zeros((L, K + 2, J + 2), dtype=F64, device=dev)
    phi[:, 1:K + 1, 1:J + 1] = torch.fft.irfft(H, n=L, dim=0)
    phi[:, 0, 1:J + 1] = phi[:, 1, 1:J + 1]
    phi[:, :K + 1, 0] = torch.roll(phi[:, :K + 1, 1], N, 0)
    half = NPOINT // 2
    x = np.concatenate([rhf[1:half + 1], -rhf[1:half + 1]])
    w = [np.prod([-x[j] / (x[i] - x[j]) for j in range(NPOINT) if j != i]) for i in range(NPOINT)]
    near, far = phi[:N, 1:K + 1, 1:half + 1], phi[N:, 1:K + 1, 1:half + 1]
    axis = near @ T(w[:half]) + far @ T(w[half:])
    phi[:N, 1:K + 1, J + 1] = axis
    phi[N:, 1:K + 1, J + 1] = axis
    return phi, coef


def _exact_source(case, seed):
    h = _hydro(case, seed)
    g = h["g"]
    J, K, dt = g.jmax, g.kmax, h["delt"]
    r = torch.tensor(g.r(), dtype=F64, device=h["rho"].device)
    rho, phi, p, om = h["rho"], h["phi"], h["p"], h["omega"]
    s, t, a = h["s"].clone(), h["t"].clone(), h["a"].clone()
    k = slice(1, K + 1)
    j, i = slice(2, J + 1), slice(1, J)          # J = 3..JMAX+1 and its inner neighbour
    rs = rho[:, k, j] + rho[:, k, i]
    s[:, k, j] += dt * (r[2:J + 1] * rs * (om[:, k, j] + om[:, k, i]) ** 2 / 8.0
                        - rs * (phi[:, k, j] - phi[:, k, i]) / (2.0 * g.delr) - (p[:, k, j] - p[:, k, i]) / g.delr)
    j, q = slice(1, J + 1), slice(0, K)          # J = 2..JMAX+1; K-1
    t[:, k, j] -= dt * (0.5 * (rho[:, k, j] + rho[:, q, j]) * (phi[:, k, j] - phi[:, q, j])
                        + p[:, k, j] - p[:, q, j]) / g.delz
    dphi = torch.roll(phi, -1, 0) - torch.roll(phi, 1, 0)
    dp = torch.roll(p, -1, 0) - torch.roll(p, 1, 0)
    a[:, k, j] -= dt * (rho[:, k, j] * dphi[:, k, j] + dp[:, k, j]) / (2.0 * g.dtheta)
    return {"s": s, "t": t, "a": a}


def _exact_star(case, seed):
    h = _hydro(case, seed)
    g, dev = h["g"], h["rho"].device
    T = functools.partial(torch.tensor, dtype=F64, device=dev)
    r, z, psi = T(g.rhf()), T(g.zhf())[:, None], T(g.psi())[:, None, None]
    sx, sy = h["rp"] * math.cos(h["ang"]), h["rp"] * math.sin(h["ang"])
    star = -(h["mass"] + h["acc"]) / torch.sqrt(
        r * r + z * z + sx * sx + sy * sy - 2.0 * r * (torch.cos(psi) * sx + torch.sin(psi) * sy))
    xx, yy = r * torch.cos(psi) - h["x"], r * torch.sin(psi) - h["y"]
    f = h["rho"] * r * (2.0 * g.delr * g.delz * g.dtheta) / torch.sqrt(xx * xx + yy * yy + z * z + 0.01 ** 2) ** 3
    c = (slice(None), slice(1, g.kmax + 1), slice(0, g.jmax + 1))   # K = 2..KMAX+1, J = 1..JMAX+1
    return {"pull": [float((f * xx)[c].sum()), float((f * yy)[c].sum())], "phi": h["phi"] + star, "starphi": star}
