"""The mode solves' tree (leaves of up to 15 z rows, nodes with BLKTRI's roots)
at the edges of its shapes: one to several levels above the leaves (KMAX 4 to
64, leaves of 1, 3, 7 and 15 rows), r systems that fill their lanes exactly,
leave one row over or nearly all rows empty (JMAX-1 = 4 .. 512 on 8, 16, 32
and 64 lanes), both lane shapes, and the orders m = 0 and m = LMAX/2 that have
no sine part (LMAX = 4).  Against the oracle's POT3 by BLKTRI's reduction:
both sum the same roots, with roundings that grow with the r operator's
condition, up to 7e-13 at JMAX 512 with KMAX 64 on the unit grid; 1e-12 as for
every grid shape."""
import pytest

import chypot
from chypot import fields
from helpers import rel_max

pytestmark = pytest.mark.gpu

torch = pytest.importorskip("torch")

SHAPES = [(5, 4, 4), (9, 8, 6), (65, 16, 4), (64, 32, 8), (66, 64, 4), (128, 4, 8), (129, 32, 4), (130, 8, 10),
          (257, 16, 4), (250, 64, 6), (256, 4, 4), (258, 8, 4), (513, 32, 4), (400, 16, 6)]


# columns of up to 511 rows (nodes with far fewer roots than rows), cells up to
# 16 times flatter than wide and the reverse
TALL = [(17, 512, 4), (33, 256, 6), (65, 512, 4), (200, 128, 8), (513, 128, 4)]


@pytest.mark.parametrize("lanes", [64, 32])
@pytest.mark.parametrize("jkl", SHAPES + TALL)
def test_tree_against_oracle(jkl, lanes):
    import pyoracle as po
    if not torch.cuda.is_available():
        pytest.skip("no HIP device")
    g = fields.unit_grid(*jkl)
    rho = fields.density_spiral_torus(g, seed=6)
    print(f"[gpu] tree {g.name} lanes {lanes}", flush=True)
    ctx = chypot.Context(0)
    pg = chypot.PreparedGrid(ctx, g)
    if lanes == 32 and g.jmax - 1 > 256:
        with pytest.raises(chypot.ChyError):
            pg.cr_lanes = 32
        return
    pg.cr_lanes = lanes
    rho_d = chypot.to_device(rho)
    phi_d = torch.zeros_like(rho_d)
    pg.solve(rho_d, phi_d, npoint=4)
    ctx.sync()
    phi = chypot.to_host(phi_d)
    pg.close()
    po.use_cyclic_reduction(True)
    try:
        want = po.solve(g, rho, npoint=4)
    finally:
        po.use_cyclic_reduction(False)
    assert rel_max(phi, want["phi"]) < 1e-12


@pytest.mark.parametrize("jkl", [(5, 4, 4), (64, 32, 24), (130, 64, 40), (257, 16, 32), (300, 8, 24)])
def test_refined_by_the_tree(jkl):
    """A refined solve that reports no corrections takes the plain solve's mode
    solves: bit for bit chy_solve's PHI, one step or two, LMAX/2 below and
    above MAXTRM (boundary values through PHI or in the spectrum); one that
    reports them still refines in binary32, within 1e-10."""
    if not torch.cuda.is_available():
        pytest.skip("no HIP device")
    g = fields.unit_grid(*jkl)
    print(f"[gpu] refined by the tree {g.name}", flush=True)
    ctx = chypot.Context(0)
    pg = chypot.PreparedGrid(ctx, g)
    rho = chypot.to_device(fields.density_spiral_torus(g, seed=8))
    plain = torch.zeros_like(rho)
    pg.solve(rho, plain, npoint=4)
    for steps in (1, 2):
        phi = torch.zeros_like(rho)
        pg.solve_refined(rho, phi, steps=steps, npoint=4)
        ctx.sync()
        assert torch.equal(phi, plain)
    phi = torch.zeros_like(rho)
    _, rel = pg.solve_refined(rho, phi, steps=2, npoint=4, report=True)
    assert 0.0 < rel[1] < 1e-5
    assert float((phi - plain).abs().max()) < 1e-10 * float(plain.abs().max())
    pg.close()


def test_refined_group_of_unlike_tunings():
    """Fields of one group on grid objects with and without the one-kernel form
    (whose buffers only some objects would have asked for by themselves)."""
    if not torch.cuda.is_available():
        pytest.skip("no HIP device")
    g = fields.unit_grid(64, 32, 64)
    print("[gpu] refined group of unlike tunings", flush=True)
    ctx = chypot.Context(0)
    for first in (0, 1):
        jobs = []
        for i in range(3):
            pg = chypot.PreparedGrid(ctx, g)
            pg.refine_fused = 32 if i == first else 0
            rho = chypot.to_device(fields.density_spiral_torus(g, seed=20 + i))
            jobs.append(dict(grid=pg, rho=rho, phi=torch.zeros_like(rho)))
        ctx.solve_batch(jobs, refine_steps=2)
        ctx.sync()
        for j in jobs:
            plain = torch.zeros_like(j["rho"])
            j["grid"].solve(j["rho"], plain)
            ctx.sync()
            assert float((j["phi"] - plain).abs().max()) < 1e-10 * float(plain.abs().max())
            j["grid"].close()


@pytest.mark.parametrize("lanes", [64, 32])
@pytest.mark.parametrize("jkl", [(64, 32, 8), (250, 8, 6), (257, 16, 4), (513, 4, 4)])
@pytest.mark.parametrize("bad", [float("nan"), float("inf")])
def test_tree_spreads_what_is_not_finite(jkl, lanes, bad):
    """One density value that is not finite leaves no finite PHI, as it does
    through the reference's sweeps, also on flat grids, where the reduction
    along r ends early for finite right-hand sides."""
    if not torch.cuda.is_available():
        pytest.skip("no HIP device")
    if lanes == 32 and jkl[0] - 1 > 256:
        pytest.skip("64 lanes only")
    g = fields.unit_grid(*jkl)
    print(f"[gpu] tree not finite {g.name} lanes {lanes}", flush=True)
    ctx = chypot.Context(0)
    pg = chypot.PreparedGrid(ctx, g)
    pg.cr_lanes = lanes
    rho = chypot.to_device(fields.density_spiral_torus(g, seed=6))
    phi = torch.zeros_like(rho)
    pg.solve(rho, phi, npoint=4)
    rho[0, 1, g.jmax // 2] = bad
    pg.pot3(rho, phi, npoint=4)
    ctx.sync()
    inner = phi[:, 1:g.kmax, 1:g.jmax]
    assert not bool(torch.isfinite(inner).any())
    pg.close()
