"""Which mode solves a refined solve takes (csrc/api.cpp refine_by_tree): the
binary64 tree where its result is no further from the exact solution of the
mode systems than the refinement's, else the refinement, whose arithmetic does
not depend on whether the per-step corrections are asked for."""
import pytest

import chypot
from chypot import fields
from helpers import rel_max
from test_gpu_cr_columns import Column, heights

pytestmark = pytest.mark.gpu

torch = pytest.importorskip("torch")


@pytest.fixture(scope="module")
def ctx():
    if not torch.cuda.is_available():
        pytest.skip("no HIP device")
    return chypot.Context(0)


def _refined(ctx, pg, rho, steps, report):
    phi = torch.zeros_like(rho)
    pg.solve_refined(rho, phi, steps=steps, npoint=4, report=report)
    ctx.sync()
    return phi


@pytest.mark.parametrize("steps", [3, 4, 8])
@pytest.mark.parametrize("jkl", [(16, 4, 4), (64, 32, 24), (130, 64, 40), (257, 16, 32), (300, 8, 24), (40, 256, 16)])
def test_three_steps_and_more_refine(ctx, jkl, steps):
    """Three steps and more run the refinement, alone and in a batch, bit for bit what they are with
    the corrections reported."""
    g = fields.unit_grid(*jkl)
    print(f"[gpu] refine {g.name} steps {steps}", flush=True)
    pgs = [chypot.PreparedGrid(ctx, g) for _ in range(2)]
    rhos = [chypot.to_device(fields.density_spiral_torus(g, seed=30 + i)) for i in range(2)]
    jobs = [dict(grid=pg, rho=r, phi=torch.zeros_like(r), npoint=4) for pg, r in zip(pgs, rhos)]
    ctx.solve_batch(jobs, refine_steps=steps)
    ctx.sync()
    for pg, rho, job in zip(pgs, rhos, jobs):
        reported = _refined(ctx, pg, rho, steps, True)
        assert torch.equal(_refined(ctx, pg, rho, steps, False), reported)
        assert torch.equal(job["phi"], reported)
    for pg in pgs:
        pg.close()


def test_three_steps_reach_the_exact_solution(ctx):
    """The refinement's limit is the exact solution of the mode systems, here the oracle's in 80 bits: an
    order of magnitude nearer than BLKTRI's roots leave the tree (2.3e-12)."""
    import pyoracle as po
    g = fields.unit_grid(64, 128, 24)
    rho = fields.density_spiral_torus(g, seed=6)
    po.use_extended(True)
    try:
        want = po.solve(g, rho, npoint=4)["phi"]
    finally:
        po.use_extended(False)
    pg = chypot.PreparedGrid(ctx, g)
    rho_d = chypot.to_device(rho)
    for steps in (3, 4):
        err = rel_max(chypot.to_host(_refined(ctx, pg, rho_d, steps, False)), want)
        print(f"[gpu] refine {g.name}: {steps} steps, {err:.1e} from the exact solution", flush=True)
        assert err < 2e-13
    pg.close()


@pytest.mark.parametrize("jkl", [(64, 32, 24), (257, 16, 32), (16, 8, 4)])
@pytest.mark.parametrize("steps", [1, 2])
def test_eigenbasis_grids_refine(ctx, jkl, steps):
    """A grid whose solver is the z eigenbasis refines in it, bit for bit what it does with the
    corrections reported."""
    g = fields.unit_grid(*jkl)
    pg = chypot.PreparedGrid(ctx, g)
    pg.mode_solver = chypot.MODES_EIGEN
    rho = chypot.to_device(fields.density_spiral_torus(g, seed=31))
    print(f"[gpu] refine, eigenbasis {g.name} steps {steps}", flush=True)
    reported = _refined(ctx, pg, rho, steps, True)
    assert torch.equal(_refined(ctx, pg, rho, steps, False), reported)
    job = dict(grid=pg, rho=rho, phi=torch.zeros_like(rho), npoint=4)
    ctx.solve_batch([job], refine_steps=steps)
    ctx.sync()
    assert torch.equal(job["phi"], reported)
    pg.close()


def test_eigenbasis_grids_keep_the_stated_accuracy(ctx):
    """Two steps stay within 1e-10 of the grid's own chy_solve, also on a graded column, whose BLKTRI
    roots are 1.3e-9 from the eigenbasis' result."""
    g = fields.unit_grid(64, 128, 24)
    pg = chypot.PreparedGrid(ctx, Column(g, heights("1.03", g.kmax + 1)))
    pg.mode_solver = chypot.MODES_EIGEN
    rho = chypot.to_device(fields.density_spiral_torus(g, seed=6))
    plain = torch.zeros_like(rho)
    pg.solve(rho, plain, npoint=4)
    err = float((_refined(ctx, pg, rho, 2, False) - plain).abs().max()) / float(plain.abs().max())
    print(f"[gpu] refine, eigenbasis, graded {g.name}: {err:.1e} from chy_solve", flush=True)
    assert err < 1e-10
    pg.close()


@pytest.mark.parametrize("jkl,growth", [((64, 32, 24), 1.3), ((64, 64, 8), 1.06), ((64, 128, 24), 1.03)])
def test_uneven_columns_refine(ctx, jkl, growth):
    """Two steps on a column whose spacing varies refine, alone and in a batch, bit for bit what they do
    with the corrections reported: within 1e-10 of the exact solution (the oracle's in 80 bits), from
    which BLKTRI's roots are 3e-10 to 1.9e-9 away."""
    import pyoracle as po
    g = fields.unit_grid(*jkl)
    c = Column(g, heights(str(growth), g.kmax + 1))
    rho = fields.density_spiral_torus(g, seed=6)
    po.use_extended(True)
    try:
        want = po.solve(c, rho, npoint=4)["phi"]
    finally:
        po.use_extended(False)
    pgs = [chypot.PreparedGrid(ctx, c) for _ in range(2)]
    rho_d = chypot.to_device(rho)
    phi = _refined(ctx, pgs[0], rho_d, 2, False)
    assert torch.equal(phi, _refined(ctx, pgs[0], rho_d, 2, True))
    jobs = [dict(grid=pg, rho=rho_d, phi=torch.zeros_like(rho_d), npoint=4) for pg in pgs]
    ctx.solve_batch(jobs, refine_steps=2)
    ctx.sync()
    assert all(torch.equal(job["phi"], phi) for job in jobs)
    err = rel_max(chypot.to_host(phi), want)
    print(f"[gpu] refine, uneven {g.name} {growth}: {err:.1e} from the exact solution", flush=True)
    assert err < 1e-10
    for pg in pgs:
        pg.close()
