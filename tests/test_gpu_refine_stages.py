"""The refinement's own kernels (binary32 mode solves, binary64 residual), which a refined solve of one
or two steps runs where the corrections are reported or the grid's solver is the z eigenbasis: their
error per step, their agreement with the one-kernel-per-plane form, and several fields per launch."""
import pytest

import chypot
from chypot import fields
from helpers import rel_max

pytestmark = pytest.mark.gpu

torch = pytest.importorskip("torch")


@pytest.fixture(scope="module")
def ctx():
    if not torch.cuda.is_available():
        pytest.skip("no HIP device")
    return chypot.Context(0)


@pytest.mark.parametrize("density", ["small_torus", "spiral"])
def test_refinement_error_per_step_256(ctx, density):
    """256x128x256 against the plain solve: the binary32 solves' ~1e-6, below 1e-10 after two steps, then
    the distance between the exact solution and the plain path's reduction (~2e-12), never nothing."""
    g = fields.unit_grid(256, 128, 256)
    rho = fields.density_small_torus(g, 1) if density == "small_torus" else fields.density_spiral_torus(g, 2)
    pg = chypot.PreparedGrid(ctx, g)
    rho_d = chypot.to_device(rho)
    plain = torch.zeros_like(rho_d)
    pg.solve(rho_d, plain)
    errs = []
    for steps in range(1, 5):
        phi = torch.zeros_like(rho_d)
        pg.solve_refined(rho_d, phi, steps=steps, report=True)
        ctx.sync()
        errs.append(float((phi - plain).abs().max()) / float(plain.abs().max()))
    pg.close()
    print(f"[gpu] refinement {density} 256x128x256: error vs plain per step " + " ".join(f"{e:.2e}" for e in errs),
          flush=True)
    assert 1e-10 < errs[0] < 1e-5
    assert 0.0 < errs[1] < 1e-10
    assert 0.0 < min(errs[2:]) and max(errs[2:]) < 1e-11


@pytest.mark.parametrize("jkl", [(256, 128, 256), (64, 32, 64), (100, 64, 32), (200, 128, 64), (40, 16, 16),
                                 (257, 8, 16)])
@pytest.mark.parametrize("steps", [1, 2])
def test_one_kernel_form_matches_the_stage_kernels(ctx, jkl, steps):
    """Every (PP, JP) the one-kernel form is built for, JMAX-1 = JP and KMAX = 8.  The binary32 r solves
    differ in method, which moves the ~1e-7 first step; two steps agree to rounding."""
    g = fields.unit_grid(*jkl)
    rho = chypot.to_device(fields.density_spiral_torus(g, seed=21))
    pg = chypot.PreparedGrid(ctx, g)
    stages, fused = torch.zeros_like(rho), torch.zeros_like(rho)
    pg.solve_refined(rho, stages, steps=steps, report=True)
    pg.refine_fused = True
    pg.solve_refined(rho, fused, steps=steps)
    ctx.sync()
    pg.close()
    err = float((fused - stages).abs().max()) / float(stages.abs().max())
    print(f"[gpu] one kernel per plane {g.name} steps {steps}: {err:.2e} from the stage kernels", flush=True)
    assert 0.0 < err < (1e-5 if steps == 1 else 2e-11)


@pytest.mark.parametrize("steps", [1, 2, 3])
@pytest.mark.parametrize("jkl,modes", [((600, 8, 24), None), ((1500, 8, 16), None), ((600, 64, 32), None),
                                       ((64, 256, 24), chypot.MODES_EIGEN), ((257, 16, 48), chypot.MODES_EIGEN)])
def test_several_fields_refine_as_one(ctx, jkl, modes, steps):
    """Three fields per launch by the binary32 kernels (grids past the tree's JMAX, eigenbasis grids), with
    another grid in the batch: each bit for bit its own solve, and near the oracle's."""
    import pyoracle as po
    g = fields.unit_grid(*jkl)
    jobs = []
    for i in range(4):
        gi = g if i < 3 else fields.unit_grid(32, 16, 64)
        pg = chypot.PreparedGrid(ctx, gi)
        if modes is not None and i < 3:
            pg.mode_solver = modes
        rho = chypot.to_device(fields.density_spiral_torus(gi, seed=70 + i))
        jobs.append(dict(grid=pg, rho=rho, phi=torch.zeros_like(rho), npoint=4, coef_mode=chypot.COEF_K2,
                         coef=torch.zeros(pg.coef_shape, dtype=torch.float64, device="cuda")))
    print(f"[gpu] several fields refine {g.name} steps {steps}", flush=True)
    for batch in (jobs[:3], jobs):  # one group, several (issued, captured, replayed)
        for _ in range(1 if batch is not jobs else 3):
            for j in batch:
                j["phi"].zero_()
            diags = ctx.solve_batch(batch, diag=True, refine_steps=steps)
            for i, j in enumerate(batch):
                phi, coef = torch.zeros_like(j["phi"]), torch.zeros_like(j["coef"])
                d, _ = j["grid"].solve_refined(j["rho"], phi, steps=steps, npoint=4, coef=coef, coef_mode=chypot.COEF_K2,
                                               diag=True)
                ctx.sync()
                assert torch.equal(j["phi"], phi) and torch.equal(j["coef"], coef), i
                assert (d.tmass, d.phichk, d.klocat) == (diags[i].tmass, diags[i].phichk, diags[i].klocat)
    want = po.solve(g, fields.density_spiral_torus(g, seed=71), npoint=4)["phi"]
    err = rel_max(chypot.to_host(jobs[1]["phi"]), want)
    print(f"[gpu] several fields refine {g.name} steps {steps}: {err:.1e} from the oracle", flush=True)
    assert err < (1e-5 if steps == 1 else 1e-10)
    for j in jobs:
        j["grid"].close()
