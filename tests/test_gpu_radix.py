"""Azimuths whose half has factors 3 and 5: the transforms' passes of 3, 5, 6,
10, 12 and 20 points, alone, with each other and with 8 and 16, for each number
of lanes per block; a few more than a block's lanes, so the last one is partly
idle.  Against the oracle's solve by the same reduction, which differs in
rounding alone (~1e-14 of the largest value here)."""
import pytest

import chypot
from chypot import fields
from helpers import rel_max

pytestmark = pytest.mark.gpu

torch = pytest.importorskip("torch")


@pytest.mark.parametrize("l", [6, 12, 20, 24, 30, 40, 60, 72, 90, 120, 144, 200, 240, 320, 400, 486, 600, 640, 800,
                               960, 1000])
def test_azimuths(l):
    import pyoracle as po
    if not torch.cuda.is_available():
        pytest.skip("no HIP device")
    g = fields.unit_grid(18, 8, l)
    print(f"[gpu] azimuths {g.name}", flush=True)
    rho = fields.density_spiral_torus(g, seed=l)
    po.use_cyclic_reduction(True)
    try:
        want = po.solve(g, rho)["phi"]
    finally:
        po.use_cyclic_reduction(False)
    ctx = chypot.Context(0)
    pg = chypot.PreparedGrid(ctx, g)
    rho_d = chypot.to_device(rho)
    phi_d = torch.full_like(rho_d, float("nan"))
    pg.solve(rho_d, phi_d)
    ctx.sync()
    got = chypot.to_host(phi_d)
    pg.close()
    assert rel_max(got[1:g.jmax, 1:g.kmax], want[1:g.jmax, 1:g.kmax]) < 1e-12


@pytest.mark.parametrize("jkl", [(18, 8, 32), (18, 8, 64), (18, 8, 128), (66, 32, 32), (130, 64, 64), (95, 128, 128),
                                 (97, 128, 128)])
def test_powers_of_two(jkl):
    """LMAX 32, 64 and 128: the splits of LMAX/2, on both sides of the number of
    lanes that decides it at 128, and each count of lanes per block: one field,
    and a batch whose blocks fill the chip, bit for bit alike."""
    import pyoracle as po
    if not torch.cuda.is_available():
        pytest.skip("no HIP device")
    g = fields.unit_grid(*jkl)
    print(f"[gpu] powers of two {g.name}", flush=True)
    rho = fields.density_spiral_torus(g, seed=7)
    po.use_cyclic_reduction(True)
    try:
        want = po.solve(g, rho)["phi"]
    finally:
        po.use_cyclic_reduction(False)
    ctx = chypot.Context(0)
    jobs = []
    for i in range(24):
        rho_d = chypot.to_device(rho if i in (0, 23) else fields.density_spiral_torus(g, seed=8))
        jobs.append(dict(grid=chypot.PreparedGrid(ctx, g), rho=rho_d, phi=torch.zeros_like(rho_d)))
    jobs[0]["grid"].solve(jobs[0]["rho"], jobs[0]["phi"])
    ctx.sync()
    alone = jobs[0]["phi"].clone()
    ctx.solve_batch(jobs)
    ctx.sync()
    got = chypot.to_host(alone)
    assert rel_max(got[1:g.jmax, 1:g.kmax], want[1:g.jmax, 1:g.kmax]) < 1e-12
    assert torch.equal(jobs[0]["phi"], alone)
    assert torch.equal(jobs[23]["phi"], alone)
    for j in jobs:
        j["grid"].close()
