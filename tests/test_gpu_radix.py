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
