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


@pytest.mark.parametrize("lanes", [64, 32])
@pytest.mark.parametrize("jkl", SHAPES)
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
