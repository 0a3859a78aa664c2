"""The z eigenbasis at the edges of its kernels' sizes: columns of 3 to 255
rows (products of 16, 32, 64 and 128 rows and the tiled one above), r systems
just inside and past each number of rows per lane (up to 1024 rows), one field
and two, orders without a sine part.  Against the oracle's 80-bit solve in the
same basis: no further from it than twice what the oracle's binary64 one is (the
operators' condition), plus 1e-13."""
import pytest

import chypot
from chypot import fields
from helpers import rel_max

pytestmark = pytest.mark.gpu

torch = pytest.importorskip("torch")


@pytest.mark.parametrize("jkl", [(5, 4, 4), (65, 8, 8), (66, 16, 6), (129, 16, 4), (130, 32, 10), (257, 64, 4),
                                 (258, 32, 4), (300, 4, 24), (513, 16, 4), (514, 8, 6), (600, 32, 4), (1025, 16, 4),
                                 (64, 128, 4), (40, 256, 4)])
def test_eigenbasis_sizes(jkl):
    import pyoracle as po
    if not torch.cuda.is_available():
        pytest.skip("no HIP device")
    g = fields.unit_grid(*jkl)
    print(f"[gpu] eigenbasis {g.name}", flush=True)
    ctx = chypot.Context(0)
    jobs = []
    for i in range(2):
        pg = chypot.PreparedGrid(ctx, g)
        pg.mode_solver = chypot.MODES_EIGEN
        rho = fields.density_spiral_torus(g, seed=30 + i)
        rho_d = chypot.to_device(rho)
        jobs.append(dict(grid=pg, rho=rho_d, phi=torch.full_like(rho_d, float("nan")), host=rho))
    jobs[0]["grid"].solve(jobs[0]["rho"], jobs[0]["phi"])
    ctx.sync()
    alone = jobs[0]["phi"][:, 1:g.kmax, 1:g.jmax].clone()
    po.use_extended(True)
    try:
        exact = po.solve(g, jobs[0]["host"])["phi"][1:g.jmax, 1:g.kmax]
    finally:
        po.use_extended(False)
    want = po.solve(g, jobs[0]["host"])["phi"][1:g.jmax, 1:g.kmax]
    got = chypot.to_host(jobs[0]["phi"])[1:g.jmax, 1:g.kmax]
    assert rel_max(got, exact) <= 2 * rel_max(want, exact) + 1e-13
    ctx.solve_batch([{k: j[k] for k in ("grid", "rho", "phi")} for j in jobs])
    ctx.sync()
    assert torch.equal(jobs[0]["phi"][:, 1:g.kmax, 1:g.jmax], alone)
    for j in jobs:
        j["grid"].close()
