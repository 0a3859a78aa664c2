"""find_force on grids of any unit of length: cells whose squared distances overflow pull with nothing, as
1/sqrt(infinity)^3 does in pot/wiggle.F:119-126, and leave the others' sum alone.  Against the oracle's
80-bit sum of the same binary64 terms, 1e-13 of the sum of their magnitudes."""
import numpy as np
import pytest

import chypot
from chypot import fields

pytestmark = pytest.mark.gpu

torch = pytest.importorskip("torch")


@pytest.mark.parametrize("scale,outer", [(1e-60, 1.0), (1.0, 1.0), (1e60, 1.0), (1.0, 1e160), (1e160, 1.0)])
def test_force_over_the_range(scale, outer):
    """outer: the factor on the outer half of the radii alone."""
    import pyoracle as po
    if not torch.cuda.is_available():
        pytest.skip("no HIP device")
    g = fields.unit_grid(48, 16, 40)
    rhf, zhf = scale * g.rhf(), scale * g.zhf()
    rhf[g.jmax // 2:] *= outer
    rho = fields.density_spiral_torus(g, seed=4)
    gs, x, y = 0.01 * scale, 0.031 * scale, -0.012 * scale
    print(f"[gpu] find_force range, scale {scale} outer {outer}", flush=True)
    (wx, wy), (ax, ay) = po.find_force(g.jmax, g.kmax, g.lmax, 4, g.delr, g.delz, g.dtheta, gs, rhf, zhf, rho, x, y)
    ctx = chypot.Context(0)
    d = chypot.ForceDesc(g.jmax, g.kmax, g.lmax, 4, g.delr, g.delz, g.dtheta, gs)
    rho_d = chypot.to_device(rho)
    rhf_d, zhf_d = torch.from_numpy(rhf).to("cuda"), torch.from_numpy(zhf).to("cuda")
    f = torch.zeros(2, dtype=torch.float64, device="cuda")
    ctx.find_force_noalloc(d, rhf_d, zhf_d, rho_d, x, y, f)  # forms its cosines on the GPU
    ctx.sync()
    assert np.isfinite([wx, wy, ax, ay]).all()
    for fx, fy in (ctx.find_force(d, rhf_d, zhf_d, rho_d, x, y), f.tolist()):
        assert abs(fx - wx) <= 1e-13 * ax and abs(fy - wy) <= 1e-13 * ay, ((fx, fy), (wx, wy), (ax, ay))
