"""COEF's amplitudes at the ends of the number range: 2 sqrt(A^2 + B^2)/|A0| as pot/pot3.f:105-132 forms
it, against the oracle.  Densities so thin that |A0| is below 1.1e-308 (2/|A0| overflows; A^2 vanishes,
so the amplitudes of the orders below LMAX/2 are zero; their sums are whole to a few 5e-324, 1e-13 of
|A0|), ordinary ones, and densities whose squares stay just finite."""
import numpy as np
import pytest

import chypot
from chypot import fields

pytestmark = pytest.mark.gpu

torch = pytest.importorskip("torch")


@pytest.mark.parametrize("lmax", [32, 48])  # a power of two, mixed radices
@pytest.mark.parametrize("scale", [1.2e-310, 1.0, 1e150])
@pytest.mark.parametrize("jk", [(16, 8), (300, 64)])  # COEF by blocks of its own, and by those of the transform
def test_amplitudes_over_the_range(jk, lmax, scale):
    import pyoracle as po
    if not torch.cuda.is_available():
        pytest.skip("no HIP device")
    g = fields.unit_grid(*jk, lmax)
    rng = np.random.default_rng(5)
    rho = np.zeros(g.shape, order="F")
    rho[1:g.jmax + 1, 1:g.kmax + 1, :] = scale * (0.5 + rng.random((g.jmax, g.kmax, lmax)))
    print(f"[gpu] COEF range {g.name} scale {scale}", flush=True)
    ctx = chypot.Context(0)
    pg = chypot.PreparedGrid(ctx, g)
    rho_d = chypot.to_device(rho)
    coef = torch.zeros(pg.coef_shape, dtype=torch.float64, device="cuda")
    pg.solve(rho_d, torch.zeros_like(rho_d), coef=coef, coef_mode=chypot.COEF_FULL)
    ctx.sync()
    pg.close()
    got = coef.cpu().numpy().transpose(3, 2, 1, 0)[1:g.jmax, 1:g.kmax, :, 0]
    # the interior lanes' raw coefficients at the ends of the grid and in the middle
    for j in (1, g.jmax // 2, g.jmax - 1):
        for k in (1, g.kmax // 2, g.kmax - 1):
            A, B = po.rfft_fwd(rho[j, k])
            x1 = abs(A[0])
            want = np.append(2.0 * np.sqrt(A[1:-1] ** 2 + B[1:-1] ** 2) / x1, abs(A[-1]) / x1)
            assert np.abs(got[j - 1, k - 1] - want).max() < 1e-13, (j, k)
    assert np.isfinite(got).all()
