"""Every call that runs BDYGEN refuses the arguments it has no meaning for:
MAXTRM outside 0..10 (the multipole table, pot/boundary.f), ISYM other than +-2
and a negative or undefined REDGE, before anything is launched (PHI keeps its
values)."""
import pytest

import chypot
from chypot import fields

pytestmark = pytest.mark.gpu

torch = pytest.importorskip("torch")

BAD = [dict(maxtrm=11), dict(maxtrm=-1), dict(isym=1), dict(isym=3), dict(isym=-8), dict(redge=-1.0),
       dict(redge=float("nan"))]


def _solve(ctx, pg, rho, phi, **kw):
    pg.solve(rho, phi, **kw)


def _refined(ctx, pg, rho, phi, **kw):
    pg.solve_refined(rho, phi, steps=2, **kw)


def _batch(ctx, pg, rho, phi, **kw):
    ctx.solve_batch([dict(grid=pg, rho=rho, phi=phi, **kw)])


def _bdygen(ctx, pg, rho, phi, **kw):
    pg.bdygen(rho, phi, **kw)


@pytest.mark.parametrize("lmax", [16, 32])  # boundary values through PHI, and in the spectrum
@pytest.mark.parametrize("call", [_solve, _refined, _batch, _bdygen])
@pytest.mark.parametrize("bad", BAD, ids=str)
def test_bdygen_arguments_refused(call, bad, lmax):
    if not torch.cuda.is_available():
        pytest.skip("no HIP device")
    g = fields.unit_grid(16, 8, lmax)
    ctx = chypot.Context(0)
    pg = chypot.PreparedGrid(ctx, g)
    rho = chypot.to_device(fields.density_spiral_torus(g, seed=3))
    phi = torch.full_like(rho, 7.0)
    with pytest.raises(chypot.ChyError) as ei:
        call(ctx, pg, rho, phi, **bad)
    assert ei.value.code == chypot.CHY_EINVAL
    ctx.sync()
    assert bool((phi == 7.0).all())
    pg.close()
