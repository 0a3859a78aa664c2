"""The mode solves' tree on columns whose z spacing is not even: graded, random and jumping cell
heights (leaves of 3 rows, levels that mix nodes with fewer roots and with all of their block's), and
evenly spaced ones that are so to rounding or to a fraction of a percent (leaves of 15 rows), against
the oracle's POT3 by BLKTRI's reduction with the same roots.

The two differ by rounding alone: a few 1e-14 at 64 rows along r, 2e-13 is four times the largest of
the spacings tried.  Evenly spaced columns may differ by what 15-row leaves in exact eigenvectors add,
1e-12 as on every grid shape."""
import numpy as np
import pytest

import chypot
from chypot import fields
from helpers import rel_max

pytestmark = pytest.mark.gpu

torch = pytest.importorskip("torch")


class Column:
    """A unit grid with cells of other heights (dz per row, scaled to the grid's height), as the
    oracle and PreparedGrid take it."""

    def __init__(self, g, dz):
        self.g = g
        self.jmax, self.kmax, self.lmax, self.shape, self.dtheta = g.jmax, g.kmax, g.lmax, g.shape, g.dtheta
        z = np.concatenate([[0.0], np.cumsum(dz)])
        self._z = (z - z[1]) / (z[-1] - z[1]) * g.z()[-1]
        self._zhf = np.append(0.5 * (self._z[:-1] + self._z[1:]), 1.5 * self._z[-1] - 0.5 * self._z[-2])

    def r(self):
        return self.g.r()

    def rhf(self):
        return self.g.rhf()

    def z(self):
        return self._z

    def zhf(self):
        return self._zhf


def heights(kind, n):
    rng = np.random.default_rng(n)
    if kind == "random":
        return 0.5 + rng.random(n)
    if kind == "jump":
        return np.where(np.arange(n) < n // 2, 1.0, 0.125)
    if kind.startswith("noise"):
        return 1.0 + float(kind[5:]) * (rng.random(n) - 0.5)
    return float(kind) ** np.arange(n)


def solve_both(jkl, kind, lanes):
    import pyoracle as po
    if not torch.cuda.is_available():
        pytest.skip("no HIP device")
    g = fields.unit_grid(*jkl)
    c = Column(g, heights(kind, g.kmax + 1))
    rho = fields.density_spiral_torus(g, seed=6)
    print(f"[gpu] column {g.name} {kind} lanes {lanes}", flush=True)
    ctx = chypot.Context(0)
    pg = chypot.PreparedGrid(ctx, c)
    pg.cr_lanes = lanes
    rho_d = chypot.to_device(rho)
    phi_d = torch.zeros_like(rho_d)
    pg.solve(rho_d, phi_d, npoint=4)
    ctx.sync()
    phi = chypot.to_host(phi_d)
    pg.close()
    po.use_cyclic_reduction(True)
    try:
        want = po.solve(c, rho, npoint=4)["phi"]
    finally:
        po.use_cyclic_reduction(False)
    err = rel_max(phi, want)
    print(f"[gpu] column {g.name} {kind} lanes {lanes}: {err:.1e} from BLKTRI's reduction", flush=True)
    return err


@pytest.mark.parametrize("lanes", [64, 32])
@pytest.mark.parametrize("jkl,kind", [((64, 4, 4), "1.5"), ((64, 8, 6), "1.3"), ((64, 16, 8), "0.7"), ((64, 16, 8), "1.6"),
                                      ((64, 32, 8), "1.03"), ((64, 32, 8), "1.3"), ((64, 32, 4), "jump"),
                                      ((64, 64, 8), "1.1"), ((64, 64, 8), "0.9"), ((64, 64, 6), "random"),
                                      ((64, 128, 8), "1.03"), ((64, 128, 6), "jump"), ((100, 256, 4), "1.01"),
                                      ((100, 256, 4), "random")])
def test_uneven_columns_against_oracle(jkl, kind, lanes):
    assert solve_both(jkl, kind, lanes) < 2e-13


@pytest.mark.parametrize("jkl,kind", [((64, 32, 8), "noise1e-14"), ((64, 64, 8), "noise1e-9"), ((100, 256, 4), "noise1e-3"),
                                      ((64, 128, 4), "noise0.009")])
def test_nearly_even_columns_against_oracle(jkl, kind):
    assert solve_both(jkl, kind, 32) < 1e-12
