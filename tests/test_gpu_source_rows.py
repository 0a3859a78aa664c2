"""SOURCE with each number of rows K per thread that the launch chooses (8, 4, 2
and 1, by how many CUs 16 would leave idle), KMAX no multiple of it: bit for
bit the oracle's, as every size is."""
import numpy as np
import pytest

import chypot
import pyoracle as po

pytestmark = pytest.mark.gpu

torch = pytest.importorskip("torch")


@pytest.mark.parametrize("jkl", [(300, 37, 250), (256, 50, 120), (130, 37, 100), (20, 3, 5)])
def test_rows_per_thread(jkl):
    if not torch.cuda.is_available():
        pytest.skip("no HIP device")
    jm, km, lm = jkl
    print(f"[gpu] chy_source_grav rows {jkl}", flush=True)
    ctx = chypot.Context(0)
    rng = np.random.default_rng(sum(jkl))
    rho, phi, omega, p, s, t, a = (np.asfortranarray(rng.standard_normal((jm + 2, km + 2, lm))) for _ in range(7))
    r = (np.arange(1, jm + 3) - 2) / jm
    d = chypot.SourceDesc(jm, km, lm, jm, km, 2, 1.0e-3, 1.0 / jm, 0.5 / km, 2 * np.pi / lm)
    sd, td, ad = (chypot.to_device(x) for x in (s, t, a))
    ctx.source_grav(d, torch.from_numpy(r).to("cuda"), *(chypot.to_device(x) for x in (rho, omega, phi, p)), sd, td, ad)
    ctx.sync()
    po.source_grav(jm, km, lm, jm, km, 2, d.delt, d.dr, d.dz, d.dtheta, r, rho, omega, phi, p, s, t, a)
    for name, got, want in (("S", sd, s), ("T", td, t), ("A", ad, a)):
        assert np.array_equal(chypot.to_host(got), want), name
