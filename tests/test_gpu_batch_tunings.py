"""Batches over grid objects of one description with unlike tunables: an item runs with its own
grid's settings, whatever comes before it, so each is bit for bit its own single solve."""
import pytest

import chypot
from chypot import fields

pytestmark = pytest.mark.gpu

torch = pytest.importorskip("torch")


@pytest.fixture(scope="module")
def ctx():
    if not torch.cuda.is_available():
        pytest.skip("no HIP device")
    return chypot.Context(0)


def _jobs(ctx, jkl, tunings):
    g = fields.unit_grid(*jkl)
    jobs = []
    for i, t in enumerate(tunings):
        pg = chypot.PreparedGrid(ctx, g)
        for name, value in t.items():
            setattr(pg, name, value)
        rho = chypot.to_device(fields.density_spiral_torus(g, seed=50 + i))
        jobs.append(dict(grid=pg, rho=rho, phi=torch.zeros_like(rho)))
    return jobs


@pytest.mark.parametrize("jkl", [(64, 32, 64), (257, 16, 48)])
@pytest.mark.parametrize("graphs", [True, False])
@pytest.mark.parametrize("steps,tunings", [
    (0, [dict(cr_lanes=32), dict(cr_lanes=64), dict(cr_lanes=32)]),
    (2, [dict(cr_lanes=64), dict(cr_lanes=32), dict(cr_lanes=32)]),
    (2, [dict(refine_fused=32), dict(refine_fused=0), dict(refine_fused=32)]),
    (1, [dict(refine_fused=0), dict(refine_fused=32), dict(refine_fused=0)]),
    (3, [dict(refine_m64=4), dict(refine_m64=-1), dict(refine_m64=8)])])
def test_unlike_tunings_keep_their_own(ctx, jkl, steps, tunings, graphs):
    print(f"[gpu] unlike tunings {jkl} steps {steps} {tunings} graphs {graphs}", flush=True)
    jobs = _jobs(ctx, jkl, tunings)
    ctx.graphs(graphs)
    for _ in range(3):  # issued, captured, replayed
        for j in jobs:
            j["phi"].zero_()
        ctx.solve_batch(jobs, refine_steps=steps)
        ctx.sync()
        for i, j in enumerate(jobs):
            alone = torch.zeros_like(j["rho"])
            if steps:
                j["grid"].solve_refined(j["rho"], alone, steps=steps)
            else:
                j["grid"].solve(j["rho"], alone)
            ctx.sync()
            assert torch.equal(j["phi"], alone), i
    ctx.graphs(True)
    for j in jobs:
        j["grid"].close()


@pytest.mark.parametrize("other", [((600, 8, 24), {}), ((64, 32, 64), dict(refine_fused=4)), ((32, 16, 64), dict(mode_solver=chypot.MODES_EIGEN))])
def test_refined_batches_allocate_for_their_own_route(ctx, other):
    """Grids whose own refined solves take the binary64 tree get no binary32 buffers for a neighbour
    in the batch that refines in binary32 (which gets them)."""
    jobs = _jobs(ctx, (64, 32, 64), [{}, {}]) + _jobs(ctx, other[0], [other[1]])
    before = [j["grid"].device_bytes for j in jobs]
    print(f"[gpu] buffers of a mixed refined batch, {other}", flush=True)
    ctx.solve_batch(jobs, refine_steps=2)
    ctx.sync()
    after = [j["grid"].device_bytes for j in jobs]
    assert after[:2] == before[:2]
    assert after[2] > before[2]
    for j in jobs:
        alone = torch.zeros_like(j["rho"])
        j["grid"].solve_refined(j["rho"], alone, steps=2)
        ctx.sync()
        assert torch.equal(j["phi"], alone)
        j["grid"].close()
