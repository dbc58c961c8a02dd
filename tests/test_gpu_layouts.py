"""What pgamd_set_layout decides: which form of the SOR kernel runs, told from the time of a
solve, since all forms return the same (needs an MI355X).  At ghost size 1 and 256 patches the form with several wavefronts per
patch takes half the time of any layout of the one-wavefront kernel."""
import numpy as np
import pytest

import gpu_testbed_poisson_gravity_amd as pg
from gpu_testbed_poisson_gravity_amd import inputs as I

pytestmark = pytest.mark.gpu
POI = 4.0 * np.pi * 1e-5
GS, N = 1, 256


@pytest.fixture(scope="module")
def batch():
    import torch

    rho, cpot, _, _ = I.plummer(N, GS, seed=5)
    return torch.as_tensor(rho).cuda(), torch.as_tensor(cpot).cuda(), torch.zeros((N, 10, 10, 10), device="cuda")


def _args():
    return pg.solver_args(sor_min_iter=150, sor_max_iter=150, sor_omega=1.49, poi_coeff=POI, graacc=False)


def _context():
    ctx = pg.Context(0)
    ctx.set_options(pot_ghost_size=GS, fuse_gravity=0)
    return ctx


def _ms(ctx, batch):
    """Shortest of ten solves."""
    import torch

    rho, cpot, out = batch
    s, best = torch.cuda.current_stream().cuda_stream, 1e9
    for _ in range(10):
        e = [torch.cuda.Event(enable_timing=True) for _ in range(2)]
        e[0].record()
        ctx.solve_device(rho, cpot, out, None, N, _args(), stream=s)
        e[1].record()
        torch.cuda.synchronize()
        best = min(best, e[0].elapsed_time(e[1]))
    return best


def test_putting_a_layout_back_restores_the_choice_of_form(batch):
    with _context() as ctx:
        own = ctx.get_layout(GS)
        before = _ms(ctx, batch)
        ctx.set_layout(GS, 1, 0)
        one = _ms(ctx, batch)
        ctx.set_layout(GS, 2, 1)
        ctx.set_layout(GS, *own)
        after = _ms(ctx, batch)
        ctx.set_layout(GS, *own)   # nothing to put back: selects that layout
        explicit = _ms(ctx, batch)
    print(f"[case] layouts: {before:.4f} ms, set {one:.4f}, put back {after:.4f}, set to the same {explicit:.4f}", flush=True)
    assert one > 1.4 * before and explicit > 1.4 * before
    assert after < 1.2 * before
