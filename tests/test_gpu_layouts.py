"""What pgamd_set_layout, pgamd_autotune and its saved table decide: which form of the SOR kernel runs, told from the time of a
solve, since all forms return the same (needs an MI355X).  At ghost size 1 and 256 patches the form with several wavefronts per
patch takes half the time of any layout of the one-wavefront kernel."""
import json

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


def _tune(ctx, batch):
    return ctx.autotune(GS, batch[0], batch[1], batch[2], N, _args(), repeats=20)


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


def test_autotuner_times_and_keeps_what_runs(batch, tmp_path):
    path = str(tmp_path / "layouts.json")
    with _context() as ctx:
        fresh = _ms(ctx, batch)
        ctx.set_layout(GS, 1, 0)
        one = _ms(ctx, batch)
        ppw, pad, ms = _tune(ctx, batch)   # chooses again
        tuned = _ms(ctx, batch)
        print(f"[case] autotune: fresh {fresh:.4f} ms, set {one:.4f}, best {ms:.4f}, tuned {tuned:.4f}", flush=True)
        assert ctx.get_layout(GS) == (ppw, pad)
        assert tuned < 1.2 * fresh and one > 1.4 * fresh
        assert 0.7 * tuned < ms < 1.2 * tuned
        ctx.autotune_save(path)
    with open(path) as f:
        table = json.load(f)
    assert table["layouts"][str(GS)] == [ppw, pad] and table["blocks_up_to"][str(GS)] >= N
    with _context() as ctx:   # a table of a context with a layout that the caller set
        ctx.set_layout(GS, 2, 0)
        ctx.autotune_save(path)
    with _context() as ctx:
        ctx.autotune_load(path)
        assert ctx.get_layout(GS) == (2, 0) and _ms(ctx, batch) > 1.4 * fresh
        table["blocks_up_to"][str(GS)] = N - 1
        with open(path, "w") as f:
            json.dump(table, f)
        ctx.autotune_load(path)   # the limit is just below this batch
        assert ctx.get_layout(GS) == (ppw, pad) and _ms(ctx, batch) > 1.4 * fresh


def test_tables_without_limits_load_with_the_default_ones(batch, tmp_path):
    path = str(tmp_path / "layouts.json")
    with _context() as ctx:
        fresh = _ms(ctx, batch)
        ctx.autotune_save(path)
        with open(path) as f:
            table = json.load(f)
        good = dict(table)
        del table["blocks_up_to"]
        with open(path, "w") as f:
            json.dump(table, f)
        ctx.set_layout(GS, 1, 0)
        ctx.autotune_load(path)
        assert _ms(ctx, batch) < 1.2 * fresh
        for bad in ({"1": -1}, {"1": "x"}, {}):
            with open(path, "w") as f:
                json.dump(dict(good, blocks_up_to=dict(bad, **{str(g): 8 for g in range(2, 6)})), f)
            with pytest.raises(pg.PgError):
                ctx.autotune_load(path)
