"""The block form of the SOR kernel (several wavefronts per patch) against the one-wavefront form, which a caller selects by
setting a layout (needs an MI355X): potentials, fluid, iteration counts and statuses must be equal bit for bit, over
starts, stopping rules, interpolation schemes, windows and the batch sizes where the form changes."""
import numpy as np
import pytest

import gpu_testbed_poisson_gravity_amd as pg
from gpu_testbed_poisson_gravity_amd import inputs as I

pytestmark = pytest.mark.gpu
POI = 4.0 * np.pi * 1e-5
DEFAULT = {1: (4, 1), 2: (2, 0), 3: (1, 0), 4: (1, 1), 5: (1, pg.LAYOUT_COMPACT)}   # the library's layouts
K = 24


def _patches(gs, special=True):
    rho, cpot, flu, _ = I.plummer(K, gs, seed=80 + gs)
    if special:
        rho[1], cpot[1] = 0.0, 0.0             # all sums zero: ties in every stopping rule
        rho[2, 1, 2, 3] = np.nan
        cpot[3, 0, 0, 0] = np.inf
        rho[4] *= 1e30                         # large sums
        rho[5], cpot[5] = 1.0, cpot[5, :1, :1, :1]
    flu[:, 1:4] = 0.05 * np.cos(np.arange(flu[:, 1:4].size)).reshape(flu[:, 1:4].shape)
    return rho, cpot, flu


def _solve(gs, at, layout, opts, args, guess=None):
    import torch

    rho, cpot, flu = _patches(gs)
    n = len(at)
    dev = lambda a: torch.as_tensor(np.ascontiguousarray(a[at])).cuda()   # noqa: E731
    G = 8 + 2 * opts.get("gra_ghost_size", 1)
    out, d_flu = torch.zeros((n, G, G, G), device="cuda"), dev(flu)
    it, st = (torch.zeros(n, dtype=torch.int32, device="cuda") for _ in range(2))
    with pg.Context(0) as ctx:
        ctx.set_options(pot_ghost_size=gs, **opts)
        if layout is not None:
            ctx.set_layout(gs, *layout)
        ctx.solve_device(dev(rho), dev(cpot), out, d_flu if args.graacc else None, n, args,
                         guess=None if guess is None else dev(guess), iters=it, status=st)
        torch.cuda.synchronize()
    return [a.cpu().numpy() for a in (out, d_flu, it, st)]


def _same(gs, n, opts, args, guess=None):
    print(f"[case] blocks gs={gs} n={n} {opts} iters {args.sor_min_iter}-{args.sor_max_iter}", flush=True)
    a = _solve(gs, np.arange(n) % K, None, opts, args, guess)
    # one patch per call: a packed wavefront goes on adding 0 * R to a patch that has stopped, which turns the infinities
    # of a non-finite patch into NaN for as long as its neighbours run
    one = [_solve(gs, [k], DEFAULT[gs], opts, args, guess) for k in range(K)]
    b = [np.concatenate(x)[np.arange(n) % K] for x in zip(*one)]
    for x, y, what in zip(a, b, ("potential", "fluid", "iterations", "status")):
        assert np.array_equal(x, y, equal_nan=x.dtype.kind == "f"), (what, np.nonzero((x != y).reshape(n, -1).any(1))[0][:9])
    return a


@pytest.mark.parametrize("gs", [1, 2, 3, 4, 5])
def test_blocks_match_one_wavefront(gs):
    R, N = 6 + 2 * gs, 8 + 2 * gs
    rng = np.random.default_rng(gs)
    run = lambda opts, guess=None, **kw: _same(gs, K, opts, pg.solver_args(**dict(   # noqa: E731
        dict(sor_min_iter=10, sor_max_iter=120, sor_omega=1.6, poi_coeff=POI, dt=0.5), **kw)), guess)
    # the stall rule down to round-off, where successive totals are close
    _, _, it, _ = run(dict(term_mode=pg.TERM_REFERENCE), sor_min_iter=10, sor_max_iter=300)
    assert it[0] < 300 and it[1] == 300
    run(dict(term_mode=pg.TERM_REFERENCE, init_mode=pg.INIT_ZERO), sor_min_iter=0, int_scheme=pg.INT_QUAD)
    for every in (1, 3):
        run(dict(term_mode=pg.TERM_RELRES, init_mode=pg.INIT_ZERO, rel_tol=1e-5, check_every=every), sor_max_iter=1000)
    run(dict(term_mode=pg.TERM_RELRES, rel_tol=0.0), sor_max_iter=40, int_scheme=pg.INT_QUAD)
    run(dict(term_mode=pg.TERM_RELRES), sor_max_iter=0)
    if gs >= 2:
        run(dict(term_mode=pg.TERM_RELRES, gra_ghost_size=2), p5=True)
        run(dict(term_mode=pg.TERM_RELRES, gra_ghost_size=2, fuse_gravity=0))
    run(dict(term_mode=pg.TERM_RELRES, gra_ghost_size=gs), graacc=False)
    # guesses, some of them rejected by the check (patch 7's is the zero field: a tie of zeros with density zero)
    scale = 1e-4 * np.where(np.arange(K) % 2, 1.0, 1e-9)[:, None, None, None]
    for mode, edge in ((pg.INIT_GUESS, R), (pg.INIT_GUESS_CUBE, N)):
        guess = (rng.standard_normal((K, edge, edge, edge)) * scale).astype(np.float32)
        guess[1] = 0.0
        run(dict(term_mode=pg.TERM_RELRES, init_mode=mode, guess_fallback_tol=0.5), guess)


@pytest.mark.parametrize("gs, n", [(1, 1025), (2, 1025), (3, 1024), (3, 1025), (4, 1024), (5, 512), (5, 513), (5, 1024)])
@pytest.mark.parametrize("rule", [pg.TERM_REFERENCE, pg.TERM_RELRES])
def test_blocks_match_at_form_changes(gs, n, rule):
    opts = dict(term_mode=rule, check_every=2)
    _same(gs, n, opts, pg.solver_args(sor_min_iter=10, sor_max_iter=80, sor_omega=1.65, poi_coeff=POI, dt=0.5))


@pytest.mark.parametrize("n", [300, 12000])
def test_mixed_batch_forms(n):
    """A mixed batch small enough for blocks at every ghost size and one with one-wavefront launches at 4 and 5."""
    import torch

    gs = (np.arange(n) % 5 + 1).astype(np.int32)
    parts = {g: _patches(g, special=False) for g in range(1, 6)}
    pick = lambda k: [parts[g][k][(i // 5) % K] for i, g in enumerate(gs)]   # noqa: E731
    res = []
    for fixed in (False, True):
        with pg.Context(0) as ctx:
            ctx.set_options(term_mode=pg.TERM_RELRES, check_every=2)
            if fixed:
                for g, lay in DEFAULT.items():
                    ctx.set_layout(g, *lay)
            plan = ctx.plan(gs)
            rho = torch.as_tensor(pg.pack(pick(0), plan.rho_off, plan.rho_floats)).cuda()
            cpot = torch.as_tensor(pg.pack(pick(1), plan.pot_in_off, plan.pot_in_floats)).cuda()
            flu = torch.as_tensor(np.stack(pick(2))).cuda()
            out = torch.zeros((n, 10, 10, 10), device="cuda")
            it, st = (torch.zeros(n, dtype=torch.int32, device="cuda") for _ in range(2))
            print(f"[case] mixed n={n} one-wavefront={fixed}", flush=True)
            ctx.solve_mixed_device(plan, rho, cpot, out, flu,
                                   pg.solver_args(sor_max_iter=80, sor_omega=1.6, poi_coeff=POI, dt=0.5), iters=it, status=st)
            torch.cuda.synchronize()
            plan.close()
        res.append([a.cpu().numpy() for a in (out, flu, it, st)])
    for x, y in zip(*res):
        assert np.array_equal(x, y, equal_nan=x.dtype.kind == "f")


@pytest.mark.parametrize("gs, n", [(3, 512), (3, 513), (5, 256), (5, 257)])
def test_fp64_forms_agree(gs, n):
    """FP64 at the batch sizes where the planes per thread change: every copy of a patch gets the same bits."""
    rho, cpot, flu, _ = I.plummer(5, gs, seed=3, dtype=np.float64)
    at = np.arange(n) % 5
    kw = dict(gs=gs, sor_min_iter=30, sor_max_iter=30, sor_omega=1.65, poi_coeff=POI, dt=0.5)
    print(f"[case] f64 blocks gs={gs} n={n}", flush=True)
    few = pg.solve_host_f64(rho, cpot, flu, **kw)
    many = pg.solve_host_f64(rho[at], cpot[at], flu[at], **kw)
    for x, y in zip(few, many):
        assert np.array_equal(x[at], y)


@pytest.mark.parametrize("gs, n", [(3, 1536), (3, 1537), (5, 768), (5, 769)])
def test_blocks_match_at_plane_changes(gs, n):
    """Batch sizes where the planes per thread change."""
    _same(gs, n, dict(term_mode=pg.TERM_REFERENCE), pg.solver_args(sor_min_iter=10, sor_max_iter=60, sor_omega=1.65,
                                                                   poi_coeff=POI, dt=0.5))


@pytest.mark.parametrize("gs", [1, 3, 5])
@pytest.mark.parametrize("what", ["zero", "nan"])
def test_blocks_are_no_slower_on_patches_that_never_stop(gs, what):
    """A patch of zeros, or with a NaN, ties at every comparison of the stall rule: the form that is chosen because it is
    faster must not spend longer than the other one on sums whose order cannot matter."""
    import torch

    n = 256
    rho, cpot, _ = _patches(gs, special=False)
    at = np.arange(n) % K
    rho, cpot = rho[at], cpot[at]
    if what == "zero":
        rho[0], cpot[0] = 0.0, 0.0
    else:
        rho[0, 1, 2, 3] = np.nan
    rho, cpot = torch.as_tensor(rho).cuda(), torch.as_tensor(cpot).cuda()
    args = pg.solver_args(sor_min_iter=10, sor_max_iter=1000, sor_omega=1.65, poi_coeff=POI, graacc=False)
    ms, res = [], []
    for fixed in (True, False):
        with pg.Context(0) as ctx:
            ctx.set_options(pot_ghost_size=gs, term_mode=pg.TERM_REFERENCE, fuse_gravity=0)
            if fixed:
                ctx.set_layout(gs, *DEFAULT[gs])
            out, it = torch.zeros((n, 10, 10, 10), device="cuda"), torch.zeros(n, dtype=torch.int32, device="cuda")
            best = 1e9
            for _ in range(5):
                e = [torch.cuda.Event(enable_timing=True) for _ in range(2)]
                e[0].record()
                ctx.solve_device(rho, cpot, out, None, n, args, iters=it, stream=torch.cuda.current_stream().cuda_stream)
                e[1].record()
                torch.cuda.synchronize()
                best = min(best, e[0].elapsed_time(e[1]))
            ms.append(best)
            res.append((out.cpu().numpy(), it.cpu().numpy()))
    print(f"[case] one {what} patch of {n}, gs={gs}: one wavefront {ms[0]:.3f} ms, blocks {ms[1]:.3f} ms", flush=True)
    assert res[0][1][0] == 1000 and np.array_equal(res[0][1], res[1][1])
    assert np.array_equal(res[0][0][1:], res[1][0][1:])
    assert ms[1] < ms[0]


@pytest.mark.parametrize("gs", [1, 3, 5])
def test_blocks_match_one_wavefront_among_subnormals(gs):
    """Fields so small that the products in the stopping rules are subnormal and round by whole units."""
    import torch

    n, g = 256, pg.geometry(gs)
    rng = np.random.default_rng(gs)
    unit = np.float32(2.0 ** -149)   # the smallest subnormal
    size = (rng.integers(1, 400, (n, 1, 1, 1))).astype(np.float32)
    cpot = torch.as_tensor((rng.standard_normal((n,) + (g["C"],) * 3) * size).astype(np.float32).round() * unit).cuda()
    rho = torch.as_tensor((rng.standard_normal((n,) + (g["R"],) * 3) * size).astype(np.float32).round() * unit / np.float32(POI)).cuda()
    differ = 0
    for tol in (0.9, 0.3, 0.1, 0.03):
        for omega in (1.3, 1.7):
            res = []
            for fixed in (True, False):
                with pg.Context(0) as ctx:
                    ctx.set_options(pot_ghost_size=gs, term_mode=pg.TERM_RELRES, rel_tol=tol, fuse_gravity=0)
                    if fixed:
                        ctx.set_layout(gs, *DEFAULT[gs])
                    out, it = torch.zeros((n, 10, 10, 10), device="cuda"), torch.zeros(n, dtype=torch.int32, device="cuda")
                    args = pg.solver_args(sor_min_iter=0, sor_max_iter=40, sor_omega=omega, poi_coeff=POI, graacc=False)
                    ctx.solve_device(rho, cpot, out, None, n, args, iters=it)
                    torch.cuda.synchronize()
                    res.append((out.cpu().numpy(), it.cpu().numpy()))
            differ += (res[0][1] != res[1][1]).sum()
            print(f"[case] subnormal gs={gs} tol={tol} omega={omega}: {np.unique(res[0][1]).size} counts, "
                  f"{(res[0][1] != res[1][1]).sum()} differ", flush=True)
    assert differ == 0
